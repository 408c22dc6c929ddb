// rANS kernels for gfx950: table construction, block-parallel encode of the
// reference's bit-wise streams, bitstream assembly and checkpointed decode.
//
// Stream format (reference core/gpu_ans.py:105-139): L = 1024, state in
// [1024, 2048), one renormalisation bit at a time; the encoder runs over the
// symbols in reverse and the emitted bit list is reversed and packed LSB-first
// into uint32 words, followed by one zero word.
//
// Parallel encode: the state after a symbol depends only on the high bits of
// the state before it, so encoder trajectories from different starting states
// merge.  A lane that owns block g tracks the interval [lo, hi] of every state
// that can enter it, starting from the full range a few symbols earlier (in
// encode order); once lo == hi the entering state is known exactly, whatever
// the true history.  If the interval has not collapsed the window grows, up to
// the end of the stream where the state is exactly L.  Results are therefore
// exact, and identical to a serial encode.
#include <climits>

#include "lq_argsort.h"
#include "lq_decode.h"
#include "lq_launch.h"
#include "lq_readpool.h"

using namespace lq;

namespace {

inline int launch_status() { return hipGetLastError() == hipSuccess ? LQ_OK : LQ_ERR_LAUNCH; }

// Compute units of the current device (cached per device; 256 on MI355X).
inline int64_t device_cus() {
    static int64_t cache[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cache[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cache[dev] = n;
    }
    return cache[dev];
}

// The table code runs on a cooperative group: a whole workgroup (one stream
// per workgroup), or one wave (one stream per wave, wave-synchronous: no
// workgroup barrier).  G::tid / G::size / G::sync are the group's lane, size
// and LDS barrier.
struct BlockGroup {
    static __device__ __forceinline__ int tid() { return (int)threadIdx.x; }
    static __device__ __forceinline__ int size() { return (int)blockDim.x; }
    static __device__ __forceinline__ void sync() { __syncthreads(); }
    static constexpr bool kWave = false;
};
struct WaveGroup {
    static __device__ __forceinline__ int tid() { return (int)(threadIdx.x & 63); }
    static __device__ __forceinline__ int size() { return 64; }
    static __device__ __forceinline__ void sync() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    static constexpr bool kWave = true;
};

// Inclusive scan over the 64 lanes of a wave in DPP moves: Hillis-Steele
// within each 16-lane row (row_shr 1, 2, 4, 8; lanes shifted in from outside
// the row read 0), then row 0's last lane added to row 1 and row 2's to row 3
// (row_bcast:15), then lane 31 added to rows 2 and 3 (row_bcast:31).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
    int v = (int)x;
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15, rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31, rows 2 and 3
    return (uint32_t)v;
}

// Sum of v over a wave (64 active lanes), in every lane.
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(v), 63);
}

// Block-wide sum of v (G::size() multiple of 64, <= 1024).
template <typename G>
__device__ int64_t block_sum(int64_t v) {
    if constexpr (G::kWave) {   // |v| < 2^42 (counts of one chunk): two halves of 21 bits, sums below 2^31
        const uint64_t lo = wave_sum((uint32_t)v & 0x1fffffu);
        const int64_t hi = (int64_t)(int32_t)wave_sum((uint32_t)(int32_t)(v >> 21));
        return hi * (int64_t)(1 << 21) + (int64_t)lo;
    }
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __shared__ int64_t part[16];
    G::sync();
    if ((G::tid() & 63) == 0) part[G::tid() >> 6] = v;
    G::sync();
    int64_t s = 0;
    for (int w = 0; w < (int)(G::size() >> 6); w++) s += part[w];
    return s;
}

// Group-wide maximum of v >= 0.
template <typename G>
__device__ int64_t block_max(int64_t v) {
    for (int o = 32; o > 0; o >>= 1) {
        const int64_t u = __shfl_xor(v, o, 64);
        v = u > v ? u : v;
    }
    if constexpr (G::kWave) return v;
    __shared__ int64_t part[16];
    G::sync();
    if ((G::tid() & 63) == 0) part[G::tid() >> 6] = v;
    G::sync();
    int64_t m = part[0];
    for (int w = 1; w < (int)(G::size() >> 6); w++) m = part[w] > m ? part[w] : m;
    return m;
}

// Bitonic sort of c[0 .. N) ascending (N a power of two, c padded with
// UINT64_MAX past the live entries).
template <typename G>
__device__ void bitonic_sort_u64(uint64_t* c, int N) {
    for (int k = 2; k <= N; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = G::tid(); t < N / 2; t += G::size()) {
                const int i = 2 * t - (t & (j - 1));   // low index of the pair: bit j clear
                const int l = i + j;
                const bool up = (i & k) == 0;
                const uint64_t x = c[i], y = c[l];
                if ((x > y) == up) { c[i] = y; c[l] = x; }
            }
            G::sync();
        }
    }
}

// adjust_pass for alphabets above 256 symbols: the members of the set
// (the first rem entries of the argsort order) that do not depend on the tie
// order, from one bitonic sort of composite (key, index) keys instead of
// per-entry rank counts.  At most one tie group straddles the cut at sorted
// position rem: the one holding positions rem - 1 and rem.  Returns (group
// uniform) whether a different subset of that group would change a frequency.
template <typename G>
__device__ bool adjust_pass_sorted(int n, const int32_t* freqs, int diff, int full, int rem, const int64_t* kk,
                                   int16_t* a, int8_t* inset, uint64_t* sk) {
    int N = 512;
    while (N < n) N <<= 1;
    for (int i = G::tid(); i < N; i += G::size())   // kk in [-(2^32 - 1), 0]: biased key in 33 bits
        sk[i] = i < n ? (((uint64_t)(kk[i] + (int64_t)4294967296LL)) << 11) | (uint64_t)i : ~0ull;
    G::sync();
    bitonic_sort_u64<G>(sk, N);
    for (int p = G::tid(); p < n; p += G::size()) {
        const int i = (int)(sk[p] & 2047u);
        a[p] = (int16_t)i;
        inset[i] = p < rem ? 1 : 0;
    }
    G::sync();
    int matters = 0;
    if (rem > 0 && rem < n && (sk[rem - 1] >> 11) == (sk[rem] >> 11)) {   // uniform
        const uint64_t kstar = sk[rem] >> 11;
        for (int p = G::tid(); p < n; p += G::size())
            if ((sk[p] >> 11) == kstar && (diff > 0 || freqs[a[p]] - full > 1)) matters = 1;
    }
    return block_sum<G>(matters) != 0;
}

// np_net_sort's network (n <= 256 keys) with the pairs in a wave's registers
// instead of LDS: element e sits in slot e / 64 of lane e % 64, as
// (key << 8) | index with keys below 2^23 (the padding's is larger), and every
// stage pairs e with e ^ m, so one lane exchange per slot and stage replaces
// the stage's LDS reads, writes and waits.  v: -key (counts or frequencies),
// vmax >= every v.  Sets inset[] of the first rem sorted entries to 1, of the
// others to 0.
__device__ void net_sort_inset(const uint32_t vin[4], uint32_t vmax, int n, int rem, int8_t* inset) {
    const int lane = WaveGroup::tid();
    uint32_t v[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int e = 64 * s + lane;
        v[s] = (e < n ? vmax - vin[s] : 0xffffffu) << 8 | (uint32_t)e;
    }
    auto stage = [&](int m) {   // m < 64, or 64, 127, 255: slot partner s, s ^ 1, s ^ 1, s ^ 3
        const int src = (lane ^ (m & 63)) << 2;
        auto cx = [&](uint32_t own, uint32_t other, bool lower) {
            const uint32_t o = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)other);
            const bool take = lower ? (own >> 8) > (o >> 8) : (o >> 8) > (own >> 8);   // equal keys stay
            return take ? o : own;
        };
        uint32_t r[4];
        if (m < 64) {
            const bool lower = (lane & (1 << (31 - __builtin_clz((unsigned)m)))) == 0;
#pragma unroll
            for (int s = 0; s < 4; s++) r[s] = cx(v[s], v[s], lower);
        } else if (m < 128) {
#pragma unroll
            for (int s = 0; s < 4; s++) r[s] = cx(v[s], v[s ^ 1], (s & 1) == 0);
        } else {
#pragma unroll
            for (int s = 0; s < 4; s++) r[s] = cx(v[s], v[s ^ 3], (s & 2) == 0);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) v[s] = r[s];
    };
    int nv = 1;
    while (nv * 8 < n) nv *= 2;
    stage(1); stage(3); stage(1); stage(7); stage(2); stage(1);
    for (int per = 2; per <= nv; per *= 2) {
        stage(8 * per - 1);
        for (int num = per / 2; num >= 2; num /= 2) stage(4 * num);
        stage(4); stage(2); stage(1);
    }
#pragma unroll
    for (int s = 0; s < 4; s++)
        if (64 * s + lane < n) inset[v[s] & 255u] = 64 * s + lane < rem ? 1 : 0;
}

// adjust_pass for one wave and at most 320 entries: the members of the set
// that do not depend on the tie order, from the rem-th smallest key kstar (all
// keys below it are in, all above out, those equal to it straddle the cut
// unless they end exactly there), found by a search over the key's bits with
// the keys in registers and a vote per entry and step.  Counting every entry's
// rank instead (n^2 LDS reads) took most of the table kernel: on alphabets of
// about 180 symbols it fell from 29.8 to 21.7 us with this search, and to 17.0
// with the network in registers (launch included).  If a different subset of the straddling group would
// change a frequency and the alphabet is at most 256 symbols with keys below
// 2^23, numpy's network order settles it here (net_sort_inset); returns (wave
// uniform) whether the caller has to.
__device__ bool adjust_pass_select(int n, const int32_t* freqs, int diff, int full, int rem, const int64_t* kk,
                                   int8_t* inset) {
    constexpr int kPer = 5;
    const int lane = WaveGroup::tid();
    uint32_t v[kPer];   // -key: counts or frequencies, below 2^32
    uint32_t any = 0;
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const int i = 64 * u + lane;
        v[u] = i < n ? (uint32_t)(-kk[i]) : 0u;
        any |= v[u];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) any |= (uint32_t)__shfl_xor((int)any, o, 64);
    any = (uint32_t)__builtin_amdgcn_readfirstlane((int)any);
    auto at_least = [&](uint32_t t) {   // entries with v >= t
        int c = 0;
#pragma unroll
        for (int u = 0; u < kPer; u++) c += __builtin_popcountll(__ballot(64 * u + lane < n && v[u] >= t));
        return c;
    };
    // the largest t with more than rem entries >= t: position rem of the
    // descending order holds t (rem < n, so t = 0 has n > rem entries)
    uint32_t t = 0;
    for (int b = 31 - __builtin_clz(any | 1u); b >= 0; b--) {
        const uint32_t c = t | (1u << b);
        if (at_least(c) > rem) t = c;
    }
    // keys above t: all in.  Equal to t: in the straddling group, or (none of
    // them before the cut) out
    const int above = t == 0xffffffffu ? 0 : at_least(t + 1u);
    const bool straddles = above < rem;
    bool mt = false;
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const int i = 64 * u + lane;
        if (i < n) {
            inset[i] = v[u] > t ? 1 : (v[u] == t && straddles ? 2 : 0);
            mt = mt || (v[u] == t && straddles && (diff > 0 || freqs[i] - full > 1));
        }
    }
    if (!__any(mt)) return false;
    if (n > 256 || any >= 1u << 23) return true;
    WaveGroup::sync();
    net_sort_inset(v, any, n, rem, inset);
    return false;
}

// One pass of the build_rans_table adjustment loop (core/gpu_ans.py:73-84)
// with m = |diff|: j = 0 .. m-1 visits order[j % n], i.e. every entry
// `full` = m / n times plus the first rem = m % n entries of the argsort order
// once more; an increment adds its visits, a decrement leaves
// max(f - visits, 1).  The argsort tie order only matters for the tie group
// straddling position rem, and only if a different subset of that group would
// change a frequency; numpy's argsort (np_argsort) runs only then.
template <typename G>
__device__ void adjust_pass(const int64_t* counts, int n, int32_t* freqs, int diff, int16_t* a, int64_t* kk,
                            int8_t* inset, NpScratch* ns, uint64_t* sk) {
    const int m = diff > 0 ? diff : -diff;
    const int full = m / n, rem = m % n;
    for (int i = G::tid(); i < n; i += G::size()) kk[i] = diff > 0 ? -counts[i] : -(int64_t)freqs[i];
    G::sync();
    bool matters;
    if constexpr (G::kWave) {
        matters = adjust_pass_select(n, freqs, diff, full, rem, kk, inset);
    } else if (n > 256 && sk) {
        matters = adjust_pass_sorted<G>(n, freqs, diff, full, rem, kk, a, inset, sk);
    } else {
        int mt = 0;
        for (int i = G::tid(); i < n; i += G::size()) {
            const int64_t ki = kk[i];
            int lt = 0, eq = 0;
            for (int j = 0; j < n; j++) { lt += kk[j] < ki; eq += kk[j] == ki; }
            const int8_t in = lt + eq <= rem ? 1 : (lt >= rem ? 0 : 2);
            inset[i] = in;
            if (in == 2 && (diff > 0 || freqs[i] - full > 1)) mt = 1;
        }
        matters = block_sum<G>(mt) != 0;
    }
    if (matters) {
        if (n <= 256) {   // numpy's network directly (np_argsort's first and only frame)
            for (int i = G::tid(); i < n; i += G::size()) { ns->k[i] = kk[i]; ns->a[i] = (int16_t)i; }
            G::sync();
            np_net_sort<G>(ns->k, ns->a, n);
            for (int p = G::tid(); p < n; p += G::size()) inset[ns->a[p]] = p < rem ? 1 : 0;
        } else {
            np_argsort<G>(kk, a, n, ns);
            for (int p = G::tid(); p < n; p += G::size()) inset[a[p]] = p < rem ? 1 : 0;
        }
        G::sync();
    }
    for (int i = G::tid(); i < n; i += G::size()) {
        const int v = full + (inset[i] == 1 ? 1 : 0);
        const int f = freqs[i];
        freqs[i] = diff > 0 ? f + v : (f - v > 1 ? f - v : 1);
    }
    G::sync();
}

// build_rans_table normalisation (core/gpu_ans.py:62-86) on LDS arrays:
// counts[n] (int64) in, freqs[n] (int32) out; a, kk, inset: n entries;
// ns: argsort scratch; sk (optional, alphabets above 256): 2048 entries.
//
// An increment pass always reaches sum == L.  In the decrement branch the
// excess is below n (only the max(., 1) bumps exceed L), so a pass whose
// excess covers all G entries with f > 1 decrements exactly those, whatever
// the order; such passes are counted in closed form and only the last,
// partial pass (excess < G) goes through adjust_pass.  The number t of full
// passes is the least t with G_t = 0 or C(t + 1) > excess, where
// G_t = #{f_i - t > 1} and C(t) = G_0 + .. + G_(t-1) = sum_i min(t, f_i - 1)
// is nondecreasing: a binary search over t in [0, max f - 1], not one pass
// per t (a single dominant symbol makes t as large as the excess).
template <typename G>
__device__ void normalise(const int64_t* counts, int n, int32_t* freqs, int16_t* a, int64_t* kk, int8_t* inset,
                          NpScratch* ns, uint64_t* sk = nullptr) {
    int64_t tl = 0;
    for (int i = G::tid(); i < n; i += G::size()) tl += counts[i];
    const int64_t total = block_sum<G>(tl);
    int64_t fl = 0;
    for (int i = G::tid(); i < n; i += G::size()) {
        int32_t f = 1;
        if (total != 0) {
            double q = (double)counts[i] / (double)total * (double)kL;   // (counts / total * L)
            int32_t t = (int32_t)q;                                       // .astype(int32)
            f = t < 1 ? 1 : t;
        }
        freqs[i] = f;
        fl += f;
    }
    const int diff = (int)(kL - block_sum<G>(fl));
    if (diff > 0) {
        adjust_pass<G>(counts, n, freqs, diff, a, kk, inset, ns, sk);
    } else if (diff < 0) {
        const int excess0 = -diff;
        int64_t fm = 0;
        for (int i = G::tid(); i < n; i += G::size()) fm = freqs[i] > fm ? freqs[i] : fm;
        const int fmax = (int)block_max<G>(fm);
        auto C = [&](int tt) {   // passes 0 .. tt-1 decrement sum_i min(tt, f_i - 1) entries in total
            int64_t c = 0;
            for (int i = G::tid(); i < n; i += G::size()) {
                const int r = freqs[i] - 1;
                c += r < tt ? r : tt;
            }
            return block_sum<G>(c);
        };
        int lo = 0, hi = fmax - 1 > 0 ? fmax - 1 : 0;   // t = fmax - 1 has G_t = 0
        while (lo < hi) {   // least t in [0, hi) with C(t + 1) > excess, else hi
            const int mid = (lo + hi) >> 1;
            if (C(mid + 1) > excess0) hi = mid; else lo = mid + 1;
        }
        const int t = lo;
        const int excess = (int)(excess0 - C(t));
        for (int i = G::tid(); i < n; i += G::size()) freqs[i] = freqs[i] - t > 1 ? freqs[i] - t : 1;
        G::sync();
        if (excess > 0) adjust_pass<G>(counts, n, freqs, -excess, a, kk, inset, ns, sk);
    }
}

// Inclusive scan of v over the block (G::size() <= 1024, multiple of 64).
template <typename G>
__device__ int block_incl_scan(int v) {
    if constexpr (G::kWave) return (int)wave_incl_scan((uint32_t)v);
    const int lane = G::tid() & 63, w = G::tid() >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    __shared__ int wsum[16];
    G::sync();
    if (lane == 63) wsum[w] = v;
    G::sync();
    for (int i = 0; i < w; i++) v += wsum[i];
    return v;
}

// out[i] = in[0] + .. + in[i-1] for i <= n (block-cooperative, any n).
template <typename G>
__device__ void exclusive_scan_array(const int32_t* in, int n, int32_t* out) {
    if constexpr (G::kWave) {   // the carry stays in registers (uniform over the wave)
        int carry = 0;
        for (int b = 0; b < n; b += 64) {
            const int i = b + G::tid();
            const int v = i < n ? in[i] : 0;
            const int incl = block_incl_scan<G>(v);
            if (i < n) out[i] = carry + incl - v;
            carry += __builtin_amdgcn_readlane(incl, 63);
        }
        if (G::tid() == 0) out[n] = carry;
        G::sync();
        return;
    }
    __shared__ int carry;
    if (G::tid() == 0) carry = 0;
    G::sync();
    for (int b = 0; b < n; b += G::size()) {
        int i = b + G::tid();
        int v = i < n ? in[i] : 0;
        int incl = block_incl_scan<G>(v);
        int c = carry;
        if (i < n) out[i] = c + incl - v;
        G::sync();
        if (G::tid() == G::size() - 1) carry = c + incl;
        G::sync();
    }
    if (G::tid() == 0) out[n] = carry;
    G::sync();
}

// ------------------------------------------------------------ chunk tables --

// WIDE = false: hist holds 16 x 256 int8-symbol bins (value + 128).
// WIDE = true:  hist holds 16 x 1024 bins from the stream's min (minmax).
template <bool WIDE>
__global__ __launch_bounds__(256) void k_chunk_tables(const uint32_t* __restrict__ hist, const int32_t* __restrict__ minmax,
                                                      lq_table* __restrict__ tables, int32_t* __restrict__ status) {
    __shared__ int64_t counts[LQ_MAXSYM];
    __shared__ int32_t freqs[LQ_MAXSYM];
    __shared__ NpScratch ns;
    __shared__ int16_t perm[LQ_MAXSYM];
    __shared__ uint32_t h[256];
    __shared__ int s_min, s_max, s_st;
    __shared__ uint32_t s_tot;
    const int64_t sid = blockIdx.x;   // chunk * 16 + stream
    const int tid = threadIdx.x;
    lq_table* T = tables + sid;
    int lo, n;
    if constexpr (!WIDE) {
        h[tid] = hist[sid * 256 + tid];
        if (tid == 0) { s_min = 256; s_max = -1; s_tot = 0; s_st = 0; }
        __syncthreads();
        if (h[tid]) { atomicMin(&s_min, tid); atomicMax(&s_max, tid); atomicAdd(&s_tot, h[tid]); }
        __syncthreads();
        if (s_max < 0) {
            if (tid == 0) { T->lo = 0; T->n_sym = 0; T->n_symbols = 0; T->status = 0; }
            return;
        }
        lo = s_min - 128 - 2;
        n = s_max - s_min + 5;
        for (int i = tid; i < n; i += 256) {
            int b = lo + i + 128;
            counts[i] = (b >= 0 && b < 256) ? (int64_t)h[b] : 0;
        }
    } else {
        const int mn = minmax[sid * 2], mx = minmax[sid * 2 + 1];
        if (mx == INT_MIN) {   // absent stream (empty coset)
            if (tid == 0) { T->lo = 0; T->n_sym = 0; T->n_symbols = 0; T->status = 0; }
            return;
        }
        lo = mn - 2;
        n = mx - mn + 5;
        if (n > kL) {   // the reference's normalisation never terminates here
            if (tid == 0) {
                T->lo = lo; T->n_sym = 0; T->n_symbols = 0; T->status = LQ_ST_ALPHABET;
                atomicOr(status + sid / LQ_STREAMS, LQ_ST_ALPHABET);
            }
            return;
        }
        if (tid == 0) { s_tot = 0; s_st = 0; }
        __syncthreads();
        uint32_t tl = 0;
        for (int i = tid; i < n; i += 256) {
            const uint32_t c = (i >= 2 && i - 2 < kL) ? hist[sid * kL + i - 2] : 0u;
            counts[i] = c;
            tl += c;
        }
        atomicAdd(&s_tot, tl);
    }
    __syncthreads();
    __shared__ int64_t kk[LQ_MAXSYM];
    __shared__ int8_t inset[LQ_MAXSYM];
    __shared__ uint64_t sk[WIDE ? 2048 : 1];   // wide alphabets: composite sort keys
    normalise<BlockGroup>(counts, n, freqs, perm, kk, inset, &ns, WIDE ? sk : nullptr);
    __shared__ int32_t cum[LQ_MAXSYM + 1];
    exclusive_scan_array<BlockGroup>(freqs, n, cum);
    for (int i = tid; i < n; i += 256) T->enc[i] = enc_pack((uint32_t)freqs[i], (uint32_t)cum[i]);
    if (tid == 0) {
        T->lo = lo;
        T->n_sym = n;
        T->n_symbols = (int32_t)s_tot;
        T->status = s_st;
        if (s_st) atomicOr(status + sid / LQ_STREAMS, s_st);
    }
}

// int8 path: one wave per stream, kTabWaves streams per workgroup; the
// stream's table built wave-synchronously (WaveGroup) in its own LDS arrays,
// with the same normalisation and tie order as k_chunk_tables<false>.
constexpr int kTabWaves = 4;
constexpr int kCap8 = 264;   // range(min - 2, max + 2) of int8 values: at most 260 symbols

// skip: when a chunk's symbols left int8 (LQ_ST_SYM_OVERFLOW, set by the launch
// before) every stream of the batch is left empty, so that the launches that
// follow do nothing.  host (nullable, host memory): the OR of the chunks' status
// words so far.
__global__ __launch_bounds__(64 * kTabWaves) void k_chunk_tables_wave(const uint32_t* __restrict__ hist,
                                                                      int64_t n_streams, lq_table* __restrict__ tables,
                                                                      int32_t* __restrict__ status, int skip,
                                                                      int64_t* __restrict__ host) {
    __shared__ int64_t counts[kTabWaves][kCap8];
    __shared__ int32_t freqs[kTabWaves][kCap8];
    __shared__ NpScratch ns[kTabWaves];
    __shared__ int16_t perm[kTabWaves][kCap8];
    __shared__ int64_t kk[kTabWaves][kCap8];
    __shared__ int8_t inset[kTabWaves][kCap8];
    __shared__ int32_t cum[kTabWaves][kCap8 + 1];
    __shared__ int s_st[kTabWaves];
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    const int64_t sid = (int64_t)blockIdx.x * kTabWaves + w;
    if (sid >= n_streams) return;   // wave-uniform; no workgroup barrier below
    lq_table* T = tables + sid;
    const uint32_t* hs = hist + sid * 256;
    uint32_t hv[4];
    int mn, mx;
    uint32_t tl = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int b = lane + 64 * j;
        hv[j] = hs[b];
        tl += hv[j];
    }
    // a bin with a count, in each quarter of the bins: first and last by ballot
    mn = 256;
    mx = -1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint64_t m = __ballot(hv[j] != 0);
        if (m) {
            mx = 64 * j + 63 - __builtin_clzll(m);
            if (mn == 256) mn = 64 * j + __builtin_ctzll(m);
        }
    }
    tl = wave_sum(tl);
    if (host && sid == 0) {
        int32_t all = 0;
        for (int64_t c = lane; c * LQ_STREAMS < n_streams; c += 64) all |= status[c];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) all |= __shfl_xor(all, o, 64);
        if (lane == 0) *host = all;
    }
    bool out = false;
    if (skip)
        for (int64_t c0 = 0; c0 * LQ_STREAMS < n_streams; c0 += 64)
            out = out || __any((c0 + lane) * LQ_STREAMS < n_streams && (status[c0 + lane] & LQ_ST_SYM_OVERFLOW));
    if (mx < 0 || out) {   // absent stream (empty coset)
        if (lane == 0) { T->lo = 0; T->n_sym = 0; T->n_symbols = 0; T->status = 0; }
        return;
    }
    const int lo = mn - 128 - 2, n = mx - mn + 5;
    // bin b is alphabet entry b - 128 - lo; the guard entries have no counts
    if (lane < 2) {
        counts[w][lane] = 0;
        counts[w][n - 1 - lane] = 0;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = lane + 64 * j - 128 - lo;
        if (i >= 2 && i < n - 2) counts[w][i] = (int64_t)hv[j];
    }
    if (lane == 0) s_st[w] = 0;
    WaveGroup::sync();
    normalise<WaveGroup>(counts[w], n, freqs[w], perm[w], kk[w], inset[w], &ns[w]);
    exclusive_scan_array<WaveGroup>(freqs[w], n, cum[w]);
    for (int i = lane; i < n; i += 64) T->enc[i] = enc_pack((uint32_t)freqs[w][i], (uint32_t)cum[w][i]);
    if (lane == 0) {
        const int st = s_st[w];
        T->lo = lo;
        T->n_sym = n;
        T->n_symbols = (int32_t)tl;
        T->status = st;
        if (st) atomicOr(status + sid / LQ_STREAMS, st);
    }
}

// ------------------------------------------------------------ chunk encode --
//
// Task = (chunk, stream st = coset * 8 + coord, block g), one lane each; a
// 256-thread workgroup holds 16 consecutive blocks x 16 streams of one chunk,
// a wave one coset of 8 blocks, so the 8 lanes of a (block, coset) read the 8
// interleaved columns of that coset one 128-byte line at a time (sym_pos
// layout).

template <typename SymT>
struct Col {
    const SymT* p;   // chunk 0 of the column; chunk k at p + 128 k (elements)
    int n;
};

template <typename SymT>
__device__ __forceinline__ Col<SymT> column(const SymT* sym, const uint32_t* blk_n1, int64_t chunk, int64_t nblk,
                                            int64_t V, int64_t h, int c, int idx) {
    uint32_t n1 = blk_n1[chunk * nblk + h];
    int64_t valid = V - h * kBlk < kBlk ? V - h * kBlk : kBlk;
    int n0 = (int)valid - (int)n1;
    Col<SymT> col;
    col.p = sym + (chunk * nblk + h) * (int64_t)kSymStride + sym_region(c, n0) + 16 * idx;
    col.n = c ? (int)n1 : n0;
    return col;
}

// f(e, b, in) for the column symbols of ranks n-1, n-2, .., 0 (the column's
// 16-symbol chunk k sits at p + 128 k); entries(chunk, hi_b, e, whole) turns a chunk
// into its 16 table entries, all read before the first is used, so a chunk's
// serial chain waits for the LDS once and not per symbol (whole: hi_b is 16, or
// 0 in lanes whose entries are not used).  b is the symbol's
// index in its chunk (a compile-time constant after unrolling); after a
// chunk's symbols done() runs.
//
// DEPTH chunks of 16-byte loads are in flight per lane: a chunk's registers
// are reloaded, for the chunk DEPTH further down, as soon as its entries are
// read.  The loads are unconditional (a lane past its last chunk reads chunk 0
// again) and the trip count is uniform over the calling lanes (votes, not
// shuffles: some of the wave's lanes may not be here): with a load under a condition, or
// with registers that move from "next" to "current", the compiler waits for
// the newest load before the symbols it was to be hidden behind (47,000 cycles
// per block and wave against 18,000 here, one wave per SIMD).
// Only a column's top chunk can be partial: it comes first, with a per-lane
// predicate (f must leave its state unchanged when in == false); after it
// lanes without chunks left are masked off.
template <int DEPTH, typename SymT, typename E, typename F, typename D>
__device__ __forceinline__ void for_each_rev(const SymT* p, int n, E&& entries, F&& f, D&& done) {
    const int k = n > 0 ? (n - 1) >> 4 : -1;   // top chunk
    if (!__any(k >= 0)) return;
    auto at = [&](int i) { return gload_chunk(p + 128 * (i > 0 ? i : 0)); };
    uint32_t e[16];
    Chunk16<SymT> buf[DEPTH];
    {
        const Chunk16<SymT> top = at(k);
#pragma unroll
        for (int j = 0; j < DEPTH; j++) buf[j] = at(k - 1 - j);
        const int hi_b = k < 0 ? 0 : n - 16 * k;
        entries(top, hi_b, e, false);
#pragma unroll
        for (int b = 15; b >= 0; b--) f(e[b], b, b < hi_b);
        done();
    }
    for (int it = 1; __any(it <= k); it += DEPTH) {
#pragma unroll
        for (int j = 0; j < DEPTH; j++) {
            const bool live = it + j <= k;
            if (!__any(live)) break;   // uniform over the calling lanes
            entries(buf[j], live ? 16 : 0, e, true);   // every lane: no merge with the old entries
            buf[j] = at(k - it - j - DEPTH);
            if (live) {
#pragma unroll
                for (int b = 15; b >= 0; b--) f(e[b], b, true);
                done();
            }
        }
    }
}

struct EncWork {  // offsets into the encode workspace
    int64_t bits, scratch, tiles, total;
};

// Streams longer than kScanTile blocks are scanned in tiles (k_scan_tiles /
// k_scan_top / k_scan_apply, then k_chunk_offsets); shorter ones by one
// workgroup per chunk (k_chunk_scan_offsets).
constexpr int kScanTile = 4096;

__host__ __device__ inline EncWork enc_layout(int64_t n_chunks, int64_t n_vectors) {
    int64_t nblk = (n_vectors + kBlk - 1) / kBlk;
    int64_t tasks = n_chunks * LQ_STREAMS * nblk;
    int64_t n_tiles = nblk > kScanTile ? n_chunks * LQ_STREAMS * ((nblk + kScanTile - 1) / kScanTile) : 0;
    EncWork w;
    w.bits = 0;
    w.scratch = ((tasks * 4 + 255) / 256) * 256;
    w.tiles = w.scratch + tasks * (int64_t)kCapW * 4;
    w.total = w.tiles + n_tiles * 8;
    return w;
}

constexpr int kEncBlocks = 16;   // blocks per encode workgroup (x 16 streams)
constexpr int kEncRing = 8;      // scratch words per lane waiting in LDS

// Grid: (block groups, chunks).
//
// On a full chip the kernel issues VALU instructions nearly all the time; with
// few blocks (a layer's prompt: one wave per SIMD or less) it waits for the
// serial chain of its 256 or so symbols, their loads and lookups.  Encode and
// offset scan, before / after the loads of for_each_rev and the branch-free
// word output below: 102 blocks 38.1 / 25.4 us, 2048 blocks 47.6 / 32.4 us,
// 131072 blocks (64 chunks of 8192 tokens) 412.7 / 364.1 us; the wide path's
// 4096 blocks 84.9 / 60 us.  The bits of three symbols (at most 30) enter a 64-bit
// accumulator, then the word they may have completed is written to the lane's
// ring in LDS whether it is complete or not (an incomplete one is written
// again, and overwritten, by the next three symbols): no branch and no
// divergence per word.  Full groups of four words leave the ring once per
// 16-symbol chunk as aligned 16-byte stores.
template <typename SymT>
__global__ __launch_bounds__(256) void k_chunk_encode(const SymT* __restrict__ sym, const uint32_t* __restrict__ blk_n1,
                                                      int64_t nblk, int64_t V, const lq_table* __restrict__ tables,
                                                      uint32_t* __restrict__ blk_bits, uint32_t* __restrict__ scratch,
                                                      uint16_t* __restrict__ blk_state) {
    // odd row stride: the 16 stream tables start in different LDS banks.
    // int8 symbols span at most 260 alphabet entries, all held in LDS.  Wide
    // (int16) alphabets reach L + 4 entries: LDS holds a window of kWin
    // entries per stream around symbol 0 (lattice coordinates centre there),
    // and the rare symbol outside it reads its entry from the table in global
    // memory, so the workgroup's LDS stays that of the int8 encoder.
    constexpr bool kWide = sizeof(SymT) == 2;
    constexpr int kWin = kWide ? 256 : 264;
    // The ring comes first: lanes without a symbol look up whatever byte their
    // chunk holds, at most 255 entries before or after their row's first.
    __shared__ struct {
        uint32_t sq[kEncRing][256];   // per-lane ring of scratch words
        uint32_t senc[LQ_STREAMS][kWin + 1];
    } sm;
    static_assert(kWin + 1 > 257 || sizeof(SymT) == 2, "any byte's lookup stays inside the table rows");
    auto& sq = sm.sq;
    auto& senc = sm.senc;
    __shared__ int slo[LQ_STREAMS], snsym[LQ_STREAMS];
    const int tid = threadIdx.x;
    const int64_t chunk = blockIdx.y;
    // wave = one coset of 8 blocks (lanes: block-major, coordinate-minor), so
    // a wave's columns hold one coset's counts and run about equally long
    const int64_t g = (int64_t)blockIdx.x * kEncBlocks + ((tid >> 3) & 15);
    const int st = ((tid >> 7) << 3) | (tid & 7);
    const lq_table* T = tables + chunk * LQ_STREAMS;
    {   // stage the tables: 16 threads per stream, its live entries only
        const int s = tid >> 4;
        const int n = T[s].n_sym, lo = T[s].lo;
        int w0 = 0;   // first alphabet entry of the stream's LDS window
        if constexpr (kWide) {
            const int w = -lo - kWin / 2;
            w0 = n <= kWin || w <= 0 ? 0 : (w < n - kWin ? w : n - kWin);
        }
        const int m = n - w0 < kWin ? n - w0 : kWin;
        for (int j = tid & 15; j < m; j += 16) senc[s][j] = encx_of(T[s].enc[j + w0]);
        if ((tid & 15) == 0) { slo[s] = lo + w0; snsym[s] = n; }
    }
    __syncthreads();
    if (g >= nblk) return;
    const int64_t task = (chunk * LQ_STREAMS + st) * nblk + g;
    if (snsym[st] == 0) {  // absent stream (empty coset)
        blk_bits[task] = 0;
        blk_state[task] = (uint16_t)kL;
        return;
    }
    const int c = st >> 3, idx = st & 7;
    const int lo_sym = slo[st];   // symbol of the window's first entry (a valid symbol)
    const uint32_t* const genc = T[st].enc;
    const int glo = T[st].lo;
    const uint32_t row = (uint32_t)(uintptr_t)(lds_u32*)&senc[st][0];   // LDS byte address of the window
    // the table entries of a chunk's first hi_b symbols (of the others: some
    // entry)
    auto entries = [&](const Chunk16<SymT>& ch, int hi_b, uint32_t e[16], bool whole) {
        if constexpr (!kWide) {
            // entry address of symbol value v: row + 4 (v - lo_sym), one 4-byte
            // dot product with the symbol's byte picked by the weights
            const int w[4] = {(int)ch.a.x, (int)ch.a.y, (int)ch.a.z, (int)ch.a.w};
            const int base = (int)row - 4 * lo_sym;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                uint32_t a = (uint32_t)__builtin_amdgcn_sdot4(w[i >> 2], 4 << (8 * (i & 3)), base, false);
                if (!whole) a = i < hi_b ? a : row;
                e[i] = *(const lds_u32*)(uintptr_t)a;
            }
        } else {
            uint32_t j[16], out = 0;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                j[i] = whole || i < hi_b ? (uint32_t)(ch.get(i) - lo_sym) : 0u;
                const uint32_t jj = j[i] < (uint32_t)kWin ? j[i] : (uint32_t)kWin - 1u;
                out |= j[i] >= (uint32_t)kWin ? 1u << i : 0u;
                e[i] = *(const lds_u32*)(uintptr_t)(row + 4u * jj);
            }
            if (out && hi_b) {   // symbols outside the window (rare)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (out & (1u << i)) e[i] = encx_of(genc[(int)j[i] + lo_sym - glo]);
            }
        }
    };
    auto nothing = []() {};

    // ---- state entering block g (encode order runs from the stream end down)
    uint32_t x = kL;
    int window = 16;   // symbols after the block; the interval collapses within 16 on typical tables
    for (;;) {
        // top of the window: `window` symbols after block g, or the stream end
        int64_t h = g + 1;
        int need = window;
        while (h < nblk) {
            int nc = column(sym, blk_n1, chunk, nblk, V, h, c, idx).n;
            if (need <= nc) break;
            need -= nc;
            h++;
        }
        const bool exact = h >= nblk;
        uint32_t lo = kL, hi = exact ? (uint32_t)kL : 2u * kL - 1u;
        const int64_t hb = exact ? nblk - 1 : h;
        for (int64_t b = hb; b > g; b--) {
            Col<SymT> col = column(sym, blk_n1, chunk, nblk, V, b, c, idx);
            const int cnt = (b == hb && !exact) ? need : col.n;
            if (lo == hi) {
                uint32_t xx = lo, k;
                for_each_rev<1>(col.p, cnt, entries, [&](uint32_t e, int, bool in) {
                    const uint32_t xn = encx_step(xx, e, &k);
                    xx = in ? xn : xx;
                }, nothing);
                lo = hi = xx;
            } else {
                for_each_rev<1>(col.p, cnt, entries, [&](uint32_t e, int, bool in) {
                    uint32_t l2 = lo, h2 = hi;
                    hull_step(l2, h2, e);
                    lo = in ? l2 : lo;
                    hi = in ? h2 : hi;
                }, nothing);
            }
        }
        if (lo == hi) { x = lo; break; }
        window *= 8;
    }

    // ---- encode block g, bits right-aligned in the task's scratch region:
    // words leave in decreasing address order from kCapW - 1
    Col<SymT> col = column(sym, blk_n1, chunk, nblk, V, g, c, idx);
    uint32_t* scr = scratch + task * (int64_t)kCapW;
    uint32_t* const qcol = &sq[0][tid];   // ring slot s at qcol[256 s]: a wave's accesses are contiguous
    // Bit accumulator (ahi:alo): the emitted bits sit at the top, newest
    // highest; a symbol's group (the k low bits of x, bit k - 1 first in the
    // final stream) enters by one funnel shift of (x:ahi:alo) right by k, two
    // v_alignbit (k <= 10; k = 0 leaves all three in place).  total counts the
    // bits; word w of the block holds bits 32 w .. 32 w + 31, so after a group
    // of symbols the word being filled has n = (total & 31) + ks bits, the top
    // n of the accumulator: bits past them are older words' and drop out.  The
    // word is bit-reversed so that its oldest bit is the most significant, as
    // the stream order wants.
    uint32_t ahi = 0u, alo = 0u, total = 0u, ks = 0u, flushed = 0u;
    auto emit = [&]() {   // ks <= 30: at most one word is completed
        const uint32_t n = (total & 31u) + ks;
        const uint32_t raw = (uint32_t)((((uint64_t)ahi << 32) | alo) >> ((0u - n) & 63u));
        qcol[256u * ((total >> 5) & (kEncRing - 1))] = __builtin_bitreverse32(raw);
        total += ks;
        ks = 0u;
    };
    auto store4 = [&]() {   // words flushed .. flushed + 3 of the block, as one 16-byte store
        const uint32_t* q = qcol + 256u * (flushed & 4u);
        *reinterpret_cast<uint4*>(scr + (kCapW - 4 - (int)flushed)) = make_uint4(q[768], q[512], q[256], q[0]);
        flushed += 4u;
    };
    // At most 127 bits wait before a chunk and its first 13 symbols add at most
    // 130, so only the last emit can meet 8 complete words, with the one it
    // fills the ring's ninth: four of them leave first (10 bits in nearly every
    // symbol: alphabets near L).
    for_each_rev<4>(col.p, col.n, entries, [&](uint32_t e, int b, bool in) {
        uint32_t k;
        const uint32_t xin = x;
        const uint32_t xn = encx_step(xin, e, &k);
        k = in ? k : 0u;
        x = in ? xn : xin;
        alo = __builtin_amdgcn_alignbit(ahi, alo, k);
        ahi = __builtin_amdgcn_alignbit(xin, ahi, k);
        ks += k;
        if (b == 0 && (total >> 5) >= flushed + (uint32_t)kEncRing) store4();
        if (b % 3 == 0) emit();
    }, [&]() {
        while ((total >> 5) >= flushed + 4u) store4();
    });
    const uint32_t nacc = total & 31u;
    if (nacc) qcol[256u * ((total >> 5) & (kEncRing - 1))] = __builtin_bitreverse32(ahi >> (32u - nacc));
    // the last, partial group's words sit in the top slots of its 16 bytes
    while (((total + 31u) >> 5) > flushed) store4();
    blk_bits[task] = total;
    blk_state[task] = (uint16_t)x;
}

// Short streams (nblk <= kScanTile), one workgroup per chunk, wave w = stream
// w: exclusive prefix of the block bit counts (64 blocks per round, a wave
// scan plus the running carry), n_bits and final state; then the chunk's word
// offsets (n_words + 1 words per present stream) and total.  Replaces
// k_chunk_scan + k_chunk_offsets for such batches.
constexpr int kScanRounds = 32;   // rounds of 64 blocks whose loads are in flight together

// chunk_base[c] = chunk_words[0] + .. + chunk_words[c - 1], by one wave.
// total (nullable, host memory): the sum of them all.
__device__ __forceinline__ void chunk_bases(const int64_t* chunk_words, int64_t n_chunks, int64_t* chunk_base, int lane,
                                            int64_t* total) {
    int64_t carry = 0;
    for (int64_t c0 = 0; c0 < n_chunks; c0 += 64) {
        const int64_t c = c0 + lane;
        const int64_t v = c < n_chunks ? __hip_atomic_load(chunk_words + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
        int64_t incl = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        if (c < n_chunks) chunk_base[c] = carry + incl - v;
        carry += __shfl(incl, 63, 64);
    }
    if (total && lane == 0) *total = carry;
}

// chunk_bases of many chunks, by one workgroup of its own.
__global__ __launch_bounds__(1024) void k_chunk_bases(const int64_t* __restrict__ chunk_words, int64_t n_chunks,
                                                      int64_t* __restrict__ chunk_base, int64_t* __restrict__ total) {
    __shared__ int64_t wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int64_t carry = 0;
    for (int64_t c0 = 0; c0 < n_chunks; c0 += 1024) {
        const int64_t c = c0 + tid, v = c < n_chunks ? chunk_words[c] : 0;
        int64_t incl = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        int64_t below = carry;
#pragma unroll
        for (int w = 0; w < 16; w++) {
            const int64_t sum = wsum[w];
            below += w < wave ? sum : 0;
            carry += sum;
        }
        if (c < n_chunks) chunk_base[c] = below + incl - v;
        __syncthreads();   // wsum is written again
    }
    if (total && tid == 0) *total = carry;
}

// Chunks up to which the scan's last workgroup makes the bases.  Every chunk pays
// for it with a release and acquire of the L2 (the scan of 300 chunks 19.1 us
// with them, 10.7 without, of 1000 chunks 46.3 and 19.5), a launch of its own
// costs about 5 us whatever the batch.
constexpr int64_t kBasesInScan = 64;

// chunk_base (nullable; counter is then a cleared word): the workgroup that
// finishes last also writes the chunks' bases.
__global__ __launch_bounds__(1024) void k_chunk_scan_offsets(const uint32_t* __restrict__ blk_bits,
                                                             const uint16_t* __restrict__ blk_state,
                                                             const lq_table* __restrict__ tables, int64_t nblk,
                                                             uint32_t* __restrict__ blk_off,
                                                             int64_t* __restrict__ stream_nbits,
                                                             int32_t* __restrict__ stream_state,
                                                             int64_t* __restrict__ stream_woff,
                                                             int64_t* __restrict__ chunk_words,
                                                             int64_t* __restrict__ chunk_base,
                                                             uint32_t* __restrict__ counter,
                                                             int64_t* __restrict__ total) {
    __shared__ int s_last;
    __shared__ int64_t s_nbits[LQ_STREAMS];
    __shared__ int s_present[LQ_STREAMS];
    const int64_t c = blockIdx.x;
    const int lane = threadIdx.x & 63, st = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t sid = c * LQ_STREAMS + st;
    const uint32_t* bb = blk_bits + sid * nblk;
    uint32_t* bo = blk_off + sid * nblk;
    uint64_t carry = 0;
    for (int64_t r0 = 0; r0 < nblk; r0 += 64 * kScanRounds) {
        uint32_t v[kScanRounds];
#pragma unroll
        for (int k = 0; k < kScanRounds; k++) {
            const int64_t b = r0 + 64 * k + lane;
            v[k] = b < nblk ? bb[b] : 0u;
        }
#pragma unroll
        for (int k = 0; k < kScanRounds; k++) {
            const uint32_t x = wave_incl_scan(v[k]);   // counts < 2^13, sums < 2^19
            const int64_t b = r0 + 64 * k + lane;
            if (b < nblk) bo[b] = (uint32_t)(carry + x - v[k]);
            carry += (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
        }
    }
    if (lane == 0) {
        const bool present = tables[sid].n_sym > 0;
        s_present[st] = present ? 1 : 0;
        s_nbits[st] = present ? (int64_t)carry : 0;
        stream_nbits[sid] = present ? (int64_t)carry : 0;
        stream_state[sid] = present ? (int32_t)blk_state[sid * nblk] : 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t w = 0;
        for (int k = 0; k < LQ_STREAMS; k++) {
            stream_woff[c * LQ_STREAMS + k] = w;
            if (s_present[k]) w += (s_nbits[k] + 31) / 32 + 1;
        }
        if (!chunk_base) {
            chunk_words[c] = w;
        } else {   // the release orders the count before the counter's step
            __hip_atomic_store(chunk_words + c, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u == gridDim.x;
        }
    }
    if (!chunk_base) return;
    __syncthreads();
    if (s_last && st == 0) chunk_bases(chunk_words, gridDim.x, chunk_base, lane, total);
}

// Tiled scan of long streams.  Tile t of stream sid covers blocks
// t * kScanTile .. + kScanTile - 1; thread i of its workgroup owns the 16
// consecutive blocks from t * kScanTile + 16 i.
__device__ __forceinline__ uint64_t block_exclusive_scan256(uint64_t v, uint64_t* part, uint64_t* total) {
    const int tid = threadIdx.x;
    part[tid] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {   // inclusive Hillis-Steele scan
        const uint64_t u = tid >= off ? part[tid - off] : 0;
        __syncthreads();
        part[tid] += u;
        __syncthreads();
    }
    *total = part[255];
    return tid ? part[tid - 1] : 0;
}

__global__ __launch_bounds__(256) void k_scan_tiles(const uint32_t* __restrict__ blk_bits, int64_t nblk, int64_t tiles,
                                                    uint64_t* __restrict__ tile_sum) {
    __shared__ uint64_t part[256];
    const int64_t sid = blockIdx.x / tiles, t = blockIdx.x % tiles;
    const uint32_t* bb = blk_bits + sid * nblk;
    const int64_t b0 = t * kScanTile + 16 * (int64_t)threadIdx.x;
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < 16; k++)
        if (b0 + k < nblk) s += bb[b0 + k];
    uint64_t tot;
    block_exclusive_scan256(s, part, &tot);
    if (threadIdx.x == 0) tile_sum[sid * tiles + t] = tot;
}

// per stream: exclusive prefix of its tile sums (in place), n_bits, final state
__global__ __launch_bounds__(256) void k_scan_top(uint64_t* __restrict__ tile_sum, int64_t tiles,
                                                  const uint16_t* __restrict__ blk_state, int64_t nblk,
                                                  const lq_table* __restrict__ tables, int64_t* __restrict__ stream_nbits,
                                                  int32_t* __restrict__ stream_state) {
    __shared__ uint64_t part[256];
    const int64_t sid = blockIdx.x;
    uint64_t* ts = tile_sum + sid * tiles;
    uint64_t carry = 0;
    for (int64_t t0 = 0; t0 < tiles; t0 += 256) {   // uniform trip count
        const int64_t t = t0 + threadIdx.x;
        const uint64_t v = t < tiles ? ts[t] : 0;
        uint64_t tot;
        const uint64_t ex = block_exclusive_scan256(v, part, &tot);
        if (t < tiles) ts[t] = carry + ex;
        carry += tot;
        __syncthreads();   // part is reused by the next round
    }
    if (threadIdx.x == 0) {
        const bool present = tables[sid].n_sym > 0;
        stream_nbits[sid] = present ? (int64_t)carry : 0;
        stream_state[sid] = present ? (int32_t)blk_state[sid * nblk] : 0;
    }
}

__global__ __launch_bounds__(256) void k_scan_apply(const uint32_t* __restrict__ blk_bits, int64_t nblk, int64_t tiles,
                                                    const uint64_t* __restrict__ tile_off, uint32_t* __restrict__ blk_off) {
    __shared__ uint64_t part[256];
    const int64_t sid = blockIdx.x / tiles, t = blockIdx.x % tiles;
    const uint32_t* bb = blk_bits + sid * nblk;
    uint32_t* bo = blk_off + sid * nblk;
    const int64_t b0 = t * kScanTile + 16 * (int64_t)threadIdx.x;
    uint32_t v[16];
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < 16; k++) {
        v[k] = b0 + k < nblk ? bb[b0 + k] : 0u;
        s += v[k];
    }
    uint64_t tot;
    uint64_t run = tile_off[sid * tiles + t] + block_exclusive_scan256(s, part, &tot);
#pragma unroll
    for (int k = 0; k < 16; k++) {
        if (b0 + k < nblk) bo[b0 + k] = (uint32_t)run;
        run += v[k];
    }
}

// per chunk: word offset of each present stream (n_words + 1 words each) and
// chunk total; one workgroup.  chunk_base: nullable.
__global__ __launch_bounds__(256) void k_chunk_offsets(const int64_t* __restrict__ stream_nbits,
                                                       const lq_table* __restrict__ tables, int64_t n_chunks,
                                                       int64_t* __restrict__ stream_woff,
                                                       int64_t* __restrict__ chunk_words,
                                                       int64_t* __restrict__ chunk_base,
                                                       int64_t* __restrict__ total) {
    for (int64_t c = threadIdx.x; c < n_chunks; c += 256) {
        int64_t nb[LQ_STREAMS];
        int ns[LQ_STREAMS];
#pragma unroll
        for (int st = 0; st < LQ_STREAMS; st++) {
            nb[st] = stream_nbits[c * LQ_STREAMS + st];
            ns[st] = tables[c * LQ_STREAMS + st].n_sym;
        }
        int64_t w = 0;
#pragma unroll
        for (int st = 0; st < LQ_STREAMS; st++) {
            stream_woff[c * LQ_STREAMS + st] = w;
            if (ns[st] > 0) w += (nb[st] + 31) / 32 + 1;
        }
        __hip_atomic_store(chunk_words + c, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!chunk_base) return;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (threadIdx.x < 64) chunk_bases(chunk_words, n_chunks, chunk_base, (int)threadIdx.x, total);
}

// One wave per (stream, group of 32 blocks).  The group owns the stream
// words whose first bit lies in its blocks' bit range; lane l assembles words
// W0 + l + 64 k, kPackU per round with all their scratch loads in flight
// (256-byte coalesced stores).  A word's first bits come from the
// right-aligned scratch of the block holding its first bit (one funnel
// shift), the rest, when the word runs past that block's end, from the first
// bits of the next block (loaded only in those lanes, merged with a select);
// the rare word that also runs past that block, or is the stream's last and
// partly past its end, is assembled block by block.  Scratch and output words
// are addressed with 32-bit byte offsets from wave-uniform bases.  The block of
// each word comes from the blocks' first owned words fw_i = ceil(off_i / 32),
// held one per lane: within a 64-word slice, the block of word w is the last
// block with fw_i <= w, i.e. the last block starting at or before the slice
// (a ballot count) unless one of the few blocks starting inside the slice
// (another ballot, walked on the scalar unit) has fw_i <= w.  The wave of a
// stream's last group also writes the zero word after the stream.  Stream bit
// positions are 32-bit (blk_off is uint32).
constexpr int kPackBlocks = 32;
constexpr int kPackU = 4;   // words per lane per round, their scratch loads all in flight

__global__ __launch_bounds__(256) void k_chunk_pack(int64_t n_streams_total, int64_t nblk, const uint32_t* __restrict__ scratch,
                                                    const uint32_t* __restrict__ blk_off,
                                                    const int64_t* __restrict__ stream_nbits,
                                                    const int64_t* __restrict__ stream_woff,
                                                    const int64_t* __restrict__ chunk_base,
                                                    const lq_table* __restrict__ tables, uint32_t* __restrict__ words) {
    __shared__ uint32_t offs[4][kPackBlocks + 2];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t gps = (nblk + kPackBlocks - 1) / kPackBlocks;   // groups per stream
    const int64_t job = (int64_t)blockIdx.x * 4 + wave;
    const int64_t sid = job / gps;
    const int64_t g0 = (job % gps) * kPackBlocks;
    if (sid >= n_streams_total || tables[sid].n_sym == 0) return;   // wave-uniform; no barrier follows
    const uint32_t nbits = (uint32_t)stream_nbits[sid];
    const int nb = (int)(nblk - g0 < kPackBlocks ? nblk - g0 : kPackBlocks);
    const uint32_t* bo = blk_off + sid * nblk;
    // offset of block g0 + i (the stream end past the last block); staged for i <= nb + 1
    auto off_glb = [&](int i) -> uint32_t { return g0 + i < nblk ? bo[g0 + i] : nbits; };
    uint32_t* of = offs[wave];
    const uint32_t myof = lane <= nb + 1 ? off_glb(lane) : 0u;
    if (lane <= nb + 1) of[lane] = myof;
    __builtin_amdgcn_wave_barrier();
    auto off_at = [&](int i) -> uint32_t { return i <= nb + 1 ? of[i] : off_glb(i); };
    // first owned word of block `lane` (blocks 0 .. nb - 1), else past every word
    const uint32_t myfw = lane < nb ? (myof + 31u) >> 5 : 0xffffffffu;
    const uint32_t W0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)((myof + 31u) >> 5));
    const uint32_t W1 = (uint32_t)__builtin_amdgcn_readlane((int)((myof + 31u) >> 5), nb);
    uint32_t* out = words + chunk_base[sid / LQ_STREAMS] + stream_woff[sid];
    // the stream's trailing zero word, from the wave of its last group
    if (g0 + nb >= nblk && lane == 0) out[((uint64_t)nbits + 31u) >> 5] = 0u;
    const uint32_t* scr0 = scratch + (sid * nblk + g0) * (int64_t)kCapW;
    constexpr uint32_t kCapBits = (uint32_t)kCapW * 32u;
    // scratch word i of the group (i < (nb + 1) * kCapW), as a 32-bit byte
    // offset from the wave-uniform base; likewise the stream's output words
    auto scr = [&](uint32_t i) -> uint32_t {
        return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(scr0) + (i << 2));
    };
    for (uint32_t wr = W0; wr < W1; wr += 64u * kPackU) {
        uint32_t lo[kPackU], hi[kPackU], clo[kPackU], chi[kPackU];
        int blk[kPackU], take[kPackU], s2[kPackU], cs[kPackU];
        uint32_t pe[kPackU];
        bool nxt[kPackU], rare[kPackU];
#pragma unroll
        for (int u = 0; u < kPackU; u++) {
            const uint32_t ws = wr + 64u * u;   // first word of the slice (wave-uniform)
            const uint32_t w = ws + lane;
            const bool ok = w < W1;
            // blocks starting at or before the slice, and inside it
            const uint64_t at = __ballot(myfw <= ws);
            uint64_t in = __ballot(myfw > ws && myfw <= ws + 63u);
            int b = __builtin_popcountll(at) - 1;
            while (in) {
                const int i = __builtin_ctzll(in);
                in &= in - 1;
                const uint32_t fwi = (uint32_t)__builtin_amdgcn_readlane((int)myfw, i);
                b = w >= fwi ? i : b;
            }
            const uint32_t p = 32u * (ok ? w : W0);
            if (!ok) b = 0;
            const uint32_t ob = of[b], oe = of[b + 1], on = of[b + 2];
            const uint32_t end = p + 32u < nbits ? p + 32u : nbits;
            const uint32_t e1 = end < oe ? end : oe;
            const uint32_t sp = kCapBits - (oe - ob) + (p - ob);   // scratch bit of p
            const uint32_t k0 = sp >> 5;
            const uint32_t i0 = (uint32_t)b * (uint32_t)kCapW + k0;
            lo[u] = scr(i0);
            hi[u] = scr(k0 + 1 < (uint32_t)kCapW ? i0 + 1 : i0);
            // a word running past its block's end continues with the first bits
            // of block b + 1 (when that block is not empty): load them in the
            // lanes that need them; they are consumed unconditionally below, so
            // no load is left pending into the next round
            const uint32_t sp1 = kCapBits - (on - oe);            // scratch bit of block b + 1's first bit
            const uint32_t k1 = sp1 >> 5;
            const bool cont = ok && e1 < end;
            nxt[u] = cont && on > oe;
            clo[u] = 0u;
            chi[u] = 0u;
            if (nxt[u]) {
                const uint32_t i1 = (uint32_t)(b + 1) * (uint32_t)kCapW + k1;
                clo[u] = scr(i1);
                chi[u] = scr(k1 + 1 < (uint32_t)kCapW ? i1 + 1 : i1);
            }
            const uint32_t e2 = end < on ? end : on;
            // rare: block b + 1 is empty, ends inside the word too, or the word
            // is the stream's last and partly past its end (its unused bits
            // must be zero); otherwise the two segments fill all 32 bits
            rare[u] = cont && e2 != p + 32u;
            blk[u] = b;
            take[u] = (int)(e1 - p);   // 1 .. 32
            s2[u] = (int)(sp & 31u);
            cs[u] = (int)(sp1 & 31u);
            pe[u] = e1;
        }
#pragma unroll
        for (int u = 0; u < kPackU; u++) {
            const uint32_t w = wr + 64u * u + lane;
            const int got = take[u];
            uint32_t res = __builtin_amdgcn_alignbit(hi[u], lo[u], (uint32_t)s2[u]) & (0xffffffffu >> ((32 - got) & 31));
            // the next block's first bits fill the rest of the word (got < 32 there)
            const uint32_t seg2 = __builtin_amdgcn_alignbit(chi[u], clo[u], (uint32_t)cs[u]) << (got & 31);
            res |= nxt[u] ? seg2 : 0u;
            if (rare[u]) {
                // block by block from block b + 1: empty blocks are skipped,
                // a block ending inside the word gives only its bits
                res &= 0xffffffffu >> ((32 - got) & 31);
                const uint32_t end = 32u * w + 32u < nbits ? 32u * w + 32u : nbits;
                uint32_t p = pe[u];
                int gb = got;
                int b = blk[u] + 1;
                while (p < end) {
                    const uint32_t ob = off_at(b), oe = off_at(b + 1);
                    if (oe > ob) {
                        const uint32_t e1 = end < oe ? end : oe;
                        const int tk2 = (int)(e1 - p);
                        const uint32_t sp = kCapBits - (oe - ob) + (p - ob);
                        const uint32_t* sc = scr0 + (int64_t)b * kCapW;
                        uint64_t y = sc[sp >> 5];
                        if ((int)(sp & 31u) + tk2 > 32) y |= (uint64_t)sc[(sp >> 5) + 1] << 32;
                        y >>= (sp & 31u);
                        res |= (tk2 == 32 ? (uint32_t)y : (uint32_t)y & ((1u << tk2) - 1u)) << gb;
                        gb += tk2;
                        p = e1;
                    }
                    b++;
                }
            }
            if (w < W1) *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(out) + (w << 2)) = res;
        }
    }
}

// ------------------------------------------------------------ chunk decode --

// Decoder LUTs of every chunk stream for decode attention (lut_entry format,
// lq_decode.h): stream st of a chunk sits at row st & 7 (the 8 LUTs of one
// coset form one LDS block) and the symbol field is the alphabet index.
__global__ __launch_bounds__(256) void k_chunk_lut(const lq_table* __restrict__ tables, uint32_t* __restrict__ lut) {
    __shared__ int32_t fr[LQ_MAXSYM];
    __shared__ int32_t cum[LQ_MAXSYM + 1];
    const int64_t sid = blockIdx.x;
    const lq_table* T = tables + sid;
    const int n = T->n_sym;
    if (n == 0) return;
    for (int i = threadIdx.x; i < n; i += 256) fr[i] = (int32_t)enc_f(T->enc[i]);
    __syncthreads();
    exclusive_scan_array<BlockGroup>(fr, n, cum);
    const uint32_t row = (uint32_t)(sid % LQ_STREAMS) & 7u;
    for (int slot = threadIdx.x; slot < kL; slot += 256) {
        int lo = 0, hi = n - 1;   // largest s with cum[s] <= slot
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (cum[mid] <= slot) lo = mid; else hi = mid - 1;
        }
        lut[sid * kL + slot] = lut_entry((uint32_t)lo, (uint32_t)(fr[lo] + slot - cum[lo]), row);
    }
}

// Inclusive maximum over the lanes below and at each lane of a wave (all 64
// active), the moves of wave_incl_scan.
__device__ __forceinline__ uint32_t wave_incl_max(uint32_t x) {
    auto up = [](uint32_t v, uint32_t u) { return u > v ? u : v; };
    int v = (int)x;
    v = (int)up((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));   // row_shr:1
    v = (int)up((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));   // row_shr:2
    v = (int)up((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));   // row_shr:4
    v = (int)up((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));   // row_shr:8
    v = (int)up((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = (int)up((uint32_t)v, (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return (uint32_t)v;
}

// The chunk decoder's LUT of one stream (lut_entry format, symbol field biased
// by `bias`), built in LDS by one wave: every symbol writes one word (its cum,
// index and frequency, ordered by cum) at its first slot, a running maximum
// hands it to the slots up to the next symbol's, and each slot's entry follows
// from it.  Lane l owns slots 16 l .. 16 l + 15.
__device__ __forceinline__ void wave_lut(const lq_table* __restrict__ T, uint32_t row, uint32_t bias, uint32_t* lut,
                                         int lane) {
    // the first 256 entries are loaded with n_sym, not after it (entries past
    // n_sym are allocated, and not used)
    uint32_t e[4];
#pragma unroll
    for (int u = 0; u < 4; u++) e[u] = T->enc[64 * u + lane];
    const int n = T->n_sym < kL ? T->n_sym : kL;
    if (n <= 0) return;   // absent stream: no lane looks its row up
    uint4* const mine = reinterpret_cast<uint4*>(lut + 16 * lane);
#pragma unroll
    for (int i = 0; i < 4; i++) mine[i] = make_uint4(0u, 0u, 0u, 0u);
    WaveGroup::sync();
    for (int j0 = 0;;) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int j = j0 + 64 * u + lane;
            const uint32_t f = enc_f(e[u]), cum = enc_c(e[u]);
            if (j < n && f) lut[cum] = (cum << 21) | ((uint32_t)j << 11) | f;
        }
        j0 += 256;
        if (j0 >= n) break;
#pragma unroll
        for (int u = 0; u < 4; u++) e[u] = j0 + 64 * u + lane < n ? T->enc[j0 + 64 * u + lane] : 0u;
    }
    WaveGroup::sync();
    uint32_t v[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint4 q = mine[i];
        v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
    }
#pragma unroll
    for (int i = 1; i < 16; i++) v[i] = v[i] > v[i - 1] ? v[i] : v[i - 1];
    const uint32_t below = (uint32_t)__shfl_up((int)wave_incl_max(v[15]), 1, 64);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const uint32_t m = lane && below > v[i] ? below : v[i];
        const uint32_t xp = (m & 0x7ffu) + (uint32_t)(16 * lane + i) - (m >> 21);
        // as lut_entry; xp >= 1 in a valid table (a malformed one gives in-range garbage)
        const int z = __clz((int)(xp | 1u)) - 21;
        const uint32_t k = z > 0 ? (uint32_t)z : 0u;
        v[i] = k | ((((m >> 11) & 1023u) + bias) << 6) | ((row * (uint32_t)kL + (((xp << k) - (uint32_t)kL) & (kL - 1u))) << 18);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) mine[i] = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}

// Whole-line chunk decoder.
//
// A wave decodes 4 consecutive blocks of one chunk at a time (a task), 16
// lanes per block: lane (block b, coset c, coordinate idx) decodes stream
// c * 8 + idx of block b with LineLane, in phases of 8 steps.  Step j of a
// phase stages the symbol index of coset-c vector `st + j` of the block at
// rank slot (st + j) % 16 of the (block, coset) staging, so no lane walks the
// coset bitmap per symbol.  After each phase the block's 16 lanes flush the
// output in whole 128-byte lines (8 vectors): a line is flushed once both
// cosets have staged every vector in it; a flushed vector's rank in its coset
// is the flushed count plus a popcount of the coset-1 bitmap below it.  A
// phase flushes at most two lines (16 consecutive vectors, 256 bytes, one
// per lane of the block's row): a second round for lines 3 and 4 left most
// of its lanes idle and cost more than the extra phases the cap adds (the
// first flushable line is always taken, so the cap never stalls the loop).
// A coset runs a phase only if the 8 vectors it stages fit the ring next to
// its unflushed ones (st - flushed <= 8).  That never blocks for good: the
// first unflushed line holds at most 8 vectors of each coset, so a coset
// that has not staged all of them has fewer than 8 unflushed and may run.
// HEADS_ALIGNED: bph is a multiple of the block size, so a block lies in one
// head.  DITHER: the chunk's dither (dither8, seed dseed[chunk]) is
// subtracted from each lattice point before scaling.
constexpr int kDecBlocks = 64;                  // blocks in flight per decode workgroup (4 per wave)
constexpr int kDecThreads = 16 * kDecBlocks;    // 1024
constexpr int kDecStage = 16;                   // staged vectors per (block, coset)
// Staging of (block b, coset c): group b * 2 + c, 16 slots of 8 u16, padded to
// 68 words so that group bases fall on banks 4 g (mod 64): the 8 groups of a
// wave write their slots j or j + 8 on disjoint banks.
constexpr int kDecGroupU16 = 136;

__device__ __forceinline__ int dpp_ror8(int v) {   // lane l <- lane l ^ 8 within each 16-lane row
    return __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false);
}

template <int OUT_DT, bool HEADS_ALIGNED, bool DITHER, bool ROT = false, bool ESC = false>
__global__ __launch_bounds__(kDecThreads) void k_chunk_decode(
        const uint32_t* __restrict__ words, const int64_t* __restrict__ chunk_base, const int64_t* __restrict__ stream_woff,
        const uint32_t* __restrict__ blk_off, const int64_t* __restrict__ stream_nbits,
        const uint16_t* __restrict__ blk_state, const uint8_t* __restrict__ coset_bits,
        const lq_table* __restrict__ tables, const uint16_t* __restrict__ scale16,
        int64_t n_chunks, int64_t n_heads, int64_t bph, int64_t nblk, int64_t span, int64_t tpw, int wpc, void* __restrict__ out,
        const int64_t* __restrict__ dseed, const float* __restrict__ signs, int lpr, float rdiv,
        const int32_t* __restrict__ esc_k, const int64_t* __restrict__ fine_off, const uint32_t* __restrict__ fine) {
    __shared__ uint32_t lut[LQ_STREAMS * kL];                               // 64 KB
    __shared__ uint32_t ring[kDecThreads / 64][kLineRing][64];              // 48 KB
    __shared__ __align__(16) uint16_t stg[kDecBlocks * 2 * kDecGroupU16];   // 34 KB
    __shared__ uint32_t bm1[kDecBlocks][kBlk / 32 + 1];                     // coset-1 bits, one zero word after each row
    const int tid = threadIdx.x;
    const float rrcp = ROT ? 1.0f / rdiv : 1.0f;   // the rotation's RN(1 / sqrt(head_dim))
    const int64_t V = n_heads * bph;
    // the workgroup's tasks (decode_split): chunk c has numbers c * span .., its
    // (nblk + 3) / 4 tasks first
    const int64_t wc = wpc > 0 ? (int64_t)blockIdx.x / wpc : 0;
    const int64_t first = wc * span + ((int64_t)blockIdx.x - wc * wpc) * tpw;
    const int64_t lim = wpc > 0 ? (wc + 1) * span : n_chunks * span;
    const int64_t last = first + tpw < lim ? first + tpw : lim;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // The workgroup walks tasks first .. last - 1, chunk by chunk; wave w builds
    // the LUT of the chunk's stream w, between two barriers, and takes the
    // chunk's tasks w, w + 16, ..  Each wave stages its own 4 blocks' bitmaps
    // and moves to its next task without waiting for the other waves.
    for (int64_t t0 = first; t0 < last;) {
    const int64_t chunk = t0 / span;
    const int64_t tend = (chunk + 1) * span < last ? (chunk + 1) * span : last;
    const int64_t tasks_end = chunk * span + (nblk + 3) / 4 < tend ? chunk * span + (nblk + 3) / 4 : tend;
    const bool lut_biased = chunk_biased(tables + chunk * LQ_STREAMS, lane);   // the LUTs' symbol fields
    if (t0 != first) __syncthreads();   // every wave is done with the previous chunk's LUTs
    {
        const lq_table* T = tables + chunk * LQ_STREAMS + wave;
        wave_lut(T, (uint32_t)wave, lut_biased ? (uint32_t)(T->lo + ((wave & 7) < 7 ? 512 : 256)) : 0u,
                 lut + wave * kL, lane);
    }
    __syncthreads();
    for (int64_t task4 = t0 + wave; task4 < tasks_end; task4 += kDecThreads / 64) {
    const int64_t gbase = (task4 - chunk * span) * 4 - wave * 4;   // block b of the workgroup: gbase + b
    __builtin_amdgcn_wave_barrier();
    for (int i = lane; i < 4 * (kBlk / 32 + 1); i += 64) {
        const int bl = wave * 4 + i / (kBlk / 32 + 1), w = i % (kBlk / 32 + 1);
        const int64_t g = gbase + bl;
        uint32_t m = 0;
        if (w < kBlk / 32 && g < nblk) {
            m = reinterpret_cast<const uint32_t*>(coset_bits + (chunk * nblk + g) * (kBlk / 8))[w];
            const int64_t lim = V - g * kBlk - 32 * w;
            m = lim >= 32 ? m : (lim <= 0 ? 0u : m & ((1u << lim) - 1u));
        }
        bm1[bl][w] = m;
    }
    __builtin_amdgcn_wave_barrier();
    {
    const int b = tid >> 4, c = (tid >> 3) & 1, idx = tid & 7, l16 = tid & 15;
    const int64_t g = gbase + b;
    if (g >= nblk) continue;   // whole blocks (16-lane rows) skip together
    const int64_t vfirst = g * kBlk;                 // first vector of the block, within the chunk
    const int valid = (int)(V - vfirst < kBlk ? V - vfirst : kBlk);
    // coset-1 count of the block from its bitmap (equal to blk_n1 for every
    // chunk the encoder wrote); counting it here ties the loop below to the
    // bitmap, so it ends even if the metadata disagrees with it
    int n1 = 0;
#pragma unroll
    for (int w = 0; w < kBlk / 32; w++) n1 += __builtin_popcount(bm1[b][w]);
    const int n = c ? n1 : valid - n1;
    const lq_table* T = tables + chunk * LQ_STREAMS;
    // escaped chunk (coarse symbols plus raw low bits, alphabets beyond L):
    // the generic path with the low bits merged in
    const int32_t* const ekc = ESC && esc_k ? esc_k + chunk * 8 : nullptr;
    bool esc = false;
    EscCoords ec;
    if (ESC && ekc) {
        ec.init(ekc, fine_off + chunk * 8, fine);
#pragma unroll
        for (int j = 0; j < 8; j++) esc = esc || ec.k[j] != 0;
    }
    const bool biased = !esc && lut_biased;
    CosetConsts cc0, cc1;   // per-coset alphabet lows, for chunks whose fields are not biased
    if (!biased) {
        cc0.init(T, 0);
        cc1.init(T + 8, 1);
    }
    float sc;
    half2_t sc2;
    const float* sgp = nullptr;   // ROT: the head's sign row
    auto set_scale = [&](int64_t head) {
        const uint16_t s16 = scale16[chunk * n_heads + head];
        sc = h2f(s16);
        const _Float16 sh = __builtin_bit_cast(_Float16, s16);
        sc2 = half2_t{sh, sh};
        if (ROT) sgp = signs + (chunk * n_heads + head) * (8 * (int64_t)lpr);
    };
    const int64_t head0 = vfirst / bph;
    set_scale(head0);
    int64_t head_end = (head0 + 1) * bph;            // first chunk vector of the next head

    const int st_id = c * 8 + idx;
    const int64_t sid = chunk * LQ_STREAMS + st_id;
    LineLane d;
    if (n > 0) {
        const int64_t task = sid * nblk + g;
        const int64_t end_bit = g + 1 < nblk ? (int64_t)blk_off[task + 1] : stream_nbits[sid];
        d.init(words + chunk_base[chunk] + stream_woff[sid], blk_off[task], end_bit, blk_state[task], lut, st_id,
               &ring[tid >> 6][0][tid & 63]);
    } else {
        d.inflight = false;
    }
    const char* const lutb = reinterpret_cast<const char*>(lut);
    using OutT = typename std::conditional<OUT_DT == LQ_F32, float, uint16_t>::type;
    OutT* const ob = reinterpret_cast<OutT*>(out) + (chunk * V + vfirst) * 8;
    const uint64_t dkey = DITHER ? mix64((uint64_t)dseed[chunk]) : 0u;
    const uint32_t* const bmr = bm1[b];
    uint16_t* const my_stg = &stg[(b * 2 + c) * kDecGroupU16 + idx];
    const int u = (l16 & 1) + 1;     // lines of the flush candidate this lane checks

    float pend[ROT ? 8 : 1];         // ROT: butterfly stages of a deferred first half-row (lanes 0..7)
    int st = 0;                      // vectors of my coset staged (symbols of my stream decoded)
    int fpos = 0, fr0 = 0, fr1 = 0;  // flushed block positions and flushed ranks per coset (block-uniform)
    d.boundary(n > 0);
    while (fpos < valid) {
        __builtin_amdgcn_wave_barrier();
        if (st < n && st - (c ? fr1 : fr0) <= kDecStage - 8) {
            // st % 8 == 0 here, so the phase's slots do not wrap; a last phase
            // with fewer than 8 symbols stages garbage in slots of ranks >= n,
            // which hold no unflushed rank (st + 8 - flushed <= 16) and are never read
            d.phase(my_stg + (st & (kDecStage - 1)) * 8, lutb);
            st = n - st < kPhase ? n : st + kPhase;
        }
        // The boundary comes between the steps and the flush: the wait for the
        // top-up also waits for older stores, and here those are a phase old
        // (before the steps it waited for the stores just issued: 131072 blocks
        // 520 us, here 493).
        d.boundary(st < n);
        __builtin_amdgcn_wave_barrier();
        const int st_o = dpp_ror8(st);
        const int s0 = c ? st_o : st, s1 = c ? st : st_o;
        // coset-1 bits of positions fpos .. fpos + 31; lanes 0 and 1 of the
        // block's row check whether the first 1 and 2 lines can be flushed (the
        // answers are monotone, so their count is the number of lines flushed)
        const int wi = fpos >> 5;
        const uint32_t W = __builtin_amdgcn_alignbit(bmr[wi + 1], bmr[wi], (uint32_t)(fpos & 31));
        const int rest = valid - fpos;
        const int np = rest < 8 * u ? rest : 8 * u;                  // 1 <= np <= 16
        const int p1 = __builtin_popcount(W << ((32 - np) & 31));   // coset-1 vectors among them
        const bool ok = 8 * (u - 1) < rest && fr0 + np - p1 <= s0 && fr1 + p1 <= s1;
        const uint64_t bal = __builtin_amdgcn_ballot_w64(ok);
        int nl = __builtin_popcountll((bal >> (tid & 48)) & 0x3ull);   // 0, 1 or 2 lines
        // ROT: a flush that starts in the middle of a 16-vector row takes one
        // line, the row's second half, so the next flushes start on a row
        // again (a 16-vector flush from the middle of a row runs the
        // butterflies of two rows for one row's stores)
        if (ROT && (fpos & 8) && nl > 1) nl = 1;
        const int F = 8 * nl < rest ? 8 * nl : rest;   // positions flushed this phase (<= 16)
        // fp32 output row of position p (fpos <= p < fpos + F): the lattice
        // point from its staged symbols, dither removed, times the head's scale
        auto lattice_y = [&](int p, float y[8]) {
            const int q = p - fpos;
            const bool cp = (W >> q) & 1u;
            const int n1b = __builtin_popcount(W & ((1u << q) - 1u));
            const int rank = cp ? fr1 + n1b : fr0 + q - n1b;
            const uint4 r = *reinterpret_cast<const uint4*>(&stg[(b * 2 + cp) * kDecGroupU16 + (rank & (kDecStage - 1)) * 8]);
            if (!HEADS_ALIGNED && vfirst + p >= head_end) {
                const int64_t head = (vfirst + p) / bph;
                head_end = (head + 1) * bph;
                set_scale(head);
            }
            if (biased) {
                lattice_biased_f32(r, cp ? 0.5f : 0.f, y);
            } else if (ESC && esc) {
                CosetConsts cs;
                cs.pick(cp, cc0, cc1);
                lattice_escaped_f32(r, cs, lut_biased, ec, vfirst + p, y);
            } else {
                CosetConsts cs;
                cs.pick(cp, cc0, cc1);
                cs.deq_f32(r, 1.0f, y);   // the lattice point itself (exact)
            }
            if constexpr (DITHER) {
                float dd[8];
                dither8(dkey, vfirst + p, dd);
#pragma unroll
                for (int j = 0; j < 8; j++) y[j] = (y[j] - dd[j]) * sc;
            } else {
#pragma unroll
                for (int j = 0; j < 8; j++) y[j] *= sc;
            }
        };
        if constexpr (ROT) {
            // Lane l16 stores the positions p == l16 (mod 16) of the flush, so a
            // 16-vector row's first half always sits in lanes 0..7 and its second
            // half in lanes 8..15.  Rows of lpr <= 8 vectors lie inside one line
            // and are rotated back whole.  When a 16-vector row's first line
            // flushes before its second, that half's butterfly stages (h <= 32)
            // wait in registers (pend) and its store is deferred; when the second
            // line comes both halves take the last stage (h = 64) together: the
            // operations and their order are those of the whole-row transform.
            for (int base = fpos & ~15; F > 0 && base < fpos + F; base += 16) {
                const int p = base + l16;
                const bool mine = p >= fpos && p < fpos + F;
                float y[8];
                if (mine) lattice_y(p, y);
                float sg[8];
                load_signs8(sgp + 8 * (l16 & (lpr - 1)), sg);
                if (lpr < 16) {
                    if (mine) {
                        rht_lanes(y, sg, l16 & (lpr - 1), lpr, rdiv, rrcp, true);
                        store8(ob, OUT_DT, p, y);
                    }
                } else {
                    const bool fh = base >= fpos && base + 8 <= fpos + F;   // the row's first line flushes now
                    const bool sh = base + 16 <= fpos + F;                   // its second line flushes now
                    if (mine) fwht_stages(y, l16 & 7, 8);
                    if (!sh) {
                        if (fh && mine) {
#pragma unroll
                            for (int j = 0; j < 8; j++) pend[j] = y[j];
                        }
                    } else {
                        if (!fh && l16 < 8) {
#pragma unroll
                            for (int j = 0; j < 8; j++) y[j] = pend[j];
                        }
                        fwht_cross(y, l16, 8);
                        div_sqrt_dim8(y, rdiv, rrcp);
#pragma unroll
                        for (int j = 0; j < 8; j++) y[j] = y[j] * sg[j];
                        store8(ob, OUT_DT, base + l16, y);
                    }
                }
            }
        } else {
            for (int r0 = 0; r0 < F; r0 += 16) {
                const int q = r0 + l16;
                if (q < F) {
                    const int p = fpos + q;
                    if (!DITHER && OUT_DT == LQ_F16 && biased) {
                        const bool cp = (W >> q) & 1u;
                        const int n1b = __builtin_popcount(W & ((1u << q) - 1u));
                        const int rank = cp ? fr1 + n1b : fr0 + q - n1b;
                        const uint4 r = *reinterpret_cast<const uint4*>(
                            &stg[(b * 2 + cp) * kDecGroupU16 + (rank & (kDecStage - 1)) * 8]);
                        if (!HEADS_ALIGNED && vfirst + p >= head_end) {
                            const int64_t head = (vfirst + p) / bph;
                            head_end = (head + 1) * bph;
                            set_scale(head);
                        }
                        const _Float16 o = cp ? (_Float16)0.5f : (_Float16)0.0f;
                        reinterpret_cast<uint4*>(ob)[p] = deq_biased_f16(r, half2_t{o, o}, sc2);
                    } else {
                        float y[8];
                        lattice_y(p, y);
                        store8(ob, OUT_DT, p, y);
                    }
                }
            }
        }
        const int f1 = __builtin_popcount(W) - __builtin_popcount((uint32_t)((uint64_t)W >> F));   // 0 <= F <= 16
        fr1 += f1;
        fr0 += F - f1;
        fpos += F;
    }
    }
    }
    t0 = tend;
    }
}

// ------------------------------------------------------- generic tables --

__global__ __launch_bounds__(256) void k_build_tables(const int64_t* __restrict__ counts, const int64_t* __restrict__ count_off,
                                                      const int32_t* __restrict__ n_sym, int32_t* __restrict__ freqs_out,
                                                      int32_t* __restrict__ cum_out, int32_t* __restrict__ lookup,
                                                      int32_t* __restrict__ status) {
    __shared__ int64_t cnt[kL];
    __shared__ int32_t fr[kL];
    __shared__ NpScratch ns;
    __shared__ int16_t perm[kL];
    __shared__ int s_st;
    const int t = blockIdx.x;
    const int n = n_sym[t];
    const int64_t o = count_off[t];
    if (n <= 0 || n > kL) {
        if (threadIdx.x == 0) status[t] = LQ_ST_ALPHABET;
        return;
    }
    for (int i = threadIdx.x; i < n; i += 256) cnt[i] = counts[o + i];
    if (threadIdx.x == 0) s_st = 0;
    __syncthreads();
    __shared__ int64_t kk[kL];
    __shared__ int8_t inset[kL];
    normalise<BlockGroup>(cnt, n, fr, perm, kk, inset, &ns);
    __shared__ int32_t cum[kL + 1];
    exclusive_scan_array<BlockGroup>(fr, n, cum);
    for (int i = threadIdx.x; i < n; i += 256) freqs_out[o + i] = fr[i];
    for (int i = threadIdx.x; i <= n; i += 256) cum_out[o + t + i] = cum[i];
    for (int slot = threadIdx.x; slot < kL; slot += 256) {   // largest s with cum[s] <= slot
        int lo = 0, hi = n - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (cum[mid] <= slot) lo = mid; else hi = mid - 1;
        }
        lookup[(int64_t)t * kL + slot] = lo;
    }
    if (threadIdx.x == 0) status[t] = s_st;
}

// ------------------------------------------------------ generic streams --

// Encode of arbitrary streams.  A stream is cut into segments of kSegSyms
// symbols, one lane each; a lane finds the exact state entering its segment as
// the chunk encoder does (an interval of states, run over a growing window of
// the symbols behind the segment until it is one state or the window reaches the
// stream's end, where the state is L), encodes the segment into its LDS column,
// and the segments' bits are joined by a scan of their counts.
//
// Workgroup b takes streams b, b + gridDim, ..  Streams of up to 64, 256, 1024
// and 4096 symbols are taken together by as many groups of 1, 4, 16 and 64 lanes
// as there are, each group writing its stream's words in place; longer ones by the
// whole workgroup, one after the other (encode_long).  One lane per stream,
// symbol by symbol, took 9278 us for 16 streams of 32768 symbols, 52 us so; one
// workgroup per stream whatever its length took 7614 us for 32768 streams of 10
// symbols, 125 for 512 of 10 and 578 for 2048 of 1000; a lane per stream 8, 8 and
// 269; so 10, 8 and 27 us.
// The tables are build_rans_table's (frequencies in [1, L], summing to L).
constexpr int kSegSyms = 64;
constexpr int kSegWords = 10 * kSegSyms / 32;   // at most 10 bits per symbol
constexpr int kSegLanes = 1024;
constexpr int kGroupSyms = 64 * kSegSyms;       // longest stream of a group of lanes

// f(entry, in) for symbols j1 - 1 .. j0, U at a time with their loads together
// (U of 8 where every lane has its own stream, i.e. its own 64-bit addresses)
template <int U, typename F>
__device__ __forceinline__ void seg_rev(const int32_t* id, const int32_t* freqs, const int32_t* cum, int j0, int j1, F&& f) {
    for (int j = j1; j > j0; j -= U) {
        uint32_t e[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int p = j - 1 - u > j0 ? j - 1 - u : j0;
            e[u] = (uint32_t)id[(uint32_t)p];
        }
#pragma unroll
        for (int u = 0; u < U; u++) e[u] = encx_of(enc_pack((uint32_t)freqs[e[u]], (uint32_t)cum[e[u]]));
#pragma unroll
        for (int u = 0; u < U; u++) f(e[u], j - 1 - u >= j0);
    }
}

// The state entering the segment that ends at e, from the symbols behind it up to
// `end`, where the state is xend: an interval of states over windows of 16, 64, ..
// `limit` symbols; 0 if that leaves more than one.
template <int U>
__device__ __forceinline__ uint32_t seg_state(const int32_t* id, const int32_t* freqs, const int32_t* cum, int e, int end,
                                              uint32_t xend, int limit) {
    if (e >= end) return xend;
    for (int window = 16; window <= limit; window *= 4) {
        const bool whole = e + window >= end;
        uint32_t lo = whole ? xend : (uint32_t)kL, hi = whole ? xend : 2u * kL - 1u;
        seg_rev<U>(id, freqs, cum, e, whole ? end : e + window, [&](uint32_t en, bool in) {
            uint32_t l2 = lo, h2 = hi;
            hull_step(l2, h2, en);
            lo = in ? l2 : lo;
            hi = in ? h2 : hi;
        });
        if (lo == hi) return lo;   // always so once the window reaches the end
    }
    return 0;
}

// Segment [b, e) of a stream, entered in state *xio, into the lane's column,
// right-aligned in the column's first *capw words; the count of its bits.  *xio:
// the state it leaves.
template <int U>
__device__ __forceinline__ uint32_t seg_encode(const int32_t* id, const int32_t* freqs, const int32_t* cum, int b, int e,
                                               uint32_t (*seg)[kSegLanes], int tid, int* capw, uint32_t* xio) {
    uint32_t x = *xio, total = 0;
    *capw = (10 * (e - b) + 31) / 32;
    int wpos = *capw - 1;
    uint64_t acc = 0;
    uint32_t nacc = 0;
    seg_rev<U>(id, freqs, cum, b, e, [&](uint32_t en, bool in) {
        uint32_t k;
        const uint32_t xin = x, xn = encx_step(xin, en, &k);
        if (in) {
            acc = (acc << k) | (((uint64_t)__builtin_bitreverse32(xin) << k) >> 32);
            nacc += k;
            total += k;
            x = xn;
            if (nacc >= 32) {
                nacc -= 32;
                seg[wpos][tid] = (uint32_t)(acc >> nacc);
                wpos = wpos > 0 ? wpos - 1 : 0;   // never below 0 with tables of the kind above
            }
        }
    });
    if (nacc) seg[wpos][tid] = (uint32_t)(acc << (32 - nacc));
    *xio = x;
    return total < 32u * (uint32_t)*capw ? total : 32u * (uint32_t)*capw;
}

// The total bits of a lane's column (right-aligned in capw words) to bits D ..
// D + total - 1 of dst; a word shared with other lanes (SHARED) is merged into
// its cleared place with an atomic.
template <bool SHARED>
__device__ __forceinline__ void seg_copy(const uint32_t (*seg)[kSegLanes], int tid, int capw, uint32_t total, int64_t D,
                                         uint32_t* dst) {
    const int sp0 = capw * 32 - (int)total;   // first bit in the column
    for (int64_t w = D >> 5; total && w <= (D + total - 1) >> 5; w++) {
        const int64_t lo = w * 32 > D ? w * 32 : D, hi = w * 32 + 32 < D + total ? w * 32 + 32 : D + total;
        const int sp = sp0 + (int)(lo - D), take = (int)(hi - lo), wi = sp >> 5, sh = sp & 31;
        uint64_t v = seg[wi][tid];
        if (sh + take > 32) v |= (uint64_t)seg[wi + 1][tid] << 32;
        const uint32_t bits = (uint32_t)(v >> sh);
        if (take == 32) dst[w] = bits;
        else if (SHARED) atomicOr(dst + w, (bits & ((1u << take) - 1u)) << (int)(lo - w * 32));
        else dst[w] = bits & ((1u << take) - 1u);   // D = 0: the last word's low bits
    }
}

// Stores of this wave have reached the L2, where the atomics of its CU work.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A stream by the whole workgroup.  Encoding runs from the stream's end, so a
// segment's place is known from the end: the joined bits are right-aligned in the
// stream's scratch words, and a last pass shifts them to the reference's layout
// (n_words + 1 words, last zero).  Streams longer than kSegLanes segments take
// that many at a time (a tile), from the end; a tile's last state is the state the
// tile behind it left.
//
// Long runs of one symbol of nearly all of L move the states round without ever
// bringing them together, so a window there only ends at the tile's end.  Lanes
// left without a state after kSegWindow symbols get it from the first wave, which
// walks the segments behind them one after the other from a known state, the
// entries of a segment loaded by its lanes: with windows to the stream's end a run
// of 262144 symbols took 271 ms, of 32768 7.5 (one lane per stream 51 and 6.4); so
// 16.2 and 1.9.
constexpr int kSegWindow = 4096;
struct LongLds {
    uint32_t wsum[kSegLanes / 64];
    uint32_t state[kSegLanes];               // entering states, 0: not known yet
    uint64_t missing[kSegLanes / 64];        // the lanes without one, per wave
    uint32_t tile_end;                       // the state the tile's last segment is entered in
};

// id: the tile's n symbols
__device__ __forceinline__ void walk_missing(const int32_t* id, const int32_t* freqs, const int32_t* cum, int n, LongLds& l) {
    const int lane = threadIdx.x & 63;
    auto entry = [&](int i) {   // of symbol `lane` of the tile's segment i
        const int p = i * kSegSyms + lane;
        const uint32_t v = (uint32_t)id[(uint32_t)(p < n ? p : n - 1)];
        return encx_of(enc_pack((uint32_t)freqs[v], (uint32_t)cum[v]));
    };
    int have = -1;   // the segment whose entries are here
    uint32_t en = 0;
    for (int w = kSegLanes / 64 - 1; w >= 0; w--) {
        const uint64_t m0 = l.missing[w];
        uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)m0) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(m0 >> 32)) << 32;
        while (m) {
            const int i = 64 * w + 63 - __builtin_clzll(m);   // behind it: segment i + 1, whose state is known
            m &= ~(1ull << (i & 63));
            if (have != i + 1) en = entry(i + 1);
            const uint32_t next = entry(i);   // in flight during the steps
            have = i;
            uint32_t x = (uint32_t)__builtin_amdgcn_readfirstlane((int)l.state[i + 1]), k;
            const int left = n - (i + 1) * kSegSyms;
            if (left >= kSegSyms) {
#pragma unroll
                for (int j = kSegSyms - 1; j >= 0; j--) x = encx_step(x, (uint32_t)__builtin_amdgcn_readlane((int)en, j), &k);
            } else {
                for (int j = left - 1; j >= 0; j--) x = encx_step(x, (uint32_t)__builtin_amdgcn_readlane((int)en, j), &k);
            }
            if (lane == 0) l.state[i] = x;
            WaveGroup::sync();
            en = next;
        }
    }
}

__device__ __forceinline__ void encode_long(const int32_t* id, const int32_t* freqs, const int32_t* cum, int64_t n,
                                            uint32_t* scr, uint32_t* out, int64_t* state_out, int64_t* nbits_out,
                                            uint32_t (*seg)[kSegLanes], LongLds& l) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t cap = (10 * n + 31) / 32 + 2;
    for (int64_t w = tid; w < cap; w += kSegLanes) scr[w] = 0u;
    const int64_t nseg = (n + kSegSyms - 1) / kSegSyms;
    int64_t done = 0;   // bits of the segments behind the current ones
    for (int64_t s1 = nseg; s1 > 0; s1 -= kSegLanes) {
        const int64_t s0 = s1 > kSegLanes ? s1 - kSegLanes : 0;
        const int32_t* const tile_id = id + s0 * kSegSyms;
        const int tn = (int)((s1 * kSegSyms < n ? s1 * kSegSyms : n) - s0 * kSegSyms);   // the tile's symbols
        const int b = tid * kSegSyms, e = b + kSegSyms < tn ? b + kSegSyms : tn;
        uint32_t total = 0, x = kL;
        int capw = 0;
        if (b < tn) x = seg_state<16>(tile_id, freqs, cum, e, tn, s1 == nseg ? (uint32_t)kL : l.tile_end, kSegWindow);
        const uint64_t missing = __ballot(x == 0);
        l.state[tid] = x;
        if (lane == 0) l.missing[wave] = missing;
        if (__syncthreads_or(missing != 0 ? 1 : 0)) {
            if (wave == 0) walk_missing(tile_id, freqs, cum, tn, l);
            __syncthreads();
            x = l.state[tid];
        }
        if (b < tn) {
            total = seg_encode<16>(tile_id, freqs, cum, b, e, seg, tid, &capw, &x);
            if (tid == 0) *state_out = l.tile_end = x;   // the last tile leaves the stream's
        }
        // bits of the segments behind mine in this tile
        const uint32_t incl = wave_incl_scan(total);
        stores_done();     // the cleared words
        __syncthreads();   // and wsum of the tile before is read
        if (lane == 63) l.wsum[wave] = incl;
        __syncthreads();
        uint32_t upto = 0, tile = 0;
#pragma unroll
        for (int w = 0; w < kSegLanes / 64; w++) {
            const uint32_t v = l.wsum[w];
            upto += w < wave ? v : 0u;
            tile += v;
        }
        const int64_t behind = done + (int64_t)(tile - (upto + incl));
        seg_copy<true>(seg, tid, capw, total, cap * 32 - behind - total, scr);
        done += tile;
    }
    stores_done();
    __syncthreads();
    const int64_t nw = (done + 31) / 32, base = cap * 32 - done;   // scratch bit of the stream's first
    for (int64_t w = tid; w < nw; w += kSegLanes) {
        const int64_t sp = base + 32 * w, wi = sp >> 5;
        const int sh = (int)(sp & 31), take = (int)(done - 32 * w < 32 ? done - 32 * w : 32);
        uint64_t v = __hip_atomic_load(scr + wi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (sh + take > 32) v |= (uint64_t)__hip_atomic_load(scr + wi + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) << 32;
        v >>= sh;
        out[w] = take == 32 ? (uint32_t)v : (uint32_t)v & ((1u << take) - 1u);
    }
    if (tid == 0) {
        out[nw] = 0u;
        *nbits_out = done;
    }
}

__global__ __launch_bounds__(kSegLanes) void k_encode_streams(
        const int32_t* __restrict__ idx, const int64_t* __restrict__ sym_off, const int64_t* __restrict__ nsym,
        const int32_t* __restrict__ freqs, const int32_t* __restrict__ cum, const int64_t* __restrict__ tab_off,
        int64_t n_streams, uint32_t* __restrict__ scratch, uint32_t* __restrict__ words,
        const int64_t* __restrict__ word_off, int64_t* __restrict__ state_out, int64_t* __restrict__ nbits_out) {
    __shared__ uint32_t seg[kSegWords][kSegLanes];   // 80 KB: a lane's bits, right-aligned in its column
    __shared__ LongLds l;
    __shared__ int s_n[kSegLanes];   // lengths of the next streams, longer ones as kGroupSyms + 1
    const int tid = threadIdx.x;
    const int64_t stride = gridDim.x;
    for (int64_t r0 = blockIdx.x; r0 < n_streams; r0 += stride * kSegLanes) {
        const int64_t left = (n_streams - r0 + stride - 1) / stride;
        const int cnt = (int)(left < kSegLanes ? left : kSegLanes);
        const int64_t len = tid < cnt ? nsym[r0 + tid * stride] : 0;
        s_n[tid] = (int)(len < kGroupSyms + 1 ? len : kGroupSyms + 1);
        const bool longer = __syncthreads_or(len > kSegSyms ? 1 : 0) != 0;
        const bool any_long = longer && __syncthreads_or(len > kGroupSyms ? 1 : 0) != 0;
        for (int lw = 0; lw <= (longer ? 6 : 0); lw += 2) {   // groups of 1 << lw lanes
            const int W = 1 << lw, gl = tid & (W - 1);
            for (int i0 = 0; i0 < cnt; i0 += kSegLanes >> lw) {
                const int i = i0 + (tid >> lw);
                const int n = i < cnt ? s_n[i] : -1;
                const bool act = n <= W * kSegSyms && n > (lw ? W / 4 * kSegSyms : -1);
                if (!__any(act)) continue;
                const int64_t t = act ? r0 + i * stride : 0;
                uint32_t* const out = words + word_off[t];
                uint32_t total = 0, x = kL;
                int capw = 0;
                const int b = gl * kSegSyms, e = b + kSegSyms < n ? b + kSegSyms : n;
                if (act && b < n) {
                    const int32_t *id = idx + sym_off[t], *F = freqs + tab_off[t], *C = cum + tab_off[t];
                    x = seg_state<8>(id, F, C, e, n, kL, 4 * kGroupSyms);   // its windows reach the end
                    total = seg_encode<8>(id, F, C, b, e, seg, tid, &capw, &x);
                }
                uint32_t incl = total;   // scan over the group; every lane of the wave is here
                for (int o = 1; o < W; o <<= 1) {
                    const uint32_t u = (uint32_t)__shfl_up((int)incl, o, 64);
                    incl += gl >= o ? u : 0u;
                }
                const uint32_t bits = (uint32_t)__shfl((int)incl, tid | (W - 1), 64);
                const uint32_t nw = (bits + 31u) / 32u;
                if (lw == 0) {
                    if (act) out[nw] = 0u;
                    seg_copy<false>(seg, tid, capw, total, 0, out);
                } else {
                    if (act)
                        for (uint32_t w = gl; w <= nw; w += W) out[w] = 0u;
                    stores_done();
                    seg_copy<true>(seg, tid, capw, total, incl - total, out);
                }
                if (act && gl == 0) {
                    state_out[t] = x;
                    nbits_out[t] = bits;
                }
            }
        }
        for (int i = 0; any_long && i < cnt; i++) {   // uniform
            if (s_n[i] <= kGroupSyms) continue;
            const int64_t t = r0 + i * stride;
            encode_long(idx + sym_off[t], freqs + tab_off[t], cum + tab_off[t], nsym[t], scratch + word_off[t],
                        words + word_off[t], state_out + t, nbits_out + t, seg, l);
        }
        __syncthreads();   // s_n is written again
    }
}

// _rans_decode_kernel semantics (core/gpu_ans.py:175-235), a workgroup per stream
// or, for short ones, a lane (lq_rans_decode_streams): renormalisation reads min(needed, n_bits - bit_pos) bits.
//
// A stream is one serial chain (every step needs the state before it), so the
// kernel is arranged around that chain's latency: tables in LDS, bits in a
// register buffer refilled from words the wave holds one per lane, the chain
// computed by all lanes alike, and everything else (symbol values, stores)
// done by 64 lanes at once from the trace of 64 steps.  A step takes one LDS
// read and a few shifts.  PAIR: the table is indexed by the slot and the next
// kAhead stream bits, and a step covers two symbols whenever the first one's
// renormalisation needs no more than those bits; it fills a CU's LDS, so it is
// taken for up to two streams per CU, and the one-symbol table (many
// workgroups per CU) beyond.  One lane per stream with the tables in global
// memory, bit by bit, took 30771 us for 16 streams of 32768 symbols,
// the chain alone 1434 us.
// The chain's tables hold for states in [L, 2L) and tables whose steps stay
// there; anything else, and the stream's last bits, take plain_steps.
//
// Long streams are first decoded in parallel.  A state holds ten bits, of which
// each step replaces some by stream bits, so decoders that start at different
// (bit, state) places of one stream mostly end in the same chain after some
// hundred symbols (measured over rounded normals of 2 to 8 bits per symbol:
// median 200 to 850, the last of 2000 starts 300 to 7000).  A tile of the stream
// is cut into kSyncLanes segments of equal bits; a lane decodes its segment from
// a guessed place, then again from the place where the lane before it ended,
// until no lane's start changes: every start is then the end of the segment
// before, from the tile's known first place on, so the chain is the serial one,
// whatever the guesses were.  Lane j's start is right after j rounds at the
// latest; lanes whose start did not change rest.  Streams that do not fall into
// step (kSyncRounds, and half the lanes by round kSyncLook: four equally likely
// symbols, for one, keep odd and even bits apart) keep the segments that are
// proven and go on serially.  The steps are those of the longest way into step
// instead of the whole stream's: 16 streams of 32768 symbols of 4 to 5 bits
// 1434 -> 239 us, of 12000 symbols 549 -> 249 us, of 200000 8589 -> 1091 us.
constexpr int kAhead = 5;
constexpr int kWordRing = 256;   // stream words in LDS
constexpr int kSyncLanes = 256;
constexpr int kSyncRounds = 128;
constexpr int kSyncLook = 16;
// Taken where the way into step is short against the stream: from 8192 symbols
// on (4200 symbols of 4 bits: 218 us serially, 332 so), more with fewer bits per
// symbol, as the way grows with about the inverse square of these (streams of 2
// to 3 bits: 16384 symbols 657 us serially, 714 so, 32768 symbols 1260 and 630).
// Not for more streams than the two-symbol table is taken for, whose waves share
// the SIMDs (600 streams of 8192 symbols: 589 us serially, 706 so).
constexpr int kSyncMin = 8192;
__device__ __forceinline__ bool sync_pays(int64_t n, int64_t nb) {
    return n >= kSyncMin && nb >= kSyncMin && (double)nb * (double)nb >= 1.5e5 * (double)n;
}

struct StreamArgs {
    const uint32_t* words;
    const int32_t *bit_off, *nbits, *init, *ndec, *lookup, *freqs, *cum, *alphabet, *tid;
    int32_t max_sym;
    const int32_t* out_off;
    int64_t* out;

    __device__ __forceinline__ void tables(int64_t t, const int32_t** lu, const int32_t** f, const int32_t** c,
                                           const int32_t** al) const {
        const int64_t tb = tid[t];
        *lu = lookup + tb * kL;
        *f = freqs + tb * max_sym;
        *c = cum + tb * max_sym;
        *al = alphabet + tb * max_sym;
    }
};

// The reference's step, from symbol i and state x with pos of the nb bits read
__device__ __forceinline__ void plain_steps(int n, int i, uint32_t x, int64_t boff, int64_t nb, int64_t pos,
                                            const uint32_t* __restrict__ wb, const int32_t* __restrict__ LU,
                                            const int32_t* __restrict__ F, const int32_t* __restrict__ C,
                                            const int32_t* __restrict__ A, int64_t* __restrict__ o, bool store) {
    for (; i < n; i++) {
        const uint32_t slot = x & (kL - 1);
        const int si = LU[slot];
        if (store) o[i] = A[si];
        x = (uint32_t)F[si] * (x >> 10) + slot - (uint32_t)C[si];
        if (x < (uint32_t)kL) {
            int64_t k = (int64_t)__clz((int)x) - 21;
            if (k > nb - pos) k = nb - pos;
            for (int64_t q = 0; q < k; q++) {
                const int64_t ab = boff + pos + q;
                x = (x << 1) | ((wb[ab >> 5] >> (ab & 31)) & 1u);
            }
            pos += k;
        }
    }
}

// The two-symbol table takes about 17 us to build and saves 0.04 us per symbol:
// 140 symbols 36 us without and 50 with it, 400 54 and 62, 600 68 and 64 to 74,
// 800 81 and 72, 4000 288 and 197.
constexpr int kPairMin = 600;

constexpr int kTileWords = 8191;   // words of a tile of the parallel decode
template <bool PAIR>
struct DecodeLds {
    // one[slot]: k | symbol index << 6 | next slot before the k bits << 16
    uint32_t one[kL];
    // two[slot << kAhead | next bits]: k1 | (64 - kAhead - k2) << 6 | next slot << 22, the
    // pair's first shift and second read; k1 = 0 and the first symbol's own k and slot
    // where it needs more than kAhead bits
    // (before that table is built: a tile's words)
    uint32_t two[PAIR ? kL << kAhead : 1];
    uint32_t ring[kWordRing];
    int32_t alph[PAIR ? kL : 1];   // the symbols' values
    uint32_t end[PAIR ? kSyncLanes : 1];
    int sum[kSyncLanes / 64], first;
    int bad;
};

// One stream, by the whole workgroup.
template <bool PAIR, int NT>
__device__ __forceinline__ void decode_stream(const uint32_t* __restrict__ wb, int64_t boff, int64_t nb, uint32_t x,
                                              const int n, const int32_t* __restrict__ LU, const int32_t* __restrict__ F,
                                              const int32_t* __restrict__ C, const int32_t* __restrict__ A,
                                              const int max_sym, int64_t* __restrict__ o, DecodeLds<PAIR>& l) {
    constexpr int64_t kTileBits = (kTileWords - 1) * 32;   // a step reads a word and the one behind it
    static_assert(kTileBits + 10 < 1 << 18, "segment ends pack a bit position and a slot into 28 bits");
    const int tid = threadIdx.x, lane = tid & 63;
    auto& one = l.one;
    auto& two = l.two;
    auto& ring = l.ring;
    auto& alph = l.alph;
    if (tid == 0) l.bad = x < (uint32_t)kL || x >= 2u * kL ? 1 : 0;
    __syncthreads();
    for (int slot = tid; slot < kL; slot += NT) {
        const int si = LU[slot];
        int64_t xp = 0;
        if (si >= 0 && si < max_sym && si < kL) xp = (int64_t)F[si] + slot - C[si];
        if (xp < 1 || xp >= 2 * kL) {
            l.bad = 1;
            one[slot] = 0u;
        } else {
            const uint32_t k = xp >= kL ? 0u : (uint32_t)(__clz((int)xp) - 21);
            one[slot] = k | ((uint32_t)si << 6) | ((((uint32_t)xp << k) - (uint32_t)kL) << 16);
        }
    }
    __syncthreads();
    int i = 0;   // symbols done
    bool pairs = false;
    const bool chain = !l.bad && nb > 0;
    if constexpr (PAIR) {
        if (chain && sync_pays(n, nb)) {   // (before the barrier behind the tile's words)
            for (int j = tid; j < kL && j < max_sym; j += kSyncLanes) alph[j] = A[j];
        }
        while (chain && sync_pays(n - i, nb)) {   // uniform
            // equal tiles of the bits that the symbols may take
            const int64_t left = nb < 10 * (int64_t)(n - i) ? nb : 10 * (int64_t)(n - i);
            const int64_t tiles = (left + kTileBits - 64) / (kTileBits - 63);
            const int p0 = (int)(boff & 31);
            // a step starts below `end`: within the tile, with its 10 bits there
            const int64_t lastp = p0 + nb - 9;
            const int64_t tend = p0 + (left + tiles - 1) / tiles;
            const int end = (int)(tend < lastp ? tend : lastp);
            const int seg = (end - p0 + kSyncLanes - 1) / kSyncLanes, cap = 4 * seg + 64;
            const int64_t first = boff >> 5, lastw = (boff + nb - 1) >> 5;
            for (int w = tid; w < (end >> 5) + 2; w += kSyncLanes)   // at most kTileWords
                two[w] = wb[first + w < lastw ? first + w : lastw];
            __syncthreads();
            const int e0 = p0 + (tid + 1) * seg, stop = e0 < end ? e0 : end;
            // a segment: the steps from (p, sl) that start before `stop` (at most cap:
            // steps may read no bits); sym: the symbol index of each
            auto walk = [&](int p, uint32_t sl, int* count, auto sym) -> uint32_t {
                int c = 0;
                auto step = [&](int j) {
                    const uint32_t e = one[sl], k = e & 63u, *w = two + (p >> 5);
                    const uint32_t v = __builtin_bitreverse32(__builtin_amdgcn_alignbit(w[1], w[0], (uint32_t)p));
                    sl = (e >> 16) + (v >> 1 >> (31u - k));
                    p += (int)k;
                    sym(c + j, (e >> 6) & 1023u);
                };
                // four at a time without a test between them while they must start below
                for (; p <= stop - 31 && c < cap; c += 4) {
#pragma unroll
                    for (int j = 0; j < 4; j++) step(j);
                }
                for (; p < stop && c < cap; c++) step(0);
                *count = c;
                return (uint32_t)p << 10 | sl;
            };
            uint32_t from = (uint32_t)(p0 + tid * seg < end ? p0 + tid * seg : end) << 10;
            if (tid == 0) from |= x - (uint32_t)kL;
            bool changed = true;
            int count = 0, rounds = 0;
            uint32_t to = 0;
            for (;;) {
                if (changed) to = walk((int)(from >> 10), from & 1023u, &count, [](int, uint32_t) {});
                l.end[tid] = to;
                if (tid == 0) l.first = kSyncLanes;
                __syncthreads();
                const uint32_t f = tid ? l.end[tid - 1] : from;
                changed = f != from;
                rounds++;
                const bool look = rounds == kSyncLook;   // (the count takes longer than the test)
                const int apart = look ? __syncthreads_count(changed ? 1 : 0) : __syncthreads_or(changed ? 1 : 0);
                if (!apart || rounds == kSyncRounds || (look && apart > kSyncLanes / 2)) break;
                from = f;
            }
            // the lanes before the first whose start would change: their segments are the chain's
            if (changed) atomicMin(&l.first, tid);
            __syncthreads();
            const int good = l.first;   // at least `rounds` of them
            const bool mine = tid < good;
            const uint32_t sum = wave_incl_scan(mine ? (uint32_t)count : 0u);
            if (lane == 63) l.sum[tid >> 6] = (int)sum;
            __syncthreads();
            int before = 0, total = 0;
            for (int w = 0; w < kSyncLanes / 64; w++) {
                if (w < (tid >> 6)) before += l.sum[w];
                total += l.sum[w];
            }
            if (mine && count > 0) {
                const int at = before + (int)sum - count, room = n - i - at;
                int64_t* q = o + i + at;
                int c2;
                walk((int)(from >> 10), from & 1023u, &c2, [&](int c, uint32_t si) {
                    if (c < room) q[c] = alph[si];
                });
            }
            const uint32_t done = l.end[good - 1];
            const int read = (int)(done >> 10) - p0;
            i = total < n - i ? i + total : n;
            boff += read;
            nb -= read;
            x = (uint32_t)kL + (done & 1023u);
            __syncthreads();   // the tile and s_end are written again
            if (good < kSyncLanes) break;
        }
        pairs = n - i >= kPairMin;   // uniform
        if (pairs) {
            for (int j = tid; j < kL << kAhead; j += 256) {
                uint32_t e = one[j >> kAhead], ks = 0u;
                const uint32_t k1 = e & 63u;
                if (k1 <= (uint32_t)kAhead) {
                    ks = k1;
                    e = one[(e >> 16) + ((uint32_t)(j & ((1 << kAhead) - 1)) >> (kAhead - k1))];
                }
                two[j] = ks | ((uint32_t)(64 - kAhead) - (e & 63u)) << 6 | (e >> 16) << 22;
            }
        }
        __syncthreads();
    }
    if (tid >= 64) return;   // the first wave decodes

    int64_t pos = 0;   // bits read
    if (chain && nb > 0 && i < n) {
        // Words from the one holding the stream's first bit (past the stream's
        // last: its last) reach the chain through a ring in LDS, topped up with
        // 64 of them per batch (load at its start, store at its end), and, within
        // a batch, a register: lane l holds the batch's l-th word, read by
        // readlane.  A batch takes at most 31 of them.
        const int64_t first = boff >> 5, lastw = (boff + nb - 1) >> 5;
        auto load = [&](int64_t w) { return wb[first + w < lastw ? first + w : lastw]; };
        ring[lane] = load(lane);
        ring[64 + lane] = load(64 + lane);
        int64_t cur = 0, filled = 128;   // words taken before this batch, words in the ring
        int r = 0;                       // words taken in this batch
        uint32_t w = 0, q = 0;
        bool more = false;
        auto open = [&]() {
            more = filled - cur < 128;   // at least 64 left
            if (more) q = load(filled + lane);
            w = ring[(cur + lane) & (kWordRing - 1)];
        };
        auto close = [&]() {
            cur += r;
            r = 0;
            if (more) {
                ring[(filled + lane) & (kWordRing - 1)] = q;
                filled += 64;
            }
        };
        BitBuf bb;
        auto refill = [&]() {   // at least 32 bits in the buffer
            if (__builtin_amdgcn_readfirstlane((int)(uint32_t)bb.buf) == 0)
                bb.push((uint32_t)__builtin_amdgcn_readlane((int)w, r++));
        };
        auto bits_read = [&]() -> int64_t {   // words taken, less the buffered bits
            return (cur + r) * 32 - (boff & 31) - (63 - __builtin_ctzll(bb.buf));
        };
        // 0, but not known to be alike in all lanes: a lookup at + zero stays in a
        // vector register until its readfirstlane (a lookup the compiler knows to
        // be uniform is read to a scalar, and waited for, at once)
        uint32_t zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        open();
        bb.init((uint32_t)__builtin_amdgcn_readlane((int)w, r++), (uint32_t)(boff & 31));
        refill();
        close();
        uint32_t slot = x - (uint32_t)kL;
        if constexpr (PAIR) {
            uint32_t ix = (slot << kAhead) | (uint32_t)(bb.buf >> (64 - kAhead));
            // 64 steps read at most 15 bits and decode at most two symbols each
            while (pairs && n - i >= 128 && nb - bits_read() >= 64 * 15 + 64) {
                open();
                uint32_t trace = 0, e = two[ix];
#pragma unroll 8
                for (int j = 0; j < 64; j++) {
                    const uint64_t v = bb.buf << (e & 63u);
                    const uint32_t rs = (e >> 6) & 63u, now = ix;
                    ix = (uint32_t)(v >> rs) + (e >> 17);
                    const uint32_t ev = two[ix + zero];   // in flight while the buffer is seen to
                    __builtin_amdgcn_sched_barrier(0);
                    trace = lane == j ? now : trace;
                    bb.buf = v << ((uint32_t)(64 - kAhead) - rs);
                    refill();
                    e = (uint32_t)__builtin_amdgcn_readfirstlane((int)ev);
                }
                close();
                const uint32_t e1 = one[trace >> kAhead], k1 = e1 & 63u;
                const bool both = k1 <= (uint32_t)kAhead;
                const uint32_t incl = wave_incl_scan(both ? 2u : 1u);
                int64_t* p = o + i + (incl - (both ? 2u : 1u));
                p[0] = A[(e1 >> 6) & 1023u];
                if (both) {
                    const uint32_t e2 = one[(e1 >> 16) + ((trace & ((1u << kAhead) - 1u)) >> (kAhead - k1))];
                    p[1] = A[(e2 >> 6) & 1023u];
                }
                i += __builtin_amdgcn_readlane((int)incl, 63);
            }
            slot = ix >> kAhead;
        }
        // one symbol per step, while a step's 10 bits are there: 64 at a time,
        // then one by one
        while (n - i >= 64 && nb - bits_read() >= 64 * 10) {
            open();
            uint32_t trace = 0, e = one[slot];
#pragma unroll 8
            for (int j = 0; j < 64; j++) {
                const uint32_t now = e;
                slot = (e >> 16) + (uint32_t)(((uint64_t)(uint32_t)(bb.buf >> 32) << (e & 63u)) >> 32);
                const uint32_t ev = one[slot + zero];
                __builtin_amdgcn_sched_barrier(0);
                trace = lane == j ? now : trace;
                bb.buf <<= (now & 63u);
                refill();
                e = (uint32_t)__builtin_amdgcn_readfirstlane((int)ev);
            }
            close();
            o[i + lane] = A[(trace >> 6) & 1023u];
            i += 64;
        }
        while (i < n && nb - bits_read() >= 10) {
            open();
            for (int j = 0; j < 64 && i < n && nb - bits_read() >= 10; j++, i++) {
                const uint32_t e = one[slot];
                if (lane == 0) o[i] = A[(e >> 6) & 1023u];
                slot = (e >> 16) + bb.take(e);
                refill();
            }
            close();
        }
        pos = bits_read();
        x = slot + (uint32_t)kL;
    }
    plain_steps(n, i, x, boff, nb, pos, wb, LU, F, C, A, o, lane == 0);
}

// Streams of at most lanes_below symbols are taken by a lane each, in the first
// lane_blocks workgroups: these do nothing else (PAIR: and then, as the others do,
// a stream of their own).  The others take the rest, one after the other.
template <bool PAIR, int NT>
__global__ __launch_bounds__(NT) void k_decode_streams(StreamArgs a, int64_t n_streams, int lanes_below, int lane_blocks) {
    __shared__ DecodeLds<PAIR> l;
    if ((int)blockIdx.x < lane_blocks) {
        // PAIR: one or two streams per workgroup, so that no CU waits for another
        const int64_t t = PAIR ? blockIdx.x + (int64_t)threadIdx.x * lane_blocks : (int64_t)blockIdx.x * NT + threadIdx.x;
        if (t < n_streams && a.ndec[t] <= lanes_below) {
            const int32_t *LU, *F, *C, *A;
            a.tables(t, &LU, &F, &C, &A);
            plain_steps(a.ndec[t], 0, (uint32_t)a.init[t], a.bit_off[t], a.nbits[t], 0, a.words, LU, F, C, A,
                        a.out + a.out_off[t], true);
        }
        if (!PAIR) return;
    }
    const int64_t first = PAIR ? blockIdx.x : (int64_t)blockIdx.x - lane_blocks;
    const int64_t stride = PAIR ? gridDim.x : (int64_t)gridDim.x - lane_blocks;
    for (int64_t t = first; t < n_streams; t += stride) {
        const int n = a.ndec[t];
        if (n <= lanes_below) continue;   // uniform
        const int32_t *LU, *F, *C, *A;
        a.tables(t, &LU, &F, &C, &A);
        decode_stream<PAIR, NT>(a.words, a.bit_off[t], a.nbits[t], (uint32_t)a.init[t], n, LU, F, C, A, a.max_sym,
                                a.out + a.out_off[t], l);
        __syncthreads();   // l is written again
    }
}

template <typename SymT>
int encode_launch(const SymT* d_sym, const uint32_t* d_blk_n1, int64_t n_chunks, int64_t n_vectors,
                  const lq_table* d_tables, void* d_work, uint32_t* d_blk_off, uint16_t* d_blk_state,
                  int64_t* d_stream_nbits, int32_t* d_stream_state, int64_t* d_stream_woff, int64_t* d_chunk_words,
                  int64_t* d_chunk_base, uint32_t* d_counter, int64_t* h_total, hipStream_t s) {
    if (n_chunks <= 0 || n_vectors <= 0) return LQ_ERR_ARG;
    const int64_t nblk = (n_vectors + kBlk - 1) / kBlk;
    EncWork w = enc_layout(n_chunks, n_vectors);
    uint32_t* bits = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(d_work) + w.bits);
    uint32_t* scratch = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(d_work) + w.scratch);
    const int64_t groups = (nblk + kEncBlocks - 1) / kEncBlocks;
    hipLaunchKernelGGL((k_chunk_encode<SymT>), dim3((unsigned)groups, (unsigned)n_chunks), dim3(256), 0, s, d_sym,
                       d_blk_n1, nblk, n_vectors, d_tables, bits, scratch, d_blk_state);
    if (nblk > kScanTile) {
        const int64_t tiles = (nblk + kScanTile - 1) / kScanTile;
        uint64_t* tsum = reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(d_work) + w.tiles);
        const dim3 tg((unsigned)(tiles * n_chunks * LQ_STREAMS));   // (stream, tile) = divmod(block, tiles)
        hipLaunchKernelGGL(k_scan_tiles, tg, dim3(256), 0, s, bits, nblk, tiles, tsum);
        hipLaunchKernelGGL(k_scan_top, dim3((unsigned)(n_chunks * LQ_STREAMS)), dim3(256), 0, s, tsum, tiles, d_blk_state,
                           nblk, d_tables, d_stream_nbits, d_stream_state);
        hipLaunchKernelGGL(k_scan_apply, tg, dim3(256), 0, s, bits, nblk, tiles, tsum, d_blk_off);
        hipLaunchKernelGGL(k_chunk_offsets, dim3(1), dim3(256), 0, s, d_stream_nbits, d_tables, n_chunks, d_stream_woff,
                           d_chunk_words, d_chunk_base, h_total);
    } else {
        const bool bases = d_chunk_base && n_chunks <= kBasesInScan;
        hipLaunchKernelGGL(k_chunk_scan_offsets, dim3((unsigned)n_chunks), dim3(64 * LQ_STREAMS), 0, s, bits,
                           d_blk_state, d_tables, nblk, d_blk_off, d_stream_nbits, d_stream_state, d_stream_woff,
                           d_chunk_words, bases ? d_chunk_base : nullptr, d_counter, h_total);
        if (d_chunk_base && !bases)
            hipLaunchKernelGGL(k_chunk_bases, dim3(1), dim3(1024), 0, s, d_chunk_words, n_chunks, d_chunk_base, h_total);
    }
    return launch_status();
}

int tables_launch(const uint32_t* d_hist, int64_t n_chunks, lq_table* d_tables, int32_t* d_status, int skip,
                  int64_t* h_status, hipStream_t s) {
    if (n_chunks <= 0) return LQ_ERR_ARG;
    const int64_t ns = n_chunks * LQ_STREAMS;
    hipLaunchKernelGGL(k_chunk_tables_wave, dim3((unsigned)((ns + kTabWaves - 1) / kTabWaves)), dim3(64 * kTabWaves), 0,
                       s, d_hist, ns, d_tables, d_status, skip, h_status);
    return launch_status();
}

ReadPool& read_pool() {
    static ReadPool p;   // trivially destroyed: the HIP runtime may be gone by then
    return p;
}

struct WriteWork {   // offsets into lq_encode_chunks' workspace
    int64_t fastdiv, sums, counter, sym, enc, total;
};

inline WriteWork write_layout(int64_t n_chunks, int64_t n_heads, int64_t bph) {
    auto al = [](int64_t b) { return (b + 255) / 256 * 256; };
    const int64_t H = n_chunks * n_heads, V = n_heads * bph, nblk = (V + kBlk - 1) / kBlk;
    WriteWork w;
    w.fastdiv = 0;   // first, and enc last: a batch that overflows hands both on
    w.sums = w.fastdiv + al(H * 4);
    w.counter = w.sums + al((4096 + H) * 8);
    w.sym = w.counter + 256;
    w.enc = w.sym + al(n_chunks * nblk * kSymStride);
    w.total = w.enc + enc_layout(n_chunks, V).total;
    return w;
}

}  // namespace

extern "C" {

int64_t lq_encode_chunks_workspace(int64_t n_chunks, int64_t n_heads, int64_t bph) {
    if (n_chunks <= 0 || n_heads <= 0 || bph <= 0) return -1;
    return write_layout(n_chunks, n_heads, bph).total;
}

int lq_encode_chunks(const void* d_x, int dtype, int64_t n_chunks, int64_t n_heads, int64_t bph, int head_dim,
                     const float* d_signs, const int64_t* d_dither_seed, const int32_t* d_chunk_bits, int scales_given,
                     float* d_sigma2, float* d_scale32, uint16_t* d_scale16, uint8_t* d_coset_bits, uint32_t* d_blk_n1,
                     void* d_deq, uint32_t* d_hist, int32_t* d_status, lq_table* d_tables, uint32_t* d_blk_off,
                     uint16_t* d_blk_state, int64_t* d_stream_nbits, int32_t* d_stream_state, int64_t* d_stream_woff,
                     int64_t* d_chunk_words, int64_t* d_chunk_base, uint32_t* d_words, int skip_overflowed, void* d_work,
                     int64_t* h_status, int64_t* h_words, hipStream_t s) {
    if (n_chunks <= 0 || n_heads <= 0 || bph <= 0 || !d_work || !d_status || !d_hist || !d_scale32 || !d_scale16 ||
        !d_chunk_base || (d_signs && d_deq))
        return LQ_ERR_ARG;
    const int64_t H = n_chunks * n_heads, V = n_heads * bph;
    const WriteWork w = write_layout(n_chunks, n_heads, bph);
    char* const base = static_cast<char*>(d_work);
    int32_t* const fastdiv = reinterpret_cast<int32_t*>(base + w.fastdiv);
    uint32_t* const counter = reinterpret_cast<uint32_t*>(base + w.counter);
    int8_t* const sym = reinterpret_cast<int8_t*>(base + w.sym);
    Clear clear;
    clear.hist = d_hist;
    clear.n_hist = n_chunks * LQ_STREAMS * 256;
    clear.status = d_status;
    clear.n_status = n_chunks;
    clear.counter = counter;
    const bool reads = h_status || h_words;
    ReadSlot slot;
    if (reads && !read_pool().take(s, &slot)) return LQ_ERR_LAUNCH;
    auto run = [&]() -> int {
        int rc = scales_given
                     ? scale_fastdiv_launch(d_scale32, H, d_signs ? (int)LQ_F32 : dtype, fastdiv, d_scale16, clear, s)
                     : head_scales_launch(d_x, dtype, n_chunks, n_heads, bph, head_dim, d_signs, d_chunk_bits,
                                          reinterpret_cast<double*>(base + w.sums), d_sigma2, d_scale32, d_scale16, fastdiv,
                                          clear, s);
        if (rc != LQ_OK) return rc;
        rc = d_signs ? lq_chunk_quantize_rht(d_x, dtype, n_chunks, n_heads, bph, head_dim, d_signs, d_scale32, sym,
                                             d_coset_bits, d_blk_n1, d_hist, d_status, d_dither_seed, s)
                     : lq_chunk_quantize(d_x, dtype, n_chunks, n_heads, bph, d_scale32, fastdiv, sym, d_coset_bits,
                                         d_blk_n1, d_hist, d_status, d_deq, dtype, d_dither_seed, s);
        if (rc != LQ_OK) return rc;
        rc = tables_launch(d_hist, n_chunks, d_tables, d_status, skip_overflowed, reads ? slot.host : nullptr, s);
        if (rc != LQ_OK) return rc;
        if (reads && !h_words && hipEventRecord(slot.event, s) != hipSuccess) return LQ_ERR_LAUNCH;
        rc = encode_launch(sym, d_blk_n1, n_chunks, V, d_tables, base + w.enc, d_blk_off, d_blk_state, d_stream_nbits,
                           d_stream_state, d_stream_woff, d_chunk_words, d_chunk_base, counter,
                           h_words ? slot.host + 1 : nullptr, s);
        if (rc != LQ_OK) return rc;
        if (h_words && hipEventRecord(slot.event, s) != hipSuccess) return LQ_ERR_LAUNCH;
        if (d_words)
            rc = lq_chunk_pack(n_chunks, V, d_tables, base + w.enc, d_blk_off, d_stream_nbits, d_stream_woff, d_chunk_base,
                               d_words, s);
        if (rc != LQ_OK || !reads) return rc;
        // The launches behind the event go on while the caller reads on.  (Those of
        // a batch whose streams were left empty run while its caller makes the wide
        // path's arrays: leaving them out, by a wait before the scan, gave such a
        // batch 0 to 10 us of 430 and cost every other small write 5 to 8 of 115.)
        if (hipEventSynchronize(slot.event) != hipSuccess) return LQ_ERR_LAUNCH;
        if (h_status) *h_status = slot.host[0];
        if (h_words) *h_words = slot.host[1];
        return LQ_OK;
    };
    const int rc = run();
    if (reads) {
        if (rc != LQ_OK) (void)hipStreamSynchronize(s);   // no launch may still write the slot
        read_pool().give(slot);
    }
    return rc;
}

int lq_encode_chunks_pack(int64_t n_chunks, int64_t n_heads, int64_t bph, const lq_table* d_tables, const void* d_work,
                          const uint32_t* d_blk_off, const int64_t* d_stream_nbits, const int64_t* d_stream_woff,
                          const int64_t* d_chunk_base, uint32_t* d_words, hipStream_t s) {
    if (n_chunks <= 0 || n_heads <= 0 || bph <= 0 || !d_work || !d_words) return LQ_ERR_ARG;
    const WriteWork w = write_layout(n_chunks, n_heads, bph);
    return lq_chunk_pack(n_chunks, n_heads * bph, d_tables, static_cast<const char*>(d_work) + w.enc, d_blk_off,
                         d_stream_nbits, d_stream_woff, d_chunk_base, d_words, s);
}

int lq_chunk_tables(const uint32_t* d_hist, int64_t n_chunks, lq_table* d_tables, int32_t* d_status, hipStream_t s) {
    return tables_launch(d_hist, n_chunks, d_tables, d_status, 0, nullptr, s);
}

int64_t lq_chunk_encode_workspace(int64_t n_chunks, int64_t n_vectors) {
    if (n_chunks <= 0 || n_vectors <= 0) return -1;
    return enc_layout(n_chunks, n_vectors).total;
}

int lq_chunk_encode(const int8_t* d_sym, const uint32_t* d_blk_n1, int64_t n_chunks, int64_t n_vectors,
                    const lq_table* d_tables, void* d_work, uint32_t* d_blk_off, uint16_t* d_blk_state,
                    int64_t* d_stream_nbits, int32_t* d_stream_state, int64_t* d_stream_woff, int64_t* d_chunk_words,
                    hipStream_t s) {
    return encode_launch(d_sym, d_blk_n1, n_chunks, n_vectors, d_tables, d_work, d_blk_off, d_blk_state, d_stream_nbits,
                         d_stream_state, d_stream_woff, d_chunk_words, nullptr, nullptr, nullptr, s);
}

int lq_chunk_encode_wide(const int16_t* d_sym, const uint32_t* d_blk_n1, int64_t n_chunks, int64_t n_vectors,
                         const lq_table* d_tables, void* d_work, uint32_t* d_blk_off, uint16_t* d_blk_state,
                         int64_t* d_stream_nbits, int32_t* d_stream_state, int64_t* d_stream_woff, int64_t* d_chunk_words,
                         hipStream_t s) {
    return encode_launch(d_sym, d_blk_n1, n_chunks, n_vectors, d_tables, d_work, d_blk_off, d_blk_state, d_stream_nbits,
                         d_stream_state, d_stream_woff, d_chunk_words, nullptr, nullptr, nullptr, s);
}

int lq_chunk_tables_wide(const uint32_t* d_hist, const int32_t* d_minmax, int64_t n_chunks, lq_table* d_tables,
                         int32_t* d_status, hipStream_t s) {
    if (n_chunks <= 0 || !d_hist || !d_minmax) return LQ_ERR_ARG;
    hipLaunchKernelGGL((k_chunk_tables<true>), dim3((unsigned)(n_chunks * LQ_STREAMS)), dim3(256), 0, s, d_hist, d_minmax,
                       d_tables, d_status);
    return launch_status();
}

int lq_chunk_pack(int64_t n_chunks, int64_t n_vectors, const lq_table* d_tables, const void* d_work,
                  const uint32_t* d_blk_off, const int64_t* d_stream_nbits, const int64_t* d_stream_woff,
                  const int64_t* d_chunk_base, uint32_t* d_words, hipStream_t s) {
    if (n_chunks <= 0 || n_vectors <= 0) return LQ_ERR_ARG;
    const int64_t nblk = (n_vectors + kBlk - 1) / kBlk;
    EncWork w = enc_layout(n_chunks, n_vectors);
    const uint32_t* scratch = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(d_work) + w.scratch);
    const int64_t ns_total = n_chunks * LQ_STREAMS;
    const int64_t jobs = ns_total * ((nblk + kPackBlocks - 1) / kPackBlocks);
    hipLaunchKernelGGL(k_chunk_pack, dim3((unsigned)((jobs + 3) / 4)), dim3(256), 0, s, ns_total, nblk, scratch,
                       d_blk_off, d_stream_nbits, d_stream_woff, d_chunk_base, d_tables, d_words);
    return launch_status();
}

static int chunk_decode_launch(const uint32_t* d_words, const int64_t* d_chunk_base, const int64_t* d_stream_woff,
                               const uint32_t* d_blk_off, const int64_t* d_stream_nbits, const uint16_t* d_blk_state,
                               const uint8_t* d_coset_bits, const lq_table* d_tables, const uint16_t* d_scale16,
                               int64_t n_chunks, int64_t n_heads, int64_t bph, uint32_t* d_lut_work, void* d_out,
                               int out_dtype, const int64_t* d_dither_seed, int head_dim, const float* d_signs,
                               const int32_t* d_esc_k, const int64_t* d_fine_off, const uint32_t* d_fine,
                               hipStream_t s) {
    if (n_chunks <= 0 || n_heads <= 0 || bph <= 0 || out_dtype < 0 || out_dtype > 2) return LQ_ERR_ARG;
    if (d_esc_k && (!d_fine_off || !d_fine)) return LQ_ERR_ARG;
    const int64_t V = n_heads * bph;
    const int64_t nblk = (V + kBlk - 1) / kBlk;
    (void)d_lut_work;   // the decoder builds its LUTs in LDS
    // One workgroup per CU, whose waves share its tasks: up to 1024 tasks (4096
    // blocks) each has a SIMD to itself.  With 64 blocks per workgroup whatever
    // the size, and the LUTs from a launch of their own, 512 blocks (a chunk of
    // 2048 tokens) took 65.2 us, 8192 blocks 72.3 and 131072 blocks 525; now
    // 39.4, 49.0 and 493.
    const DecodeSplit cut = decode_split(n_chunks, (nblk + 3) / 4, device_cus());
    const dim3 grid((unsigned)cut.grid);
    const bool aligned = bph % kBlk == 0;
    const int lpr = d_signs ? head_dim / 8 : 1;
    const float div = d_signs ? (float)sqrt((double)head_dim) : 1.0f;
    // escaped chunks get their own instantiations (the escape constants would
    // otherwise cost registers in every decoder)
#define LQ_DECODE_E(DT, AL, DI, RO, ES)                                                                           \
    hipLaunchKernelGGL((k_chunk_decode<DT, AL, DI, RO, ES>), grid, dim3(kDecThreads), 0, s, d_words, d_chunk_base,      \
                       d_stream_woff, d_blk_off, d_stream_nbits, d_blk_state, d_coset_bits, d_tables, d_scale16,       \
                       n_chunks, n_heads, bph, nblk, cut.span, cut.tpw, cut.wpc, d_out, d_dither_seed, d_signs, lpr, div, \
                       d_esc_k, d_fine_off, d_fine)
#define LQ_DECODE(DT, AL, DI, RO)                                                                                 \
    do {                                                                                                          \
        if (d_esc_k) LQ_DECODE_E(DT, AL, DI, RO, true); else LQ_DECODE_E(DT, AL, DI, RO, false);                  \
    } while (0)
#define LQ_DECODE_DT(DT, RO)                                                                                      \
    do {                                                                                                          \
        if (d_dither_seed) { if (aligned) LQ_DECODE(DT, true, true, RO); else LQ_DECODE(DT, false, true, RO); }   \
        else { if (aligned) LQ_DECODE(DT, true, false, RO); else LQ_DECODE(DT, false, false, RO); }               \
    } while (0)
    if (d_signs) {
        if (out_dtype == LQ_F16) LQ_DECODE_DT(LQ_F16, true);
        else if (out_dtype == LQ_BF16) LQ_DECODE_DT(LQ_BF16, true);
        else LQ_DECODE_DT(LQ_F32, true);
    } else {
        if (out_dtype == LQ_F16) LQ_DECODE_DT(LQ_F16, false);
        else if (out_dtype == LQ_BF16) LQ_DECODE_DT(LQ_BF16, false);
        else LQ_DECODE_DT(LQ_F32, false);
    }
#undef LQ_DECODE_DT
#undef LQ_DECODE
#undef LQ_DECODE_E
    return launch_status();
}

int lq_chunk_decode(const uint32_t* d_words, const int64_t* d_chunk_base, const int64_t* d_stream_woff,
                    const uint32_t* d_blk_off, const int64_t* d_stream_nbits, const uint16_t* d_blk_state,
                    const uint8_t* d_coset_bits, const uint32_t* d_blk_n1, const lq_table* d_tables,
                    const uint16_t* d_scale16, int64_t n_chunks, int64_t n_heads, int64_t bph, uint32_t* d_lut_work,
                    void* d_out, int out_dtype, const int64_t* d_dither_seed, hipStream_t s) {
    (void)d_blk_n1;   // the decoder counts each block's coset-1 vectors from the bitmap
    return chunk_decode_launch(d_words, d_chunk_base, d_stream_woff, d_blk_off, d_stream_nbits, d_blk_state,
                               d_coset_bits, d_tables, d_scale16, n_chunks, n_heads, bph, d_lut_work, d_out, out_dtype,
                               d_dither_seed, 0, nullptr, nullptr, nullptr, nullptr, s);
}

int lq_chunk_decode_escaped(const uint32_t* d_words, const int64_t* d_chunk_base, const int64_t* d_stream_woff,
                            const uint32_t* d_blk_off, const int64_t* d_stream_nbits, const uint16_t* d_blk_state,
                            const uint8_t* d_coset_bits, const lq_table* d_tables, const uint16_t* d_scale16,
                            int64_t n_chunks, int64_t n_heads, int64_t bph, int head_dim, const float* d_signs,
                            const int32_t* d_esc_k, const int64_t* d_fine_off, const uint32_t* d_fine,
                            uint32_t* d_lut_work, void* d_out, int out_dtype, const int64_t* d_dither_seed, hipStream_t s) {
    if (!d_esc_k || !d_fine_off || !d_fine) return LQ_ERR_ARG;
    if (d_signs && (head_dim < 8 || head_dim > 128 || (head_dim & (head_dim - 1)) || bph <= 0 || bph % (head_dim / 8)))
        return LQ_ERR_ARG;
    return chunk_decode_launch(d_words, d_chunk_base, d_stream_woff, d_blk_off, d_stream_nbits, d_blk_state,
                               d_coset_bits, d_tables, d_scale16, n_chunks, n_heads, bph, d_lut_work, d_out, out_dtype,
                               d_dither_seed, d_signs ? head_dim : 0, d_signs, d_esc_k, d_fine_off, d_fine, s);
}

int lq_chunk_decode_rht(const uint32_t* d_words, const int64_t* d_chunk_base, const int64_t* d_stream_woff,
                        const uint32_t* d_blk_off, const int64_t* d_stream_nbits, const uint16_t* d_blk_state,
                        const uint8_t* d_coset_bits, const lq_table* d_tables, const uint16_t* d_scale16,
                        int64_t n_chunks, int64_t n_heads, int64_t bph, int head_dim, const float* d_signs,
                        uint32_t* d_lut_work, void* d_out, int out_dtype, const int64_t* d_dither_seed, hipStream_t s) {
    if (!d_signs || head_dim < 8 || head_dim > 128 || (head_dim & (head_dim - 1)) || bph <= 0 || bph % (head_dim / 8))
        return LQ_ERR_ARG;
    return chunk_decode_launch(d_words, d_chunk_base, d_stream_woff, d_blk_off, d_stream_nbits, d_blk_state,
                               d_coset_bits, d_tables, d_scale16, n_chunks, n_heads, bph, d_lut_work, d_out, out_dtype,
                               d_dither_seed, head_dim, d_signs, nullptr, nullptr, nullptr, s);
}

int lq_chunk_luts(const lq_table* d_tables, int64_t n_chunks, uint32_t* d_lut, hipStream_t s) {
    if (n_chunks <= 0 || !d_tables || !d_lut) return LQ_ERR_ARG;
    hipLaunchKernelGGL(k_chunk_lut, dim3((unsigned)(n_chunks * LQ_STREAMS)), dim3(256), 0, s, d_tables, d_lut);
    return launch_status();
}

int lq_build_tables(const int64_t* d_counts, const int64_t* d_count_off, const int32_t* d_n_sym, int32_t n_tables,
                    int32_t* d_freqs, int32_t* d_cum, int32_t* d_lookup, int32_t* d_status, hipStream_t s) {
    if (n_tables <= 0) return LQ_ERR_ARG;
    hipLaunchKernelGGL(k_build_tables, dim3((unsigned)n_tables), dim3(256), 0, s, d_counts, d_count_off, d_n_sym, d_freqs,
                       d_cum, d_lookup, d_status);
    return launch_status();
}

int lq_rans_encode_streams(const int32_t* d_idx, const int64_t* d_sym_off, const int64_t* d_n, const int32_t* d_freqs,
                           const int32_t* d_cum, const int64_t* d_tab_off, int32_t n_streams, uint32_t* d_scratch,
                           uint32_t* d_words, const int64_t* d_word_off, int64_t* d_state, int64_t* d_nbits,
                           hipStream_t s) {
    if (n_streams <= 0) return LQ_ERR_ARG;
    const int64_t cus = device_cus();   // one workgroup per CU (its LDS)
    hipLaunchKernelGGL(k_encode_streams, dim3((unsigned)(n_streams < cus ? n_streams : cus)), dim3(kSegLanes), 0, s, d_idx,
                       d_sym_off, d_n, d_freqs, d_cum, d_tab_off, (int64_t)n_streams, d_scratch, d_words, d_word_off, d_state,
                       d_nbits);
    return launch_status();
}

int lq_rans_decode_streams(const int32_t* d_bits, const int32_t* d_bit_off, const int32_t* d_nbits, const int32_t* d_init,
                           const int32_t* d_ndec, const int32_t* d_lookup, const int32_t* d_freqs, const int32_t* d_cum,
                           const int32_t* d_alphabet, const int32_t* d_tid, int32_t max_sym, const int32_t* d_out_off,
                           int32_t n_streams, int64_t* d_out, hipStream_t s) {
    if (n_streams <= 0 || max_sym <= 0) return LQ_ERR_ARG;
    const StreamArgs a = {reinterpret_cast<const uint32_t*>(d_bits), d_bit_off, d_nbits, d_init, d_ndec, d_lookup, d_freqs,
                          d_cum, d_alphabet, d_tid, max_sym, d_out_off, d_out};
    const int64_t cus = device_cus();
    const int64_t n = n_streams;
    // A lane per stream takes 0.7 us per symbol whatever the number of streams (up
    // to some 30000); a workgroup per stream 0.08 or less, but about 10 us for its
    // tables, and the CUs hold a few thousand at most.  us, lane / workgroup:
    // 16 streams of 10 symbols 10.0 / 12.6, of 24 17.8 / 12.6; 512 of 32
    // 21.2 / 22.9, of 64 40 / 38 (two at a time per CU), of 200 112 / 77; 2048 of
    // 10 9.3 / 12.0, of 24 18.8 / 16.6; 4096 of 64 43 / 40, of 128 93 / 47; 8192 of
    // 128 90 / 95, of 256 169 / 118; 16384 of 256 172 / 227; 32768 of 256 204 / 437.
    if (n <= 2 * cus) {   // the two-symbol tables fill a CU's LDS
        hipLaunchKernelGGL((k_decode_streams<true, 256>), dim3((unsigned)n), dim3(256), 0, s, a, n, n <= cus ? 16 : 48,
                           (int)(n < cus ? n : cus));
    } else {
        const int64_t least = n <= 4 * cus ? 8 : 16;
        const int64_t below = n >= 32768 ? INT_MAX : (n * n >> 18 > least ? n * n >> 18 : least);
        // four waves build the tables faster while a CU has room for them, one wave
        // leaves room for more streams (1024 of 64 symbols 20.3 us with four, 27
        // with one; 2000 of 64 38 and 24.5, of 4000 590 and 338)
        if (n <= 4 * cus) {
            const int lane_blocks = (int)((n + 255) / 256);
            hipLaunchKernelGGL((k_decode_streams<false, 256>), dim3((unsigned)(lane_blocks + n)), dim3(256), 0, s, a, n,
                               (int)below, lane_blocks);
        } else {
            const int lane_blocks = (int)((n + 63) / 64);
            const int64_t rest = below == INT_MAX ? 0 : (n < 32 * cus ? n : 32 * cus);
            hipLaunchKernelGGL((k_decode_streams<false, 64>), dim3((unsigned)(lane_blocks + rest)), dim3(64), 0, s, a, n,
                               (int)below, lane_blocks);
        }
    }
    return launch_status();
}

}  // extern "C"
