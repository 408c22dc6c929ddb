// Launches shared between the library's translation units (host side): the
// write path as one call (lq_encode_chunks) is made of them.
#pragma once

#include "latticequant_amd.h"

namespace lq {

// Words cleared on the side by the first launch of a write: the histograms,
// the chunks' status words and one counter.
struct Clear {
    uint32_t* hist = nullptr;
    int64_t n_hist = 0;
    int32_t* status = nullptr;
    int64_t n_status = 0;
    uint32_t* counter = nullptr;
};

// lq_head_scales (signs null) or lq_head_scales_rht
int head_scales_launch(const void* x, int dtype, int64_t n_chunks, int64_t n_heads, int64_t bph, int head_dim,
                       const float* signs, const int32_t* bits, double* work, float* sigma2, float* scale32,
                       uint16_t* scale16, int32_t* fastdiv, const Clear& clear, hipStream_t s);

// lq_scale_fastdiv, and the fp16 copies of the scales (scale16 nullable)
int scale_fastdiv_launch(const float* scale32, int64_t n, int dtype, int32_t* fastdiv, uint16_t* scale16,
                         const Clear& clear, hipStream_t s);

// How the chunk decoder's work is cut into workgroups.  A chunk has per_chunk
// tasks; a workgroup takes up to 16 of one chunk at a time (a round) and builds
// the chunk's LUTs first, which is counted as one round more (its waves wait for
// each other there).  Either every chunk is cut into equal parts, wpc workgroups
// of tpw tasks each, as many as fit the CUs at once (wpc > 0), or the whole batch
// is cut into one run of rounds per CU, which may cross chunk boundaries (wpc = 0;
// a chunk then has `span` task numbers, per_chunk rounded up to whole rounds).
// More chunks than CUs leave the last wave of equal parts nearly empty, so the
// rounds of the longest CU decide: 257 chunks of 64 tasks 458 us as 257 parts,
// 314 us in runs; 256 chunks 271 us as parts.
struct DecodeSplit {
    int64_t span, tpw;
    int wpc;
    int64_t grid;
};

inline DecodeSplit decode_split(int64_t n_chunks, int64_t per_chunk, int64_t cus) {
    const auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    const int64_t parts = n_chunks < cus ? cus / n_chunks : 1, tpw = up(per_chunk, parts), wpc = up(per_chunk, tpw);
    const int64_t by_parts = up(n_chunks * wpc, cus) * (up(tpw, 16) + 1);
    const int64_t rounds = up(per_chunk, 16), run = up(n_chunks * rounds, cus);
    const int64_t by_runs = run + 1 + (run + rounds - 2) / rounds;   // a run crosses at most that many boundaries
    if (by_parts <= by_runs) return {per_chunk, tpw, (int)wpc, n_chunks * wpc};
    return {16 * rounds, 16 * run, 0, up(n_chunks * rounds, run)};
}

}  // namespace lq
