"""Batches at the edges of the launch rules: how the blocks of a batch are cut
into workgroups (quantizer, decoder) and how a head's partial sums are added
must not show in any output."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _x(C, H, T, hd, seed, dtype=torch.float16):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(C, 1, H, T, hd, generator=g)
    x[..., :2] *= 6.0
    return x.to(dtype).cuda()


# blocks per chunk x chunks: a task is 4 blocks, a workgroup walks the tasks of
# one part of a chunk, or (many or uneven chunks) crosses chunk boundaries
@pytest.mark.parametrize("C,H,T,hd", [
    (1, 1, 3, 8),          # less than one block
    (1, 2, 260, 128),      # 17 blocks: a task of one block
    (3, 8, 203, 128),      # a partial last block, three parts per chunk
    (300, 1, 40, 64),      # more chunks than compute units
    (100, 8, 260, 128),    # 17 tasks per chunk, two parts
    (7, 8, 2100, 128),     # 132 tasks per chunk over 36 parts
    (129, 2, 1024, 128),   # one part of 16 tasks per chunk
    (300, 1, 2080, 128),   # 17 tasks per chunk, more chunks than CUs: runs of whole rounds over chunk boundaries
])
def test_decode_parts_gpu(C, H, T, hd):
    """Every chunk decoded in the batch equals the chunk decoded alone, and the
    oracle's rows at both ends of the batch."""
    from latticequant_amd import codec
    x = _x(C, H, T, hd, C + T)
    enc, _ = codec.encode_batch(x, 4)
    out = codec.decode_batch(enc)
    for c in sorted({0, 1 % C, C // 2, C - 1}):
        assert torch.equal(out[c], codec.decode_batch(enc.select(c))[0])
    for c in {0, C - 1}:
        ch = O.compress_chunk(x[c].cpu().numpy(), 4, scales_f32=enc.scale32.view(C, -1)[c].cpu().numpy())
        base, nw = int(enc.chunk_base[c]), int(enc.chunk_words[c])
        assert np.array_equal(enc.words[base:base + nw].cpu().numpy().view(np.uint32), ch.bitstream)
        assert np.array_equal(out[c].cpu().numpy(), O.decompress_chunk(ch))


# heads x vectors per head: 1, 8, 512, 513 .. partial sums per head (one per 512
# vectors, about 4096 in all)
@pytest.mark.parametrize("C,H,T,dtype", [
    (1, 3, 33, torch.float16), (1, 8, 256, torch.bfloat16), (1, 4, 16400, torch.float16), (1, 1, 33000, torch.float16),
])
def test_scale_parts_gpu(C, H, T, dtype):
    """sigma^2 against 64-bit sums: the partial sums are 64-bit, so one fp32
    rounding (2^-24) is all that may separate them, twice that being allowed
    for the sum's own rounding falling on the other side."""
    from latticequant_amd import codec
    x = _x(C, H, T, 128, T, dtype)
    _, _, _, s2 = codec.quantize_batch(x, 4, with_sigma2=True)
    want = x.double().square().mean((-1, -2)).reshape(-1)
    assert float(((s2.double() - want) / want).abs().max()) <= 2.0 ** -23


# blocks in the launch: 1, 2 .. 8 blocks per quantizer workgroup, and counts one
# off a multiple
@pytest.mark.parametrize("C,H,T", [(1, 1, 32), (2, 1, 1025), (1, 8, 4100), (2, 8, 4096), (9, 8, 1500), (20, 8, 3300)])
@pytest.mark.parametrize("deq", [False, True])
def test_quantizer_workgroups_gpu(C, H, T, deq):
    """Histograms, counts and symbols do not depend on the blocks per
    workgroup: the batch equals its chunks encoded one at a time (other launch
    shapes), word for word."""
    from latticequant_amd import codec
    x = _x(C, H, T, 128, 7 * T)
    enc, d = codec.encode_batch(x, 4, deq_out=deq)
    for c in sorted({0, C - 1}):
        one, d1 = codec.encode_batch(x[c:c + 1], 4, deq_out=deq)
        base, nw = int(enc.chunk_base[c]), int(enc.chunk_words[c])
        assert nw == int(one.chunk_words[0])
        assert torch.equal(enc.words[base:base + nw], one.words[:nw])
        assert torch.equal(enc.coset_bits[c], one.coset_bits[0]) and torch.equal(enc.blk_n1[c], one.blk_n1[0])
        if deq:
            assert torch.equal(d[c], d1[0])


def _tie_heavy(rng, n, kind):
    if kind == 0:
        return rng.integers(1, 4, n)                                  # three counts: large tie groups
    if kind == 1:
        return (1 + 2000 * np.exp(-0.5 * ((np.arange(n) - n / 2) / (0.1 * n + 1)) ** 2)).astype(np.int64)
    if kind == 2:
        return np.where(rng.random(n) < 0.02, 100000, rng.integers(1, 3, n))   # an excess: the decrement branch
    return rng.integers(1, 4, n) * (1 << 22) + (rng.random(n) < 0.5)  # keys beyond 2^23


@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_int8_tables_tie_order_gpu(kind):
    """Every table of the int8 path against the oracle (numpy's argsort order
    on ties) at alphabets of 5 .. 260 symbols, around the network's sizes (8,
    16, .. 256) and the wave's quarters."""
    from latticequant_amd import codec, _lib as L
    rng = np.random.default_rng(kind)
    spans = [1, 2, 3, 4, 5, 11, 12, 13, 27, 28, 59, 60, 61, 100, 123, 124, 125, 150, 187, 188, 200, 220, 251, 252, 253,
             255, 256, 64, 65, 128, 192, 230]
    hist = np.zeros((len(spans), 256), np.int64)
    for i, m in enumerate(spans):
        b0 = int(rng.integers(0, 256 - m + 1))
        hist[i, b0:b0 + m] = _tie_heavy(rng, m, kind)
    C = len(spans) // 16
    d = torch.from_numpy(hist.astype(np.uint32).view(np.int32)).cuda()
    tables = torch.zeros(C * 16 * L.TABLE_BYTES, dtype=torch.uint8, device="cuda")
    st = torch.zeros(C, dtype=torch.int32, device="cuda")
    L.check(L.lib().lq_chunk_tables(d.data_ptr(), C, tables.data_ptr(), st.data_ptr(), L.stream_ptr(d.device)),
            "lq_chunk_tables")
    t = tables.view(torch.int32).view(-1, L.TABLE_BYTES // 4).cpu().numpy()
    assert not st.any()
    for i, m in enumerate(spans):
        b0 = int(np.flatnonzero(hist[i])[0])
        lo, n = b0 - 128 - 2, m + 4
        assert (int(t[i, 0]), int(t[i, 1])) == (lo, n)
        counts = np.zeros(n, np.int64)
        counts[2:-2] = hist[i, b0:b0 + m]
        want = O.build_rans_table(counts, list(range(lo, lo + n))).freqs
        got = t[i, 4:4 + n].view(np.uint32)
        assert np.array_equal(got & 0x7ff, want), (kind, m)
        assert np.array_equal((got >> 11) & 0x3ff, (np.cumsum(want) - want) & 0x3ff)


def _stream(rng, n, spread):
    s = np.rint(rng.normal(0.0, spread, n)).astype(np.int64) if spread else np.zeros(n, np.int64)
    lo, hi = (int(s.min()), int(s.max())) if n else (0, 0)
    pad = 2 if spread else 0    # spread 0: one symbol with all of L, no bits
    counts = np.bincount(s - lo, minlength=hi - lo + 1)
    alphabet = list(range(lo - pad, hi + pad + 1))
    return s, np.concatenate([np.zeros(pad, np.int64), counts if n else np.ones(1, np.int64), np.zeros(pad, np.int64)]), alphabet


# lengths around a segment (64), the window behind it (16, 64), a decoder batch
# (64, 128) and a tile of segments (65536); spreads from no bits per symbol to
# alphabets near L
@pytest.mark.parametrize("spread", [0.0, 0.3, 3.0, 40.0, 100.0])
def test_stream_coder_lengths_gpu(spread):
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(int(10 * spread) + 1)
    lens = [0, 1, 2, 15, 16, 17, 63, 64, 65, 80, 127, 128, 129, 191, 192, 193, 500, 1000, 4097, 65535, 65536, 65537, 70001]
    parts = [_stream(rng, n, spread) for n in lens]
    tabs = gpu_ans.build_rans_tables([p[1] for p in parts], [p[2] for p in parts])
    enc = gpu_ans.rans_encode_many([p[0] for p in parts], tabs)
    for (s, counts, alphabet), (words, state, nbits) in zip(parts, enc):
        want = O.rans_encode(s, O.build_rans_table(counts, alphabet))
        assert (state, nbits) == (int(want[1]), int(want[2])), len(s)
        assert np.array_equal(words, want[0]), len(s)
    streams = [gpu_ans.RANSStream(w, nb, st, len(p[0]), t) for (w, st, nb), p, t in zip(enc, parts, tabs)]
    for got, p in zip(gpu_ans.gpu_rans_decode(streams), parts):
        assert np.array_equal(got, p[0]), len(p[0])
    # more streams than the two-symbol tables are taken for
    many = gpu_ans.gpu_rans_decode([streams[i % 19] for i in range(600)])
    for i, got in enumerate(many):
        assert np.array_equal(got, parts[i % 19][0])


# streams of every group width (64, 256, 1024, 4096 symbols and one past each)
# side by side in one launch: fewer streams than CUs, several per workgroup, more
# than a workgroup's lanes
@pytest.mark.parametrize("m", [40, 700, 40 + 256 * 1024])
def test_stream_encoder_groups_gpu(m):
    from latticequant_amd import _lib as L
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(m)
    lens = [0, 1, 10, 63, 64, 65, 200, 255, 256, 257, 700, 1023, 1024, 1025, 3000, 4095, 4096, 4097, 5000]
    if m > 4096:
        lens = [n for n in lens if n <= 65] + [257]
    kinds = [_stream(rng, n, sp) for sp in (0.0, 0.4, 3.0, 100.0) for n in lens]
    tabs = gpu_ans.build_rans_tables([k[1] for k in kinds], [k[2] for k in kinds])
    want = [O.rans_encode(s, O.build_rans_table(c, a)) for s, c, a in kinds]
    order = rng.integers(0, len(kinds), m)
    order[:min(m, len(kinds))] = np.arange(min(m, len(kinds)))
    n = np.array([len(kinds[k][0]) for k in order], np.int64)
    cap = (10 * n + 31) // 32 + 2
    sym_off, word_off = (np.concatenate([[0], np.cumsum(v)[:-1]]) for v in (n, cap))
    tsz = np.array([t.n_symbols + 1 for t in tabs])
    toff = np.concatenate([[0], np.cumsum(tsz)[:-1]])

    def dev(a, dt):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dt).cuda()

    idx = dev(np.concatenate([kinds[k][0] - kinds[k][2][0] for k in order]), torch.int32)
    so, ln, to, wo = (dev(a, torch.int64) for a in (sym_off, n, toff[order], word_off))
    fr = dev(np.concatenate([np.append(t.freqs, 0) for t in tabs]), torch.int32)
    cu = dev(np.concatenate([t.cumfreqs for t in tabs]), torch.int32)
    scr, words = (torch.full((int(cap.sum()) + 8,), -9, dtype=torch.int32, device="cuda") for _ in range(2))
    st, nb = (torch.full((m,), -1, dtype=torch.int64, device="cuda") for _ in range(2))
    L.check(L.lib().lq_rans_encode_streams(idx.data_ptr(), so.data_ptr(), ln.data_ptr(), fr.data_ptr(), cu.data_ptr(),
                                           to.data_ptr(), m, scr.data_ptr(), words.data_ptr(), wo.data_ptr(),
                                           st.data_ptr(), nb.data_ptr(), L.stream_ptr(idx.device)), "encode")
    words, st, nb = words.cpu().numpy().view(np.uint32), st.cpu().numpy(), nb.cpu().numpy()
    assert np.array_equal(st, np.array([int(want[k][1]) for k in order]))
    assert np.array_equal(nb, np.array([int(want[k][2]) for k in order]))
    for i in list(range(min(m, 700))) + list(rng.integers(0, m, 3000)):
        w = want[order[i]][0]
        assert np.array_equal(words[word_off[i]:word_off[i] + len(w)], w), (i, n[i])
    assert (words[int(cap.sum()):] == 0xfffffff7).all()


def test_stream_encoder_many_short_time_gpu():
    """8192 streams of 10 symbols take about the time of 16 (one lane each);
    with a workgroup each they took 160 times as long."""
    us = [_encode_us(np.array([3, 4, 1]), np.arange(10) % 3, m)[0] for m in (16, 8192)]
    assert us[1] < 10 * us[0], us


def _encode_us(counts, idx, m):
    """Time of lq_rans_encode_streams for m copies of one stream, in
    microseconds, and the (state, bits) of the last."""
    from latticequant_amd import _lib as L
    from latticequant_amd.core import gpu_ans
    tab = gpu_ans.build_rans_tables([counts], [list(range(len(counts)))])[0]
    n, cap = len(idx), (10 * len(idx) + 31) // 32 + 2

    def dev(a, dt):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dt).cuda()

    d_idx, so = dev(np.tile(idx, m), torch.int32), dev(np.arange(m) * n, torch.int64)
    ln, to, wo = dev(np.full(m, n), torch.int64), dev(np.zeros(m), torch.int64), dev(np.arange(m) * cap, torch.int64)
    fr, cu = dev(np.append(tab.freqs, 0), torch.int32), dev(tab.cumfreqs, torch.int32)
    scr, words = (torch.zeros(cap * m, dtype=torch.int32, device="cuda") for _ in range(2))
    st, nb = (torch.zeros(m, dtype=torch.int64, device="cuda") for _ in range(2))
    us = _us(lambda: L.check(L.lib().lq_rans_encode_streams(
        d_idx.data_ptr(), so.data_ptr(), ln.data_ptr(), fr.data_ptr(), cu.data_ptr(), to.data_ptr(), m, scr.data_ptr(),
        words.data_ptr(), wo.data_ptr(), st.data_ptr(), nb.data_ptr(), L.stream_ptr(d_idx.device)), "encode"), 5)
    return us, (int(st[-1]), int(nb[-1]))


# runs over which states do not come together: one symbol with all of L, one of
# nearly all of it, runs of such a symbol between others, cut at tile ends
@pytest.mark.parametrize("n", [4097, 5000, 20000, 65536, 65537, 140000])
def test_stream_encoder_runs_gpu(n):
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(n)
    runs = np.zeros(n, np.int64)
    runs[rng.integers(0, n, 12)] = 1
    half = np.where((np.arange(n) // (n // 3 + 1)) % 2 == 1, rng.integers(-3, 4, n), 0)
    syms = [np.zeros(n, np.int64), np.zeros(n, np.int64), runs, half]
    alphabets = [[0], [-2, -1, 0, 1, 2], [0, 1], list(range(-5, 6))]
    counts = [np.array([np.count_nonzero(s == a) for a in al]) for s, al in zip(syms, alphabets)]
    enc = gpu_ans.rans_encode_many(syms, gpu_ans.build_rans_tables(counts, alphabets))
    for i, (s, c, al, (words, state, nbits)) in enumerate(zip(syms, counts, alphabets, enc)):
        want = O.rans_encode(s, O.build_rans_table(c, al))
        assert (state, nbits) == (int(want[1]), int(want[2])), i
        assert np.array_equal(words, want[0]), i


@pytest.mark.parametrize("counts", [[7], [0, 0, 7, 0, 0]])
def test_stream_encoder_one_symbol_time_gpu(counts):
    """Four times as many equal symbols take about four times as long (with
    windows to the stream's end: sixteen times, and more than one lane)."""
    n = 60000
    short, long = (_encode_us(np.array(counts), np.full(m, len(counts) // 2), 1)[0] for m in (n, 4 * n))
    assert long < 7 * short, (short, long)


# alphabets of nearly L symbols, all about equally likely: nearly every symbol
# takes 10 bits, the most a 16-symbol chunk can add to the encoder's ring of words
@pytest.mark.parametrize("T", [256, 1031])
def test_wide_encoder_ten_bits_per_symbol_gpu(T):
    from latticequant_amd import codec
    g = torch.Generator().manual_seed(T)
    x = ((torch.rand(1, 2, T, 128, generator=g) - 0.5) * 990).to(torch.float16)
    x[..., 7::8] *= 2   # the last coordinate's symbol is half of it
    scale = torch.ones(2)
    enc, _ = codec.encode_batch(x.cuda()[None], 4, scale32=scale, wide=True, escape=False)
    ch = O.compress_chunk(x.numpy(), 4, scales_f32=scale.numpy())
    base, nw = int(enc.chunk_base[0]), int(enc.chunk_words[0])
    assert int(enc.stream_nbits.min()) > 9.5 * 0.4 * T * 2 * 16   # both cosets of every coordinate
    assert np.array_equal(enc.words[base:base + nw].cpu().numpy().view(np.uint32), ch.bitstream)
    assert np.array_equal(codec.decode_batch(enc)[0].cpu().numpy(), O.decompress_chunk(ch))


# the parallel decode: from 8192 symbols on (more with few bits per symbol), in
# tiles of about 262000 bits; streams of four equally likely symbols move by two
# bits per step, so starts on an odd bit never fall into step and the proven
# segments go on serially; fewer symbols than the stream holds, and fewer bits
# than the symbols take; beyond two streams per CU all goes serially
@pytest.mark.parametrize("many", [False, True])
def test_stream_decoder_parallel_gpu(many):
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(11)
    parts = [_stream(rng, n, sp) for n, sp in [(8191, 3.0), (8192, 3.0), (30000, 0.6), (8203, 30.0), (33000, 9.0),
                                               (70001, 4.0), (150000, 0.7), (131072, 12.0), (90000, 1.0)]]
    four = [np.repeat(np.arange(4), n // 4) for n in (16384, 40004, 262144)]
    for f in four:
        rng.shuffle(f)
        parts.append((f.astype(np.int64), np.full(4, len(f) // 4, np.int64), [0, 1, 2, 3]))
    tabs = gpu_ans.build_rans_tables([p[1] for p in parts], [p[2] for p in parts])
    assert all((t.freqs == 256).all() for t in tabs[-3:])
    enc = gpu_ans.rans_encode_many([p[0] for p in parts], tabs)
    streams, want = [], []
    for (w, st, nb), p, t in zip(enc, parts, tabs):
        for n in (len(p[0]), len(p[0]) - 1, 8192, 8400):
            n = min(n, len(p[0]))
            streams.append(gpu_ans.RANSStream(w, nb, st, n, t))
            want.append(p[0][:n])
        # the symbols whose bits are all there: a step takes at most 10
        cut = nb * 2 // 3
        streams.append(gpu_ans.RANSStream(w, cut, st, cut // 10, t))
        want.append(p[0][:cut // 10])
    if many:   # small streams fill the launch
        streams += [streams[0]] * 520
        want += [want[0]] * 520
    for i, (got, ref) in enumerate(zip(gpu_ans.gpu_rans_decode(streams), want)):
        assert np.array_equal(got, ref), (i, len(ref))


def _decode_case(rng, m, lens):
    """m streams of lengths drawn from lens (each of them once at least), of a few
    tables, as (streams, wanted symbols)."""
    from latticequant_amd.core import gpu_ans
    parts = [_stream(rng, n, 3.0) for n in lens]
    tabs = gpu_ans.build_rans_tables([p[1] for p in parts], [p[2] for p in parts])
    enc = gpu_ans.rans_encode_many([p[0] for p in parts], tabs)
    one = [gpu_ans.RANSStream(w, nb, st, len(p[0]), t) for (w, st, nb), p, t in zip(enc, parts, tabs)]
    order = np.concatenate([np.arange(len(lens)), rng.integers(0, len(lens), m - len(lens))])
    rng.shuffle(order)
    return [one[i] for i in order], [parts[i][0] for i in order]


# around the numbers of streams at which the launch changes (one and two per CU,
# four per CU, 32768), with streams on both sides of the length below which a lane
# takes a stream: 16, 48, 8, 16, 64 (4100 streams), every length from 32768 on
@pytest.mark.parametrize("m", [20, 256, 257, 512, 513, 1024, 1025, 2100, 4100, 32767, 32768])
def test_stream_decoder_launches_gpu(m):
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(m)
    lens = [1, 8, 9, 15, 16, 17, 47, 48, 49, 64, 65, 128, 599, 600, 700] if m < 4096 else [1, 7, 16, 64, 65, 90]
    streams, want = _decode_case(rng, m, lens)
    got = gpu_ans.gpu_rans_decode(streams)
    assert np.array_equal(np.concatenate(got), np.concatenate(want))


@pytest.mark.parametrize("m,n,times", [(8192, 10, 1.6), (32768, 64, 1.8)])
def test_stream_decoder_many_short_time_gpu(m, n, times):
    """Short streams take about the time of 64 of them, however many there are: a
    lane each (with a workgroup each 2.2 and 5 times as long)."""
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(n)
    us = []
    for k in (64, m):
        streams, _ = _decode_case(rng, k, [n])
        prep = gpu_ans.prepare_gpu_decode(streams)
        if k == 64 and n > 16:   # 64 streams of this length a lane each: 0.7 us per symbol
            us.append(0.7 * n)
            continue
        us.append(_us(lambda: gpu_ans.run_gpu_decode_kernel(prep)))
    assert us[1] < times * us[0], us


def test_stream_decoder_truncated_gpu():
    """A stream with fewer bits than its symbols need is decoded to its length
    with the reference's rule (a step reads min(needed, bits left)), from any
    state, as the plain step written out below."""
    from latticequant_amd.core import gpu_ans
    rng = np.random.default_rng(5)
    s, counts, alphabet = _stream(rng, 700, 9.0)
    tab = gpu_ans.build_rans_tables([counts], [alphabet])[0]
    words, state, nbits = gpu_ans.rans_encode_many([s], [tab])[0]
    cases = [(nbits, state, 700), (nbits - 1, state, 700), (nbits // 2, state, 700), (9, state, 60), (0, state, 40),
             (nbits, 1024, 700), (nbits, 77, 700), (nbits, state, 760)]
    streams = [gpu_ans.RANSStream(words, nb, st, n, tab) for nb, st, n in cases]
    for (nb, st, n), got in zip(cases, gpu_ans.gpu_rans_decode(streams)):
        x, pos, want = st, 0, []
        for _ in range(n):
            slot = x & 1023
            si = int(tab.lookup[slot])
            want.append(tab.alphabet[si])
            x = (int(tab.freqs[si]) * (x >> 10) + slot - int(tab.cumfreqs[si])) & 0xffffffff
            if x < 1024:
                k = min((32 - x.bit_length()) - 21, nb - pos)
                for q in range(pos, pos + k):
                    x = (x << 1) | (int(words[q >> 5]) >> (q & 31) & 1)
                pos += max(k, 0)
        assert np.array_equal(got, np.array(want)), (nb, st, n)


@pytest.mark.parametrize("C,T", [(1, 40), (3, 1100), (70, 64), (2, 16400)])
@pytest.mark.parametrize("wide", ["auto", False])
@pytest.mark.parametrize("arena", ["own", "bound", "given"])
def test_write_call_sizes_gpu(C, T, wide, arena):
    """The write's one native call: chunk bases and total (one workgroup and
    the tiled scan of long streams, more chunks than a wave's lanes), in an
    arena of its exact size, at the bound, and the caller's."""
    from latticequant_amd import codec
    x = _x(C, 8, T, 128, C * T)
    given = torch.full((codec.words_bound(C, 8 * T * 16),), -7, dtype=torch.int32, device="cuda")
    kw = {"own": {}, "bound": {"exact_size": False}, "given": {"words_out": given}}[arena]
    enc, _ = codec.encode_batch(x, 4, wide=wide, **kw)
    cw = enc.chunk_words.cpu()
    assert torch.equal(enc.chunk_base.cpu(), torch.cumsum(cw, 0) - cw)
    total = int(cw.sum())
    if arena == "own":
        assert enc.words.numel() == total + 2
    if arena == "given":
        assert enc.words.data_ptr() == given.data_ptr() and bool((given[total:] == -7).all())
    c = C - 1
    ch = O.compress_chunk(x[c].cpu().numpy(), 4, scales_f32=enc.scale32.view(C, -1)[c].cpu().numpy())
    base = int(enc.chunk_base[c])
    assert np.array_equal(enc.words[base:base + int(cw[c])].cpu().numpy().view(np.uint32), ch.bitstream)
    given_scales, _ = codec.encode_batch(x, 4, scale32=enc.scale32, wide=wide)
    assert torch.equal(given_scales.words[:total], enc.words[:total])
    assert torch.equal(given_scales.scale16, enc.scale16)


def _us(f, n=20):
    """Median time of f's work on the GPU, in microseconds."""
    ts = []
    for i in range(n + 3):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        f()
        b.record()
        b.synchronize()
        ts.append(a.elapsed_time(b) * 1e3)
    return sorted(ts[3:])[n // 2]


# chunk bases by the scan's last workgroup (up to 64 chunks) and by a launch of
# their own, 1024 chunks at a time
@pytest.mark.parametrize("C", [64, 65, 1024, 1025, 2500])
def test_write_call_bases_gpu(C):
    from latticequant_amd import codec
    x = _x(C, 1, 5, 8, C)
    enc, _ = codec.encode_batch(x, 4)
    cw = enc.chunk_words.cpu()
    assert torch.equal(enc.chunk_base.cpu(), torch.cumsum(cw, 0) - cw)
    assert enc.words.numel() == int(cw.sum()) + 2
    one, _ = codec.encode_batch(x[C - 1:], 4)
    assert torch.equal(enc.words[int(enc.chunk_base[-1]):-2], one.words[:-2])


def test_write_call_many_chunks_time_gpu():
    """The one call does what its launches made one by one do, whose chunk
    bases come from torch.cumsum: with 16384 chunks of one block the GPU may not
    take longer by more than a fifth (with a release and an acquire of the L2
    per chunk it took a third longer; 4 % without)."""
    from latticequant_amd import codec, _lib as L
    C, V = 16384, 128
    x = _x(C, 1, 8, 128, 1)
    lib, s = L.lib(), L.stream_ptr(x.device)
    arena = torch.zeros(codec.words_bound(C, V), dtype=torch.int32, device="cuda")
    e, _ = codec.encode_batch(x, 4, words_out=arena, wide=False)
    want = arena.clone()

    def dev(n, dt):
        return torch.empty(int(n), dtype=dt, device="cuda")

    sym, work = dev(C * L.LQ_SYM_STRIDE, torch.int8), dev(lib.lq_chunk_encode_workspace(C, V), torch.uint8)
    fd, sums, cw = dev(C, torch.int32), dev(4096 + C, torch.float64), torch.zeros(C + 1, dtype=torch.int64, device="cuda")

    def launches():
        e.hist.zero_(), e.status.zero_()
        L.check(lib.lq_head_scales(x.data_ptr(), L.LQ_F16, C, 1, V, e.bits.data_ptr(), sums.data_ptr(), e.sigma2.data_ptr(),
                                   e.scale32.data_ptr(), e.scale16.data_ptr(), fd.data_ptr(), s), "scales")
        L.check(lib.lq_chunk_quantize(x.data_ptr(), L.LQ_F16, C, 1, V, e.scale32.data_ptr(), fd.data_ptr(), sym.data_ptr(),
                                      e.coset_bits.data_ptr(), e.blk_n1.data_ptr(), e.hist.data_ptr(), e.status.data_ptr(),
                                      None, L.LQ_F16, None, s), "quantize")
        L.check(lib.lq_chunk_tables(e.hist.data_ptr(), C, e.tables.data_ptr(), e.status.data_ptr(), s), "tables")
        L.check(lib.lq_chunk_encode(sym.data_ptr(), e.blk_n1.data_ptr(), C, V, e.tables.data_ptr(), work.data_ptr(),
                                    e.blk_off.data_ptr(), e.blk_state.data_ptr(), e.stream_nbits.data_ptr(),
                                    e.stream_state.data_ptr(), e.stream_woff.data_ptr(), cw[1:].data_ptr(), s), "encode")
        base = torch.cumsum(cw[:C], 0)
        L.check(lib.lq_chunk_pack(C, V, e.tables.data_ptr(), work.data_ptr(), e.blk_off.data_ptr(),
                                  e.stream_nbits.data_ptr(), e.stream_woff.data_ptr(), base.data_ptr(), arena.data_ptr(),
                                  s), "pack")

    arena.zero_()
    one = _us(lambda: codec.encode_batch(x, 4, words_out=arena, wide=False))
    arena.zero_()
    apart = _us(launches)
    assert torch.equal(arena, want)
    assert one < 1.2 * apart, (one, apart)


def test_write_call_capture_gpu():
    """Without dither the write into a caller's arena is launches only: a graph of
    it gives the eager words on every replay, with new input too.  With dither
    seeds, which come from the host, a capture is refused (a recorded copy would
    read its staging memory again at every replay)."""
    from latticequant_amd import codec
    x = _x(2, 4, 300, 128, 1)
    arena = torch.zeros(codec.words_bound(2, 4 * 300 * 16), dtype=torch.int32, device="cuda")
    codec.encode_batch(x, 4, words_out=arena, wide=False)   # (the rates' tensor is made outside the graph)
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        enc, _ = codec.encode_batch(x, 4, words_out=arena, wide=False)
    for seed in (1, 2, 3):
        x.copy_(_x(2, 4, 300, 128, seed))
        want, _ = codec.encode_batch(x, 4)
        n = int(want.chunk_words.sum())
        arena.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(arena[:n], want.words[:n]) and torch.equal(enc.chunk_base, want.chunk_base)
    refused = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(refused, stream=side):
            codec.encode_batch(x, 4, words_out=arena, wide=False, dither_seed=[5, 6])
    torch.cuda.synchronize()
    again, _ = codec.encode_batch(x, 4)
    assert torch.equal(again.words[:n], want.words[:n])   # (the slack words have no value)


def test_write_call_overflow_leaves_arena_gpu():
    """One chunk of three outside int8: the batch is coded once, on int16
    symbols; words past its bitstreams are not touched."""
    from latticequant_amd import codec
    x = _x(3, 2, 600, 128, 3)
    x[1, 0, 0, :, 0] *= 400.0
    bound = codec.words_bound(3, 2 * 600 * 16)
    given = torch.full((bound,), -7, dtype=torch.int32, device="cuda")
    enc, _ = codec.encode_batch(x, 5, words_out=given)
    assert enc.extra["wide"]
    ref, _ = codec.encode_batch(x, 5, wide=True)
    total = int(ref.chunk_words.sum())
    assert torch.equal(enc.chunk_words, ref.chunk_words)
    assert torch.equal(given[:total], ref.words[:total]) and bool((given[total:] == -7).all())
    assert torch.equal(codec.decode_batch(enc), codec.decode_batch(ref))


@pytest.mark.parametrize("rotated", [False, True])
@pytest.mark.parametrize("given", [False, True])
def test_write_call_overflow_once_gpu(rotated, given, monkeypatch):
    """A batch that leaves int8 is tried on int8 once, and the int16 path takes over
    its scales, their fast-division words and sigma^2: the batch is the one
    wide=True writes."""
    from latticequant_amd import _lib as L, codec
    x = _x(2, 4, 300, 128, 9)
    x[1, 0, 2, 7] *= 2000.0
    signs = (torch.randint(0, 2, (8, 128), generator=torch.Generator().manual_seed(2)) * 2 - 1).float().cuda()
    rows = codec.rotate_rows(x, signs, inverse=False) if rotated else x
    s32, s16, _, s2 = codec.quantize_batch(rows, 5, with_sigma2=True)
    kw = {"scale32": s32 if given else None, "dither_seed": [3, 4] if rotated else None}
    want, _ = codec.encode_batch(rows, 5, wide=True, **kw)
    calls, lib = [], L.lib()
    for name in ("lq_encode_chunks", "lq_encode_chunks_pack", "lq_scale_fastdiv", "lq_head_scales"):
        f = getattr(lib, name)
        monkeypatch.setattr(lib, name, lambda *a, f=f, name=name: calls.append(name) or f(*a))

    got, _ = codec.encode_batch(x, 5, rht_signs=signs if rotated else None, **kw)
    monkeypatch.undo()
    assert got.extra["wide"] and calls == ["lq_encode_chunks"]
    assert torch.equal(got.scale32, s32) and torch.equal(got.scale16, s16)
    assert got.sigma2 is None if given else torch.equal(got.sigma2, s2)
    n = int(want.chunk_words.sum())
    assert torch.equal(got.words[:n], want.words[:n]) and torch.equal(got.chunk_words, want.chunk_words)
    for f in ("coset_bits", "blk_n1", "blk_off", "blk_state", "stream_nbits", "stream_state", "stream_woff", "chunk_base"):
        assert torch.equal(getattr(got, f), getattr(want, f)), f


def test_write_call_threads_gpu():
    """Calls from more threads at once than read-back slots are kept (16), on their
    own streams, each with its read-back; every call ends and gives its words."""
    import threading
    from latticequant_amd import codec
    n, rounds = 20, 4
    xs = [_x(2, 4, 300 + 7 * i, 128, i) for i in range(n)]
    want = [codec.encode_batch(x, 4)[0] for x in xs]
    torch.cuda.synchronize()
    bad, done = [], []
    together = threading.Barrier(n, timeout=60)

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(rounds):
                    together.wait()
                    e, _ = codec.encode_batch(xs[i], 4)
                    s.synchronize()
                    if not (torch.equal(e.words[:-2], want[i].words[:-2]) and torch.equal(e.chunk_base, want[i].chunk_base)):
                        bad.append(i)
                    done.append(i)
            s.synchronize()
        except Exception as e:   # a thread's exception would not fail the test by itself
            bad.append(e)
            together.abort()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad and len(done) == n * rounds


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,hd,steps", [
    (1, 8, 128, [1, 1, 1, 5, 1, 1, 16, 1]),      # decode steps, buffers growing
    (2, 3, 64, [127, 1, 128, 1]),                # 1016 vectors per head, then 1024: the general path between
    (1, 1, 8, [1, 2, 1000, 1023, 1024, 1]),      # one vector per token, up to the limit and past it
    (3, 2, 24, [7, 1, 340]),                     # head_dim not a power of two
])
def test_direct_updates_gpu(B, H, hd, steps, dtype, monkeypatch):
    """update()'s one-launch form against the general one (quantize, then
    append), taken exactly where it should be: rows, scales, sigma^2 and
    bitstreams, with K and V at their own rates, from contiguous, transposed and
    misaligned tensors, zero heads."""
    from latticequant_amd.allocation.eval_alloc import VariableRateKVCache
    g = torch.Generator().manual_seed(hd)
    kv = []
    for i, T in enumerate(steps):
        t = torch.randn(2, B, H, T, hd, generator=g) * 3.0
        t[:, 0, 0] *= 0.0 if i == 1 else 1.0
        t[1, :, -1] *= 1e-4
        t = t.to(dtype).cuda()
        k, v = t[0], t[1]
        if i % 3 == 1:      # as attention layers hand them over: (B, T, H, hd) transposed
            k, v = (a.transpose(1, 2).contiguous().transpose(1, 2) for a in (k, v))
        if i % 3 == 2:      # rows that start 2 or 4 bytes past a 16-byte boundary
            k = torch.cat([k.new_zeros(1), k.reshape(-1)])[1:].view(k.shape)
        kv.append((k, v))

    # the one-launch form takes heads of up to 1023 vectors, up to 2^14 in all, on
    # 16-byte boundaries
    bph = [k.shape[2] * hd // 8 for k, _ in kv]
    want_direct = [n <= 1023 and n * B * H <= 1 << 14 and (not k.is_contiguous() or k.data_ptr() % 16 == 0)
                   for n, (k, _) in zip(bph, kv)]
    assert any(want_direct) and not all(want_direct)
    took = []
    update_direct = VariableRateKVCache._update_direct

    def recorded(*a):
        r = update_direct(*a)
        took.append(r is not None)
        return r

    def fill(direct):
        monkeypatch.setattr(VariableRateKVCache, "_update_direct", recorded if direct else lambda *a: None)
        c = VariableRateKVCache([{"K": 3, "V": 5}, {"K": 4, "V": 4}], eval_only_no_entropy=False)
        outs = []
        for k, v in kv:
            for layer in range(2):
                outs.append([t.clone() for t in c.update(k, v, layer)])
        return c, outs

    a, oa = fill(True)
    assert took == [d for d in want_direct for _ in range(2)]   # two layers
    b, ob = fill(False)
    for (ka, va), (kb, vb) in zip(oa, ob):
        assert torch.equal(ka, kb) and torch.equal(va, vb)
    assert a.total_vectors == b.total_vectors and a.compressed_bytes() == b.compressed_bytes()
    for la, lb in zip(a._layers(), b._layers()):
        for ca, cb in zip(la.chunks, lb.chunks):
            assert torch.equal(ca.gpu_bitstream, cb.gpu_bitstream) and torch.equal(ca.coset_packed, cb.coset_packed)
            assert torch.equal(ca.scales, cb.scales) and torch.equal(ca.encoded.sigma2, cb.encoded.sigma2)
            assert torch.equal(a._decompress_chunk(ca), b._decompress_chunk(cb))


@pytest.mark.parametrize("T,chans,factor", [
    (16, 1, 400.0),      # one block, one vector of every token outside the records' range
    (48, 128, 400.0),    # every vector is an exception (256 of a block: the count saturates)
    (2064, 3, 40.0),     # several per token, a half tile at the end
    (4096, 40, 12.0),    # about one vector in three
])
@pytest.mark.parametrize("which", ["k", "v", "both"])
def test_attention_exceptions_gpu(T, chans, factor, which):
    """Attention over prefixes with many exception vectors, in K, in V and in
    both, against float64 attention over the rows the dequantiser writes for
    the same prefix (it reads every exception on its own).  The step rounds
    each weight of P V to fp16 (2^-11 of it) and its output (2^-11), so it lies
    within 2^-10 of sum_t p_t |v_t|; a fifth of that for the fp32 scores."""
    from latticequant_amd import codec
    from latticequant_amd.llm import resident
    B, H, group, tail = 2, 2, 4, 5
    g = torch.Generator().manual_seed(T + chans)
    kv = torch.randn(2, B, H, T, 128, generator=g)
    pick = torch.randperm(128, generator=g)[:chans]
    for i in range(2):
        if which in ("both", "kv"[i]):
            kv[i][..., pick] *= factor
    if which != "v":
        kv[0] *= 0.05     # keep the scores of outlier channels in range of a soft maximum
    kv = kv.half().cuda()
    q = torch.randn(B, H * group, 1, 128, generator=g).half().cuda()
    tl = torch.randn(2, B, H, tail, 128, generator=g).half().cuda()
    res = []
    for i in range(2):
        # coordinates up to 900: outlier channels far outside [-16, 15], and below
        # 1024, up to which fp16 holds every half-integer (the kernel's operands
        # are fp16; larger coordinates are rounded before the scale)
        s32 = torch.full((B * H,), float(kv[i].abs().max()) / 900.0, device="cuda")
        r = resident.ResidentKV(B * H, T)
        r.append(kv[i], s32, s32.half())
        res.append(r)
    assert int(res[0].n_exc) + int(res[1].n_exc) > 0
    out = resident.resident_decode_attention(res[0], res[1], q, tl[0], tl[1])
    k, v = (torch.cat([r.dequant(torch.float32).view(B, H, T, 128).half(), tl[i]], 2).double()
            for i, r in enumerate(res))
    qq = q.double().view(B, H, group, 128)
    p = torch.matmul(qq, k.transpose(-1, -2).contiguous()) / 128 ** 0.5
    w = p.softmax(-1)
    err = (out.double().view(B, H, group, 128) - torch.matmul(w, v)).abs().amax(-1) / torch.matmul(w, v.abs()).amax(-1)
    assert float(err.max()) < 1.2 * 2.0 ** -10


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("H,bph", [(1, 512), (1, 1025), (3, 515), (2, 20 * 512 + 7)])
def test_quantizer_integer_output_gpu(dtype, wide, H, bph):
    """Launches without a dequantised output keep the lattice points as biased
    integers and load a block ahead; those with one keep floats and load none.
    Both give the same symbols, bitmaps, counts, histograms or ranges, and
    status, up to coordinates beyond every symbol range, infinities and NaN,
    and at ragged ends."""
    from latticequant_amd import _lib as L
    C, V, nblk = 2, H * bph, (H * bph + 511) // 512
    g = torch.Generator().manual_seed(bph)
    x = torch.randn(C, V, 8, generator=g) * 2.0 ** torch.randint(-3, 5, (C, V, 1), generator=g)
    x[:, ::3] = torch.round(x[:, ::3] * 2) / 2                     # grid points: ties
    x[0, 7::61] = torch.randn(x[0, 7::61].shape, generator=g) * 30000    # chunk 0 overflows, chunk 1 does not
    x[0, 11::97, 3] = float("inf")
    x[0, 13::89, 5] = float("-inf")
    x[0, 17::101, 0] = float("nan")
    if dtype != torch.float16:
        x[0, 19::103] = torch.randn(x[0, 19::103].shape, generator=g) * 1e7
    x = x.to(dtype).cuda().contiguous()
    scale = torch.full((C * H,), 0.75, device="cuda")
    code, lib, s = L.dtype_code(dtype), L.lib(), L.stream_ptr(x.device)
    fd = torch.empty(C * H, dtype=torch.int32, device="cuda")
    L.check(lib.lq_scale_fastdiv(scale.data_ptr(), C * H, code, fd.data_ptr(), s), "lq_scale_fastdiv")

    def run(out):
        sym = torch.zeros(C * nblk * L.LQ_SYM_STRIDE * (2 if wide else 1), dtype=torch.int8, device="cuda")
        cb = torch.zeros(C * nblk * 64, dtype=torch.uint8, device="cuda")
        n1 = torch.zeros(C * nblk, dtype=torch.int32, device="cuda")
        st = torch.zeros(C, dtype=torch.int32, device="cuda")
        if wide:
            tab = torch.tensor([2 ** 31 - 1, -2 ** 31], dtype=torch.int32).repeat(C * 16).cuda()
        else:
            tab = torch.zeros(C * 16 * 256, dtype=torch.int32, device="cuda")
        f = lib.lq_chunk_quantize_wide if wide else lib.lq_chunk_quantize
        L.check(f(x.data_ptr(), code, C, H, bph, scale.data_ptr(), fd.data_ptr(), sym.data_ptr(), cb.data_ptr(),
                  n1.data_ptr(), tab.data_ptr(), st.data_ptr(), L.ptr(out), code, None, s), "lq_chunk_quantize")
        return sym, cb, n1, tab, st

    lean, full = run(None), run(torch.empty_like(x))
    # rows of a group's unused places keep what an earlier block staged there,
    # so the staging is compared through the counts' ranges: symbols by column
    for a, b in zip(lean[1:], full[1:]):
        assert torch.equal(a, b)
    assert lean[4].cpu().tolist() == [lean[4][0].item(), 0] and lean[4][0].item() != 0
    w = torch.int16 if wide else torch.int8
    a, b = (t.view(w).view(C * nblk, -1).cpu() for t in (lean[0], full[0]))
    n1 = lean[2].cpu()
    for k in range(C * nblk):
        valid = min(512, V - (k % nblk) * 512)
        one = int(n1[k])
        base = 0
        for n in (valid - one, one):
            for q in range(0, n, 16):
                m = min(16, n - q)
                ga, gb = (t[k, base:base + 128].view(8, 16)[:, :m] for t in (a, b))
                assert torch.equal(ga, gb), (k, q)
                base += 128
