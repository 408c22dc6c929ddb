"""The work this framework is measured on: calls of its public entry points as
programs that keep a compressed KV cache make them.

A case is a dict of plain values.  `kind` names the entry points it calls:

  update    CompressedKVCache.update, the decode step of a model: one new token
            (a few, with speculative decoding) in every layer
  write     codec.encode_batch: a prompt's K and V of one layer (with the
            dequantised rows that go to attention), or a whole cache at once
  read      codec.decode_batch: one chunk or a whole cache back to K / V rows
  wide      codec.encode_batch + decode_batch of heavy-tailed K at low rates,
            whose symbols leave int8
  rotated   encode_rotated + decode_rotated: the long-context path (per-head
            Hadamard rotation, subtractive dither)
  prompt    ResidentKVCache: a prompt's update, then one decode step (update and
            attend)
  attend    resident_decode_attention: a decode step over a long prefix
  fixed     compress_fixed_rate + fused_decompress_chunk: the fixed-rate form
  streams   core.gpu_ans: rans_encode_many + gpu_rans_decode of one chunk's
            coordinate streams on host arrays, as the stand-alone coder is called

Shapes are the Llama-3.1-8B GQA shape (8 kv heads, 32 query heads, head_dim 128)
and the 4-head shape of the variable-rate workload; the drawn cases spread tokens,
heads, chunks, rates and element types over the same ranges.
"""
import math

import numpy as np
import torch

HD = 128
_DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_SIZE = {"fp16": 2, "bf16": 2, "fp32": 4}


def listed():
    return [
        # one generated token: every layer's update of a fresh cache (the smallest calls; launches and host time)
        {"name": "token_update", "kind": "update", "layers": 32, "heads": 8, "tokens": 1, "bits": 4, "dtype": "bf16"},
        # a short chat prompt, one layer's K and V, a length that fills no tile
        {"name": "write_short", "kind": "write", "chunks": 2, "heads": 8, "tokens": 203, "bits": 4, "dtype": "bf16",
         "deq": True},
        # an ordinary prompt, one layer's K and V
        {"name": "write_layer", "kind": "write", "chunks": 2, "heads": 8, "tokens": 4096, "bits": 4, "dtype": "fp16",
         "deq": True},
        # a whole 32-layer cache of 8192 tokens compressed at once (the repository's headline workload)
        {"name": "write_cache", "kind": "write", "chunks": 64, "heads": 8, "tokens": 8192, "bits": 4, "dtype": "fp16",
         "deq": False},
        # one chunk read back, as a cache that decompresses layer by layer does
        {"name": "read_chunk", "kind": "read", "chunks": 1, "heads": 8, "tokens": 2048, "bits": 4, "dtype": "bf16"},
        # a whole 32-layer cache of 8192 tokens read back at once (the headline workload's other direction)
        {"name": "read_cache", "kind": "read", "chunks": 64, "heads": 8, "tokens": 8192, "bits": 4, "dtype": "fp16"},
        # a layer's heavy-tailed K at 3 bits (variable-rate schedules): int16 symbols, alphabets beyond 256
        {"name": "wide_layer", "kind": "wide", "chunks": 2, "heads": 4, "tokens": 16384, "bits": 3, "dtype": "fp16"},
        # rotated and dithered long-context chunk, batch 8, both directions
        {"name": "rotated_chunk", "kind": "rotated", "batch": 8, "heads": 8, "tokens": 4096, "bits": 4,
         "dtype": "fp16"},
        # a prompt into the resident cache of one layer and the first decode step over it
        {"name": "resident_prompt", "kind": "prompt", "heads": 8, "group": 4, "tokens": 2050, "bits": 4,
         "dtype": "fp16"},
        # a decode step over a 32k prefix
        {"name": "attend_long", "kind": "attend", "batch": 1, "heads": 8, "group": 4, "tokens": 32768, "tail": 128,
         "bits": 4},
        # fixed-rate round trip of one layer's K (no entropy coding)
        {"name": "fixed_layer", "kind": "fixed", "heads": 8, "tokens": 2048, "bits": 4, "dtype": "fp16"},
        # one chunk's 16 coordinate streams through the stand-alone coder (a 512-token layer of 8 heads)
        {"name": "coder_streams", "kind": "streams", "streams": 16, "symbols": 32768, "spread": 3.5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["update", "write", "write", "read", "read", "wide", "rotated", "prompt", "attend", "fixed",
                       "streams"])
    heads = rng.choice([2, 4, 8, 8])
    bits = rng.choice([3, 4, 4, 5])
    dtype = rng.choice(["fp16", "bf16"])
    if kind == "update":
        return {"kind": kind, "layers": rng.randint(4, 32), "heads": heads, "tokens": rng.choice([1, 1, 1, 2, 5]),
                "bits": bits, "dtype": dtype}
    if kind in ("write", "read"):
        if kind == "write" and rng.random() < 0.15:
            dtype = "fp32"
        chunks = rng.choice([1, 2, 2, 8, 28, 64])
        tokens = _log(rng, 17, 8192)
        c = {"kind": kind, "chunks": chunks, "heads": heads, "tokens": tokens, "bits": bits, "dtype": dtype}
        if kind == "write":
            c["deq"] = chunks <= 2
        return c
    if kind == "wide":
        return {"kind": kind, "chunks": rng.choice([1, 2, 4]), "heads": rng.choice([4, 8]),
                "tokens": _log(rng, 500, 16384), "bits": 3, "dtype": dtype}
    if kind == "rotated":
        return {"kind": kind, "batch": rng.choice([1, 2, 8]), "heads": heads, "tokens": _log(rng, 100, 8192),
                "bits": bits, "dtype": dtype}
    if kind == "prompt":
        return {"kind": kind, "heads": heads, "group": rng.choice([1, 4, 7]), "tokens": _log(rng, 200, 8192),
                "bits": bits, "dtype": dtype}
    if kind == "attend":
        return {"kind": kind, "batch": rng.choice([1, 1, 2, 4]), "heads": heads, "group": rng.choice([1, 4, 8]),
                "tokens": 16 * _log(rng, 8, 2048), "tail": rng.randint(1, 143), "bits": bits}
    if kind == "fixed":
        return {"kind": kind, "heads": heads, "tokens": _log(rng, 128, 8192), "bits": bits, "dtype": dtype}
    return {"kind": "streams", "streams": rng.choice([1, 8, 16, 32]), "symbols": _log(rng, 500, 32768),
            "spread": rng.uniform(1.0, 12.0)}


# ------------------------------------------------------------------ inputs --

def _kv(shape, seed, dtype, outliers=4, factor=10.0):
    """Rows of K / V (.., heads, tokens, 128): N(0, 1) with a few outlier
    channels per head, as rotary keys show them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for c in range(shape[0]):   # chunk by chunk: no fp32 copy of a whole cache
        t = torch.randn(shape[1:], generator=g, device="cuda")
        if outliers:
            pick = torch.rand(shape[1:-2] + (HD,), generator=g, device="cuda").argsort(-1) < outliers
            t *= torch.where(pick, factor, 1.0)[..., None, :]
        out[c] = t
    return out


def _heavy(shape, seed, dtype):
    """Student-t (3 degrees of freedom) rows with 8 outlier channels x20 per head."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    z = torch.randn(shape, generator=g, device="cuda")
    chi = torch.randn((3,) + shape, generator=g, device="cuda").square_().sum(0)
    t = z / (chi / 3.0).sqrt()
    pick = torch.rand(shape[:-2] + (HD,), generator=g, device="cuda").argsort(-1) < 8
    t *= torch.where(pick, 20.0, 1.0)[..., None, :]
    return t.clamp_(-60000, 60000).to(dtype)


def _write_input(case, seed):
    return _kv((case["chunks"], 1, case["heads"], case["tokens"], HD), seed, _DT[case["dtype"]])


def _attend_inputs(case, seed):
    b, h, t, tail = case["batch"], case["heads"], case["tokens"], case["tail"]
    kv = _kv((2, b, h, t, HD), seed, torch.float16, outliers=0)
    tl = _kv((2, b, h, tail, HD), seed + 1, torch.float16, outliers=0)
    q = _kv((b, h * case["group"], 1, HD), seed + 2, torch.float16, outliers=0)
    return kv, tl, q


def _prompt_inputs(case, seed):
    h, t = case["heads"], case["tokens"]
    dt = _DT[case["dtype"]]
    kv = _kv((2, 1, h, t, HD), seed, dt, outliers=2, factor=4.0)
    new = _kv((2, 1, h, 1, HD), seed + 1, dt, outliers=0)
    q = _kv((1, h * case["group"], 1, HD), seed + 2, dt, outliers=0)
    return kv, new, q


def _stream_symbols(case, seed):
    rng = np.random.default_rng(seed)
    return [np.rint(rng.normal(0.0, case["spread"] * (1.0 + 0.1 * i), case["symbols"])).astype(np.int64)
            for i in range(case["streams"])]


def _arena(case):
    """The bitstream arena a writing program keeps, at its upper bound (cleared,
    so that the words past the bitstreams have a value)."""
    from latticequant_amd import codec
    vectors = case.get("batch", 1) * case["heads"] * case["tokens"] * HD // 8
    return torch.zeros(codec.words_bound(case.get("chunks", 1), vectors), dtype=torch.int32, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "update":
        dt = _DT[case["dtype"]]
        kv = _kv((2 * case["layers"], 1, case["heads"], case["tokens"], HD), seed, dt)
        return {"case": case, "kv": [(kv[2 * i], kv[2 * i + 1]) for i in range(case["layers"])]}
    if kind == "write":
        return {"case": case, "x": _write_input(case, seed), "arena": _arena(case)}
    if kind == "read":
        from latticequant_amd import codec
        enc, _ = codec.encode_batch(_write_input(case, seed), case["bits"])
        return {"case": case, "enc": enc}
    if kind == "wide":
        return {"case": case, "x": _heavy((case["chunks"], 1, case["heads"], case["tokens"], HD), seed,
                                          _DT[case["dtype"]]), "arena": _arena(case)}
    if kind == "rotated":
        from latticequant_amd.llm import rotated
        x = _kv((1, case["batch"], case["heads"], case["tokens"], HD), seed, _DT[case["dtype"]])
        rotated.prepare_signs(x.shape, [3], [0], x.device)
        return {"case": case, "x": x, "arena": _arena(case)}
    if kind == "prompt":
        kv, new, q = _prompt_inputs(case, seed)
        return {"case": case, "kv": kv, "new": new, "q": q}
    if kind == "attend":
        from latticequant_amd import codec
        from latticequant_amd.llm import resident
        kv, tl, q = _attend_inputs(case, seed)
        res = []
        for i in range(2):
            enc, _ = codec.encode_batch(kv[i][None], case["bits"])
            res.append(resident.from_chunk(kv[i], enc))
        work = resident.attn_workspace(case["batch"] * case["heads"], case["group"], case["tokens"], case["tail"],
                                       device=q.device)
        return {"case": case, "k": res[0], "v": res[1], "q": q, "tail": tl, "work": work}
    if kind == "fixed":
        return {"case": case, "x": _kv((1, case["heads"], case["tokens"], HD), seed, _DT[case["dtype"]], outliers=0)}
    from latticequant_amd.core import gpu_ans
    syms = _stream_symbols(case, seed)
    counts, alphabets = [], []
    for s in syms:   # the alphabet of a chunk's stream: min - 2 .. max + 2
        lo, hi = int(s.min()) - 2, int(s.max()) + 2
        alphabets.append(list(range(lo, hi + 1)))
        counts.append(np.bincount(s - lo, minlength=hi - lo + 1).astype(np.int64))
    return {"case": case, "syms": syms, "tables": gpu_ans.build_rans_tables(counts, alphabets)}


# -------------------------------------------------------------------- pass --

def _batch_outputs(enc, deq=None):
    """The compressed form: every field but the tables, whose unused entries
    are not defined (the bitstreams depend on every used one)."""
    out = {"words": enc.words, "scale32": enc.scale32, "scale16": enc.scale16, "coset_bits": enc.coset_bits,
           "blk_n1": enc.blk_n1, "blk_off": enc.blk_off, "blk_state": enc.blk_state, "nbits": enc.stream_nbits,
           "state": enc.stream_state, "woff": enc.stream_woff, "chunk_words": enc.chunk_words}
    if deq is not None:
        out["deq"] = deq
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "update":
        from latticequant_amd.llm.compressed_kv_cache import CompressedKVCache
        cache = CompressedKVCache(case["bits"])
        return [cache.update(k, v, i) for i, (k, v) in enumerate(state["kv"])]
    if kind == "write":
        from latticequant_amd import codec
        return _batch_outputs(*codec.encode_batch(state["x"], case["bits"], deq_out=case["deq"],
                                                  words_out=state["arena"]))
    if kind == "read":
        from latticequant_amd import codec
        return codec.decode_batch(state["enc"], out_dtype=_DT[case["dtype"]])
    if kind == "wide":
        from latticequant_amd import codec
        enc, _ = codec.encode_batch(state["x"], case["bits"], words_out=state["arena"])
        return {**_batch_outputs(enc), "rows": codec.decode_batch(enc, out_dtype=state["x"].dtype)}
    if kind == "rotated":
        from latticequant_amd.llm import rotated
        enc, _ = rotated.encode_rotated(state["x"], case["bits"], [3], [0], words_out=state["arena"])
        return {**_batch_outputs(enc), "rows": rotated.decode_rotated(enc, out_dtype=state["x"].dtype)}
    if kind == "prompt":
        from latticequant_amd.llm.resident_cache import ResidentKVCache
        cache = ResidentKVCache(case["bits"])
        k, v = cache.update(state["kv"][0], state["kv"][1], 0)
        cache.update(state["new"][0], state["new"][1], 0)
        return {"k": k, "v": v, "out": cache.attend(0, state["q"])}
    if kind == "attend":
        from latticequant_amd.llm import resident
        return resident.resident_decode_attention(state["k"], state["v"], state["q"], state["tail"][0],
                                                  state["tail"][1], work=state["work"])
    if kind == "fixed":
        from latticequant_amd.llm.compressed_kv_cache import compress_fixed_rate
        from latticequant_amd.llm.fused_triton_merge import fused_decompress_chunk
        # the packed and fallback rows, whose number depends on the values, come back as the rows merged from them
        ch = compress_fixed_rate(state["x"], case["bits"])
        return {"mask": ch.repr_mask, "scales": ch.scales, "rows": fused_decompress_chunk(ch)}
    from latticequant_amd.core import gpu_ans
    enc = gpu_ans.rans_encode_many(state["syms"], state["tables"])
    streams = [gpu_ans.RANSStream(bitstream=w, n_bits=nb, initial_state=st, n_symbols=len(s), table=t)
               for (w, st, nb), s, t in zip(enc, state["syms"], state["tables"])]
    # the words, whose number depends on the values, come back as the symbols decoded from all of them
    return {"state": np.array([e[1] for e in enc]), "bits": np.array([e[2] for e in enc]),
            "symbols": gpu_ans.gpu_rans_decode(streams)}


# ------------------------------------------------------------------- floor --

# operations of one 8-dim vector: two roundings of D8 (8 rounds, 8 differences,
# 8 costs, 8 sums, 8 compares each), the choice and the scaling; one rANS step
# (a few integer operations) per coordinate
_QUANT = 100
_CODE = 8 * 6


def work(case):
    kind = case["kind"]
    if kind == "streams":
        n = case["streams"] * case["symbols"]
        bits = max(1.0, math.log2(case["spread"] * 4.13))   # entropy of a rounded normal
        return {"bytes": n * 8 + n * bits / 8 * 2 + n * 8, "flops": 2 * n * 6}
    el = _SIZE.get(case.get("dtype"), 2)
    rows = case["heads"] * case["tokens"] * case.get("chunks", 1) * case.get("batch", 1)
    n = rows * HD
    comp = n * (case["bits"] - 0.5) / 8        # bitstream and side information
    if kind == "update":
        n *= 2 * case["layers"]
        return {"bytes": 2 * n * el, "flops": n // 8 * _QUANT}
    if kind == "write":
        return {"bytes": n * el * (2 if case["deq"] else 1) + comp, "flops": n // 8 * (_QUANT + _CODE)}
    if kind == "read":
        return {"bytes": n * el + comp, "flops": n // 8 * (_CODE + 8)}
    if kind in ("wide", "rotated"):
        rot = n * 14 * 2 if kind == "rotated" else 0
        return {"bytes": 2 * n * el + 2 * comp, "flops": n // 8 * (_QUANT + 2 * _CODE + 8) + rot}
    if kind == "prompt":
        qh = case["heads"] * case["group"]
        return {"bytes": 4 * n * el + 2 * comp + 2 * n * 5 // 8,
                "flops": 2 * n // 8 * (_QUANT + _CODE) + 4 * qh * case["tokens"] * HD}
    if kind == "attend":
        qh = case["heads"] * case["batch"] * case["group"]
        tail = 2 * case["batch"] * case["heads"] * case["tail"] * HD * 2
        return {"bytes": 2 * n * case["bits"] // 8 + tail + 4 * qh * HD,
                "flops": 4 * qh * (case["tokens"] + case["tail"]) * HD}
    return {"bytes": 2 * n * el + 2 * n * case["bits"] // 8, "flops": n // 8 * (_QUANT + 30)}


def tolerance(case):
    """Lattice points, bitstreams and the rows rounded from them have one right
    value; attention sums in another order and rounds its probabilities."""
    if case["kind"] in ("attend", "prompt"):
        return {"rel": 2e-3}
    return "exact"


# ------------------------------------------------------- 64-bit reference --

def _d8(x):
    r = x.round()
    e = x - r
    odd = (r.sum(-1) % 2).abs() > 0.5
    j = e.abs().argmax(-1, keepdim=True)
    step = torch.where(e.gather(-1, j) < 0, -1.0, 1.0).to(x.dtype)
    return r.scatter_add(-1, j, step * odd[..., None])


def _e8(x):
    a = _d8(x)
    b = _d8(x - 0.5) + 0.5
    near = (x - a).square().sum(-1) <= (x - b).square().sum(-1)
    return torch.where(near[..., None], a, b)


def _points(x, bits):
    """(lattice points, scale32, scale16) of (.., heads, tokens, 128) rows, one
    scale per head, in 64 bits (the scales as they are stored)."""
    shp = x.shape
    v = x.double().reshape(shp[:-2] + (-1, 8))
    s = (2 * math.pi * math.e * v.square().mean((-1, -2)) * 4.0 ** -bits).sqrt()
    s32 = s.float().double()[..., None, None]
    return _e8(v / s32).reshape(shp), s32, s32.half().double()


def _attention(q, k, v, group):
    """q (b, hq, 1, 128), k / v (b, h, t, 128), in 64 bits."""
    b, hq = q.shape[:2]
    qq = q.double().reshape(b, hq // group, group, HD)
    p = torch.matmul(qq, k.double().transpose(-1, -2).contiguous()) / math.sqrt(HD)
    return torch.matmul(p.softmax(-1), v.double()).reshape(b, hq, 1, HD)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("write", "read"):
        if case["chunks"] * case["heads"] * case["tokens"] > 1 << 18:
            return None                              # a whole cache: minutes in 64 bits
        x = _write_input(case, seed)
        q, s32, s16 = _points(x, case["bits"])
        if kind == "read":
            return q * s16
        out = dict.fromkeys(("words", "scale32", "scale16", "coset_bits", "blk_n1", "blk_off", "blk_state", "nbits",
                             "state", "woff", "chunk_words"))
        out["scale32"] = s32.reshape(-1)
        if case["deq"]:
            out["deq"] = q * s32
        return out
    if kind == "update":
        st = prepare(case, seed)
        res = []
        for k, v in st["kv"]:
            pair = []
            for x in (k, v):
                q, s32, _ = _points(x, case["bits"])
                pair.append(q * s32)
            res.append(tuple(pair))
        return res
    if kind == "attend":
        kv, tl, q = _attend_inputs(case, seed)
        rows = []
        for i in range(2):
            p, _, s16 = _points(kv[i], case["bits"])
            rows.append(torch.cat([(p * s16).half(), tl[i]], 2))
        return _attention(q, rows[0], rows[1], case["group"])
    if kind == "prompt":
        kv, new, q = _prompt_inputs(case, seed)
        n = max(case["tokens"] - 128, 0) // 16 * 16     # tokens past the fp16 tail, in blocks of 16
        rows, att = [], []
        for i in range(2):
            x = kv[i]
            pre = x[:, :, :0]
            if n:
                p, _, s16 = _points(x[:, :, :n], case["bits"])
                pre = p * s16
            rows.append(torch.cat([pre.double(), x[:, :, n:].double()], 2))
            # the step's flush (16 more tokens once the tail is 16 over) has its own scales
            t = torch.cat([x[:, :, n:], new[i]], 2)
            m = (t.shape[2] - 128) // 16 * 16 if t.shape[2] >= 144 else 0
            mid = t[:, :, :0]
            if m:
                p, _, s16 = _points(t[:, :, :m], case["bits"])
                mid = (p * s16).half()
            att.append(torch.cat([pre.half(), mid.half(), t[:, :, m:].half()], 2))
        return {"k": rows[0], "v": rows[1], "out": _attention(q.half(), att[0], att[1], case["group"])}
    if kind == "fixed":
        q, _, s16 = _points(_kv((1, case["heads"], case["tokens"], HD), seed, _DT[case["dtype"]], outliers=0),
                            case["bits"])
        return {"mask": None, "scales": s16.reshape(-1), "rows": q * s16}
    return None     # bitstreams and symbols: whole numbers, compared exactly
