"""The work a user of the KV codec has it do, as cases that can be timed and compared.

Seven kinds of call, each over the ranges that a decode server or a prefill meets:

  hook          sp_hip_roundtrip_cells: the post-decode hook over the cells a step wrote
  ship_attn     sp_hip_attn_decode / sp_hip_attn_decode_seqs over ship records
  ship_codec    sp_hip_write_* then sp_hip_read_* of the ship cache
  sqfree_attn   sp_hip_sqfree_attn_decode(_seqs)
  sqfree_codec  sp_hip_sqfree_write_layer then sp_hip_sqfree_read_layer
  hier_attn     sp_hip_hier_attn_decode(_seqs)
  hier_codec    sp_hip_hier_write_layer then sp_hip_hier_read_layer

`exact` restates the record formats in plain torch (the codec's float32 steps one
rounding each, as the format defines them) and takes everything after the records in
64 bits.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "shannon-prime-llama_amd"))
import sp_hip as S  # noqa: E402

HIER_SK, HIER_BITS, HIER_RBITS = 30, (5, 5), 2
SQ_BITS, SQ_RBITS = (5, 4, 4, 4, 5), 3


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one decoded token's K and V through the post-decode hook, V transposed as
        # llama.cpp keeps it: the smallest call, once per layer and token
        dict(name="hook_token_hd128", kind="hook", hd=128, heads=8, cells=1, v_trans=True, dtype="f16"),
        # a decode step of an 8B-shaped model at 32K: every one of its 32 layers
        dict(name="decode_hd128_32k", kind="ship_attn", hd=128, bands="bridge", heads=8, n_q=32, n_seq=1, ctx=32768,
             ragged=False, layers=32, want="out"),
        # a serving step: 12 chats of unequal length in one unified cache (one layer pair)
        dict(name="decode_hd128_batch", kind="ship_attn", hd=128, bands="bridge", heads=8, n_q=32, n_seq=12, ctx=4500,
             ragged=True, layers=2, want="out"),
        # the MHA, head_dim 96 configuration: 16 concurrent sequences of 4096
        dict(name="decode_hd96_batch", kind="ship_attn", hd=96, bands="bridge", heads=32, n_q=32, n_seq=16, ctx=4096,
             ragged=False, layers=2, want="out"),
        # a 1B-shaped model (head_dim 64, the bridge's bands for it) at the 4096 positions
        # the reference quotes its fused op on
        dict(name="decode_hd64_4k", kind="ship_attn", hd=64, bands="bridge", heads=8, n_q=32, n_seq=1, ctx=4096,
             ragged=False, layers=4, want="out"),
        # head_dim 256 on the ship path, an odd context
        dict(name="decode_hd256_8k", kind="ship_attn", hd=256, bands="bridge", heads=8, n_q=16, n_seq=1, ctx=8191,
             ragged=False, layers=2, want="out"),
        # bulk prefill compression and reconstruction, the headline workload
        dict(name="bulk_hd128", kind="ship_codec", hd=128, bands="bridge", heads=8, layers=32, n_tok=32768, start=0,
             dtype="f16", via="all"),
        # a prompt chunk of a head_dim 64 model through the layer calls, float32 rows
        dict(name="chunk_hd64_f32", kind="ship_codec", hd=64, bands="bridge", heads=8, layers=4, n_tok=1999, start=777,
             dtype="f32", via="layer"),
        # the aggressive path's prefill and its reconstruction, a 16K prompt of one layer
        dict(name="sqfree_chunk", kind="sqfree_codec", sk=115, v_one=True, heads=4, layers=1, n_tok=16384, start=0,
             dtype="f16"),
        # its decode step at batch 4
        dict(name="sqfree_decode_batch", kind="sqfree_attn", sk=115, v_one=True, heads=4, n_q=32, n_seq=4, ctx=16384,
             ragged=False, layers=2, want="out"),
        # a 2048-token prefill chunk through the hierarchical path
        dict(name="hier_chunk", kind="hier_codec", heads=8, layers=1, n_tok=2048, start=4096, dtype="f16"),
        # the long-context decode step: 8 sequences of 128K
        dict(name="hier_decode_batch", kind="hier_attn", heads=8, n_q=16, n_seq=8, ctx=131072, ragged=False, layers=1,
             want="out"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _attn_shape(rng, most, heads, longest):
    """Sequences and context so that n_seq * ctx stays within `most` positions per KV head."""
    n_seq = rng.choice([1, 1, 2, 3, 5, 8, 13, 16])
    ctx = _log(rng, 100, max(101, min(longest, most // (n_seq * heads))))
    return dict(n_seq=n_seq, ctx=ctx, ragged=rng.random() < 0.7, layers=rng.choice([1, 2]),
                want=rng.choice(["out", "out", "out", "both", "scores"]))


def draw(rng):
    kind = rng.choice(["hook", "ship_attn", "ship_attn", "ship_codec", "ship_codec", "sqfree_attn", "sqfree_codec",
                       "hier_attn", "hier_codec"])
    dtype = rng.choice(["f16", "f16", "f32"])
    if kind == "hook":
        hd = rng.choice([64, 128, 128, 256])
        return dict(kind=kind, hd=hd, heads=rng.choice([4, 8]), cells=_log(rng, 1, 1600), v_trans=rng.random() < 0.6,
                    dtype=dtype)
    if kind == "ship_attn":
        hd, bands = rng.choice([(64, "bridge"), (64, "ship"), (96, "bridge"), (128, "bridge"), (128, "bridge"),
                                (256, "bridge")])
        heads = rng.choice([2, 4, 8, 8, 16] if hd != 96 else [8, 32])
        g = rng.choice([1, 2, 3, 4, 4, 8]) if hd != 96 else rng.choice([1, 1, 4])
        c = dict(kind=kind, hd=hd, bands=bands, heads=heads, n_q=heads * g)
        c.update(_attn_shape(rng, 1 << 19, heads, 60000))
        return c
    if kind == "ship_codec":
        hd, bands = rng.choice([(64, "bridge"), (64, "ship"), (96, "bridge"), (128, "bridge"), (256, "bridge")])
        heads, layers = rng.choice([2, 4, 8, 32]), rng.choice([1, 2, 4])
        return dict(kind=kind, hd=hd, bands=bands, heads=heads, layers=layers, n_tok=_log(rng, 1, 8192),
                    start=rng.choice([0, 0, 1, 129, 1000]), dtype=dtype, via=rng.choice(["all", "layer"]))
    if kind in ("sqfree_attn", "sqfree_codec"):
        sk, v_one = rng.choice([(115, True), (115, True), (115, False), (77, False)])
        c = dict(kind=kind, sk=sk, v_one=v_one)
        if kind == "sqfree_codec":
            c.update(heads=rng.choice([2, 4, 8]), layers=1, n_tok=_log(rng, 1, 16384), start=rng.choice([0, 1, 1000]),
                     dtype=dtype)
        else:
            heads = rng.choice([2, 4, 8])
            c.update(heads=heads, n_q=heads * rng.choice([1, 3, 4, 8, 8]))
            c.update(_attn_shape(rng, 1 << 18, heads, 40000))
        return c
    if kind == "hier_codec":
        return dict(kind=kind, heads=rng.choice([1, 4, 8]), layers=1, n_tok=_log(rng, 1, 4096),
                    start=rng.choice([0, 1, 4096]), dtype=dtype)
    heads = rng.choice([1, 4, 8])
    c = dict(kind=kind, heads=heads, n_q=heads * rng.choice([1, 2, 2, 4, 8]))
    c.update(_attn_shape(rng, 1 << 21, heads, 131072))
    return c


# ---------------------------------------------------------------------------
# shapes
# ---------------------------------------------------------------------------

def _spans(n, nb):
    size = n // nb
    return [(b * size, n - b * size if b == nb - 1 else size) for b in range(nb)]


def _band_bytes(n, bits):
    return sum(2 + (sz * b + 7) // 8 for (_, sz), b in zip(_spans(n, len(bits)), bits))


def _ship_bits(case):
    """The bridge's default bands by head_dim; "ship" is 5/5/4/3 and 3 at any width."""
    if case["hd"] >= 128 or case.get("bands") == "ship":
        return (5, 5, 4, 3), (3,)
    return (5, 4, 4), (5,)


def _hd(case):
    return 128 if case["kind"].startswith("sqfree") else 256 if case["kind"].startswith("hier") else case["hd"]


def _record_bytes(case):
    kind = case["kind"]
    if kind.startswith("sqfree"):
        nr = 154 - case["sk"]
        tail = 4 + (nr * SQ_RBITS + 7) // 8 + (nr + 7) // 8
        return _band_bytes(case["sk"], SQ_BITS) + tail, _band_bytes(case["sk"], (3,) if case["v_one"] else SQ_BITS) + tail
    if kind.startswith("hier"):
        b = _band_bytes(HIER_SK, HIER_BITS) + 4 + 300 * HIER_RBITS // 8
        return b, b
    kb, vb = ((5, 5, 4, 3), (3,)) if kind == "hook" else _ship_bits(case)
    return _band_bytes(case["hd"], kb), _band_bytes(case["hd"], vb)


def _sequences(case):
    """Starts and lengths of an attention case: equal sequences end to end, or ragged ones
    (down to a quarter of ctx) at whatever cells the unified cache had free."""
    n, ctx = case["n_seq"], case["ctx"]
    if not case["ragged"]:
        return [i * ctx for i in range(n)], [ctx] * n
    starts, lens, at = [], [], 3
    for i in range(n):
        lens.append(max(1, ctx - ((i * 5) % n) * 3 * ctx // (4 * n) - i))
        starts.append(at)
        at += lens[-1] + 7 + 2 * i
    return starts, lens


def _max_seq(case):
    """Cells of the cache: llama.cpp pads its KV size to a multiple of 256."""
    if "ctx" in case:
        starts, lens = _sequences(case)
        n = starts[-1] + lens[-1]
    elif case["kind"] == "hook":
        n = 3_900_000 // (case["heads"] * case["hd"]) - 255  # the tensors come back whole
    else:
        n = case["start"] + case["n_tok"]
    return (n + 255) // 256 * 256


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _rope(x, pos):
    """x [positions, heads, hd] rotated pairwise (i, i + hd/2), theta 500000."""
    half = x.shape[-1] // 2
    inv = 500000.0 ** (-torch.arange(half, device="cuda", dtype=torch.float64) * 2.0 / x.shape[-1])
    ang = pos.double()[:, None] * inv[None, :]
    c, s = torch.cos(ang).float()[:, None, :], torch.sin(ang).float()[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], dim=-1)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _kv_rows(case, seed, layer, n):
    """K and V rows [n, heads, hd] of one layer: N(0,1) with rotary positions for K on the
    ship path (a per-channel log-normal scale at head_dim 96), heavy-tailed outlier
    channels on the aggressive path, N(0,1) at head_dim 256's hierarchical path."""
    g = _generator(seed * 1009 + layer)
    heads, hd = case["heads"], _hd(case)
    dt = torch.float32 if case.get("dtype") == "f32" else torch.float16
    out = []
    for is_v in (0, 1):
        x = torch.empty((n, heads, hd), dtype=dt, device="cuda")
        chan = torch.exp(0.5 * torch.randn((1, heads, hd), generator=g, device="cuda")) if hd == 96 else None
        outlier = torch.randint(hd, (heads, 4), generator=g, device="cuda")
        for r0 in range(0, n, 1 << 17):
            m = min(1 << 17, n - r0)
            y = torch.randn((m, heads, hd), generator=g, device="cuda")
            if chan is not None:
                y = y * chan
            elif case["kind"].startswith("sqfree"):
                t = torch.randn((m, heads, 4), generator=g, device="cuda")
                chi = torch.randn((m, heads, 4, 4), generator=g, device="cuda").square().sum(-1)
                y.scatter_(2, outlier[None].expand(m, -1, -1), 3.0 * t / torch.sqrt(chi / 4.0))
            elif not is_v and not case["kind"].startswith("hier"):
                y = _rope(y, torch.arange(r0, r0 + m, device="cuda"))
            x[r0:r0 + m] = y.to(dt)
        out.append(x)
    return out


def _queries(case, seed, layer):
    g = _generator(seed * 1009 + 500 + layer)
    return torch.randn((case["n_seq"], case["n_q"], _hd(case)), generator=g, device="cuda")


def _predictors(case, seed):
    """One fp16 predictor [300, 30] per (layer, head), as a calibrated model loads them."""
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((case["layers"] * case["heads"], 300, HIER_SK)) * 0.05).astype(np.float16)


def _cells(case, seed):
    """The cells a step wrote: scattered over the unified cache, each once."""
    g = _generator(seed * 1009 + 900)
    return torch.randperm(_max_seq(case), generator=g, device="cuda")[:case["cells"]].to(torch.int32)


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

class _Memory:
    """Device memory as an array that torch can look at."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "|u1", "data": (ptr, False), "version": 3}


def _records(cache, ptr, shape):
    """A cache's records as a tensor over its own memory, which the tensor keeps alive."""
    t = torch.as_tensor(_Memory(ptr, shape), device="cuda")
    if t.data_ptr() != ptr:
        raise RuntimeError("the records were copied")
    t.cache = cache
    return t


def _p(t):
    return C.c_void_p(t.data_ptr())


def _ints(v):
    return (C.c_int * len(v))(*v)


def _cache(case, seed, max_seq, layers):
    stream = torch.cuda.current_stream().cuda_stream
    kind, heads, hd = case["kind"], case["heads"], _hd(case)
    if kind.startswith("sqfree"):
        cfg = S.config(hd, layers, heads, k_bits=SQ_BITS, v_bits=(3,) if case["v_one"] else SQ_BITS)
        return S.SqfreeCache(cfg, max_seq, rbits=SQ_RBITS, spinor=True, sk_k=case["sk"], stream=stream)
    if kind.startswith("hier"):
        order = _squarefree_first(330)
        cache = S.HierCache(S.config(hd, layers, heads), 330, order[:HIER_SK], order[HIER_SK:],
                            S.band_config(HIER_SK, HIER_BITS), HIER_RBITS, max_seq, layers * heads, stream=stream)
        cache.upload_W(_predictors(case, seed).view(np.uint16))
        return cache
    kb, vb = ((5, 5, 4, 3), (3,)) if kind == "hook" else _ship_bits(case)
    return S.ShipCache(S.config(hd, layers, heads, k_bits=kb, v_bits=vb), max_seq, stream)


def prepare(case, seed):
    L, kind = S.lib(), case["kind"]
    heads, hd, ms = case["heads"], _hd(case), _max_seq(case)
    layers = case.get("layers", 1)
    cache = _cache(case, seed, ms, layers)
    dt = S.DTYPE_F32 if case.get("dtype") == "f32" else S.DTYPE_F16
    st = dict(cache=cache, calls=[])  # calls: (function, arguments) of one pass; out: what it returns
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    row = heads * hd
    kB, vB = _record_bytes(case)
    if kind.endswith("attn"):
        write = {"ship_attn": L.sp_hip_write_layer, "sqfree_attn": L.sp_hip_sqfree_write_layer,
                 "hier_attn": L.sp_hip_hier_write_layer}[kind]
        one = {"ship_attn": L.sp_hip_attn_decode, "sqfree_attn": L.sp_hip_sqfree_attn_decode,
               "hier_attn": L.sp_hip_hier_attn_decode}[kind]
        many = {"ship_attn": L.sp_hip_attn_decode_seqs, "sqfree_attn": L.sp_hip_sqfree_attn_decode_seqs,
                "hier_attn": L.sp_hip_hier_attn_decode_seqs}[kind]
        starts, lens = _sequences(case)
        n_q, scale = case["n_q"], C.c_float(1.0 / math.sqrt(hd))
        st["q"] = [_queries(case, seed, i) for i in range(layers)]
        st["keep"] = a, b = _ints(starts), _ints(lens)
        st["out"] = {}
        if case["want"] != "scores":
            st["out"]["out"] = [torch.zeros_like(q) for q in st["q"]]
        if case["want"] != "out":
            st["out"]["scores"] = [torch.zeros(n_q * sum(lens), device="cuda") for _ in range(layers)]
        for i in range(layers):
            k, v = _kv_rows(case, seed, i, ms)
            S.check(write(cache.ref, i, 0, ms, _p(k), _p(v), row, S.DTYPE_F16), "write")
            sc = _p(st["out"]["scores"][i]) if "scores" in st["out"] else None
            o = _p(st["out"]["out"][i]) if "out" in st["out"] else None
            if case["n_seq"] == 1 and starts[0] == 0:
                st["calls"].append((one, (cache.ref, i, lens[0], _p(st["q"][i]), n_q, scale, sc, o, stream)))
            else:
                st["calls"].append((many, (cache.ref, i, case["n_seq"], C.cast(a, C.c_void_p), C.cast(b, C.c_void_p),
                                           _p(st["q"][i]), n_q, scale, sc, o, stream)))
            torch.cuda.synchronize()  # k and v are given back
        return st
    shape = (layers * heads, ms)
    rec = [_records(cache, cache.c.d_k_cache, shape + (kB,)), _records(cache, cache.c.d_v_cache, shape + (vB,))]
    if kind == "hook":
        k, v = _kv_rows(case, seed, 0, ms)
        k, v = k.view(ms, row), v.view(ms, row)
        v = v.t().contiguous() if case["v_trans"] else v
        st["cells"] = cells = _cells(case, seed)
        vs = (1, ms) if case["v_trans"] else (row, 1)
        st["calls"].append((L.sp_hip_roundtrip_cells, (cache.ref, 0, _p(cells), len(cells), _p(k), row, _p(v), vs[0],
                                                       vs[1], dt, -1, stream)))
        st["out"] = {"k": k, "v": v, "records": rec}
        return st
    n, p0 = case["n_tok"], case["start"]
    rows = [_kv_rows(case, seed, i, n) for i in range(layers)]
    if kind == "ship_codec" and case["via"] == "all":
        src = [torch.stack([r[j].transpose(0, 1) for r in rows]).contiguous() for j in (0, 1)]
        dst = [torch.zeros_like(t) for t in src]
        st["src"] = src
        st["calls"] += [(L.sp_hip_write_all, (cache.ref, p0, n, _p(src[0]), _p(src[1]), dt)),
                        (L.sp_hip_read_all, (cache.ref, p0, n, _p(dst[0]), _p(dst[1]), dt, -1))]
    else:
        write, read = {"ship_codec": (L.sp_hip_write_layer, L.sp_hip_read_layer),
                       "sqfree_codec": (L.sp_hip_sqfree_write_layer, L.sp_hip_sqfree_read_layer),
                       "hier_codec": (L.sp_hip_hier_write_layer, L.sp_hip_hier_read_layer)}[kind]
        dst = [[torch.zeros_like(t) for t in r] for r in rows]
        st["src"] = rows
        more = (-1,) if kind == "ship_codec" else ()
        st["calls"] += [(write, (cache.ref, i, p0, n, _p(r[0]), _p(r[1]), row, dt)) for i, r in enumerate(rows)]
        st["calls"] += [(read, (cache.ref, i, p0, n, _p(r[0]), _p(r[1]), row, dt) + more) for i, r in enumerate(dst)]
    st["out"] = {"rows": dst, "records": rec}
    return st


def run(st):
    for fn, args in st["calls"]:
        if fn(*args) != 0:
            raise RuntimeError(S.last_error())
    return st["out"]


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def work(case):
    heads, hd, layers = case["heads"], _hd(case), case.get("layers", 1)
    kB, vB = _record_bytes(case)
    if case["kind"].endswith("attn"):
        lens = _sequences(case)[1]
        pos, q = sum(lens), case["n_seq"] * case["n_q"] * hd
        out, sc = case["want"] != "scores", case["want"] != "out"
        b = heads * pos * (kB + (vB if out else 0)) + 4 * q * (2 if out else 1) + (4 * case["n_q"] * pos if sc else 0)
        return {"bytes": layers * b, "flops": layers * 2 * case["n_q"] * pos * hd * (2 if out else 1)}
    es = 4 if case["dtype"] == "f32" else 2
    n = layers * heads * (case["cells"] if case["kind"] == "hook" else case["n_tok"])
    # each vector read, its record written, and the way back (the hook keeps the record at hand)
    b = n * (4 * hd * es + (1 if case["kind"] == "hook" else 2) * (kB + vB))
    f = n * 4 * hd * math.log2(hd) + (n * 4 * 300 * HIER_SK * 2 if case["kind"].startswith("hier") else 0)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # records and reconstructions are defined bit for bit; attention sums in 32 bits
    # (up to 7e-7 from the 64-bit result, measured; this is about four times that, and
    # "max" the like for single entries)
    if case["kind"].endswith("attn"):
        return {"rel": 3e-6, "max": 5e-5}
    return "exact"


# ---------------------------------------------------------------------------
# the formats in plain torch
# ---------------------------------------------------------------------------

def _squarefree_first(n):
    sf = [all((i + 1) % (d * d) for d in range(2, int(math.isqrt(i + 1)) + 1)) for i in range(n)]
    return [i for i in range(n) if sf[i]] + [i for i in range(n) if not sf[i]]


def _transform(x):
    """The Vilenkin-Hartley transform of the rows of x, in x's own type, one rounding a step."""
    n, stride, f32 = x.shape[-1], 1, x.dtype == torch.float32
    num = (lambda v: float(np.float32(v))) if f32 else float
    root = (lambda v: float(np.float32(1.0) / np.sqrt(np.float32(v)))) if f32 else (lambda v: 1.0 / math.sqrt(v))
    pow2, m = n & (n - 1) == 0, n
    for p in (2, 3, 5, 7, 11):
        while m % p == 0:
            g = x.reshape(-1, n // (stride * p), p, stride)
            out = torch.empty_like(g)
            for k in range(p):
                if pow2:
                    out[:, :, k] = g[:, :, 0] + g[:, :, 1] if k == 0 else g[:, :, 0] - g[:, :, 1]
                    continue
                acc = torch.zeros_like(g[:, :, 0])
                for j in range(p):
                    a = 2.0 * math.pi * ((k * j) % p) / p
                    acc = acc + num(math.cos(a) + math.sin(a)) * g[:, :, j]
                out[:, :, k] = acc * root(p)
            x, stride, m = out.reshape(-1, n), stride * p, m // p
    return x * root(n) if pow2 else x


def _over(x, v):
    """x / v, rounded once (a plain number on the right would become a product)."""
    return x / torch.full((1,), v, dtype=x.dtype, device=x.device)


def _tree_sum(x):
    """Row sums in the 256-slot order of the format's reductions."""
    s = torch.zeros((x.shape[0], 256), device=x.device)
    for i in range(0, x.shape[1], 256):
        part = x[:, i:i + 256]
        s[:, :part.shape[1]] += part
    h = 128
    while h:
        s = s[:, :h] + s[:, h:2 * h]
        h //= 2
    return s[:, :1]


def _bands(x, bits):
    """What the band quantizer keeps of the rows of x: (code * stored scale) in 64 bits."""
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    for (off, sz), b in zip(_spans(x.shape[1], len(bits)), bits):
        band, top = x[:, off:off + sz], float((1 << (b - 1)) - 1)
        ss = _over(band.abs().amax(1, keepdim=True), top).half().float()
        inv = torch.where(ss > 0, torch.ones_like(ss) / ss, torch.zeros_like(ss))
        out[:, off:off + sz] = torch.round(band * inv).clamp(-top, top).double() * ss.double()
    return out


def _residual(dev, bits, hier):
    """What the residual quantizer keeps of the rows of dev, in 64 bits."""
    mag = _over(_tree_sum(dev.abs()), float(dev.shape[1])).clamp_min(1e-12)
    levels = 1 << bits
    step = _over(2.0 * (mag if hier else mag * float(bits)), float(levels - 1))
    at = dev * (torch.ones_like(step) / step) + 0.5 * (levels - 1)
    lv = (torch.round(at) if hier else torch.trunc(at + 0.5)).clamp(0, levels - 1)
    return (lv.double() - 0.5 * (levels - 1)) * step.double()


def _mobius(n):
    out, d = 1, 2
    while n > 1:
        if n % d == 0:
            n //= d
            if n % d == 0:
                return 0
            out = -out
        d += 1
    return out


def _coefficients(case, x, is_v, W):
    """The transform coefficients (64 bits) that the records of rows x [n, hd] stand for."""
    hd = x.shape[1]
    x = x.float()
    if not case["kind"].startswith(("sqfree", "hier")):
        kb, vb = ((5, 5, 4, 3), (3,)) if case["kind"] == "hook" else _ship_bits(case)
        c = _transform(x)
        if is_v:
            return _bands(c, vb)
        order = torch.tensor(_squarefree_first(hd), device=x.device)
        out = torch.empty(c.shape, dtype=torch.float64, device=x.device)
        out[:, order] = _bands(c[:, order], kb)
        return out
    hier = case["kind"].startswith("hier")
    pad = 330 if hier else 154
    c = _transform(torch.cat([x, _over(_tree_sum(x), float(hd)).expand(-1, pad - hd)], 1))
    order = _squarefree_first(pad)
    sk = HIER_SK if hier else case["sk"]
    skel, rest = torch.tensor(order[:sk], device=x.device), torch.tensor(order[sk:], device=x.device)
    bits = HIER_BITS if hier else (3,) if is_v and case["v_one"] else SQ_BITS
    s32 = c[:, skel]
    s64 = _bands(s32, bits)
    out = torch.empty(c.shape, dtype=torch.float64, device=x.device)
    out[:, skel] = s64
    if hier:
        w = torch.from_numpy(W).to(x.device)
        pred = torch.zeros((x.shape[0], len(rest)), device=x.device)
        for s in range(sk):
            pred = pred + w[:, s].float() * s32[:, s:s + 1]
        out[:, rest] = s64 @ w.double().t().contiguous() + _residual(c[:, rest] - pred, HIER_RBITS, True)
        return out
    slot = {c_: i for i, c_ in enumerate(order[:sk])}
    M = torch.zeros((sk, len(rest)), dtype=torch.float64, device=x.device)
    pred = torch.zeros((x.shape[0], len(rest)), device=x.device)
    for r, c_ in enumerate(order[sk:]):
        for d in range(1, c_ + 1):
            if (c_ + 1) % d == 0 and d - 1 in slot and _mobius((c_ + 1) // d):
                M[slot[d - 1], r] = _mobius((c_ + 1) // d)
                pred[:, r] = pred[:, r] + float(_mobius((c_ + 1) // d)) * s32[:, slot[d - 1]]
    a = c[:, rest]
    flip = (a + pred).abs() < (a - pred).abs()
    dev = torch.where(flip, a + pred, a - pred)
    p64 = s64 @ M
    out[:, rest] = torch.where(flip, -p64, p64) + _residual(dev, SQ_RBITS, False)
    return out


def _rebuilt(case, x, is_v, W):
    """The rows that reading the records of rows x back gives, in 64 bits."""
    c = _coefficients(case, x, is_v, W)
    T = _transform(torch.eye(c.shape[1], dtype=torch.float64, device=c.device)).contiguous()
    return c @ T[:, :x.shape[1]].contiguous()


def exact(case, seed):
    kind, heads, hd, layers = case["kind"], case["heads"], _hd(case), case.get("layers", 1)
    W = _predictors(case, seed) if kind.startswith("hier") else [None] * (layers * heads)

    def rebuilt(x, is_v, layer):  # [n, heads, hd]
        y = torch.empty(x.shape, dtype=torch.float64, device="cuda")
        for h in range(heads):
            for r0 in range(0, x.shape[0], 1 << 18):
                y[r0:r0 + (1 << 18), h] = _rebuilt(case, x[r0:r0 + (1 << 18), h], is_v, W[layer * heads + h])
        return y

    if kind == "hook":
        ms, at = _max_seq(case), _cells(case, seed).long()
        both = []
        for is_v, x in enumerate(_kv_rows(case, seed, 0, ms)):
            y = x.double()
            y[at] = rebuilt(x[at], is_v, 0)
            y = y.view(ms, heads * hd)
            both.append(y.t().contiguous() if is_v and case["v_trans"] else y)
        return {"k": both[0], "v": both[1], "records": None}
    if not kind.endswith("attn"):
        rows = [[rebuilt(x, is_v, i) for is_v, x in enumerate(_kv_rows(case, seed, i, case["n_tok"]))]
                for i in range(layers)]
        if case.get("via") == "all":
            rows = [torch.stack([r[j].transpose(0, 1) for r in rows]).contiguous() for j in (0, 1)]
        return {"rows": rows, "records": None}
    starts, lens = _sequences(case)
    n_q, g = case["n_q"], case["n_q"] // heads
    out, scores = [], []
    for i in range(layers):
        k, v = _kv_rows(case, seed, i, _max_seq(case))
        q = _queries(case, seed, i).double() * float(np.float32(1.0 / math.sqrt(hd)))
        o = torch.empty((case["n_seq"], n_q, hd), dtype=torch.float64, device="cuda")
        sc = [torch.empty((n_q, n), dtype=torch.float64, device="cuda") for n in lens]
        for h in range(heads):
            for s, (a, n) in enumerate(zip(starts, lens)):
                kk = _rebuilt(case, k[a:a + n, h], 0, W[i * heads + h])
                x = q[s, h * g:(h + 1) * g].contiguous() @ kk.t().contiguous()
                sc[s][h * g:(h + 1) * g] = x
                if case["want"] != "scores":
                    vv = _rebuilt(case, v[a:a + n, h], 1, W[i * heads + h])
                    o[s, h * g:(h + 1) * g] = torch.softmax(x, dim=1) @ vv
        out.append(o)
        scores.append(torch.cat([x.reshape(-1) for x in sc]))
    got = {}
    if case["want"] != "scores":
        got["out"] = out
    if case["want"] != "out":
        got["scores"] = scores
    return got
