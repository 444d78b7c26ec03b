"""The hier codec's block-per-tile kernels (sp_hier_split.hip), and the one-wave kernels
that take the large fp16 calls: records and reconstructions bit for bit against the
oracle, and the two against each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import oracle_py as O  # noqa: E402
import sp_hip as S  # noqa: E402
import workloads as W  # noqa: E402
from gpu_util import d2h, dev, p  # noqa: E402
from test_gpu_attn import say  # noqa: E402

HD, PAD, B = 256, 330, 103


def _cache(H, max_seq, seed=21):
    sk, tg = O.hier_geometry(PAD)
    Wm = W.hier_W(H, len(tg), len(sk), seed=seed)
    hc = S.HierCache(S.config(HD, 1, H), PAD, sk, tg, S.band_config(len(sk), [5, 5]), 2, max_seq, H,
                     stream=torch.cuda.current_stream().cuda_stream)
    hc.upload_W(Wm)
    return hc, Wm


def _records(hc, H, max_seq):
    torch.cuda.synchronize()
    return [d2h(q, H * max_seq * B).reshape(H, max_seq, B) for q in (hc.c.d_k_cache, hc.c.d_v_cache)]


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,start", [(1, 0), (1, 5), (63, 1), (64, 16), (65, 3), (130, 2), (200, 15)])
def test_layer_calls_match_oracle(n, start, f32):
    """K and V of two heads through the layer calls: tile edges, record runs at every kind of
    address (103-byte records from byte 103 * start of an odd-length slot), rows of infinities
    and NaN among them, nothing written outside the run."""
    say(f"hier split n={n} start={start} f32={f32}")
    H, ms = 2, start + n + 3
    hc, Wm = _cache(H, ms)
    k16, v16 = W.cfg5_kv(n_heads=H, n_pos=n, hd=HD, seed=n)
    for x in (k16, v16):
        x[0, n // 2, 7] = np.inf
        x[1, n - 1, 200] = np.nan
        x[1, 0, :] = 0
    xs = [x.astype(np.float32) * np.float32(1 + 2.0 ** -12) if f32 else x for x in (k16, v16)]
    rows = [np.ascontiguousarray(x.transpose(1, 0, 2)).reshape(n, H * HD) for x in xs]
    t = [dev(r if f32 else r.view(np.uint16)) for r in rows]
    dt = S.DTYPE_F32 if f32 else S.DTYPE_F16
    S.check(S.lib().sp_hip_hier_write_layer(hc.ref, 0, start, n, p(t[0]), p(t[1]), H * HD, dt))
    got = _records(hc, H, ms)
    out = [torch.zeros((n, H, HD), dtype=torch.float32 if f32 else torch.float16, device="cuda") for _ in range(2)]
    S.check(S.lib().sp_hip_hier_read_layer(hc.ref, 0, start, n, p(out[0]), p(out[1]), H * HD, dt))
    torch.cuda.synchronize()
    sk, tg = O.hier_geometry(PAD)
    bc = O.band_config(len(sk), [5, 5])
    for side in range(2):
        for h in range(H):
            if f32:
                ref = O.hier_compress_f32(xs[side][h], HD, PAD, sk, tg, bc, Wm[h], 2)
            else:
                ref = O.hier_compress_f16(xs[side][h].view(np.uint16), HD, PAD, sk, tg, bc, Wm[h], 2)
            np.testing.assert_array_equal(got[side][h, start:start + n], ref)
            assert not got[side][h, start + n:].any() and not got[side][h, :start].any()
            rec = O.hier_decompress_f32(ref, HD, PAD, sk, tg, bc, Wm[h], 2)
            o = out[side][:, h].cpu().numpy()
            r = rec if f32 else rec.astype(np.float16)
            np.testing.assert_array_equal(np.isnan(o), np.isnan(r))
            bits = np.uint32 if f32 else np.uint16
            np.testing.assert_array_equal(np.where(np.isnan(o), 0, o).view(bits), np.where(np.isnan(r), 0, r).view(bits))
    hc.free()


def test_large_calls_match_small_ones():
    """8 heads, K and V, eight tiles per CU (8185 positions on 256 CUs, a ragged last tile): whole
    calls (the one-wave kernels, two whole rounds of a tile per SIMD where the block-per-tile
    ones take eight of a tile per CU: the rule's line is 3.2 to one) against calls of 1000
    positions (the block-per-tile kernels), and the whole call's first and last records of a
    head against the oracle."""
    H, step = 8, 1000
    n = 32 * torch.cuda.get_device_properties(0).multi_processor_count - 7
    say(f"hier split vs lane n={n}")
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = [torch.randn((n, H * HD), generator=g, device="cuda").half() for _ in range(2)]
    (whole, Wm), (parts, _) = _cache(H, n), _cache(H, n)
    L = S.lib()
    S.check(L.sp_hip_hier_write_layer(whole.ref, 0, 0, n, p(x[0]), p(x[1]), H * HD, S.DTYPE_F16))
    for a in range(0, n, step):
        m = min(step, n - a)
        S.check(L.sp_hip_hier_write_layer(parts.ref, 0, a, m, p(x[0][a:]), p(x[1][a:]), H * HD, S.DTYPE_F16))
    recs = _records(whole, H, n)
    for a, b in zip(recs, _records(parts, H, n)):
        np.testing.assert_array_equal(a, b)
    sk, tg = O.hier_geometry(PAD)
    ends = np.r_[0:70, n - 70:n]
    for side in range(2):
        for h in (0, H - 1):
            rows = x[side].view(n, H, HD)[:, h].cpu().numpy()[ends]
            ref = O.hier_compress_f16(np.ascontiguousarray(rows).view(np.uint16), HD, PAD, sk, tg, O.band_config(len(sk), [5, 5]), Wm[h], 2)
            np.testing.assert_array_equal(recs[side][h, ends], ref)
    y = [torch.zeros_like(x[0]) for _ in range(4)]
    S.check(L.sp_hip_hier_read_layer(whole.ref, 0, 0, n, p(y[0]), p(y[1]), H * HD, S.DTYPE_F16))
    for a in range(0, n, step):
        m = min(step, n - a)
        S.check(L.sp_hip_hier_read_layer(parts.ref, 0, a, m, p(y[2][a:]), p(y[3][a:]), H * HD, S.DTYPE_F16))
    torch.cuda.synchronize()
    for i in range(2):
        assert torch.equal(y[i].view(torch.int16), y[2 + i].view(torch.int16))
    whole.free()
    parts.free()
