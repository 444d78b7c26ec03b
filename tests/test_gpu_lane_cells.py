"""Layer calls of the one-vector-per-lane codec kernels at record runs of every address class:
even-sized records (26 to 76 bytes) from any cell of odd- and even-length slots, tile edges,
rows of infinities and NaN; records and reconstructions bit for bit against the oracle, and
nothing written outside the run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import oracle_py as O  # noqa: E402
import sp_hip as S  # noqa: E402
import workloads as W  # noqa: E402
from gpu_util import d2h, dev, p  # noqa: E402
from test_gpu_attn import say  # noqa: E402

SHIP = [(64, [5, 4, 4], [5]), (64, [5, 5, 4, 3], [3]), (96, [5, 4, 4], [5]), (128, [5, 5, 4, 3], [3])]
RUNS = [(1, 0), (1, 1), (63, 1), (64, 2), (65, 3), (130, 1)]


def _inputs(hd, H, n, f32):
    kv = W.cfg1_kv(n_heads=H, n_pos=n, hd=hd, seed=hd + n)
    for x in kv:
        x[0, n // 2, 7] = np.inf
        x[H - 1, n - 1, hd - 1] = np.nan
        x[H - 1, 0, :] = 0
    xs = [x.astype(np.float32) * np.float32(1 + 2.0 ** -12) if f32 else x for x in kv]
    return xs, [dev((r if f32 else r.view(np.uint16)).transpose(1, 0, 2).reshape(n, H * hd)) for r in xs]


def _records(cc, B, H, ms):
    torch.cuda.synchronize()
    return [d2h(q, H * ms * b).reshape(H, ms, b) for q, b in zip((cc.c.d_k_cache, cc.c.d_v_cache), B)]


def _same(got, ref, f32):
    bits = np.uint32 if f32 else np.uint16
    nan = np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(np.where(nan, 0, got).view(bits), np.where(nan, 0, ref).view(bits))


def _check(cc, write, read, compress, decompress, B, hd, n, start, f32):
    H, ms = 2, start + n + 3
    xs, t = _inputs(hd, H, n, f32)
    dt = S.DTYPE_F32 if f32 else S.DTYPE_F16
    S.check(write(cc.ref, 0, start, n, p(t[0]), p(t[1]), H * hd, dt))
    out = [torch.full((n, H, hd), 7.0, dtype=torch.float32 if f32 else torch.float16, device="cuda") for _ in range(2)]
    S.check(read(cc, start, n, p(out[0]), p(out[1]), H * hd, dt))
    both = _records(cc, B, H, ms)
    for side in range(2):
        for h in range(H):
            ref = compress[side](xs[side][h])
            np.testing.assert_array_equal(both[side][h, start:start + n], ref)
            assert not both[side][h, :start].any() and not both[side][h, start + n:].any()
            rec = decompress[side](ref)
            _same(out[side][:, h].cpu().numpy(), rec if f32 else rec.astype(np.float16), f32)
    # one side alone gives what both gave
    alone = [torch.full_like(o, 7.0) for o in out]
    for side in range(2):
        a = [None, None]
        a[side] = p(t[side])
        S.check(write(cc.ref, 0, start, n, a[0], a[1], H * hd, dt))
        a[side] = p(alone[side])
        S.check(read(cc, start, n, a[0], a[1], H * hd, dt))
    for b, c in zip(both, _records(cc, B, H, ms)):
        np.testing.assert_array_equal(b, c)
    for o, c in zip(out, alone):
        _same(c.cpu().numpy(), o.cpu().numpy(), f32)
    cc.free()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,start", RUNS)
@pytest.mark.parametrize("hd,kb,vb", SHIP)
def test_ship_layer(hd, kb, vb, n, start, f32):
    say(f"lane cells ship hd={hd} k={kb} v={vb} n={n} start={start} f32={f32}")
    cc = S.ShipCache(S.config(hd, 1, 2, k_bits=kb, v_bits=vb), start + n + 3,
                     stream=torch.cuda.current_stream().cuda_stream)
    bcs, orders = [O.band_config(hd, kb), O.band_config(hd, vb)], [O.mobius_order(hd), None]

    def comp(s):
        return lambda x: O.ship_compress_f32(x, bcs[s], orders[s]) if f32 else \
            O.ship_compress_f16(x.view(np.uint16), bcs[s], orders[s])

    def dec(s):
        return lambda r: O.ship_decompress_f32(r, bcs[s], orders[s])

    def read(c, start, n, k, v, stride, dt):
        return S.lib().sp_hip_read_layer(c.ref, 0, start, n, k, v, stride, dt, -1)

    _check(cc, S.lib().sp_hip_write_layer, read, [comp(0), comp(1)], [dec(0), dec(1)],
           [b.total_bytes for b in bcs], hd, n, start, f32)


@pytest.mark.parametrize("n,start", RUNS)
@pytest.mark.parametrize("v_bits", [[5, 4, 4, 4, 5], [3]])
def test_sqfree_layer(v_bits, n, start):
    hd, k_bits = 128, [5, 4, 4, 4, 5]
    say(f"lane cells sqfree v={v_bits} n={n} start={start}")
    cc = S.SqfreeCache(S.config(hd, 1, 2, k_bits=k_bits, v_bits=v_bits), start + n + 3, rbits=3, spinor=True, sk_k=115,
                       stream=torch.cuda.current_stream().cuda_stream)
    km = O.Knight(154, 115)
    bcs = [O.band_config(115, k_bits), O.band_config(115, v_bits)]

    def comp(s):
        return lambda x: O.sqfree_compress_f16(x.view(np.uint16), hd, km, bcs[s], 3, True)

    def dec(s):
        return lambda r: O.sqfree_decompress_f32(r, hd, km, bcs[s], 3, True)

    def read(c, start, n, k, v, stride, dt):
        return S.lib().sp_hip_sqfree_read_layer(c.ref, 0, start, n, k, v, stride, dt)

    _check(cc, S.lib().sp_hip_sqfree_write_layer, read, [comp(0), comp(1)], [dec(0), dec(1)],
           [cc.c.bytes_per_pos_k, cc.c.bytes_per_pos_v], hd, n, start, False)


@pytest.mark.parametrize("kind", ["ship", "sqfree", "hier"])
def test_sides_read_into_one_buffer(kind):
    """Both sides of a read in one buffer: interleaved rows (K and V of a token side by side)
    give what separate buffers give; the same rows for both end with V's, as two reads would."""
    H, n, start = 2, 150, 1
    hd = 256 if kind == "hier" else 128
    ms = start + n + 3
    say(f"lane cells one buffer {kind}")
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "ship":
        cc = S.ShipCache(S.config(hd, 1, H), ms, stream=stream)
        write, rd = S.lib().sp_hip_write_layer, S.lib().sp_hip_read_layer
        tail = (-1,)
    elif kind == "sqfree":
        b = [5, 4, 4, 4, 5]
        cc = S.SqfreeCache(S.config(hd, 1, H, k_bits=b, v_bits=b), ms, rbits=3, spinor=True, sk_k=77, stream=stream)
        write, rd, tail = S.lib().sp_hip_sqfree_write_layer, S.lib().sp_hip_sqfree_read_layer, ()
    else:
        sk, tg = O.hier_geometry(330)
        cc = S.HierCache(S.config(hd, 1, H), 330, sk, tg, S.band_config(len(sk), [5, 5]), 2, ms, H, stream=stream)
        cc.upload_W(W.hier_W(H, len(tg), len(sk), seed=4))
        write, rd, tail = S.lib().sp_hip_hier_write_layer, S.lib().sp_hip_hier_read_layer, ()
    w = H * hd
    t = [dev(x.view(np.uint16).transpose(1, 0, 2).reshape(n, w)) for x in W.cfg1_kv(n_heads=H, n_pos=n, hd=hd, seed=3)]
    S.check(write(cc.ref, 0, start, n, p(t[0]), p(t[1]), w, S.DTYPE_F16))
    ref = [torch.zeros((n, w), dtype=torch.int16, device="cuda") for _ in range(2)]
    S.check(rd(cc.ref, 0, start, n, p(ref[0]), p(ref[1]), w, S.DTYPE_F16, *tail))
    mixed = torch.zeros((n, 2, w), dtype=torch.int16, device="cuda")
    S.check(rd(cc.ref, 0, start, n, p(mixed), p(mixed[0, 1]), 2 * w, S.DTYPE_F16, *tail))
    one = torch.zeros((n, w), dtype=torch.int16, device="cuda")
    S.check(rd(cc.ref, 0, start, n, p(one), p(one), w, S.DTYPE_F16, *tail))
    torch.cuda.synchronize()
    assert torch.equal(mixed[:, 0], ref[0]) and torch.equal(mixed[:, 1], ref[1])
    assert torch.equal(one, ref[1]) and not torch.equal(ref[0], ref[1])
    cc.free()


@pytest.mark.parametrize("hd,n", [(128, 8300), (256, 4200)])
def test_large_fp32_runs_off_a_dword(hd, n):
    """8 heads of fp32 rows from cell 1 (V records off a dword) past one round of the lane kernels'
    blocks on 256 CUs, where the general kernels take them, K and V and V alone, against the
    same rows in calls of 1000 (the lane kernels)."""
    H = 8
    say(f"lane cells large fp32 hd={hd} n={n}")
    g = torch.Generator(device="cuda")
    g.manual_seed(hd)
    x = [torch.randn((n, H * hd), generator=g, device="cuda") for _ in range(2)]
    st = torch.cuda.current_stream().cuda_stream
    whole, parts = (S.ShipCache(S.config(hd, 1, H), n + 2, stream=st) for _ in range(2))
    L, B = S.lib(), [whole.c.k_bands.total_bytes, whole.c.v_bands.total_bytes]
    y = [torch.zeros_like(x[0]) for _ in range(5)]
    S.check(L.sp_hip_write_layer(whole.ref, 0, 1, n, p(x[0]), p(x[1]), H * hd, S.DTYPE_F32))
    S.check(L.sp_hip_read_layer(whole.ref, 0, 1, n, p(y[0]), p(y[1]), H * hd, S.DTYPE_F32, -1))
    S.check(L.sp_hip_read_layer(whole.ref, 0, 1, n, None, p(y[4]), H * hd, S.DTYPE_F32, -1))
    for a in range(0, n, 1000):
        m = min(1000, n - a)
        S.check(L.sp_hip_write_layer(parts.ref, 0, 1 + a, m, p(x[0][a:]), p(x[1][a:]), H * hd, S.DTYPE_F32))
        S.check(L.sp_hip_read_layer(parts.ref, 0, 1 + a, m, p(y[2][a:]), p(y[3][a:]), H * hd, S.DTYPE_F32, -1))
    for a, b in zip(_records(whole, B, H, n + 2), _records(parts, B, H, n + 2)):
        np.testing.assert_array_equal(a, b)
    for a, b in ((0, 2), (1, 3), (4, 3)):
        assert torch.equal(y[a].view(torch.int32), y[b].view(torch.int32))
    whole.free()
    parts.free()
