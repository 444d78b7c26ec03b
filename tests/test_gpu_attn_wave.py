"""The matrix-core decode attention (k_attn_wave) over every record layout it serves,
against the oracle (scores and softmax . V within 1e-3 relative, elementwise): the
launch shapes (blocks of 4, 8 and 16 waves, one or several tiles per wave, a sequence
that is one block), records at odd cells, GQA 1-8, and scores that outgrow a wave's
first tile."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import oracle_py as O  # noqa: E402
import sp_hip as S  # noqa: E402
import workloads as W  # noqa: E402
from gpu_util import dev, empty_f32, host, p, stream  # noqa: E402
from test_gpu_attn import rel_close, say  # noqa: E402
from test_gpu_attn_seqs import _check  # noqa: E402

BRIDGE, SHIP = ((5, 4, 4), (5,)), ((5, 5, 4, 3), (3,))
LAYOUTS = [(64, BRIDGE), (64, SHIP), (96, BRIDGE), (128, SHIP), (256, SHIP)]


def _cache(hd, bands, H, n, seed, mobius=True, ramp=None):
    """A one-layer cache of n written cells (and two unwritten ones) and the oracle's records."""
    k16, v16 = W.cfg3_kv(n_heads=H, n_pos=n, hd=hd, seed=seed)
    if ramp is not None:
        k16 = (k16.astype(np.float32) * ramp[None, :, None]).astype(np.float16)
    cc = S.ShipCache(S.config(hd, 1, H, k_bits=bands[0], v_bits=bands[1], mobius=mobius), n + 2,
                     stream=torch.cuda.current_stream().cuda_stream)
    rows = [dev(np.ascontiguousarray(x.transpose(1, 0, 2)).view(np.uint16)) for x in (k16, v16)]
    S.check(S.lib().sp_hip_write_layer(cc.ref, 0, 0, n, p(rows[0]), p(rows[1]), H * hd, S.DTYPE_F16))
    torch.cuda.synchronize()
    kbc, vbc = O.band_config(hd, list(bands[0])), O.band_config(hd, list(bands[1]))
    order = O.mobius_order(hd) if mobius else None
    kr = O.ship_compress_f16(k16.reshape(-1, hd).view(np.uint16), kbc, order).reshape(H, n, -1)
    vr = O.ship_compress_f16(v16.reshape(-1, hd).view(np.uint16), vbc).reshape(H, n, -1)
    return cc, kbc, vbc, order, kr, vr


def _run(hd, bands, H, n_q, starts, lens, mobius=True, ramp=None):
    n = max(s + m for s, m in zip(starts, lens))
    cc, kbc, vbc, order, kr, vr = _cache(hd, bands, H, n, hd + n, mobius, ramp)
    q = np.stack([W.cfg2_q(n_q=n_q, hd=hd, pos=m, seed=3 + i) for i, m in enumerate(lens)])
    scale = 1.0 / math.sqrt(hd)

    def ref(i, s0, m):
        return O.attn_decode(q[i], kr[:, s0:s0 + m], vr[:, s0:s0 + m], H, m, kbc, vbc, order, scale)
    _check(S.lib().sp_hip_attn_decode_seqs, cc.ref, 0, starts, lens, q, n_q, hd, scale, ref)
    cc.free()


@pytest.mark.parametrize("G", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("hd,bands", LAYOUTS)
def test_odd_cells_and_tile_edges(hd, bands, G):
    """Sequences at odd cells of 2-mod-4-byte records (and of an odd cache length), at the
    edges of tiles and of 4-, 8- and 16-wave blocks."""
    starts = [1, 2, 7, 70, 131, 500, 3]
    lens = [1, 63, 64, 65, 300, 1025, 1027 if G < 5 else 513]
    say(f"wave attn hd={hd} bands={bands} G={G}")
    _run(hd, bands, 2, 2 * G, starts, lens, mobius=G != 3)
    _run(hd, bands, 2, 2 * G, [5], [511], mobius=G != 3)  # 8 tiles: one block, nothing to merge


@pytest.mark.parametrize("hd,bands,H,G,n_seq,n", [
    (64, BRIDGE, 8, 2, 16, 2100),    # two tiles per wave, 16-wave blocks, three of a sequence's 33 tiles left over
    (64, SHIP, 8, 8, 16, 3090),      # eight heads: blocks of four waves
    (96, BRIDGE, 32, 1, 12, 1000),   # more sequences x KV heads than arrival counters: two launches
    (96, BRIDGE, 8, 5, 16, 3100),
    (128, SHIP, 8, 4, 16, 3100),     # four tiles per wave at 168 registers
    (128, SHIP, 8, 8, 4, 4200),      # eight heads at head_dim 128: one tile per wave, nine 8-wave blocks
    (256, SHIP, 8, 2, 16, 1100),
    (256, SHIP, 4, 6, 16, 2110),
])
def test_several_tiles_per_wave(hd, bands, H, G, n_seq, n):
    """Enough tiles that waves walk several, over overlapping ranges. K grows 40-fold along the
    cells, so later tiles' weights outgrow the scale a wave took from its first tile (2^15
    over [2^5, 2^6): scores more than 6.2 above its maximum) and its sums are rescaled."""
    say(f"wave attn tiles hd={hd} bands={bands} H={H} G={G} n_seq={n_seq} n={n}")
    starts = [(37 * i) % 150 for i in range(n_seq)]
    lens = [n - 13 * i for i in range(n_seq)]
    m = max(s + k for s, k in zip(starts, lens))
    _run(hd, bands, H, H * G, starts, lens, ramp=np.linspace(0.2, 8.0, m, dtype=np.float32))


def test_long_single_sequence_head_dim_64():
    """One sequence of 130 16-wave blocks over two KV heads, two tiles per wave or one."""
    hd, H, n_q, n = 64, 2, 4, 140001
    say(f"wave attn hd={hd} n={n}")
    cc, kbc, vbc, order, kr, vr = _cache(hd, BRIDGE, H, n, 9)
    q = W.cfg2_q(n_q=n_q, hd=hd, pos=n, seed=4)
    scale = 1.0 / math.sqrt(hd)
    s_ref, o_ref = O.attn_decode(q, kr, vr, H, n, kbc, vbc, order, scale)
    sc, out, qt = empty_f32(n_q * n), empty_f32(n_q * hd), dev(q)
    S.check(S.lib().sp_hip_attn_decode(cc.ref, 0, n, p(qt), n_q, C.c_float(scale), p(sc), p(out), stream()))
    rel_close(host(sc).reshape(n_q, n), s_ref)
    rel_close(host(out).reshape(n_q, hd), o_ref)
    cc.free()


@pytest.mark.parametrize("G,n", [(1, 37001), (8, 37001), (4, 80000)])
def test_scores_alone_of_long_sequences(G, n):
    """One sequence past 9/8 of a round at head_dim 128: the scores alone go in blocks of 16 waves of
    several tiles (two of 4632 tiles, three of 10000), with an output in other shapes; the
    same scores bit for bit."""
    hd, H = 128, 8
    n_q = H * G
    say(f"wave attn scores alone G={G} n={n}")
    cc = S.ShipCache(S.config(hd, 1, H), n, stream=torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda")
    g.manual_seed(n + G)
    k, v = (torch.randn((n, H * hd), generator=g, device="cuda").half() for _ in range(2))
    S.check(S.lib().sp_hip_write_layer(cc.ref, 0, 0, n, p(k), p(v), H * hd, S.DTYPE_F16))
    q = torch.randn((n_q, hd), generator=g, device="cuda")
    for mb in (-1, 2):
        both, alone, out = empty_f32(n_q * n), empty_f32(n_q * n), empty_f32(n_q * hd)
        args = (cc.ref, 0, n, p(q), n_q, C.c_float(1.0 / math.sqrt(hd)))
        S.check(S.lib().sp_hip_attn_decode_bands(*args, p(both), p(out), mb, stream()))
        S.check(S.lib().sp_hip_attn_decode_bands(*args, p(alone), None, mb, stream()))
        assert torch.equal(both.view(torch.int32), alone.view(torch.int32))
        assert bool(torch.isfinite(out).all()) and bool((out != 0).any())
    cc.free()
