"""The matrix-core decode attention's powers of two (k_attn_wave: the scale of a head's fp16
weights and of its query) where what they scale is tiny or a wave's first tiles have no values,
and its softmax reference where a later best score has no value; against the oracle (1e-3
relative, elementwise)."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import oracle_py as O  # noqa: E402
import sp_hip as S  # noqa: E402
from gpu_util import dev, empty_f32, host, p, stream  # noqa: E402
from test_gpu_attn import rel_close, say  # noqa: E402
from test_gpu_attn_seqs import _arr  # noqa: E402
from test_gpu_attn_wave import BRIDGE, LAYOUTS, SHIP  # noqa: E402


def _run(hd, bands, H, n_q, score, v_amp, n_seq=1, q_scale=1.0, broken=()):
    """n_seq equal sequences over the same cells: position t scores score[t] for every query head
    and its V row is v_amp[t] * N(0, 1). The cache has cells for all of them (its workspace is
    sized by them), so they go out in one launch. broken: (position, K value, V value) put into
    a row's element."""
    n = len(score)
    rng = np.random.default_rng(hd + n)
    u = rng.standard_normal((H, 1, hd)) / 10
    k16 = (u * np.asarray(score)[None, :, None]).astype(np.float16)
    v16 = (rng.standard_normal((H, n, hd)) * np.asarray(v_amp)[None, :, None]).astype(np.float16)
    for t, kv, vv in broken:
        k16[:, t, 3], v16[:, t, hd - 2] = kv, vv
    kbc, vbc, order = O.band_config(hd, list(bands[0])), O.band_config(hd, list(bands[1])), O.mobius_order(hd)
    kr = O.ship_compress_f16(k16.reshape(-1, hd).view(np.uint16), kbc, order).reshape(H, n, -1)
    vr = O.ship_compress_f16(v16.reshape(-1, hd).view(np.uint16), vbc).reshape(H, n, -1)
    scale = 1.0 / math.sqrt(hd)
    # along u, as long as makes the lowest score what it should be
    q = np.repeat(u[:, 0], n_q // H, axis=0).astype(np.float32)
    at = int(np.argmin(score))
    got = O.attn_decode(q, kr[:, at:at + 1], vr[:, at:at + 1], H, 1, kbc, vbc, order, scale, want_out=False)[0]
    q = (q * (score[at] / got) * q_scale).astype(np.float32)
    s_ref, o_ref = O.attn_decode(q, kr, vr, H, n, kbc, vbc, order, scale)

    cc = S.ShipCache(S.config(hd, 1, H, k_bits=bands[0], v_bits=bands[1]), n_seq * n + 2,
                     stream=torch.cuda.current_stream().cuda_stream)
    rows = [dev(np.ascontiguousarray(x.transpose(1, 0, 2)).view(np.uint16)) for x in (k16, v16)]
    S.check(S.lib().sp_hip_write_layer(cc.ref, 0, 0, n, p(rows[0]), p(rows[1]), H * hd, S.DTYPE_F16))
    (_, starts), (_, lens) = a, b = _arr([0] * n_seq), _arr([n] * n_seq)
    qt, sc, out = dev(np.tile(q, (n_seq, 1))), empty_f32(n_seq * n_q * n), empty_f32(n_seq * n_q * hd)
    S.check(S.lib().sp_hip_attn_decode_seqs(cc.ref, 0, n_seq, starts, lens, p(qt), n_q, C.c_float(scale), p(sc), p(out),
                                            stream()))
    g_s, g_o = host(sc).reshape(n_seq, n_q, n), host(out).reshape(n_seq, n_q, hd)
    cc.free()
    assert np.isfinite(g_s).all() and np.isfinite(g_o).all()
    for i in {0, n_seq - 1}:
        rel_close(g_s[i], s_ref)
        rel_close(g_o[i], o_ref)


@pytest.mark.parametrize("G", [2, 7])
@pytest.mark.parametrize("hd,bands", LAYOUTS)
def test_every_weight_tiny(hd, bands, G):
    """The best position's V record is zero and the others score 84 lower: the tile's largest
    weight is about 2^-122, whose normalising power of two is past the fp32 range."""
    say(f"wave attn tiny weights hd={hd} bands={bands} G={G}")
    _run(hd, bands, 2, 2 * G, [1.0] + [-83.0] * 63, [0.0] + [1.0] * 63)


@pytest.mark.parametrize("hd,bands", LAYOUTS)
def test_tiny_query(hd, bands):
    """A query of about 1e-36 (2^-120): its normalising power of two is past the fp32 range."""
    say(f"wave attn tiny query hd={hd} bands={bands}")
    _run(hd, bands, 2, 6, np.linspace(-1.0, 1.0, 200), np.ones(200), q_scale=1e-36)


# two or more tiles per wave on 256 CUs
SEVERAL = [(64, BRIDGE, 8, 2, 16, 2100), (64, SHIP, 8, 8, 16, 3090), (96, BRIDGE, 8, 5, 16, 3100),
           (96, BRIDGE, 32, 1, 12, 1100), (128, SHIP, 8, 4, 16, 3100), (256, SHIP, 8, 2, 16, 1100),
           (256, SHIP, 4, 6, 16, 2110)]


@pytest.mark.parametrize("lower", [10.0, 20.0])
@pytest.mark.parametrize("hd,bands,H,G,n_seq,n", SEVERAL)
def test_first_tiles_without_values(hd, bands, H, G, n_seq, n, lower):
    """Seven tiles of eight have zero V records; the eighth's scores are 10 or 20 lower and its V
    records small (scales of about 2^-6): all that the output consists of."""
    say(f"wave attn no values first hd={hd} bands={bands} H={H} G={G} n={n} lower={lower}")
    eighth = np.arange(n) // 64 % 8 == 7
    score = np.where(eighth, -lower, -0.5) + np.random.default_rng(n).uniform(-0.5, 0.5, n)
    _run(hd, bands, H, H * G, score, np.where(eighth, 0.05, 0.0), n_seq)


@pytest.mark.parametrize("above", [40.0, 95.0])
@pytest.mark.parametrize("hd,bands,H,G,n_seq,n", SEVERAL)
def test_later_best_position_without_values(hd, bands, H, G, n_seq, n, above):
    """One position of the eighth tile scores 40 or 95 above its wave's first tile (past the range
    of the fp32 exponential) with a zero V record; the output consists of a few positions of
    the seventeenth that score 3 below it."""
    say(f"wave attn best without values hd={hd} bands={bands} H={H} G={G} n={n} above={above}")
    score, v_amp = np.full(n, -above), np.ones(n)
    score[7 * 64 + 21], v_amp[7 * 64 + 21] = -0.5, 0.0
    score[16 * 64 + 5:16 * 64 + 9] = -3.5
    _run(hd, bands, H, H * G, score, v_amp, n_seq)


@pytest.mark.parametrize("hd,bands,H,G,n_seq,n", SEVERAL)
def test_rows_that_are_not_finite(hd, bands, H, G, n_seq, n):
    """K and V rows with an infinity or a NaN, in the first, a middle and the last tile: their bands'
    scales are not finite, which reads as 0, at positions that would have scored among the best."""
    say(f"wave attn rows not finite hd={hd} bands={bands} H={H} G={G} n={n}")
    score = np.linspace(-3.0, -0.5, n)
    _run(hd, bands, H, H * G, score, np.ones(n), n_seq,
         broken=[(5, np.inf, 1.0), (9, 1.0, -np.inf), (n // 2, -np.inf, np.inf), (n // 2 + 1, 1.0, np.nan), (n - 2, 1.0, np.inf),
                 (n - 1, np.inf, np.nan)])
