"""The sqfree attention's matrix-core products over groups of four query heads: group sizes
that leave rows of the last group unused, at tile edges, against the oracle."""
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
from test_gpu_sqfree_attn import _sqfree_cache, rel_close, say  # noqa: E402


@pytest.mark.parametrize("groups", ["auto", "one"])
@pytest.mark.parametrize("sk,v_bits,H,G,n_kv,runs", [
    (77, [5, 4, 4, 4, 5], 2, 8, 129, 1), (77, [5, 4, 4, 4, 5], 1, 4, 63, 0), (115, [5, 4, 4, 4, 5], 2, 7, 65, 1),
    (115, [3], 1, 6, 191, 1), (115, [3], 2, 1, 257, 2), (115, [5, 4, 4, 4, 5], 1, 8, 128, 0)])
def test_head_groups(sk, v_bits, H, G, n_kv, runs, groups, monkeypatch):
    if runs:
        monkeypatch.setenv("SP_HIP_SQFREE_ATTN_RUNS", str(runs))
    if groups == "one":
        monkeypatch.setenv("SP_HIP_SQFREE_ATTN_GROUPS", "1")
    say(f"sqfree attn head groups sk={sk} v_bits={v_bits} H={H} G={G} n_kv={n_kv} runs={runs} groups={groups}")
    hd, n_q = 128, H * G
    cc, km, kbc, vbc, kp, vp = _sqfree_cache(sk, v_bits, H, n_kv, seed=sk + n_kv)
    q = W.cfg2_q(n_q=n_q, hd=hd, pos=n_kv, seed=G)
    scale = 1.0 / math.sqrt(hd)
    s_ref, o_ref = O.sqfree_attn_decode(q, kp, vp, H, n_kv, hd, km, kbc, vbc, 3, True, scale)
    qt, sc, out = dev(q), empty_f32(n_q * n_kv), empty_f32(n_q * hd)
    S.check(S.lib().sp_hip_sqfree_attn_decode(cc.ref, 1, n_kv, p(qt), n_q, C.c_float(scale), p(sc), p(out), stream()))
    rel_close(host(sc).reshape(n_q, n_kv), s_ref)
    rel_close(host(out).reshape(n_q, hd), o_ref)
    assert np.isfinite(host(out)).all()
    cc.free()
