"""The sqfree attention's products, on the matrix cores over groups of four query heads (group
sizes that leave rows of the last group unused) and on the vector unit for one and two heads,
at tile edges, against the oracle."""
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
    (115, [3], 1, 6, 191, 1), (115, [3], 2, 1, 257, 2), (115, [5, 4, 4, 4, 5], 1, 8, 128, 0),
    (77, [5, 4, 4, 4, 5], 2, 2, 193, 1), (77, [5, 4, 4, 4, 5], 2, 1, 65, 1), (115, [3], 2, 2, 320, 2)])
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


@pytest.mark.parametrize("sk,v_bits,G", [(115, [3], 1), (115, [5, 4, 4, 4, 5], 2), (77, [5, 4, 4, 4, 5], 1), (77, [5, 4, 4, 4, 5], 2)])
def test_vector_and_matrix_scores_are_the_same_bits(sk, v_bits, G):
    """16 sequences of 8 KV heads in one call (3072 tiles: the vector unit on 256 CUs) and each by
    itself (the matrix cores): the same scores, and outputs within the order of their sums."""
    hd, H, n_seq, n = 128, 8, 16, 1500
    n_q, ms = H * G, n_seq * 100 + n
    say(f"sqfree attn vector and matrix sk={sk} v_bits={v_bits} G={G}")
    cc = S.SqfreeCache(S.config(hd, 1, H, k_bits=[5, 4, 4, 4, 5], v_bits=v_bits), ms, rbits=3, spinor=True, sk_k=sk,
                       stream=torch.cuda.current_stream().cuda_stream)
    L, g = S.lib(), torch.Generator(device="cuda")
    g.manual_seed(sk + G)
    k, v = (torch.randn((ms, H * hd), generator=g, device="cuda").half() for _ in range(2))
    S.check(L.sp_hip_sqfree_write_layer(cc.ref, 0, 0, ms, p(k), p(v), H * hd, S.DTYPE_F16))
    starts = np.arange(n_seq, dtype=np.int32) * 100
    lens = np.full(n_seq, n, dtype=np.int32) - np.arange(n_seq, dtype=np.int32)
    q = torch.randn((n_seq, n_q, hd), generator=g, device="cuda")

    def run(i0, m):
        tot = n_q * int(lens[i0:i0 + m].sum())
        sc, out = empty_f32(tot), empty_f32(m * n_q * hd)
        S.check(L.sp_hip_sqfree_attn_decode_seqs(cc.ref, 0, m, C.c_void_p(starts[i0:].ctypes.data), C.c_void_p(lens[i0:].ctypes.data),
                                                 p(q[i0]), n_q, C.c_float(1.0 / math.sqrt(hd)), p(sc), p(out), stream()))
        return host(sc), host(out)

    s_all, o_all = run(0, n_seq)
    one = [run(i, 1) for i in range(n_seq)]
    np.testing.assert_array_equal(s_all.view(np.uint32), np.concatenate([o[0] for o in one]).view(np.uint32))
    rel_close(o_all, np.concatenate([o[1] for o in one]))
    cc.free()
