"""Dense GEMMs on MFMA-tiled weights through the device entry points, at the
edges of the schedules' tiles, against the oracle.

(The host GEMM entry points multiply row-major weights, so the schedules that
read tiled weights are reached here, with the flag.) The bars are the GEMM's:
max-rel 1e-3 against the oracle's fp32 result and err/esc 1e-4 against the
exact value.
"""
import numpy as np
import pytest

from helpers import acts, err_esc, fp4_weights, fp8_weights, max_rel
from test_gpu_tiled import dev_pack

pytestmark = pytest.mark.gpu


def gemm_tiled(hip, fmt, w, ws, c, s, round_out=0):
    """[M, O] of the tiled-weight GEMM; the row after the last must stay untouched"""
    L = hip.lib()
    (M, K), O = c.shape, w.shape[0]
    _, _, (tw, tws) = dev_pack(hip, fmt, w, ws, O, K)
    dws = tws if fmt == 0 else hip.DevBuf.from_array(ws)
    dc, ds = hip.DevBuf.from_array(c), hip.DevBuf.from_array(s)
    guard = np.full((M + 1, O), -7.5, np.float32)
    do = hip.DevBuf.from_array(guard)
    fn = L.apus_hip_fp4_gemm_dev if fmt == 0 else L.apus_hip_fp8_gemm_dev
    hip._check(fn(tw.ptr, dws.ptr, dc.ptr, ds.ptr, do.ptr, M, O, K, hip.W_TILED | round_out), "gemm")
    hip._check(L.apus_hip_synchronize(), "sync")
    out = do.to_array(np.float32, (M + 1, O))
    assert np.all(out[M] == -7.5)
    return out[:M]


def check(got, oracle, fmt, w, ws, c, s):
    gemm, truth = (oracle.fp4_gemm, oracle.fp4_truth) if fmt == 0 else (oracle.fp8_gemm, oracle.fp8_truth)
    t, esc = truth(w, ws, c, s)
    assert max_rel(got, gemm(w, ws, c, s)) <= 1e-3
    assert err_esc(got, t, esc) <= 1e-4


@pytest.mark.parametrize("K", (1024, 2048, 4096, 8192))
@pytest.mark.parametrize("M", (9, 16, 17, 32, 33, 64))
def test_narrow_tiled(hip, oracle, rng, M, K):
    """The narrow schedule (FP8, 9..64 rows): tile scales that differ along K,
    at K = 1024 too, where a wave's two groups share a word of scale bytes with
    the next wave's."""
    O = 256
    w, ws = fp8_weights(rng, O, K)
    c, s = oracle.act_quant(acts(rng, M, K, 2.0))
    check(gemm_tiled(hip, 1, w, ws, c, s), oracle, 1, w, ws, c, s)
