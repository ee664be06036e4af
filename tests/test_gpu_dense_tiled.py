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
@pytest.mark.parametrize("M", (9, 16, 17, 32, 33, 48, 49, 64))
def test_narrow_tiled(hip, oracle, rng, M, K):
    """The narrow schedule (FP8, 9..64 rows): tile scales that differ along K,
    at K = 1024 too, where a wave's two groups share a word of scale bytes with
    the next wave's."""
    O = 256
    w, ws = fp8_weights(rng, O, K)
    c, s = oracle.act_quant(acts(rng, M, K, 2.0))
    check(gemm_tiled(hip, 1, w, ws, c, s), oracle, 1, w, ws, c, s)


def gemm_rows(hip, fmt, w, ws, c, s, round_out=0):
    """the same GEMM on row-major weights (the register-ring tile schedule)"""
    L = hip.lib()
    (M, K), O = c.shape, w.shape[0]
    bufs = [hip.DevBuf.from_array(v) for v in (w, ws, c, s)]
    do = hip.DevBuf(M * O * 4)
    fn = L.apus_hip_fp4_gemm_dev if fmt == 0 else L.apus_hip_fp8_gemm_dev
    hip._check(fn(*(b.ptr for b in bufs), do.ptr, M, O, K, round_out), "gemm")
    hip._check(L.apus_hip_synchronize(), "sync")
    return do.to_array(np.float32, (M, O))


@pytest.mark.parametrize("fmt,M,O,K", [
    (1, 500, 14336, 1024), (0, 449, 14336, 1024),      # 256 x 128 tiles
    (1, 120, 28672, 1024), (0, 380, 10240, 2048),      # 128 x 128
    (1, 65, 16384, 1024), (1, 200, 8192, 2048),        # 64 x 128, 256 workgroups
    (0, 150, 6144, 1024), (1, 129, 5760, 2048), (1, 300, 8192, 1024),   # 64 x 128: 144, 135; more than 256
    (1, 300, 12288, 1024), (0, 300, 12288, 1024),      # 64 x 128 for 288 tiles of 128 x 128
    (1, 520, 1536, 1024), (0, 1040, 384, 1024), (1, 577, 2048, 1024),   # even groups of row blocks: 9, 17, 10
    (1, 66, 128, 8192), (0, 9, 128, 1024), (1, 129, 384, 4096), (0, 64, 256, 4096), (0, 70, 128, 2048),  # 64 x 64
    (1, 1000, 1024, 4096),
])
def test_block_schedule(hip, oracle, rng, fmt, M, O, K):
    """Every tile of the block schedule, at ragged row counts: the bits of the
    register-ring tile schedule (one chain per output in both), and the
    oracle's values in sampled rows and columns."""
    w, ws = (fp4_weights if fmt == 0 else fp8_weights)(rng, O, K)
    c, s = oracle.act_quant(acts(rng, M, K, 2.0))
    got = gemm_tiled(hip, fmt, w, ws, c, s)
    assert np.array_equal(got.view(np.uint32), gemm_rows(hip, fmt, w, ws, c, s).view(np.uint32))
    rows = np.unique(np.r_[0, M - 1, rng.integers(0, M, 6)])
    cols = slice(O - 128, O)
    wsc = ws[cols] if fmt == 0 else ws[-1:]
    check(got[rows, cols], oracle, fmt, np.ascontiguousarray(w[cols]), np.ascontiguousarray(wsc), c[rows], s[rows])


def test_block_schedule_unaligned_out(hip, oracle, rng):
    """Output rows that 16-byte stores cannot take: the tile schedule, same bits."""
    M, O, K = 70, 128, 1024
    L = hip.lib()
    w, ws = fp8_weights(rng, O, K)
    c, s = oracle.act_quant(acts(rng, M, K))
    _, _, (tw, _) = dev_pack(hip, 1, w, ws, O, K)
    dws, dc, ds = (hip.DevBuf.from_array(v) for v in (ws, c, s))
    do = hip.DevBuf(M * O * 4 + 16)
    hip._check(L.apus_hip_fp8_gemm_dev(tw.ptr, dws.ptr, dc.ptr, ds.ptr, do.ptr + 4, M, O, K, hip.W_TILED | 1), "gemm")
    hip._check(L.apus_hip_synchronize(), "sync")
    got = do.to_array(np.float32, (M * O + 4,))[1:1 + M * O].reshape(M, O)
    want = gemm_tiled(hip, 1, w, ws, c, s, 1)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("what", ["w", "ws", "codes", "scales"])
@pytest.mark.parametrize("fmt,M", [(0, 20), (0, 70), (1, 20), (1, 70)])
def test_unaligned_operands(hip, rng, fmt, M, what):
    """Operands at 4-byte offsets, which the narrow and block schedules' loads
    to LDS do not take: the tile schedule, the bits of the same GEMM on
    row-major weights."""
    O, K = 256, 2048
    L = hip.lib()
    w, ws = (fp4_weights if fmt == 0 else fp8_weights)(rng, O, K)
    c, s = hip.act_quant(acts(rng, M, K))
    _, _, (tw, tws) = dev_pack(hip, fmt, w, ws, O, K)
    bufs = {"w": (tw, w.nbytes), "ws": (tws, ws.nbytes) if fmt == 0 else (hip.DevBuf.from_array(ws), ws.nbytes),
            "codes": (hip.DevBuf.from_array(c), c.nbytes), "scales": (hip.DevBuf.from_array(s), s.nbytes)}
    b, n = bufs[what]
    moved = hip.DevBuf(n + 16)
    hip._check(L.apus_hip_d2d(moved.ptr + 4, b.ptr, n), "d2d")
    ptr = {k: v[0].ptr for k, v in bufs.items()} | {what: moved.ptr + 4}
    do = hip.DevBuf(M * O * 4)
    fn = L.apus_hip_fp4_gemm_dev if fmt == 0 else L.apus_hip_fp8_gemm_dev
    hip._check(fn(ptr["w"], ptr["ws"], ptr["codes"], ptr["scales"], do.ptr, M, O, K, hip.W_TILED), "gemm")
    hip._check(L.apus_hip_synchronize(), "sync")
    got = do.to_array(np.float32, (M, O))
    # FP8 tile scales come by 4-byte loads: no other path for them
    want = (gemm_tiled if fmt == 1 and what == "ws" else gemm_rows)(hip, fmt, w, ws, c, s)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
