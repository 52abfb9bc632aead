"""The int8 GEMM whose workgroups split K over their waves (gemm_split16_kernel) at the edges of its tiles and rounds, bit for
bit against the oracle: rows and tokens short of and past 16, block counts short of, at and past its 16- and 32-block rounds,
tile heights 4, 8, 16 and 32, several targets, residuals, SwiGLU, per-block and per-token scales, and its automatic choice
(K > 1536, few tokens) with one workgroup per CU and more (4100 x 1568: past its limit for per-block q8 SwiGLU)."""
import numpy as np
import pytest

import oracle as O
from conftest import bits_equal
from edgelm_amd import elmh as E

pytestmark = pytest.mark.gpu


def up(ctx, w):
    return ctx.upload(w.dtype, w.rows, w.cols, w.data, w.scales)


# (rows, second target's rows, K, T, forced): forced runs it below its automatic range too
CASES = [(17, 0, 32, 5, True), (70, 33, 480, 31, True), (64, 16, 512, 16, True), (100, 0, 544, 17, True),
         (48, 64, 1056, 33, True), (130, 40, 1600, 9, False), (96, 0, 2112, 48, False), (40, 24, 8224, 6, False),
         (24, 0, 16512, 7, False), (300, 4000, 1568, 16, False), (4100, 64, 1568, 17, False),
         (2100, 0, 2048, 17, False)]


@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c[:4])) for c in CASES])
@pytest.mark.parametrize("dt", [O.Q8, O.Q4])
def test_gemm_split_exact(ctx, dt, case, monkeypatch):
    n, n2, k, T, forced = case
    if forced:
        monkeypatch.setenv("ELMH_GEMM_KERNEL", "split")
    r = np.random.default_rng(n + k + T)
    ws = [O.make_weight(r.normal(0, 0.05, (m, k)).astype(np.float32), dt) for m in (n, n2) if m]
    wu = O.make_weight(r.normal(0, 0.05, (n, k)).astype(np.float32), dt)
    dws, du = [up(ctx, w) for w in ws], up(ctx, wu)
    x = r.normal(0, 1, (T, k)).astype(np.float32)
    res = [r.normal(0, 1, (T, n)).astype(np.float32)] + [None] * (len(ws) - 1)
    print(f"[gpu] split gemm dt={dt} {case}", flush=True)
    for g, w in zip(ctx.matmul(x, dws, res, act=E.ACT_INT8), O.cpu_matmul(x, ws, res, act_quant=True)):
        assert bits_equal(g, w)
    assert bits_equal(ctx.swiglu(x, dws[0], du, act=E.ACT_INT8), O.cpu_swiglu(x, ws[0], wu, act_quant=True))
    for T1 in (T, 1):
        x1 = np.ascontiguousarray(x[:T1])
        got = ctx.matmul(x1, dws, None, act=E.ACT_INT8_TOKEN)
        for g, w in zip(got, ws):
            assert bits_equal(g, O.matmul_a8_token(x1, w)), f"token T={T1}"
    g, u = O.matmul_a8_token(x, ws[0]), O.matmul_a8_token(x, wu)
    want = np.array([O.silu(float(v)) for v in g.ravel()], np.float32).reshape(g.shape) * u
    assert bits_equal(ctx.swiglu(x, dws[0], du, act=E.ACT_INT8_TOKEN), want)
    for d in dws + [du]:
        d.free()
