"""RMSNORM alone and fused with the GEMM's quantizer at wide rows (four rows per workgroup up to
K = 2048, one past it), bit for bit against the oracle: the edges of the two ranges, odd numbers of
32-blocks, token counts that leave padded slots."""
import numpy as np
import pytest

import oracle as O
from conftest import bits_equal
from edgelm_amd import elmh as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [2048, 2080, 4096, 8160, 8192])
@pytest.mark.parametrize("T", [5, 37])
def test_rmsnorm_quantized_wide_rows(ctx, k, T):
    r = np.random.default_rng(k + T)
    ws = [O.make_weight(r.normal(0, 0.05, (m, k)).astype(np.float32), O.Q4) for m in (48, 20)]
    wu = O.make_weight(r.normal(0, 0.05, (48, k)).astype(np.float32), O.Q4)
    dws = [ctx.upload(w.dtype, w.rows, w.cols, w.data, w.scales) for w in ws + [wu]]
    x = (r.normal(0, 1, (T, k)) * np.exp(r.normal(0, 2, (T, 1)))).astype(np.float32)
    x[0, 32:64] = 0
    nw = r.normal(1, 0.2, k).astype(np.float32)
    xn = O.rmsnorm(x, nw, 1e-5)
    bx, bn, bh = (ctx.buffer(a.nbytes).upload(a) for a in (x, nw, np.zeros_like(x)))
    by = [ctx.buffer(T * m * 4) for m in (48, 20)]
    print(f"[gpu] rmsnorm + quantizer K={k} T={T}", flush=True)
    ctx.rmsnorm_dev(bx.ptr, bn.ptr, bh.ptr, T, k, 1e-5)
    assert bits_equal(bh.download(x.shape, np.float32), xn)
    ctx.rmsnorm_matmul_dev(bx.ptr, bn.ptr, 1e-5, T, k, dws[:2], [b.ptr for b in by], None, act=E.ACT_INT8)
    for b, w in zip(by, O.cpu_matmul(xn, ws, None, act_quant=True)):
        assert bits_equal(b.download(w.shape, np.float32), w)
    ctx.rmsnorm_swiglu_dev(bx.ptr, bn.ptr, 1e-5, T, k, dws[0], dws[2], by[0].ptr, act=E.ACT_INT8)
    assert bits_equal(by[0].download((T, 48), np.float32), O.cpu_swiglu(xn, ws[0], wu, act_quant=True))
    for b in [bx, bn, bh] + by:
        b.free()
    for d in dws:
        d.free()
