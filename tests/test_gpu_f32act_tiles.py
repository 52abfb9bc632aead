"""The f32-activation kernels at the sizes where their dispatch or tiles turn, bit for bit against the oracle: the LDS-tile
GEMM's four tiles with ragged rows, tokens and row lengths (K past and short of whole 16s, 32s and 128s, K below 4), several
targets, and the long-row one-token q4 GEMV with one and several row sets per workgroup, RMSNORM inside and outside."""
import numpy as np
import pytest

import oracle as O
from conftest import bits_equal
from edgelm_amd import elmh as E

pytestmark = pytest.mark.gpu


def up(ctx, w):
    return ctx.upload(w.dtype, w.rows, w.cols, w.data, w.scales)


def weight(r, n, k, dt):
    return O.make_weight(r.normal(0, 0.05, (n, k)).astype(np.float32), dt)


# (rows, K, T): 64 x 32 tiles (512 workgroups; two steps and six, which use both buffers again), 64 x 16, 32 x 16, 16 x 8
TILES = [(2000, 96, 505), (2000, 352, 505), (1030, 160, 490), (1000, 288, 126), (70, 544, 9), (33, 2080, 2), (17, 32, 3)]


@pytest.mark.parametrize("shape", TILES, ids=["x".join(map(str, s)) for s in TILES])
@pytest.mark.parametrize("dt", [O.Q8, O.Q4])
def test_f32act_gemm_tiles(ctx, dt, shape):
    n, k, T = shape
    r = np.random.default_rng(n + k)
    for kk in [k] + ([k - 1, k - 18, k - 30] if dt == O.Q8 else []):
        ws = [weight(r, n, kk, dt), weight(r, 40, kk, dt)]
        x = r.normal(0, 1, (T, kk)).astype(np.float32)
        res = r.normal(0, 1, (T, n)).astype(np.float32)
        dws = [up(ctx, w) for w in ws]
        print(f"[gpu] f32act gemm tiles dt={dt} {n}x{kk} T={T}", flush=True)
        got = ctx.matmul(x, dws, [res, None], act=E.ACT_F32)
        for g, w in zip(got, O.cpu_matmul(x, ws, [res, None], act_quant=False)):
            assert bits_equal(g, w), f"K={kk}"
        wu = weight(r, n, kk, dt)
        du = up(ctx, wu)
        assert bits_equal(ctx.swiglu(x, dws[0], du, act=E.ACT_F32), O.cpu_swiglu(x, ws[0], wu, act_quant=False)), f"swiglu K={kk}"
        for d in dws + [du]:
            d.free()


# (rows, K, T): pairs of tokens (gemm_f32act_kernel), K past its 2048-element chunk, K % 4 and an odd last token, several row groups
PAIRS = [(12300, 90, 3), (24600, 2077, 2), (1540, 61, 33), (16400, 37, 7)]


@pytest.mark.parametrize("shape", PAIRS, ids=["x".join(map(str, s)) for s in PAIRS])
@pytest.mark.parametrize("dt", [O.Q8, O.Q4])
def test_f32act_gemm_pairs_of_tokens(ctx, dt, shape):
    n, k, T = shape
    k = k if dt == O.Q8 else k // 32 * 32
    r = np.random.default_rng(n + k)
    ws = [weight(r, n, k, dt), weight(r, 40, k, dt)]
    x = r.normal(0, 1, (T, k)).astype(np.float32)
    res = r.normal(0, 1, (T, n)).astype(np.float32)
    dws = [up(ctx, w) for w in ws]
    print(f"[gpu] f32act gemm pairs of tokens dt={dt} {n}x{k} T={T}", flush=True)
    for g, w in zip(ctx.matmul(x, dws, [res, None], act=E.ACT_F32), O.cpu_matmul(x, ws, [res, None], act_quant=False)):
        assert bits_equal(g, w)
    wu = weight(r, n, k, dt)
    du = up(ctx, wu)
    assert bits_equal(ctx.swiglu(x, dws[0], du, act=E.ACT_F32), O.cpu_swiglu(x, ws[0], wu, act_quant=False))
    for d in dws + [du]:
        d.free()


def test_f32act_gemm_rows_shorter_than_a_chain(ctx):
    r = np.random.default_rng(3)
    for k in (1, 2, 3, 4, 5, 7):
        w = weight(r, 20, k, O.Q8)
        x = r.normal(0, 1, (5, k)).astype(np.float32)
        d = up(ctx, w)
        assert bits_equal(ctx.matmul(x, [d], None, act=E.ACT_F32)[0], O.cpu_matmul(x, [w], None, act_quant=False)[0]), f"K={k}"
        d.free()


# (rows, K): 3, 2 and 1 row sets of a 256-thread workgroup, more than 256 groups, an odd number of groups
WIDE = [(200, 2080), (90, 2720), (77, 4096), (100, 8192), (72, 8224), (41, 14336)]


@pytest.mark.parametrize("shape", WIDE, ids=["x".join(map(str, s)) for s in WIDE])
def test_f32act_long_row_gemv(ctx, shape):
    n, k = shape
    r = np.random.default_rng(n)
    ws = [weight(r, n, k, O.Q4), weight(r, 24, k, O.Q4)]
    wu = weight(r, n, k, O.Q4)
    dws, du = [up(ctx, w) for w in ws], up(ctx, wu)
    x = r.normal(0, 1, (1, k)).astype(np.float32)
    res = r.normal(0, 1, (1, n)).astype(np.float32)
    print(f"[gpu] f32act long rows {n}x{k}", flush=True)
    got = ctx.matmul(x, dws, [res, None], act=E.ACT_F32)
    for g, w in zip(got, O.cpu_matmul(x, ws, [res, None], act_quant=False)):
        assert bits_equal(g, w)
    assert bits_equal(ctx.swiglu(x, dws[0], du, act=E.ACT_F32), O.cpu_swiglu(x, ws[0], wu, act_quant=False))
    if k <= 8192:  # RMSNORM in the call
        nw = r.normal(1, 0.1, k).astype(np.float32)
        xn = O.rmsnorm(x, nw, 1e-5)
        bx, bn, by = ctx.buffer(x.nbytes).upload(x), ctx.buffer(nw.nbytes).upload(nw), ctx.buffer(n * 4)
        ctx.rmsnorm_matmul_dev(bx.ptr, bn.ptr, 1e-5, 1, k, [dws[0]], [by.ptr], None, act=E.ACT_F32)
        assert bits_equal(by.download((1, n), np.float32), O.cpu_matmul(xn, [ws[0]], None, act_quant=False)[0])
        ctx.rmsnorm_swiglu_dev(bx.ptr, bn.ptr, 1e-5, 1, k, dws[0], du, by.ptr, act=E.ACT_F32)
        assert bits_equal(by.download((1, n), np.float32), O.cpu_swiglu(xn, ws[0], wu, act_quant=False))
        for b in (bx, bn, by):
            b.free()
    for d in dws + [du]:
        d.free()


# (rows of each target, K, RMSNORM inside, SwiGLU): several tiles per workgroup (more than 512 tiles), the last workgroups with one
# fewer, targets whose boundary a workgroup crosses between two of its tiles; 1, 2 and 3 row sets, 256 threads and more
TILED = [((4200, 1003, 40), 4128, True, False), ((24600, 100), 2080, True, False), ((8300,), 2752, True, True), ((8311,), 4096, False, True),
         ((8200, 4100, 16), 4096, False, False), ((4130, 8), 10272, False, False), ((4100,), 8192, True, True)]


@pytest.mark.parametrize("case", TILED, ids=["x".join(map(str, c[0] + (c[1],))) for c in TILED])
def test_f32act_long_row_gemv_several_tiles_a_workgroup(ctx, case):
    rows, k, norm, sw = case
    r = np.random.default_rng(rows[0] + k)

    def w(n):
        return O.make_weight(r.standard_normal((n, k), dtype=np.float32) * np.float32(0.05), O.Q4)

    ws = [w(n) for n in rows] + ([w(rows[0])] if sw else [])
    dws = [up(ctx, v) for v in ws]
    x = r.normal(0, 1, (1, k)).astype(np.float32)
    nw = r.normal(1, 0.1, k).astype(np.float32)
    xin = O.rmsnorm(x, nw, 1e-5) if norm else x
    bx, bn = ctx.buffer(x.nbytes).upload(x), ctx.buffer(nw.nbytes).upload(nw)
    by = [ctx.buffer(4 * n) for n in rows]
    print(f"[gpu] f32act long rows, several tiles: {case}", flush=True)
    if sw:
        if norm:
            ctx.rmsnorm_swiglu_dev(bx.ptr, bn.ptr, 1e-5, 1, k, dws[0], dws[1], by[0].ptr, act=E.ACT_F32)
        else:
            ctx.swiglu_dev(bx.ptr, 1, k, dws[0], dws[1], by[0].ptr, act=E.ACT_F32)
        want = [O.cpu_swiglu(xin, ws[0], ws[1], act_quant=False)]
    else:
        if norm:
            ctx.rmsnorm_matmul_dev(bx.ptr, bn.ptr, 1e-5, 1, k, dws, [b.ptr for b in by], None, act=E.ACT_F32)
        else:
            ctx.matmul_dev(bx.ptr, 1, k, dws, [b.ptr for b in by], None, act=E.ACT_F32)
        want = O.cpu_matmul(xin, ws, None, act_quant=False)
    for b, v in zip(by, want):
        assert bits_equal(b.download(v.shape, np.float32), v)
    for b in [bx, bn] + by:
        b.free()
    for d in dws:
        d.free()


def test_f32act_gemm_more_workgroups_than_a_grid(ctx):
    """One row and 67 million tokens as SwiGLU: 4.2 million workgroups of 512 threads, more than one launch is given (2^22), so a
    second one takes the last 589 tokens. x repeats a pattern of tokens, so every token's output is known."""
    k, pat, T = 4, 1 << 20, 16 * ((1 << 22) + 37) - 3
    r = np.random.default_rng(8)
    wg, wu = weight(r, 1, k, O.Q8), weight(r, 1, k, O.Q8)
    dg, du = up(ctx, wg), up(ctx, wu)
    x = r.normal(0, 1, (pat, k)).astype(np.float32)
    bx, by = ctx.buffer(T * k * 4), ctx.buffer(T * 4)
    bx.upload(x)
    for t in range(pat, T, pat):
        ctx.memcpy_d2d(bx.ptr + t * k * 4, bx.ptr, min(pat, T - t) * k * 4)
    print(f"[gpu] f32act gemm of {T} tokens", flush=True)
    ctx.swiglu_dev(bx.ptr, T, k, dg, du, by.ptr, act=E.ACT_F32)
    got = by.download((T,), np.float32).view(np.int32)
    want = O.cpu_swiglu(x, wg, wu, act_quant=False).ravel().view(np.int32)
    for t in range(0, T, pat):
        assert np.array_equal(got[t:t + pat], want[:min(pat, T - t)]), t
    for b in (bx, by):
        b.free()
    dg.free(), du.free()
