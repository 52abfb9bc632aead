"""The chunk attention kernels that share a kv head's rows (attention_rows_kernel, 4 and 8 rows a workgroup, head sizes up to 64
and over) and the workgroup-per-row kernel (attention_step_kernel) at the edges of their tiles, bit for bit against the oracle:
head sizes 16 does not divide, groups that the rows of a workgroup straddle, positions around the 16-, 64- and 256-position
steps, and a last token whose key and value are NaN and infinite, which no earlier token may see. Past the positions whose
score rows those keep in LDS, and for key caches off 16 bytes: attention_kernel."""
import numpy as np
import pytest

import oracle as O
from conftest import bits_equal

pytestmark = pytest.mark.gpu

# (n_heads, n_kv, head_dim, max_ctx, pos0, T): 4 rows (T * heads / 8 < 1024), 8 rows, one workgroup per row (<= 256)
SHAPES = [(8, 2, 128, 400, 0, 65), (12, 4, 96, 330, 250, 33), (6, 2, 100, 90, 3, 61), (5, 1, 256, 100, 15, 60), (16, 4, 4, 70, 0, 64),
          (32, 8, 64, 300, 1, 257), (32, 8, 20, 300, 0, 257),
          # 8 rows at head sizes over 64, a ragged last group of them; over 128 the dims take two passes
          (32, 8, 128, 300, 1, 257), (32, 8, 100, 300, 0, 257), (32, 8, 192, 300, 0, 257),
          # chunks whose score rows only attention_kernel keeps in LDS
          (4, 1, 64, 10100, 10020, 65), (4, 1, 128, 10100, 10020, 65),
          (8, 8, 80, 1100, 1020, 3), (4, 1, 128, 80, 0, 64),
          (9, 3, 64, 80, 60, 5), (9, 3, 64, 200, 126, 2), (9, 3, 64, 200, 126, 3), (4, 1, 64, 400, 300, 64)]  # 128 positions, past them


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("rope", [True, False])
def test_chunk_attention_bit_exact(ctx, shape, rope):
    nh, nkv, hd, mc, pos0, T = shape
    r = np.random.default_rng(nh * 1000 + hd + T)
    tab = O.rope_table(hd, mc, 10000.0) if rope else None
    kc, vc = (r.normal(0, 1, (nkv, mc, hd)).astype(np.float32) for _ in range(2))
    q = r.normal(0, 1, (T, nh * hd)).astype(np.float32)
    k, v = (r.normal(0, 1, (T, nkv * hd)).astype(np.float32) for _ in range(2))
    k[-1, ::2] = np.nan
    v[-1, ::3], v[-1, 1::3] = np.inf, np.nan
    vc[:, pos0 + T:] = np.nan  # past the chunk
    up = lambda a: ctx.buffer(a.nbytes).upload(a)  # noqa: E731
    bufs = [up(a) for a in (q, k, v, kc, vc)] + [ctx.buffer(q.nbytes)] + ([up(tab[0]), up(tab[1])] if rope else [])
    bq, bk, bv, bkc, bvc, bo = bufs[:6]
    print(f"[gpu] chunk attention {shape} rope={rope}", flush=True)
    ctx.attention_dev(bq.ptr, bk.ptr, bv.ptr, bo.ptr, T, pos0, nh, nkv, hd, bkc.ptr, bvc.ptr, mc,
                      *([bufs[6].ptr, bufs[7].ptr] if rope else [None, None]))
    want = O.attention(q, k, v, pos0, nh, nkv, kc, vc, tab)
    got = bo.download(q.shape, np.float32)
    assert bits_equal(got[:-1], want[:-1])
    assert np.array_equal(np.isnan(got[-1]), np.isnan(want[-1]))
    n = pos0 + T - 1
    assert bits_equal(bkc.download(kc.shape, np.float32)[:, :n], kc[:, :n])
    assert bits_equal(bvc.download(vc.shape, np.float32)[:, :n], vc[:, :n])
    for b in bufs:
        b.free()


@pytest.mark.parametrize("T", [257, 512])
def test_chunk_attention_writes_the_gemm_operand(ctx, T):
    """Head size 64 with 4096 (token, head) pairs or more: the rows kernel hands its output over quantized (16 heads: 4 rows
    a workgroup at 257 tokens, 8 at 512)."""
    nh, nkv, hd, mc, pos0 = 16, 8, 64, 600, 7
    r = np.random.default_rng(T)
    tab = O.rope_table(hd, mc, 10000.0)
    kc, vc = (r.normal(0, 1, (nkv, mc, hd)).astype(np.float32) for _ in range(2))
    q = r.normal(0, 1, (T, nh * hd)).astype(np.float32)
    k, v = (r.normal(0, 1, (T, nkv * hd)).astype(np.float32) for _ in range(2))
    w = O.make_weight(r.normal(0, 0.05, (72, nh * hd)).astype(np.float32), O.Q4)
    dw = ctx.upload(w.dtype, w.rows, w.cols, w.data, w.scales)
    up = lambda a: ctx.buffer(a.nbytes).upload(a)  # noqa: E731
    bufs = [up(a) for a in (q, k, v, kc, vc, *tab)] + [ctx.buffer(q.nbytes), ctx.buffer(T * 72 * 4)]
    bq, bk, bv, bkc, bvc, bc, bs, bo, by = bufs
    print(f"[gpu] chunk attention + matmul T={T}", flush=True)
    ctx.attention_matmul_dev(bq.ptr, bk.ptr, bv.ptr, bo.ptr, T, pos0, nh, nkv, hd, bkc.ptr, bvc.ptr, mc, bc.ptr, bs.ptr, dw, by.ptr)
    assert ctx.attention_matmul_fused()
    att = O.attention(q, k, v, pos0, nh, nkv, kc, vc, tab)
    assert bits_equal(bo.download(q.shape, np.float32), att)
    assert bits_equal(by.download((T, 72), np.float32), O.cpu_matmul(att, [w], None, act_quant=True)[0])
    for b in bufs:
        b.free()
    dw.free()


@pytest.mark.parametrize("nh,nkv,hd", [(4, 2, 128), (3, 1, 100), (2, 1, 256), (4, 4, 16)])
def test_step_attention_bit_exact(ctx, nh, nkv, hd):
    """One token, its position in device memory, around the 16-, 64- and 1024-position steps and the 64 value rows in flight;
    the cache past the step's position is NaN."""
    mc = 1200
    r = np.random.default_rng(hd + mc)
    tab = O.rope_table(hd, mc, 10000.0)
    up = lambda a: ctx.buffer(a.nbytes).upload(a)  # noqa: E731
    for pos in (0, 1, 15, 16, 63, 64, 65, 127, 128, 129, 191, 192, 700, 1023, 1024, 1100):
        kc, vc = (r.normal(0, 1, (nkv, mc, hd)).astype(np.float32) for _ in range(2))
        kc[:, pos:], vc[:, pos:] = np.nan, np.nan
        q = r.normal(0, 1, (1, nh * hd)).astype(np.float32)
        k, v = (r.normal(0, 1, (1, nkv * hd)).astype(np.float32) for _ in range(2))
        bufs = [up(a) for a in (q, k, v, kc, vc, *tab, np.array([pos], np.int32))] + [ctx.buffer(q.nbytes)]
        bq, bk, bv, bkc, bvc, bc, bs, bp, bo = bufs
        print(f"[gpu] step attention {nh, nkv, hd, mc} position {pos}", flush=True)
        ctx.attention_step_dev(bq.ptr, bk.ptr, bv.ptr, bo.ptr, bp.ptr, nh, nkv, hd, bkc.ptr, bvc.ptr, mc, bc.ptr, bs.ptr)
        want = O.attention(q, k, v, pos, nh, nkv, kc, vc, tab)
        assert bits_equal(bo.download(q.shape, np.float32), want)
        n = pos + 1
        assert bits_equal(bkc.download(kc.shape, np.float32)[:, :n], kc[:, :n])
        assert bits_equal(bvc.download(vc.shape, np.float32)[:, :n], vc[:, :n])
        for b in bufs:
            b.free()


@pytest.mark.parametrize("nh,nkv,hd", [(4, 2, 128), (6, 2, 20)])
@pytest.mark.parametrize("pos,T,step", [(0, 1, True), (90, 1, True), (90, 1, False), (70, 33, False), (30, 3, False)])
def test_attention_key_cache_off_16_bytes(ctx, nh, nkv, hd, pos, T, step):
    """A key cache that starts 4 bytes off: the kernels that copy its rows 16 bytes at a time leave it to attention_kernel,
    for one token with the append inside."""
    mc = 110
    r = np.random.default_rng(hd + pos + T)
    tab = O.rope_table(hd, mc, 10000.0)
    up = lambda a: ctx.buffer(a.nbytes).upload(a)  # noqa: E731
    kc, vc = (r.normal(0, 1, (nkv, mc, hd)).astype(np.float32) for _ in range(2))
    q = r.normal(0, 1, (T, nh * hd)).astype(np.float32)
    k, v = (r.normal(0, 1, (T, nkv * hd)).astype(np.float32) for _ in range(2))
    off = np.concatenate([np.zeros(1, np.float32), kc.ravel()])
    bufs = [up(a) for a in (q, k, v, off, vc, *tab, np.array([pos], np.int32))] + [ctx.buffer(q.nbytes)]
    bq, bk, bv, bkc, bvc, bc, bs, bp, bo = bufs
    print(f"[gpu] attention, key cache off 16 bytes: {nh, nkv, hd} position {pos} T={T} step={step}", flush=True)
    if step:
        ctx.attention_step_dev(bq.ptr, bk.ptr, bv.ptr, bo.ptr, bp.ptr, nh, nkv, hd, bkc.ptr + 4, bvc.ptr, mc, bc.ptr, bs.ptr)
    else:
        ctx.attention_dev(bq.ptr, bk.ptr, bv.ptr, bo.ptr, T, pos, nh, nkv, hd, bkc.ptr + 4, bvc.ptr, mc, bc.ptr, bs.ptr)
    want = O.attention(q, k, v, pos, nh, nkv, kc, vc, tab)
    assert bits_equal(bo.download(q.shape, np.float32), want)
    assert bits_equal(bkc.download(off.shape, np.float32)[1:].reshape(kc.shape), kc)
    assert bits_equal(bvc.download(vc.shape, np.float32), vc)
    for b in bufs:
        b.free()
