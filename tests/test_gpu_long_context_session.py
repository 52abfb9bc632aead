"""Decode steps of a Session (and one-token calls) whose cache is too long for one workgroup's LDS: the step that is captured as a HIP graph keeps
its score rows in global memory, which the first (op by op) step has to have made, as nothing is allocated in a capture."""
import numpy as np
import pytest

import oracle as O
from conftest import bits_equal
from edgelm_amd import elmh as E
from edgelm_amd import host
from edgelm_amd import synth as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [64, 16])
def test_steps_replay_over_a_cache_past_lds(tmp_path, monkeypatch, hd):
    ctx = 30016
    path = str(tmp_path / "m.elm")
    S.write_model(path, dict(S.TINY, dim=2 * hd, n_heads=2, n_kv_heads=1, head_dim=hd, max_seq=ctx), "q4", seed=5, sd=0.15, embed_sd=0.5)
    m = host.Model(path)
    mine = host.Session(m, "hip,cpu", max_ctx=ctx, max_batch=8, act_quant=True)
    monkeypatch.setenv("EDGELM_HIP_GRAPHS", "0")
    eager = host.Session(m, "hip,cpu", max_ctx=ctx, max_batch=8, act_quant=True)
    for i, t in enumerate((3, 7, 1, 9, 4)):  # op by op, captured, replayed
        print(f"[gpu] head size {hd}, {ctx} positions: step {i}", flush=True)
        toks = np.array([t], np.int32)
        assert bits_equal(mine.forward(toks), eager.forward(toks)), f"step {i}"
    mine.close(), eager.close()


def test_one_token_call_captured_without_a_step_before_it():
    """A one-token call at a short position is captured as it is, with nothing run before it: the rows that the same step would
    need over the whole cache are made outside captures only."""
    nh, nkv, hd, mc, pos = 4, 2, 128, 32768, 70
    r = np.random.default_rng(3)
    tab = O.rope_table(hd, mc, 10000.0)
    kc, vc = (r.normal(0, 1, (nkv, mc, hd)).astype(np.float32) for _ in range(2))
    q = r.normal(0, 1, (1, nh * hd)).astype(np.float32)
    k, v = (r.normal(0, 1, (1, nkv * hd)).astype(np.float32) for _ in range(2))
    with E.Context(0) as c:
        up = lambda a: c.buffer(a.nbytes).upload(a)  # noqa: E731
        bufs = [up(a) for a in (q, k, v, kc, vc, *tab)] + [c.buffer(q.nbytes)]
        bq, bk, bv, bkc, bvc, bc, bs, bo = bufs
        print(f"[gpu] one-token attention captured first, {mc} positions", flush=True)
        c.graph_begin()
        c.attention_dev(bq.ptr, bk.ptr, bv.ptr, bo.ptr, 1, pos, nh, nkv, hd, bkc.ptr, bvc.ptr, mc, bc.ptr, bs.ptr)
        g = c.graph_end()
        want = O.attention(q, k, v, pos, nh, nkv, kc, vc, tab)
        for _ in range(3):
            c.graph_launch(g)
            assert bits_equal(bo.download(q.shape, np.float32), want)
        c.graph_destroy(g)
        for b in bufs:
            b.free()
