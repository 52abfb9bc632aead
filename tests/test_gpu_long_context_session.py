"""Decode steps of a Session whose cache is too long for one workgroup's LDS: the step that is captured as a HIP graph keeps
its score rows in global memory, which the first (op by op) step has to have made, as nothing is allocated in a capture."""
import numpy as np
import pytest

from conftest import bits_equal
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
