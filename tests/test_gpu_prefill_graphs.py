"""Prefill forwards replayed as HIP graphs (last-row logits, one graph per length and first position) with fresh tokens
every round, against a session with prefill graphs off: a replay must attend over the new tokens of every position, not
over what an earlier forward left in the buffers. Sessions that ask for every row's logits never replay a prefill, so the
logits here are the last row's."""
import numpy as np
import pytest

from conftest import bits_equal
from edgelm_amd import host
from edgelm_amd import synth as S

pytestmark = pytest.mark.gpu

# head size 64 (attention fused into the o projection's call) and 16 (the general attention kernel)
HD64 = dict(S.TINY, dim=128, n_heads=2, n_kv_heads=1, head_dim=64, max_seq=256)


@pytest.mark.parametrize("cfg", [HD64, S.TINY], ids=["hd64", "hd16"])
@pytest.mark.parametrize("act", [True, False], ids=["int8", "f32"])
def test_prefill_graph_replays_fresh_tokens(tmp_path, monkeypatch, cfg, act):
    path = str(tmp_path / "m.elm")
    S.write_model(path, cfg, "q4", seed=77, sd=0.15, embed_sd=0.5)
    m = host.Model(path)
    mine = host.Session(m, "hip,cpu", max_ctx=96, max_batch=32, act_quant=act)
    monkeypatch.setenv("EDGELM_HIP_PREFILL_GRAPHS", "0")
    eager = host.Session(m, "hip,cpu", max_ctx=96, max_batch=32, act_quant=act)
    r = np.random.default_rng(5)
    for rnd in range(4):  # op by op, captured, replayed, replayed
        mine.reset(), eager.reset()
        for n in (24, 24, 1, 7):
            toks = r.integers(0, cfg["vocab"], n).astype(np.int32)
            print(f"[gpu] prefill graphs round {rnd}: {n} tokens at position {mine.pos()}", flush=True)
            a, b = mine.forward(toks), eager.forward(toks)
            assert bits_equal(a, b), f"round {rnd}, {n} tokens: max diff {np.abs(a - b).max()}"
    mine.close(), eager.close()
