"""Kept logits of a generation that fills its pinned slots several times over
(a vocabulary wide enough that a run of steps is a few), launch by launch and
as graph replays, a second generation on the same session, and one whose last
run is partial; every logit against the oracle."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.direct import DeviceModel, Session
from oracle import cpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")


@pytest.mark.parametrize("use_graph", [True, False])
def test_kept_logits_in_runs(use_graph):
    m = synth.mistral_model(64, 1, 2, 1, 32, 128, 70000, seed=13)  # 280 kB of logits a step: runs of three
    s = Session(DeviceModel(m), 64, 8)
    for tokens in (1, 31, 17):
        print(f"graph {use_graph} tokens {tokens}", flush=True)
        prompt = synth.token_ids(tokens, 5, 70000)
        got = s.generate(prompt, tokens, keep_logits=True, use_graph=use_graph)
        want_tokens, want_logits = cpu.OracleRun(m, 64).generate(list(prompt), tokens, keep_logits=True)
        assert got.token_ids == want_tokens
        assert np.array_equal(got.logits, np.stack(want_logits))
