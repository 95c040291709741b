"""GPU parity of the few-tile attention (one head's keys dealt to eight
waves) against the oracle: a layer's rows, exact, at key counts that leave
waves without a step, one step each, and uneven runs; long carried texts;
values and keys whose digits send a tile to the wider paths."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.direct import DeviceModel, Session
from oracle import cpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")


# A first range and a second over the keys it left. Head size 256 takes the
# path at 400 rows (four value passes) and the one-row routine at 130.
@pytest.mark.parametrize("hd,heads,kv,ranges", [
    (64, 8, 2, (2, 3)), (64, 4, 4, (64, 17)), (64, 8, 8, (150, 33)), (128, 8, 2, (15, 49)), (128, 4, 1, (63, 66)),
    (128, 8, 2, (513, 70)), (256, 8, 1, (400, 130))])
def test_split_attention_ranges(hd, heads, kv, ranges):
    print(f"head size {hd} heads {heads}/{kv} ranges {ranges}", flush=True)
    n = sum(ranges)
    m = synth.mistral_model(256, 2, heads, kv, hd, 512, 512, seed=hd + n)
    check(m, ranges)


# Layer 0's norm weights scaled so that its values, or its queries and keys
# alone (through their weights' rows), need a fourth or fifth digit.
@pytest.mark.parametrize("times", [1 << 7, 1 << 10, 1 << 14])
def test_split_attention_wide_values(times):
    m = synth.mistral_model(512, 2, 8, 2, 64, 512, 512, seed=77)
    key = synth.PREFIX + "layers.0.input_layernorm.weight"
    m.tensors[key] = (m.tensors[key].astype(np.int64) * times).clip(-2 ** 31, 2 ** 31 - 1).astype(np.int32)
    check(m, (40, 30))


def check(m, ranges):
    n = sum(ranges)
    ids = synth.token_ids(7, n, m.vocab)
    s = Session(DeviceModel(m), n + 5, max(ranges))
    got, pos = [], 0
    for r in ranges:
        rows, _ = s.layer_range(ids[pos:pos + r], pos)
        got.append(rows)
        pos += r
    got = np.concatenate(got, axis=1)
    _, want = cpu.OracleRun(m, n + 5).pass_rows(list(ids), 0, keep_layers=True)
    for layer in range(m.num_layers):
        assert np.array_equal(got[layer], want[layer]), layer
