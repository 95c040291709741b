"""GPU parity of gemma-dense's Q16.16 projections on the matrix cores (two
digit planes per value) against the oracle: one- and two-digit weights up to
the ends of their range, a weight that needs a third digit and a width the
tiles do not take (both stay on the per-row kernel), and row counts at the
edges of the dispatch and of the token tiles; every layer's rows exact."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.direct import DeviceModel, Session
from oracle import cpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")


@pytest.mark.parametrize("kind", ["one", "two", "ends", "three"])
@pytest.mark.parametrize("ple,rows", [(64, 23), (64, 24), (128, 33), (64, 70), (32, 40)])
def test_ple_projections(kind, ple, rows):
    print(f"{kind} ple {ple} rows {rows}", flush=True)
    rng = np.random.default_rng(ple + rows)
    shape = synth.gemma_shape(256, 2, 4, 1, 64, 512, ple, softcap=30.0)
    m = synth.gemma_model(shape, 512, seed=3 + rows)
    for name, t in m.tensors.items():
        if "per_layer_model_projection" in name or "per_layer_input_gate" in name or \
                ("per_layer_projection" in name and "norm" not in name):
            lo, hi = {"one": (-128, 128), "two": (-3000, 3000)}.get(kind, (-32896, 32640))
            w = rng.integers(lo, hi, t.shape).astype(np.int32)
            if kind == "three":
                w.flat[0] = 32640
            m.tensors[name] = w
    ids = synth.token_ids(5, rows, m.vocab)
    got, _ = Session(DeviceModel(m), rows, rows).layer_pass(ids)
    _, want = cpu.OracleRun(m, rows).pass_rows(list(ids), 0, keep_layers=True)
    for layer in range(m.num_layers):
        assert np.array_equal(got[layer], want[layer]), layer


def test_model_device_bytes_count_the_planes():
    # Two planes of one byte per value and a 32-bit shift per row, rows padded
    # to whole 16-row tiles, for each of the three kinds of matrix; weights
    # that need a third digit get none.
    shape = synth.gemma_shape(256, 2, 4, 1, 64, 512, 64, softcap=30.0)
    for wide in (False, True):
        m = synth.gemma_model(shape, 512, seed=2)
        if wide:
            m.tensors[synth.PREFIX + "layers.1.per_layer_input_gate.weight"].flat[5] = 1 << 20
        dm = DeviceModel(m)
        before = dm.device_bytes()
        Session(dm, 8, 1)
        assert dm.device_bytes() == before
        Session(dm, 8, 8)
        planes = lambda rows, cols: rows * (2 * cols + 4)
        want = planes(2 * 64, 256) + 2 * planes(256, 64) + (1 if wide else 2) * planes(64, 256)
        assert dm.device_bytes() == before + want
