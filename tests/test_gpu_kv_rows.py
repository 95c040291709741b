"""Carried keys in and out of the transposed K cache, position rows on the
host's side: what was written comes back, at tile edges, offsets and blocks
longer than the device staging, and nothing around it changes."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.direct import DeviceModel, Session

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def session():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")
    m = synth.mistral_model(64, 1, 6, 3, 32, 64, 64, seed=5)  # kv rows of 96 values
    return Session(DeviceModel(m), 45000, 1)


@pytest.mark.parametrize("pos0,count", [(0, 1), (31, 2), (7, 31), (64, 33), (100, 1000), (3, 44997)])
def test_written_keys_come_back(session, pos0, count):
    rng = np.random.default_rng(count)
    mark = [rng.integers(-2 ** 31, 2 ** 31, (45000, 96)).astype(np.int32) for _ in range(2)]
    session.write_kv(0, 0, *mark)
    want = [a.copy() for a in mark]
    rows = [rng.integers(-2 ** 31, 2 ** 31, (count, 96)).astype(np.int32) for _ in range(2)]
    session.write_kv(0, pos0, *rows)
    for a, b in zip(want, rows):
        a[pos0:pos0 + count] = b
    got = session.read_kv(0, pos0, count)
    assert all(np.array_equal(a, b) for a, b in zip(got, rows))
    got = session.read_kv(0, 0, 45000)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
