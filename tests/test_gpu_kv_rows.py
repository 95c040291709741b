"""Carried keys in and out of the transposed K cache, position rows on the
host's side: what was written comes back, at tile edges, offsets and blocks
longer than the device staging, and nothing around it changes."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.direct import DeviceModel, Session

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def session():
    return make_session(1)


def make_session(layers):
    native.check(native.lib().q8gpu_init(), "q8gpu_init")
    m = synth.mistral_model(64, layers, 6, 3, 32, 64, 64, seed=5)  # kv rows of 96 values
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


def test_reads_from_several_threads():
    # Each thread its own layer and block length, so that the staging is
    # shared and grows between the calls.
    s = make_session(4)
    rng = np.random.default_rng(1)
    keys = [[rng.integers(-2 ** 31, 2 ** 31, (9000, 96)).astype(np.int32) for _ in range(2)] for _ in range(4)]
    for layer, (k, v) in enumerate(keys):
        s.write_kv(layer, 0, k, v)

    def read(layer):
        for i in range(40):
            p, n = 17 * i + layer, 100 + 1500 * layer + 31 * i
            k, v = s.read_kv(layer, p, n)
            if not (np.array_equal(k, keys[layer][0][p:p + n]) and np.array_equal(v, keys[layer][1][p:p + n])):
                return False
        return True

    with ThreadPoolExecutor(4) as ex:
        assert all(ex.map(read, range(4)))
