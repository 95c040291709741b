"""GPU parity of the products of few tokens (16 x 16 and 32 x 32 tiles, the
waves sharing one tile's k steps) against the oracle, every output exact."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.tensor import Q8Matrix
from oracle import cpu
from test_gpu_q8_product import per_block_matrix, product_ws, rand_activations

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")


# Token counts at the edges of both tile shapes and of their dispatch; rows
# that leave the last 16-row tile partial or a 32-row tile half empty; one k
# step, fewer steps than waves, and step counts that leave waves uneven.
@pytest.mark.parametrize("tokens,rows,cols", [(2, 1, 64), (16, 17, 64), (13, 200, 4160), (17, 16, 128), (32, 33, 576),
                                              (33, 250, 4160), (64, 144, 1088), (65, 48, 192), (16, 4100, 256),
                                              (31, 48, 14336)])
@pytest.mark.parametrize("kind", ["row", "unit", "tiny", "same", "spread4"])
def test_few_token_products(tokens, rows, cols, kind):
    print(f"{kind} tokens {tokens} rows {rows} cols {cols}", flush=True)
    rng = np.random.default_rng(tokens * 31 + rows + cols)
    if kind == "row":
        raw = synth.q8_matrix(synth.tensor_seed(19, rows), rows, cols, synth.scale_base_for(cols), True)
    else:
        raw = per_block_matrix(rng, rows, cols, kind)
    m = Q8Matrix.from_bytes(raw, rows, cols)
    for bits in (7, 16, 22, 32):  # one to five activation digits
        x = rand_activations(rng, tokens, cols, bits)
        if bits < 32:
            x = np.clip(x, -(1 << (bits - 1)), (1 << (bits - 1)) - 1).astype(np.int32)
        assert np.array_equal(product_ws(m, x), cpu.linear_q8(x, raw))


# Where the tiled GEMM takes over: past three tiles of 32 rows and tokens per
# CU (256) with row scales, four up to 64 tokens, five with per-block scales.
@pytest.mark.parametrize("scales,rows,tokens,few", [
    ("row", 4096, 16, True), ("row", 4096, 192, True), ("row", 4096, 193, False), ("row", 4096, 256, False),
    ("row", 16384, 64, True), ("row", 16416, 64, False), ("row", 28672, 32, True), ("row", 28672, 33, False),
    ("block", 4096, 320, True), ("block", 4096, 321, False), ("block", 28672, 32, True), ("block", 28672, 33, False),
    ("unfolded", 4096, 2048, True)])
def test_few_token_rule(scales, rows, tokens, few):
    raw = synth.q8_matrix(3, rows, 64, synth.scale_base_for(64), scales == "row")
    m = Q8Matrix.from_bytes(raw, rows, 64)
    if scales == "block":
        m.prepare_matrix_cores()
    assert m.route(tokens).startswith("few") == few, m.route(tokens)


def test_products_past_one_launch_stay_on_the_vector_path():
    # 300000 unfolded rows and 60000 tokens (a 72 GB result) are 17.6 M tiles
    # of 256 threads, past the 2^32 threads of a launch.
    m = Q8Matrix.from_bytes(synth.q8_matrix(3, 300000, 64, synth.scale_base_for(64), False), 300000, 64)
    assert m.route(50000) == "few 32x32, 4 waves"
    assert m.route(60000) == "per token"
