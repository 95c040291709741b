"""GPU parity of the tiled multi-token products' ends of blocks: sums rounded
in double (ties, saturation, and the blocks that are redone wide), partial
row and token tiles, the 128-token per-block shape and its two-pass form for
four and five activation digits, every output exact against the oracle."""
import numpy as np
import pytest

from iris_amd import native
from iris_amd.tensor import Q8Matrix
from oracle import cpu
from test_gpu_q8_product import per_block_matrix, product_ws, rand_activations

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")


def row_matrix(rng, rows, cols, bits):
    """Random weights, every scale of row r the f16 bits[r % len(bits)]."""
    nb = cols // 32
    raw = np.empty((rows, nb, 34), dtype=np.uint8)
    scale = np.array(bits, dtype=np.uint16)[np.arange(rows) % len(bits)]
    raw[:, :, :2] = scale.view(np.uint8).reshape(rows, 1, 2)
    raw[:, :, 2:] = rng.integers(0, 256, (rows, nb, 32), dtype=np.uint8)
    return raw.reshape(rows, nb * 34)


# 600 tokens x 4160 rows: more 64-token per-block workgroups than CUs, so the
# 128-token shape runs, its last row and token tiles partial; 257 x 4100: the
# 64-token shapes, the last 16-row tile partial too.
@pytest.mark.parametrize("tokens,rows,cols", [(600, 4160, 128), (257, 4100, 192)])
@pytest.mark.parametrize("kind", ["halves", "largest", "same", "spread4"])
def test_tiled_product_ends(tokens, rows, cols, kind):
    print(f"{kind} tokens {tokens} rows {rows} cols {cols}", flush=True)
    rng = np.random.default_rng(tokens + rows + cols)
    if kind == "halves":  # +-0.5 and 2^-24: every other sum is a tie, either sign
        raw = row_matrix(rng, rows, cols, [0x3800, 0xB800, 0x0001])
    elif kind == "largest":  # the largest f16, either sign, beside a zero
        raw = row_matrix(rng, rows, cols, [0x7BFF, 0xFBFF, 0x0000])
    else:
        raw = per_block_matrix(rng, rows, cols, kind)
    m = Q8Matrix.from_bytes(raw, rows, cols)
    m.prepare_matrix_cores()
    for bits in (7, 16, 22, 32):  # one to five activation digits
        x = rand_activations(rng, tokens, cols, bits)
        if bits < 32:
            x = np.clip(x, -(1 << (bits - 1)), (1 << (bits - 1)) - 1).astype(np.int32)
        assert np.array_equal(product_ws(m, x), cpu.linear_q8(x, raw))
