"""GPU parity of the tiled multi-token products' ends of blocks: sums rounded
in double (ties, saturation, and the blocks that are redone wide), partial
row and token tiles, the 128-token per-block shape and its two-pass form for
four and five activation digits; each launch shape by name, over k loops that
wrap its ring. Outputs exact against the oracle."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.tensor import Q8Matrix
from oracle import cpu
from test_gpu_q8_product import grouped_activations, per_block_matrix, product_ws, rand_activations

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
# 128-token shape runs, its last row and token tiles partial; 300 x 4100: the
# 64-token shapes, the last 16-row tile partial too; 257 x 4100: the same with
# row scales, the few-token product per block.
@pytest.mark.parametrize("tokens,rows,cols", [(600, 4160, 128), (257, 4100, 192), (300, 4100, 192)])
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


def check_route(m, raw, tokens, cols, route):
    """The product takes `route`, and the outputs of the edge rows and 160
    more, over token groups of one to five digits, are the oracle's."""
    print(f"{route}: tokens {tokens} rows {m.rows} cols {cols}", flush=True)
    assert m.route(tokens) == route
    rng = np.random.default_rng(tokens + m.rows + cols)
    x = grouped_activations(rng, tokens, cols)
    sel = np.unique(np.r_[0, m.rows - 17:m.rows, rng.choice(m.rows, 160)])
    assert np.array_equal(product_ws(m, x)[:, sel], cpu.linear_q8(x, raw[sel]))


# Short and long k loops, odd step counts (no split), and rows long enough
# for the deeper rings; 603 tokens hold a group of each digit count.
@pytest.mark.parametrize("rows,cols,route", [
    (1400, 192, "tiled 128x64"), (1400, 4160, "tiled 128x64"), (1400, 256, "tiled 128x64 split"),
    (1400, 4224, "tiled 128x64 split"), (1400, 8192, "tiled 128x64 split deep"), (3300, 192, "tiled 128x128"),
    (3300, 4160, "tiled 128x128"), (3300, 256, "tiled 128x128 split"), (3300, 4224, "tiled 128x128 split"),
    (3300, 8192, "tiled 128x128 split deep"), (6700, 256, "tiled 256x128"), (6700, 4224, "tiled 256x128"),
    (13400, 4160, "tiled 256x128")])
def test_row_scale_shapes(rows, cols, route):
    raw = synth.q8_matrix(synth.tensor_seed(21, rows), rows, cols, synth.scale_base_for(cols), True)
    check_route(Q8Matrix.from_bytes(raw, rows, cols), raw, 603, cols, route)


@pytest.mark.parametrize("kind,planes,rows,tokens", [
    ("tiny", 2, 2200, "128x64"), ("same", 3, 2200, "128x64"), ("same", 3, 3300, "128x128"),
    ("spread4", 3, 3300, "128x128"), ("spread12", 4, 700, "64x64"), ("widest", 6, 700, "64x64")])
@pytest.mark.parametrize("cols", [128, 1088, 4224])
def test_folded_shapes(kind, planes, rows, tokens, cols):
    raw = per_block_matrix(np.random.default_rng(rows + cols), rows, cols, kind)
    b = raw.reshape(rows, cols // 32, 34)
    b[:, :, 2:][b[:, :, 2:] == 0x80] = 0x81  # no -128: the widest matrices then always fold
    m = Q8Matrix.from_bytes(raw, rows, cols)
    m.prepare_matrix_cores()
    check_route(m, raw, 603, cols, f"folded {tokens}, {planes} planes")


# Matrices as uploaded, one scale per block: both tile sides, shared by eight
# waves and, past one tile per CU, by four; four digits and more stay on the
# vector path.
@pytest.mark.parametrize("kind,rows,tokens,route", [
    ("same", 100, 16, "few 16x16, 8 waves"), ("same", 4200, 16, "few 16x16, 4 waves"),
    ("same", 300, 603, "few 32x32, 8 waves"), ("same", 1100, 603, "few 32x32, 4 waves"),
    ("spread4", 1100, 603, "few 32x32, 4 waves"), ("spread12", 300, 70, "per token")])
@pytest.mark.parametrize("cols", [64, 1088])
def test_unfolded_shapes(kind, rows, tokens, route, cols):
    raw = per_block_matrix(np.random.default_rng(rows + cols), rows, cols, kind)
    check_route(Q8Matrix.from_bytes(raw, rows, cols), raw, tokens, cols, route)


def test_wide_row_scales_through_the_tiles():
    # Scales from zero and subnormals up to f16 exponent 30 (2^40 in Q.24),
    # both signs, against magnitudes from 8 to 32 bits: sums rounded in
    # double, and blocks past 2^42 redone wide.
    rng = np.random.default_rng(31)
    rows, cols, tokens = 8400, 256, 96
    bits = (rng.integers(0, 2, 512) << 15) | (rng.integers(0, 31, 512) << 10) | rng.integers(0, 1024, 512)
    bits[:3] = [0, 0x8000, 0x0001]  # zero, negative zero, the smallest subnormal
    raw = row_matrix(rng, rows, cols, bits)
    m = Q8Matrix.from_bytes(raw, rows, cols)
    assert m.route(tokens).startswith("tiled")
    x = np.concatenate([rand_activations(rng, 1, cols, int(b)) for b in np.linspace(8, 32, tokens).astype(int)])
    assert np.array_equal(product_ws(m, x), cpu.linear_q8(x, raw))
