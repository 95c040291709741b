"""GPU parity of the few-tile attention (one head's keys dealt to eight
waves) against the oracle: a layer's rows, exact, at key counts that leave
waves without a step, one step each, and uneven runs; long carried texts;
values whose digits send a tile to the one-row routine, and queries or keys
of four digits, in the split and the four-head workgroups."""
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


# Layer 0's norm weights scaled so that its queries, keys and values need a
# fourth or fifth digit: every workgroup takes the one-row routine there.
@pytest.mark.parametrize("times", [1 << 7, 1 << 10, 1 << 14])
def test_split_attention_wide_values(times):
    m = synth.mistral_model(512, 2, 8, 2, 64, 512, 512, seed=77)
    key = synth.PREFIX + "layers.0.input_layernorm.weight"
    m.tensors[key] = (m.tensors[key].astype(np.int64) * times).clip(-2 ** 31, 2 ** 31 - 1).astype(np.int32)
    check(m, (40, 30))


# One side of layer 0's scores a thousand times as large and the other as
# small: four digits of queries or of keys against values of at most three,
# and scores that spread the weights. 530 rows of 32 heads and 520 of 16 at
# head size 256 are 272 and 132 four-head workgroups; the others are split.
@pytest.mark.parametrize("wide,other", [("q", "k"), ("k", "q")])
@pytest.mark.parametrize("hd,heads,kv,ranges", [(64, 8, 2, (40, 30)), (64, 4, 4, (150, 17)), (64, 32, 8, (530,)),
                                                (128, 8, 2, (70, 20)), (256, 8, 1, (400,)), (256, 16, 2, (520,))])
def test_four_digit_queries_or_keys(hd, heads, kv, ranges, wide, other):
    print(f"wide {wide} head size {hd} heads {heads}/{kv} ranges {ranges}", flush=True)
    n = sum(ranges)
    m = synth.mistral_model(512, 1, heads, kv, hd, 512, 512, seed=78)
    w = {p: m.tensors[synth.PREFIX + f"layers.0.self_attn.{p}_proj.weight"] for p in "qkv"}
    b = w[wide].reshape(w[wide].shape[0], -1, 34)
    b[:, :, 1] += 10 << 2  # the f16 exponent: times 2^10
    b = w[other].reshape(w[other].shape[0], -1, 34)
    b[:, :, 0], b[:, :, 1] = 8 + np.arange(b.shape[0])[:, None] % 8, 0  # about 2^-21
    # The digits, from the oracle: positions after 0 only rotate the pairs.
    ids = synth.token_ids(7, n, m.vocab)
    x = cpu.OracleRun(m, 16).embed(ids)
    norm = m.values(m.layer_name(0, "input_layernorm.weight"))
    x = np.stack([cpu.rms_norm(r, norm, m.shape.norm_eps) for r in x])
    top = {p: np.abs(cpu.linear_q8(x, w[p]).astype(np.int64)).reshape(n, -1, hd) for p in "qkv"}
    pair = {p: np.hypot(t[:, :, 0::2], t[:, :, 1::2]) for p, t in top.items()}  # rotation keeps it
    tiles = [pair[wide][t:t + 16].max(axis=(0, 2)).min() for t in range(0, n, 16)]
    assert min(tiles) > 2 ** 0.5 * 0x7F7F7F and pair[wide].max() < 0x7F7F7F7F
    assert pair[other].max() <= 0x7F7F7F and top["v"].max() <= 0x7F7F7F
    check(m, ranges)


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
