"""GPU parity of the multi-row attention where every score a row sees
saturates at the lowest i32: its first maximum is then its first visible key,
which keeps the residual weight (crates/det-num/src/ops.rs:233-261,
466-481). Head 0's keys are its queries negated, so that a row's score on its
own key is -|q|^2 / sqrt(head size); three- and four-digit queries, the
split and the four-head workgroups, and unscaled scores, the oracle's digits
and scores checked first and every row compared exactly."""
import numpy as np
import pytest

from iris_amd import native, synth
from iris_amd.direct import DeviceModel, Session
from iris_amd.model import PREFIX
from oracle import cpu

pytestmark = pytest.mark.gpu

LOWEST = -2 ** 31
THREE_DIGITS = 0x7F7F7F  # the largest value of three signed byte digits


@pytest.fixture(scope="module", autouse=True)
def device():
    native.check(native.lib().q8gpu_init(), "q8gpu_init")


def normed_rows(m, ids):
    x = cpu.OracleRun(m, 16).embed(ids)
    w = m.values(m.layer_name(0, "input_layernorm.weight"))
    return np.stack([cpu.rms_norm(r, w, m.shape.norm_eps) for r in x])


def opposed_mistral(heads, top):
    """A one-layer model whose head 0 has q = (c, 0, c, 0, ..) and k = -q
    before the rotation, c a single product of the token's row, and the ids
    of its tokens in falling order of |c|, which is about `top` at most."""
    hd, H = 64, 512
    m = synth.mistral_model(H, 1, heads, heads, hd, 512, 256, seed=heads)
    wq, wk = (m.tensors[PREFIX + f"layers.0.self_attn.{p}_proj.weight"] for p in "qk")
    base = wq[0].copy()
    for r in range(hd):
        blocks = [w[r].reshape(-1, 34) for w in (wq, wk)]
        for b, sign in zip(blocks, (1, -1)):
            q = base.reshape(-1, 34)[:, 2:].view(np.int8) if r % 2 == 0 else np.zeros((H // 32, 32), np.int8)
            b[:] = base.reshape(-1, 34)
            b[:, 2:] = (sign * q).astype(np.int8).view(np.uint8)
    ids = np.arange(m.vocab)
    c = np.abs(cpu.linear_q8(normed_rows(m, ids), wq[:1]).astype(np.int64)[:, 0])
    bits = int(wq[0, 0]) | int(wq[0, 1]) << 8
    scale = np.float16(np.array([bits], np.uint16).view(np.float16)[0] * (top / c.max()))
    bits = int(np.array([scale]).view(np.uint16)[0])
    for w in (wq, wk):
        b = w[:hd].reshape(hd, -1, 34)
        b[:, :, 0], b[:, :, 1] = bits & 0xFF, bits >> 8
    return m, ids[np.argsort(-c)]


# 530 rows of 32 heads: 272 four-head workgroups; 20 rows: one head each.
@pytest.mark.parametrize("heads,rows", [(4, 20), (32, 530)])
@pytest.mark.parametrize("top,digits", [(THREE_DIGITS * 0.99, 3), (1.2e8, 4)])
def test_lowest_scores_keep_the_first_key(heads, rows, top, digits):
    m, order = opposed_mistral(heads, top)
    ids = np.resize(order, rows)
    ids[:3] = order[0]  # three rows that see only saturated scores
    x = normed_rows(m, ids)
    q, k, v = (cpu.linear_q8(x, m.tensors[PREFIX + f"layers.0.self_attn.{p}_proj.weight"]) for p in "qkv")
    lim = {2: 0x7F7F, 3: THREE_DIGITS, 4: 0x7F7F7F7F}
    assert lim[digits - 1] < np.abs(q).max() <= lim[digits] and np.abs(v).max() <= THREE_DIGITS
    s = m.shape
    f = np.array(s.rope_inverse_frequencies)
    q, k = ([cpu.rotate_consecutive_pairs(a[p, :64], f, p) for p in range(3)] for a in (q, k))
    for p in range(3):
        for j in range(p + 1):
            assert cpu.lib().dn_scaled_score(q[p], k[j], 64, s.attention_scale_q32) == LOWEST
    check(m, ids)


def test_lowest_unscaled_scores_keep_the_first_key():
    # gemma-dense: the norms of the heads carry the size, the keys' negated.
    shape = synth.gemma_shape(256, 1, 4, 4, 64, 512, 64, softcap=30.0)
    m = synth.gemma_model(shape, 512, seed=9)
    at = PREFIX + "layers.0.self_attn."
    m.tensors[at + "k_proj.weight"] = m.tensors[at + "q_proj.weight"].copy()
    m.tensors[at + "q_norm.weight"] = np.full(64, 1_700_000, np.int32)
    m.tensors[at + "k_norm.weight"] = np.full(64, -1_700_000, np.int32)
    ids = synth.token_ids(3, 20, m.vocab)
    row = cpu.linear_q8(normed_rows(m, ids[:1]), m.tensors[at + "q_proj.weight"])[0]
    for h in range(4):
        q, k = (cpu.rms_norm(row[64 * h:64 * h + 64], m.tensors[at + f"{p}_norm.weight"], shape.norm_eps) for p in "qk")
        assert np.abs(q).max() <= THREE_DIGITS
        assert cpu.lib().dn_requantize(int(np.dot(q.astype(np.int64), k.astype(np.int64)))) == LOWEST
    check(m, ids)


def check(m, ids):
    print(f"{m.family} heads {m.shape.num_attention_heads} rows {len(ids)}", flush=True)
    got, _ = Session(DeviceModel(m), len(ids), len(ids)).layer_pass(ids)
    _, want = cpu.OracleRun(m, len(ids)).pass_rows(list(ids), 0, keep_layers=True)
    assert np.array_equal(got[0], want[0])
