"""The measured cases: what a user of this library has it do.

Four kinds of call, each through a public entry point:

- ``product``: one exact Q8_0 x Q16.16 product. ``entry`` is "device" (device
  pointers on a stream, q8gpu_product_device_ws, the matrix prepared for the
  matrix cores as a long-lived program does) or "host" (the drop-in
  q8gpu_product through ``tensor.linear_slab_from_source``: host rows in and
  out, the matrix as uploaded).
- ``stage``: one layer over one range of rows with the keys of the positions
  before it carried in (``Session.layer_stage``), and the range's own keys
  read back, as a chain's layer stage does.
- ``chain``: every layer over one range with its rows and per-layer SHA-256
  checkpoints (``Session.layer_pass``).
- ``generate``: greedy generation (``Session.generate``): the prompt pass and
  then one pass per token, replayed as a graph, with every selection's logits.

Weights are Gaussian, quantised to Q8_0 the way a GGUF file's are (a block's
scale is its largest magnitude / 127, as f16: ``scales`` "block"), or with one
scale for a whole row as this repository's benchmark has them ("row").
Activations are rows of unit variance, what a norm leaves.

Every result is an integer that the reference's arithmetic fixes bit for bit,
so every tolerance is exact.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from iris_amd import native, scalars, synth
from iris_amd.direct import DeviceModel, Session
from iris_amd.model import PREFIX, MistralShape, Model
from iris_amd.tensor import Q8Matrix, linear_slab_from_source

ONE = 65536

# Layer shapes of this repository's two benchmark models.
MISTRAL = dict(hidden=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, vocab=32000)
GEMMA = dict(hidden=2048, heads=8, kv_heads=1, head_dim=256, ffn=16384, vocab=256000, ple=256)


def listed():
    return [
        # The smallest product of a decode step at Gemma-2B shape: the output
        # projection of one token. Latency and the launch count.
        dict(name="gemv_2048x2048_block", kind="product", entry="device", tokens=1, cols=2048, rows=2048, scales="block"),
        # One token through one feed-forward projection at Mistral-7B shape,
        # the benchmark's GEMV (one scale per row).
        dict(name="gemv_4096x14336_row", kind="product", entry="device", tokens=1, cols=4096, rows=14336, scales="row"),
        # A handful of tokens (a short prompt, a draft to verify) through the
        # down projection of a GGUF matrix.
        dict(name="product_13tok_14336x4096_block", kind="product", entry="device", tokens=13, cols=14336, rows=4096,
             scales="block"),
        # A short ragged prompt through the stacked q, k and v projections.
        dict(name="product_77tok_4096x6144_row", kind="product", entry="device", tokens=77, cols=4096, rows=6144,
             scales="row"),
        # The drop-in product as the reference's host side calls it, for a
        # short prompt: host buffers, a GGUF matrix as uploaded.
        dict(name="host_24tok_4096x4096_block", kind="product", entry="host", tokens=24, cols=4096, rows=4096,
             scales="block"),
        # The gate and up products of a 2048-row pass, for both layouts.
        dict(name="gemm_2048tok_4096x28672_row", kind="product", entry="device", tokens=2048, cols=4096, rows=28672,
             scales="row"),
        dict(name="gemm_2048tok_4096x28672_block", kind="product", entry="device", tokens=2048, cols=4096, rows=28672,
             scales="block"),
        # One layer of a chain over a short ragged range late in a text.
        dict(name="stage_45rows_at_1500", kind="stage", rows=45, start=1500, scales="block"),
        # One layer of a chain over a 512-row range in mid-text.
        dict(name="stage_512rows_at_512", kind="stage", rows=512, start=512, scales="row"),
        # The teacher-forced chain pass with its checkpoints, two layers deep.
        dict(name="chain_2048rows_2layers", kind="chain", rows=2048, layers=2, scales="row"),
        # Greedy decoding at Mistral-7B shape, four layers and the head.
        dict(name="decode_mistral_512_32", kind="generate", family="mistral", layers=4, prompt=512, tokens=32,
             scales="row"),
        # Greedy decoding at Gemma-2B shape, four layers and the tied head.
        dict(name="decode_gemma_128_32", kind="generate", family="gemma", layers=4, prompt=128, tokens=32,
             scales="block"),
    ]


def _log(rng, lo, hi, step=1):
    """A size in [lo, hi], uniform in its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    scales = rng.choice(["row", "block"])
    kind = rng.choice(["product", "product", "product", "stage", "stage", "chain", "generate"])
    if kind == "product":
        entry = rng.choice(["device", "device", "host"])
        cols = rng.choice([2048, 4096, 14336, _log(rng, 512, 16384, 32)])
        rows = _log(rng, 1024, min(28672, 4096 * 28672 // cols))
        tokens = 1 if rng.random() < 0.25 else _log(rng, 2, 512 if entry == "host" else 2048)
        if entry == "host" and scales == "block":
            tokens = min(tokens, 64)
        return dict(kind="product", entry=entry, tokens=tokens, cols=cols, rows=rows, scales=scales)
    if kind == "stage":
        return dict(kind="stage", rows=_log(rng, 2, 1024), start=rng.randrange(0, 2048), scales=scales)
    if kind == "chain":
        return dict(kind="chain", rows=_log(rng, 64, 2048 if scales == "row" else 768), layers=2, scales=scales)
    return dict(kind="generate", family=rng.choice(["mistral", "gemma"]), layers=rng.choice([2, 3, 4]),
                prompt=_log(rng, 4, 512), tokens=rng.randrange(8, 33), scales=scales)


# ------------------------------------------------------------------ inputs


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + salt * 7919 + 1) & 0x7FFFFFFFFFFF)
    return g


def _q8(seed, salt, rows, cols, scales, sigma):
    """Gaussian weights as Q8_0 bytes [rows, cols/32*34] on the GPU."""
    g = _gen(seed, salt)
    nb = cols // 32
    out = torch.empty((rows, nb, 34), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 26) // cols)
    for r0 in range(0, rows, step):
        n = min(step, rows - r0)
        w = torch.randn((n, nb, 32), device="cuda", generator=g) * sigma
        top = w.abs().amax(dim=2, keepdim=True)
        if scales == "row":
            top = top.amax(dim=1, keepdim=True).expand(n, nb, 1)
        d = (top / 127).to(torch.float16).contiguous()
        q = torch.clamp(torch.round(w / d.float()), -127, 127).to(torch.int8)
        out[r0:r0 + n, :, :2] = d.view(torch.uint8).view(n, nb, 2)
        out[r0:r0 + n, :, 2:] = q.view(torch.uint8)
    return out.view(rows, nb * 34)


def _host_q8(seed, salt, rows, cols, scales, sigma=None):
    return _q8(seed, salt, rows, cols, scales, sigma or 1.0 / math.sqrt(cols)).cpu().numpy()


def _rows(seed, salt, n, width, sigma=1.0):
    """Q16.16 rows, Gaussian of the given standard deviation."""
    x = torch.randn((n, width), device="cuda", generator=_gen(seed, salt)) * (sigma * ONE)
    return torch.round(x).to(torch.int32)


def _norm(seed, salt, width):
    x = torch.rand(width, device="cuda", generator=_gen(seed, salt))
    return (ONE + torch.floor((x - 0.5) * 16384)).to(torch.int32).cpu().numpy()


def _ids(seed, n, vocab):
    return torch.randint(0, vocab, (n,), device="cuda", generator=_gen(seed, 3)).cpu().numpy().astype(np.int64)


def _mistral(seed, layers, scales, vocab):
    m = MISTRAL
    h, f = m["hidden"], m["ffn"]
    q, kv = m["heads"] * m["head_dim"], m["kv_heads"] * m["head_dim"]
    shape = MistralShape(
        hidden_size=h, num_hidden_layers=layers, num_attention_heads=m["heads"], num_key_value_heads=m["kv_heads"],
        head_dim=m["head_dim"], intermediate_size=f, vocab_size=vocab, norm_eps=scalars.f32_to_acc_bits(1e-5),
        attention_scale_q32=scalars.attention_scale_q32(m["head_dim"]),
        rope_inverse_frequencies=scalars.plain_rope_inverse_frequencies(1_000_000, m["head_dim"]),
        max_positions=32768, tied_head=False)
    t = {PREFIX + "embed_tokens.weight": _host_q8(seed, 10, vocab, h, scales, 1.0),
         PREFIX + "norm.weight": _norm(seed, 11, h),
         PREFIX + "lm_head.weight": _host_q8(seed, 12, vocab, h, scales)}
    for layer in range(layers):
        at, s = f"{PREFIX}layers.{layer}.", 100 + 20 * layer
        for i, (name, r, c) in enumerate(_mistral_matrices()):
            t[at + name] = _host_q8(seed, s + i, r, c, scales)
        t[at + "input_layernorm.weight"] = _norm(seed, s + 10, h)
        t[at + "pre_feedforward_layernorm.weight"] = _norm(seed, s + 11, h)
    return Model("mistral-dense", shape, t)


def _mistral_matrices():
    m = MISTRAL
    h, f = m["hidden"], m["ffn"]
    q, kv = m["heads"] * m["head_dim"], m["kv_heads"] * m["head_dim"]
    return [("self_attn.q_proj.weight", q, h), ("self_attn.k_proj.weight", kv, h), ("self_attn.v_proj.weight", kv, h),
            ("self_attn.o_proj.weight", h, q), ("mlp.gate_proj.weight", f, h), ("mlp.up_proj.weight", f, h),
            ("mlp.down_proj.weight", h, f)]


def _gemma(seed, layers, scales):
    m = GEMMA
    h, f, p, v = m["hidden"], m["ffn"], m["ple"], m["vocab"]
    q, kv = m["heads"] * m["head_dim"], m["kv_heads"] * m["head_dim"]
    shape = synth.gemma_shape(h, layers, m["heads"], m["kv_heads"], m["head_dim"], v, p, eps=1e-6, rope_sliding=10_000,
                              rope_full=10_000, softcap=30.0, tied_head=True)

    def values(salt, rows, cols):
        return _rows(seed, salt, rows, cols, 1.0 / math.sqrt(cols)).cpu().numpy()

    t = {PREFIX + "embed_tokens.weight": _host_q8(seed, 10, v, h, scales),
         PREFIX + "embed_tokens_per_layer.weight": _host_q8(seed, 13, v, layers * p, scales, 1.0 / 16),
         PREFIX + "per_layer_model_projection.weight": values(14, layers * p, h),
         PREFIX + "per_layer_projection_norm.weight": _norm(seed, 15, p),
         PREFIX + "norm.weight": _norm(seed, 11, h)}
    for layer in range(layers):
        at, s = f"{PREFIX}layers.{layer}.", 100 + 30 * layer
        for i, (name, r, c) in enumerate([("self_attn.q_proj.weight", q, h), ("self_attn.k_proj.weight", kv, h),
                                          ("self_attn.v_proj.weight", kv, h), ("self_attn.o_proj.weight", h, q),
                                          ("mlp.gate_proj.weight", f, h), ("mlp.up_proj.weight", f, h),
                                          ("mlp.down_proj.weight", h, f)]):
            t[at + name] = _host_q8(seed, s + i, r, c, scales)
        t[at + "per_layer_input_gate.weight"] = values(s + 8, p, h)
        t[at + "per_layer_projection.weight"] = values(s + 9, h, p)
        for i, (name, width) in enumerate([("input_layernorm", h), ("post_attention_layernorm", h),
                                           ("pre_feedforward_layernorm", h), ("post_feedforward_layernorm", h),
                                           ("post_per_layer_input_norm", h), ("self_attn.q_norm", m["head_dim"]),
                                           ("self_attn.k_norm", m["head_dim"])]):
            t[at + name + ".weight"] = _norm(seed, s + 12 + i, width)
    return Model("gemma-dense", shape, t)


# ------------------------------------------------------------------ the calls


def prepare(case, seed):
    native.check(native.lib().q8gpu_init(), "q8gpu_init")
    if case["kind"] == "product":
        m = Q8Matrix.from_bytes(_host_q8(seed, 1, case["rows"], case["cols"], case["scales"]), case["rows"], case["cols"])
        x = _rows(seed, 2, case["tokens"], case["cols"])
        if case["entry"] == "host":
            return dict(case=case, matrix=m, x=x.cpu().numpy())
        ws = None
        if case["tokens"] > 1:
            m.prepare_matrix_cores()
            ws = torch.empty(native.lib().q8gpu_workspace_bytes(m.handle, case["tokens"]), dtype=torch.uint8,
                             device="cuda")
        out = torch.empty((case["tokens"], case["rows"]), dtype=torch.int32, device="cuda")
        return dict(case=case, matrix=m, x=x, out=out, ws=ws)
    if case["kind"] == "stage":
        n, start = case["rows"], case["start"]
        dm = DeviceModel(_mistral(seed, 1, case["scales"], 256))
        dm.model.tensors = {}
        session = Session(dm, start + n, n)
        k, v = _carried(seed, start)
        if start:
            session.write_kv(0, 0, k.cpu().numpy(), v.cpu().numpy())
        return dict(case=case, dm=dm, session=session, x=_rows(seed, 2, n, MISTRAL["hidden"]).cpu().numpy())
    if case["kind"] == "chain":
        dm = DeviceModel(_mistral(seed, case["layers"], case["scales"], 4096))
        dm.model.tensors = {}
        return dict(case=case, dm=dm, session=Session(dm, case["rows"], case["rows"]), ids=_ids(seed, case["rows"], 4096))
    if case["family"] == "mistral":
        dm = DeviceModel(_mistral(seed, case["layers"], case["scales"], MISTRAL["vocab"]))
    else:
        dm = DeviceModel(_gemma(seed, case["layers"], case["scales"]))
    dm.model.tensors = {}
    session = Session(dm, case["prompt"] + case["tokens"], case["prompt"])
    return dict(case=case, dm=dm, session=session, ids=_ids(seed, case["prompt"], dm.model.vocab))


def _carried(seed, start):
    width = MISTRAL["kv_heads"] * MISTRAL["head_dim"]
    return _rows(seed, 4, start, width), _rows(seed, 5, start, width)


def run(state):
    case = state["case"]
    if case["kind"] == "product":
        if case["entry"] == "host":
            return linear_slab_from_source(state["x"], state["matrix"])
        ws = state["ws"]
        native.check(native.lib().q8gpu_product_device_ws(
            state["matrix"].handle, state["x"].data_ptr(), case["tokens"], state["out"].data_ptr(),
            None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(),
            torch.cuda.current_stream().cuda_stream), "product")
        return state["out"]
    session = state["session"]
    if case["kind"] == "stage":
        out = session.layer_stage(0, state["x"], case["start"])
        k, v = session.read_kv(0, case["start"], case["rows"])
        return {"rows": out, "k": k, "v": v}
    if case["kind"] == "chain":
        rows, hashes = session.layer_pass(state["ids"])
        return {"rows": rows, "hashes": np.array([list(bytes.fromhex(h)) for h in hashes], dtype=np.uint8)}
    got = session.generate(state["ids"], case["tokens"], keep_logits=True)
    return {"logits": got.logits, "ids": np.array(got.token_ids, dtype=np.int64)}


def _layer_work(rows, start):
    """(weight bytes, K and V bytes, flops) of one Mistral-7B-shape layer."""
    m = MISTRAL
    weights = sum(r * c for _, r, c in _mistral_matrices())
    kvw, qw = m["kv_heads"] * m["head_dim"], m["heads"] * m["head_dim"]
    pairs = rows * start + rows * (rows + 1) // 2
    return weights * 34 // 32, 2 * 4 * kvw * (start + rows), 2 * rows * weights + 4 * pairs * qw


def work(case):
    if case["kind"] == "product":
        t, c, r = case["tokens"], case["cols"], case["rows"]
        return {"bytes": r * c * 34 // 32 + 4 * t * (c + r), "flops": 2 * t * r * c}
    if case["kind"] in ("stage", "chain"):
        n = case["rows"]
        w, kv, fl = _layer_work(n, case.get("start", 0))
        layers = case.get("layers", 1)
        return {"bytes": layers * (w + kv + 4 * n * MISTRAL["hidden"]) + 4 * n * MISTRAL["hidden"], "flops": layers * fl}
    p, t, n = case["prompt"], case["tokens"], case["layers"]
    m = MISTRAL if case["family"] == "mistral" else GEMMA
    kvw, qw = m["kv_heads"] * m["head_dim"], m["heads"] * m["head_dim"]
    weights = (2 * qw + 2 * kvw) * m["hidden"] + 3 * m["ffn"] * m["hidden"]
    layer = weights * 34 // 32
    values = weights
    head = m["vocab"] * m["hidden"]
    if case["family"] == "gemma":
        layer += 3 * 4 * m["ple"] * m["hidden"]
        values += 3 * m["ple"] * m["hidden"]
    passes = t - 1  # the last selection runs no pass
    ctx = passes * p + passes * (passes + 1) // 2
    pairs = p * (p + 1) // 2 + ctx
    return {"bytes": n * (layer * (1 + passes) + 8 * kvw * (p + ctx)) + t * (head * 34 // 32 + 4 * m["vocab"]),
            "flops": n * (2 * (p + passes) * values + 4 * pairs * qw) + 2 * t * head}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------ 64 bits


def _dequantised(raw, rows, cols):
    b = raw.view(rows, cols // 32, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).view(rows, cols)


def _weights(seed, salt, rows, cols, scales, sigma=None):
    return _dequantised(_q8(seed, salt, rows, cols, scales, sigma or 1.0 / math.sqrt(cols)), rows, cols)


def _exact_layer(seed, layer, scales, x, k_old, v_old):
    """One Mistral-7B-shape layer in float64, values (not Q16.16 integers)."""
    m, s = MISTRAL, 100 + 20 * layer
    n, start = x.shape[0], k_old.shape[0]
    hd, heads, kvh = m["head_dim"], m["heads"], m["kv_heads"]
    w = [lambda i=i, r=r, c=c: _weights(seed, s + i, r, c, scales) for i, (_, r, c) in enumerate(_mistral_matrices())]

    def norm(v, salt):
        g = torch.from_numpy(_norm(seed, salt, m["hidden"])).to(v.device).double() / ONE
        return v * torch.rsqrt((v * v).mean(dim=1, keepdim=True) + 1e-5) * g

    inv = 1_000_000.0 ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    angle = torch.arange(start, start + n, device="cuda", dtype=torch.float64)[:, None] * inv[None, :]
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]

    def rotate(v):
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], dim=-1).flatten(-2)

    h = norm(x, s + 10)
    q = rotate((h @ w[0]().T).view(n, heads, hd))
    k = rotate((h @ w[1]().T).view(n, kvh, hd))
    v = (h @ w[2]().T).view(n, kvh, hd)
    keys = torch.cat([k_old.view(start, kvh, hd), k])
    vals = torch.cat([v_old.view(start, kvh, hd), v])
    mask = torch.arange(start + n, device="cuda")[None, :] > torch.arange(start, start + n, device="cuda")[:, None]
    ctx = torch.empty((n, heads, hd), dtype=torch.float64, device="cuda")
    for i in range(heads):
        scores = (q[:, i] @ keys[:, i * kvh // heads].T) / math.sqrt(hd)
        ctx[:, i] = scores.masked_fill(mask, float("-inf")).softmax(dim=1) @ vals[:, i * kvh // heads]
    x = x + ctx.view(n, -1) @ w[3]().T
    h = norm(x, s + 11)
    gate = h @ w[4]().T
    return x + (gate * torch.sigmoid(gate) * (h @ w[5]().T)) @ w[6]().T, k.reshape(n, -1), v.reshape(n, -1)


def exact(case, seed):
    """The values without rounding to Q16.16 (in its units). None for
    generation: a later logit depends on which of two near-equal logits the
    selections before it took."""
    if case["kind"] == "product":
        x = _rows(seed, 2, case["tokens"], case["cols"]).double()
        return x @ _weights(seed, 1, case["rows"], case["cols"], case["scales"]).T
    if case["kind"] == "generate":
        return None
    if case["kind"] == "stage":
        x = _rows(seed, 2, case["rows"], MISTRAL["hidden"]).double() / ONE
        k, v = _carried(seed, case["start"])
        out, k, v = _exact_layer(seed, 0, case["scales"], x, k.double() / ONE, v.double() / ONE)
        return {"rows": out * ONE, "k": k * ONE, "v": v * ONE}
    width = MISTRAL["kv_heads"] * MISTRAL["head_dim"]
    none = torch.empty((0, width), dtype=torch.float64, device="cuda")
    ids = torch.from_numpy(_ids(seed, case["rows"], 4096)).cuda()
    x = _weights(seed, 10, 4096, MISTRAL["hidden"], case["scales"], 1.0)[ids]
    rows = []
    for layer in range(case["layers"]):
        x, _, _ = _exact_layer(seed, layer, case["scales"], x, none, none)
        rows.append(x * ONE)
    return {"rows": torch.stack(rows), "hashes": None}
