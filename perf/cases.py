"""Workloads of the quantized MatVec path, as programs that use this package run them: the cases whose times are
compared when a kernel changes.

A case is a dict of plain values. `listed()` gives the fixed ones, `draw(rng)` another of the same ranges,
`prepare(case, seed)` what a program holds before the call (resident matrices, groups, captured steps, inputs), `run(state)`
one pass through the public entry points, `work(case)` the bytes and operations no implementation can do
without, `tolerance(case)` how far two correct implementations may differ and `exact(case, seed)` the outputs in
64 bits from plain torch.

Kinds:
  matvec       one resident matrix, one activation vector (device pointers, or the synchronous host-buffer call)
  group        several matrices of one shape in one launch, one vector each (K formats: the Q8_K integer product)
  batch        one matrix over several positions (short prompts, drafts, prefill): FP32 activations for the legacy
               formats, the Q8_K integer product for the K formats
  group_batch  a K-format group sharing one input over several positions (gate and up of a prefill)
  attention    grouped attention of one query position over a cached prefix
  token        a whole decode token of a small Qwen-shaped model, captured once and replayed, logits read back
"""
from __future__ import annotations

import math

import numpy as np
import torch

import satori_amd as S
from satori_amd.decode import DecoderConfig, DeviceDecoder

FORMATS = {"q8_0": S.BlockQuantization.Q8_0, "q4_0": S.BlockQuantization.Q4_0, "q4_k": S.BlockQuantization.Q4_K,
           "q6_k": S.BlockQuantization.Q6_K}
BLOCK_BYTES = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210)}
HIDDEN, KV, FFN, HEADS, KV_HEADS, HEAD_DIM = 1536, 256, 8960, 12, 2, 128  # the 1.5B decoder's widths
EPSILON, ROPE_BASE = 1e-6, 1e6

# The most a drawn case may do, which is what the largest listed ones do.
MOST_WEIGHTS = 11008 * 4096
MOST_PRODUCTS = MOST_WEIGHTS * 256
MOST_GROUP_BYTES = 64 * 4718592


def listed() -> list[dict]:
    return [
        # The smallest call: a host program's Ternary2MatVec.Execute on a small matrix (copies, launch, wait).
        {"name": "t2_host_1024", "kind": "matvec", "format": "ternary2", "block": 64, "rows": 1024, "columns": 1024,
         "call": "host"},
        # The reference's own benchmark shape, one resident matrix: a projection of a ternary model's decode step.
        {"name": "t2_4096", "kind": "matvec", "format": "ternary2", "block": 128, "rows": 4096, "columns": 4096,
         "call": "device"},
        # The same shape over a model's worth of matrices in one launch, streamed from HBM.
        {"name": "t2_group_64", "kind": "group", "format": "ternary2", "block": 128, "rows": 4096, "columns": 4096,
         "members": 64},
        # One Q8_0 projection with FP32 activations.
        {"name": "q8_0_4096", "kind": "matvec", "format": "q8_0", "block": 0, "rows": 4096, "columns": 4096,
         "call": "device"},
        # A short prompt (or a draft to verify) through a Q8_0 projection.
        {"name": "q8_0_batch_12", "kind": "batch", "format": "q8_0", "rows": 4096, "columns": 4096, "positions": 12},
        # A prefill chunk through a Q4_0 up projection.
        {"name": "q4_0_batch_256", "kind": "batch", "format": "q4_0", "rows": 11008, "columns": 4096,
         "positions": 256},
        # Gate and up of one decode position: a Q4_K group on the Q8_K integer path.
        {"name": "q4k_gate_up", "kind": "group", "format": "q4_k", "block": 0, "rows": FFN, "columns": HIDDEN,
         "members": 2},
        # A few positions at once through a Q4_K projection (speculative decoding, the last tokens of a prompt).
        {"name": "q4k_batch_5", "kind": "batch", "format": "q4_k", "rows": 4096, "columns": 4096, "positions": 5},
        # Gate and up of a full prefill chunk.
        {"name": "q4k_prefill_256", "kind": "group_batch", "format": "q4_k", "rows": FFN, "columns": HIDDEN,
         "members": 2, "positions": 256},
        # The down projection of a prefill chunk that does not fill its last tile.
        {"name": "q6k_prefill_200", "kind": "batch", "format": "q6_k", "rows": HIDDEN, "columns": FFN,
         "positions": 200},
        # Attention of one decode position at the end of a 4096-token context.
        {"name": "attention_4096", "kind": "attention", "heads": HEADS, "kv_heads": KV_HEADS, "head_dim": HEAD_DIM,
         "tokens": 4096},
        # A whole decode token in the middle of a conversation.
        {"name": "token_6_layers", "kind": "token", "layers": 6, "vocab": 32000, "position": 1500},
    ]


def _log(rng, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _shape(rng, fmt: str, most: int) -> tuple[int, int]:
    """Rows and columns over their ranges: any row count, whole blocks of columns (any count for Ternary2)."""
    unit = 1 if fmt == "ternary2" else BLOCK_BYTES[fmt][0]
    while True:
        rows = _log(rng, 256, 14336)
        columns = max(2 * unit, _log(rng, 512, 14336) // unit * unit)
        if rows * columns <= most:
            return rows, columns


def draw(rng) -> dict:
    kind = rng.choice(["matvec", "matvec", "group", "batch", "batch", "batch", "group_batch", "attention", "token"])
    if kind == "matvec":
        fmt = rng.choice(["ternary2", "ternary2", "q8_0", "q4_0", "q4_k", "q6_k"])
        rows, columns = _shape(rng, fmt, MOST_WEIGHTS)
        return {"kind": kind, "format": fmt, "block": rng.choice([64, 128, 256]) if fmt == "ternary2" else 0,
                "rows": rows, "columns": columns, "call": rng.choice(["device", "device", "host"])}
    if kind == "group":
        fmt = rng.choice(["ternary2", "q4_k", "q6_k"])
        rows, columns = _shape(rng, fmt, MOST_WEIGHTS)
        members = min(_log(rng, 2, 64), max(2, MOST_GROUP_BYTES // (rows * columns)))
        return {"kind": kind, "format": fmt, "block": rng.choice([64, 128, 256]) if fmt == "ternary2" else 0,
                "rows": rows, "columns": columns, "members": members}
    if kind == "batch":
        fmt = rng.choice(["q8_0", "q4_0", "q4_k", "q6_k"])
        rows, columns = _shape(rng, fmt, MOST_WEIGHTS)
        return {"kind": kind, "format": fmt, "rows": rows, "columns": columns,
                "positions": min(_log(rng, 2, 256), MOST_PRODUCTS // (rows * columns))}
    if kind == "group_batch":
        fmt = rng.choice(["q4_k", "q6_k"])
        members = rng.choice([2, 3])
        rows, columns = _shape(rng, fmt, MOST_WEIGHTS // members)
        return {"kind": kind, "format": fmt, "rows": rows, "columns": columns, "members": members,
                "positions": _log(rng, 16, 256)}
    if kind == "attention":
        kv_heads = rng.choice([1, 2, 4, 8])
        return {"kind": kind, "heads": kv_heads * rng.choice([1, 2, 4, 6]), "kv_heads": kv_heads,
                "head_dim": rng.choice([64, 96, 128]), "tokens": _log(rng, 16, 8192)}
    return {"kind": "token", "layers": rng.randint(2, 6), "vocab": _log(rng, 8000, 32000),
            "position": _log(rng, 32, 4000)}


# ---- inputs, from the seed alone ----

def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _bytes(t: torch.Tensor) -> torch.Tensor:
    """The bytes of a tensor's elements, as a new last dimension."""
    return t.contiguous().view(torch.uint8).reshape(*t.shape, t.element_size())


def _weights(g, fmt: str, rows: int, columns: int, block: int = 0):
    """A payload quantized from N(0, 0.02) weights (Ternary2: N(0, 1)) and its decoded weights' 64-bit parts: a
    function that gives them [rows][columns]."""
    if fmt == "ternary2":
        blocks = -(-columns // block)
        w = torch.zeros(rows, blocks * block, device="cuda")
        w[:, :columns] = _normal(g, rows, columns)
        w = w.reshape(rows, blocks, block)
        counts = torch.full((blocks, 1), block, device="cuda")
        counts[-1] = columns - (blocks - 1) * block
        scale = w.abs().sum(-1, keepdim=True) / counts
        code = torch.where(w > 0.5 * scale, 1, torch.where(w < -0.5 * scale, 2, 0)).to(torch.uint8)
        c4 = code.reshape(rows, blocks, block // 4, 4)
        packed = c4[..., 0] | (c4[..., 1] << 2) | (c4[..., 2] << 4) | (c4[..., 3] << 6)
        payload = torch.cat([_bytes(scale.squeeze(-1)), packed], dim=-1)
        sign = torch.where(code == 1, 1.0, torch.where(code == 2, -1.0, 0.0))

        def decode():
            return (sign.double() * scale.double()).reshape(rows, -1)[:, :columns]
        return payload, decode
    elements = BLOCK_BYTES[fmt][0]
    w = _normal(g, rows, columns // elements, elements, scale=0.02)
    if fmt == "q8_0":
        d = (w.abs().amax(-1, keepdim=True) / 127).half()
        q = (w / d.float()).round().clamp(-127, 127)
        payload = torch.cat([_bytes(d.squeeze(-1)), q.to(torch.int8).view(torch.uint8)], dim=-1)
        return payload, lambda: (q.double() * d.double()).reshape(rows, columns)
    if fmt == "q4_0":
        top = w.gather(-1, w.abs().argmax(-1, keepdim=True))
        d = (top / -8).half()
        q = (w / d.float()).round().clamp(-8, 7) + 8
        b = q.to(torch.uint8)
        payload = torch.cat([_bytes(d.squeeze(-1)), b[..., :16] | (b[..., 16:] << 4)], dim=-1)
        return payload, lambda: ((q.double() - 8) * d.double()).reshape(rows, columns)
    if fmt == "q4_k":
        sub = w.reshape(*w.shape[:2], 8, 32)
        low = sub.amin(-1).clamp(max=0)
        step = (sub.amax(-1) - low) / 15
        d = (step.amax(-1, keepdim=True) / 63).half()
        dmin = (-low.amin(-1, keepdim=True) / 63).half()
        s = (step / d.float()).round().clamp(1, 63)
        m = (-low / dmin.float()).round().clamp(0, 63)
        q = ((sub + (dmin.float() * m)[..., None]) / (d.float() * s)[..., None]).round().clamp(0, 15)
        si, mi, qi = s.to(torch.uint8), m.to(torch.uint8), q.to(torch.uint8)
        scales = torch.cat([si[..., :4] | ((si[..., 4:] >> 4) << 6), mi[..., :4] | ((mi[..., 4:] >> 4) << 6),
                            (si[..., 4:] & 15) | ((mi[..., 4:] & 15) << 4)], dim=-1)
        qs = (qi[..., 0::2, :] | (qi[..., 1::2, :] << 4)).reshape(*w.shape[:2], 128)
        payload = torch.cat([_bytes(d.squeeze(-1)), _bytes(dmin.squeeze(-1)), scales, qs], dim=-1)

        def decode():
            return ((d.double() * s.double())[..., None] * q.double()
                    - (dmin.double() * m.double())[..., None]).reshape(rows, columns)
        return payload, decode
    sub = w.reshape(*w.shape[:2], 16, 16)  # Q6_K
    step = sub.abs().amax(-1) / 31
    d = (step.amax(-1, keepdim=True) / 127).half()
    s = (step / d.float()).round().clamp(1, 127)
    q = (sub / (d.float() * s)[..., None]).round().clamp(-32, 31)
    k = (q + 32).to(torch.uint8).reshape(*w.shape[:2], 2, 4, 32)
    low, high = k & 15, k >> 4
    ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4), low[..., 1, :] | (low[..., 3, :] << 4)], dim=-1)
    qh = high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) | (high[..., 3, :] << 6)
    payload = torch.cat([ql.reshape(*w.shape[:2], 128), qh.reshape(*w.shape[:2], 64),
                         s.to(torch.int8).view(torch.uint8), _bytes(d.squeeze(-1))], dim=-1)
    return payload, lambda: ((d.double() * s.double())[..., None] * q.double()).reshape(rows, columns)


def _inputs(case: dict, seed: int):
    """The payloads (with their decoders) and activations of a matrix case, the same for prepare() and exact()."""
    g = _generator(seed)
    kind, fmt, rows, columns = case["kind"], case["format"], case["rows"], case["columns"]
    members = case.get("members", 1)
    distinct = [_weights(g, fmt, rows, columns, case.get("block", 0)) for _ in range(min(members, 4))]
    if fmt == "ternary2":
        x = torch.rand(members, columns, generator=g, device="cuda") * 2 - 1
    elif kind == "group":
        x = _normal(g, 1, columns)  # the members of a K group share their input
    else:
        x = _normal(g, case.get("positions", 1), columns)
    return distinct, x


# ---- what a program keeps ----

class _State:
    """Resident objects of one program, released in order when it is dropped."""

    def __init__(self):
        self.owned = []      # disposed from the last to the first
        self.tensors = []    # device memory the launches point into

    def own(self, thing):
        self.owned.append(thing)
        return thing

    def __del__(self):
        while self.owned:
            self.owned.pop().dispose()


def _create(ctx, fmt: str, rows: int, columns: int, block: int, payload: torch.Tensor):
    data = payload.reshape(-1).cpu().numpy()
    if fmt == "ternary2":
        return ctx.create_ternary2(rows, columns, block, data)
    return ctx.create(data, S.QuantizedMatrixShape(rows, columns, FORMATS[fmt]))


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind == "attention":
        return _prepare_attention(case, seed)
    if kind == "token":
        return _prepare_token(case, seed)
    state = _State()
    state.kind = kind
    fmt, rows, columns, block = case["format"], case["rows"], case["columns"], case.get("block", 0)
    distinct, x = _inputs(case, seed)
    if kind == "matvec" and case["call"] == "host":
        state.x, state.y = x.reshape(-1).cpu().numpy(), np.zeros(rows, np.float32)
        if fmt == "ternary2":
            state.matrix = S.Ternary2Matrix.from_packed(rows, columns, block, distinct[0][0].reshape(-1).cpu().numpy())
            state.own(state.matrix.device())
        else:
            state.matrix = state.own(_create(S.default_context(), fmt, rows, columns, block, distinct[0][0]))
        state.host = True
        return state
    state.host = False
    ctx = S.default_context()
    members, positions = case.get("members", 1), case.get("positions", 1)
    first = [state.own(_create(ctx, fmt, rows, columns, block, payload)) for payload, _ in distinct]
    matrices = first + [state.own(first[k % len(first)].clone()) for k in range(len(first), members)]
    state.tensors.append(x)
    state.y = [torch.zeros(positions, rows, device="cuda") for _ in range(members)]
    state.positions = positions
    if kind in ("group", "group_batch"):
        inputs = [x[k % x.shape[0]].data_ptr() if kind == "group" else x.data_ptr() for k in range(members)]
        state.group = state.own(S.HipGroup(ctx, matrices, inputs, [y.data_ptr() for y in state.y], fmt != "ternary2"))
    else:
        state.matrix, state.px, state.py = matrices[0], x.data_ptr(), state.y[0].data_ptr()
    return state


def _prepare_attention(case: dict, seed: int):
    state = _State()
    state.kind = "attention"
    state.tensors += _attention_inputs(case, seed)
    state.out = torch.zeros(case["heads"] * case["head_dim"], device="cuda")
    state.ops = S.DeviceOps(S.default_context())
    state.arguments = (*(t.data_ptr() for t in state.tensors), case["heads"], case["kv_heads"], case["head_dim"],
                       case["tokens"], state.out.data_ptr())
    return state


def _attention_inputs(case: dict, seed: int):
    g = _generator(seed)
    width = case["kv_heads"] * case["head_dim"]
    return (_normal(g, case["heads"] * case["head_dim"]), _normal(g, case["tokens"], width),
            _normal(g, case["tokens"], width))


ROLES = {"q": (HIDDEN, HIDDEN, "q4_k"), "k": (KV, HIDDEN, "q4_k"), "v": (KV, HIDDEN, "q4_k"),
         "o": (HIDDEN, HIDDEN, "q4_k"), "gate": (FFN, HIDDEN, "q4_k"), "up": (FFN, HIDDEN, "q4_k"),
         "down": (HIDDEN, FFN, "q6_k")}


def _token_inputs(case: dict, seed: int):
    """Per layer: the payloads and decoders by role, the norm and bias vectors and the cached prefix."""
    g = _generator(seed)
    for _ in range(case["layers"]):
        weights = {role: _weights(g, fmt, rows, columns) for role, (rows, columns, fmt) in ROLES.items()}
        vectors = {"attn_norm": torch.rand(HIDDEN, generator=g, device="cuda") + 0.5,
                   "ffn_norm": torch.rand(HIDDEN, generator=g, device="cuda") + 0.5,
                   "q_bias": _normal(g, HIDDEN, scale=0.1), "k_bias": _normal(g, KV, scale=0.1),
                   "v_bias": _normal(g, KV, scale=0.1)}
        yield (weights, vectors, _normal(g, case["position"], KV, scale=0.5),
               _normal(g, case["position"], KV, scale=0.5))
    yield _weights(g, "q6_k", case["vocab"], HIDDEN), torch.rand(HIDDEN, generator=g, device="cuda") + 0.5


def _prepare_token(case: dict, seed: int):
    state = _State()
    state.kind = "token"
    ctx = state.own(S.HipContext(0))
    layers, vectors, caches = [], [], []
    for item in _token_inputs(case, seed):
        if len(item) == 2:
            payload, output_norm = item[0][0], item[1]
            output = state.own(_create(ctx, "q6_k", case["vocab"], HIDDEN, 0, payload))  # tied to the embedding
            break
        weights, vec, keys, values = item
        layers.append({role: state.own(_create(ctx, fmt, rows, columns, 0, weights[role][0]))
                       for role, (rows, columns, fmt) in ROLES.items()})
        state.tensors += vec.values()
        vectors.append({name: t.data_ptr() for name, t in vec.items()})
        caches.append((keys.cpu().numpy(), values.cpu().numpy()))
    state.tensors.append(output_norm)
    config = DecoderConfig(hidden=HIDDEN, heads=HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM, ffn=FFN, epsilon=EPSILON,
                           rope_base=ROPE_BASE, max_tokens=case["position"] + 1)
    torch.cuda.synchronize()
    state.decoder = state.own(DeviceDecoder(ctx, config, layers, vectors, output_norm.data_ptr(), output, output))
    for layer, (keys, values) in enumerate(caches):
        ctx.upload(state.decoder.keys[layer], keys)
        ctx.upload(state.decoder.values[layer], values)
    state.step = state.own(state.decoder.capture(seed % case["vocab"], case["position"], folded=True))
    return state


def run(state):
    if state.kind == "token":
        state.step.execute()
        return state.decoder.read_logits()
    if state.kind == "attention":
        state.ops.grouped_attention(*state.arguments)
        return state.out
    if state.host:
        if isinstance(state.matrix, S.Ternary2Matrix):
            S.Ternary2MatVec.execute(state.matrix, state.x, state.y)
        else:
            state.matrix.execute(state.x, state.y)
        return state.y
    if state.kind == "group":
        state.group.execute()
    elif state.kind == "group_batch":
        state.group.execute_batch(state.positions)
    elif state.kind == "batch":
        state.matrix.execute_batch_device(state.px, state.positions, state.py)
    else:
        state.matrix.execute_device(state.px, state.py)
    return state.y


# ---- what cannot be done without ----

def _payload_bytes(fmt: str, rows: int, columns: int, block: int = 0) -> int:
    if fmt == "ternary2":
        return rows * -(-columns // block) * (4 + block // 4)
    elements, size = BLOCK_BYTES[fmt]
    return rows * (columns // elements) * size


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "attention":
        n = case["tokens"] * case["kv_heads"] * case["head_dim"]
        return {"bytes": 8 * n + 8 * case["heads"] * case["head_dim"],
                "flops": 4 * case["tokens"] * case["heads"] * case["head_dim"]}
    if kind == "token":
        shapes = case["layers"] * list(ROLES.values()) + [(case["vocab"], HIDDEN, "q6_k")]
        cache = case["layers"] * (case["position"] + 1) * KV
        return {"bytes": sum(_payload_bytes(f, r, c) for r, c, f in shapes) + 8 * cache + 4 * case["vocab"],
                "flops": sum(2 * r * c for r, c, _ in shapes) + 4 * case["layers"] * (case["position"] + 1) * HIDDEN}
    rows, columns, members, positions = case["rows"], case["columns"], case.get("members", 1), case.get("positions", 1)
    payload = _payload_bytes(case["format"], rows, columns, case.get("block", 0))
    inputs = members if kind == "group" and case["format"] == "ternary2" else 1
    return {"bytes": members * payload + 4 * positions * (inputs * columns + members * rows),
            "flops": 2 * members * positions * rows * columns}


def tolerance(case: dict) -> dict:
    # FP32 sums over one row, in any order: 0.7e-7 to 1.6e-7 against 64 bits measured, and twice that between two
    # orders. A whole token measured 1.3e-7 too, but it passes every layer's activations through Q8_K, where one
    # different last bit can move a code by a step: 1/127 of its block's largest value, about 6e-4 of the norm of a
    # 1,536-wide vector.
    if case["kind"] == "token":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-6, "max": 1e-5}


# ---- the outputs in 64 bits ----

def _q8k(x: torch.Tensor) -> torch.Tensor:
    """FP32 vectors [positions][columns] after Q8_K (Q8KCodec.QuantizeBlock): code * scale in 64 bits. The code is
    round-to-nearest-even of the FP32 product with -127 / (the block's first element of largest magnitude)."""
    blocks = x.reshape(x.shape[0], -1, 256)
    top = blocks.gather(-1, blocks.abs().argmax(-1, keepdim=True))
    inverse = (-127.0 / top.double()).float()  # divided in 64 bits, so rounded once
    codes = (blocks * inverse).round().clamp(max=127)
    return (codes.double() * (1.0 / inverse.double()).float().double()).reshape(x.shape)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "token":
        return _exact_token(case, seed)
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        return _attention64(q, k, v, case["heads"], case["kv_heads"], case["head_dim"])
    distinct, x = _inputs(case, seed)
    integer = case["format"] in ("q4_k", "q6_k") and kind != "matvec"
    x64 = _q8k(x) if integer else x.double()
    members = case.get("members", 1)
    out = []
    decoded = [decode() for _, decode in distinct]
    for k in range(members):
        w = decoded[k % len(decoded)]
        if kind == "group":
            out.append((x64[k % x64.shape[0]][None] @ w.T))
        else:
            out.append(x64 @ w.T)
    if kind == "matvec" and case["call"] == "host":
        return out[0].reshape(-1)
    return out


def _attention64(q, k, v, heads: int, kv_heads: int, head_dim: int):
    group = heads // kv_heads
    tokens = k.shape[0]
    qh = q.reshape(kv_heads, group, head_dim)
    kh = k.reshape(tokens, kv_heads, head_dim).permute(1, 2, 0).contiguous()
    vh = v.reshape(tokens, kv_heads, head_dim).permute(1, 0, 2).contiguous()
    out = [torch.softmax(qh[h] @ kh[h] / math.sqrt(head_dim), dim=-1) @ vh[h] for h in range(kv_heads)]
    return torch.stack(out).reshape(-1)


def _exact_token(case: dict, seed: int):
    """The token in 64 bits, each operator's output rounded to FP32 where the decoder stores it (Q8_K codes are made
    from those)."""
    f32 = lambda t: t.float().double()  # noqa: E731
    position, token = case["position"], seed % case["vocab"]
    items = list(_token_inputs(case, seed))
    (_, decode_output), output_norm = items.pop()
    output = decode_output()

    def norm(t, w):
        return f32(t / torch.sqrt((t * t).mean() + EPSILON) * w.double())

    def project(decode, t):
        return f32(decode() @ _q8k(t.float()[None])[0])

    half = HEAD_DIM // 2
    angle = position / ROPE_BASE ** (2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / HEAD_DIM)
    sn, cs = torch.sin(angle), torch.cos(angle)

    def rope(t):
        a, b = t.reshape(-1, HEAD_DIM)[:, :half], t.reshape(-1, HEAD_DIM)[:, half:]
        return f32(torch.cat([a * cs - b * sn, a * sn + b * cs], dim=-1).reshape(-1))

    r = f32(output[token])
    for weights, vec, keys, values in items:
        decoders = {role: d for role, (_, d) in weights.items()}
        h = norm(r, vec["attn_norm"])
        q, k, v = (f32(project(decoders[n], h) + vec[n + "_bias"].double()) for n in ("q", "k", "v"))
        keys64 = torch.cat([keys.double(), rope(k)[None]])
        values64 = torch.cat([values.double(), v[None]])
        attended = f32(_attention64(rope(q), keys64, values64, HEADS, KV_HEADS, HEAD_DIM))
        r = f32(r + project(decoders["o"], attended))
        h = norm(r, vec["ffn_norm"])
        gate, up = project(decoders["gate"], h), project(decoders["up"], h)
        r = f32(r + project(decoders["down"], f32(gate * torch.sigmoid(gate) * up)))
    return output @ _q8k(norm(r, output_norm).float()[None])[0]
