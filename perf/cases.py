"""Timing cases: the calls a serving program makes on the Gated DeltaNet path, through the
public entry points (`GDNBackend` and `torch.ops.lightdelta.*`), under the library's default
settings.

A case is a dict of plain values.  Its `kind` says which call it is:
  decode   one decode or speculative-verify step of a stack of layers (`layers` calls), with
           `commit` the accepted states copied back to their home slots (`copy_state`)
  conv     the same step with the causal conv1d in front (`decode_conv`)
  copies   a batch of requests swapped out of the state pools and in again at other slots
           (gather, scatter), states duplicated (`copy_state`) and freed slots cleared
  prefill  prompts of `prompts` sequences in one call, lengths between `low` and `high`

Activations come as a layer hands them over: qkv and gate are column slices of one buffer, a
and b of another.  q, k, v, gate, a, b ~ N(0, 1) in bf16, A_log ~ U(-1, 1), states ~ 0.02 N(0, 1)
in fp32.  Batches hold a padding request now and then, as a captured batch size does.
"""

from __future__ import annotations

import math

import torch

from lightdelta_amd import ops  # noqa: F401  -- registers torch.ops.lightdelta
from lightdelta_amd.backend import GDNBackend
from lightdelta_amd.config import BackendConfig

DIM = 128
EPS = 1e-6


def listed():
    return [
        # One request of a small model (4/8 heads): the latency of a single call.
        _decode("decode_b1_small", batch=1, heads=4, v_heads=8),
        # The decode step of an ordinary batch, one layer.
        _decode("decode_b32", batch=32),
        # The step of a full batch through several layers, whose states (1.6 GB) no cache holds.
        _decode("decode_b128_layers6", batch=128, layers=6),
        # Speculative verify of up to 4 tokens a request, then the commit of the accepted state.
        _decode("verify_b64_t4_commit", batch=64, width=4, commit=True),
        # The serving layer's step (conv1d and recurrence in one call), an odd batch with a
        # padding request, 16/48 heads, parameters in bf16 as a bf16 checkpoint has them.
        _decode("conv_b37_hv48", kind="conv", batch=37, v_heads=48, bf16=True, padding=1),
        # The same with speculative tokens (a conv state of 3 + 2 columns).
        _decode("conv_verify_b11_t3", kind="conv", batch=11, width=3),
        # Preemption: 96 requests out of the pools and in again.
        dict(name="copies_96", kind="copies", rows=96, v_heads=32),
        # One long new prompt: what time to first token waits for.
        _prefill("prefill_1x4096", prompts=1, low=4096, high=4096, initial=0.0),
        # A full batch of equal prompts that continue from a state (chunked prefill of a server).
        _prefill("prefill_32x1024", prompts=32, low=1024, high=1024),
        # Many short prompts of unequal length.
        _prefill("prefill_512x8to56", prompts=512, low=8, high=56, initial=0.5),
        # Very short extensions of running requests.
        _prefill("prefill_200x1to20", prompts=200, low=1, high=20),
        # A mixed batch: lengths from one token to thousands, 16/48 heads, bf16 parameters.
        _prefill("prefill_13x1to3000_hv48", prompts=13, low=1, high=3000, v_heads=48, bf16=True,
                 initial=0.5),
    ]


def _decode(name, batch, kind="decode", heads=16, v_heads=32, width=1, layers=1, commit=False,
            bf16=False, padding=0):
    return dict(name=name, kind=kind, batch=batch, heads=heads, v_heads=v_heads, width=width,
                layers=layers, commit=commit, bf16=bf16, padding=padding)


def _prefill(name, prompts, low, high, heads=16, v_heads=32, bf16=False, initial=1.0):
    return dict(name=name, kind="prefill", prompts=prompts, low=low, high=high, heads=heads,
                v_heads=v_heads, bf16=bf16, initial=initial)


def draw(rng):
    def log_int(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    heads, v_heads = rng.choice([(4, 8), (16, 32), (16, 32), (16, 48), (8, 16)])
    kind = rng.choice(["decode", "conv", "copies", "prefill", "prefill", "prefill"])
    if kind == "copies":
        case = dict(kind=kind, rows=log_int(1, 96), v_heads=v_heads)
    elif kind == "prefill":
        # tokens over three decades, prompts from one to as many as that allows
        tokens = log_int(16, 20000)
        prompts = min(log_int(1, 512), max(1, tokens // 4))
        mean = max(1, tokens // prompts)
        spread = rng.choice([0, mean // 2, mean - 1])
        case = _prefill("", prompts, mean - spread, mean + spread, heads, v_heads,
                        rng.random() < 0.3, rng.choice([0.0, 0.5, 1.0]))
    else:
        width = rng.choice([1, 1, 1, 2, 3, 4])
        batch = log_int(1, 128 // width)
        case = _decode("", batch, kind, heads, v_heads, width, 1,
                       kind == "decode" and width > 1 and rng.random() < 0.5,
                       rng.random() < 0.3, 1 if batch > 4 and rng.random() < 0.3 else 0)
    case.pop("name", None)
    return case


# ---- inputs ------------------------------------------------------------------------------


def _lengths(case):
    """Prompt lengths, spread evenly in the logarithm from `low` to `high` and shuffled (the
    same for every seed)."""
    n, low, high = case["prompts"], case["low"], case["high"]
    if low == high:
        return [low] * n
    if high < 8 * low:
        values = [round(low + (high - low) * (i + 0.5) / n) for i in range(n)]
    else:
        values = [round(math.exp(math.log(low) + math.log(high / low) * (i + 0.5) / n))
                  for i in range(n)]
    gen = torch.Generator().manual_seed(n)
    return [values[i] for i in torch.randperm(n, generator=gen).tolist()]


class _Source:
    """Random tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        x = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std,
                                                                          generator=self.gen)
        return x if dtype == torch.float32 else x.to(dtype)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda")

    def perm(self, n):
        return torch.randperm(n, generator=self.gen, device="cuda")


def _layer(src, case, tokens, slots):
    """One layer's activations, parameters and state pool."""
    heads, v_heads = case["heads"], case["v_heads"]
    param = torch.bfloat16 if case["bf16"] else torch.float32
    cols, gate_cols = (2 * heads + v_heads) * DIM, v_heads * DIM
    qkvz = src.normal(tokens, cols + gate_cols, dtype=torch.bfloat16)
    ba = src.normal(tokens, 2 * v_heads, dtype=torch.bfloat16)
    return dict(
        qkv=qkvz[:, :cols], gate=qkvz[:, cols:].view(tokens, v_heads, DIM),
        a=ba[:, v_heads:], b=ba[:, :v_heads],
        a_log=src.uniform(v_heads) * 2 - 1,
        dt_bias=src.normal(v_heads, std=0.1).to(param),
        weight=(1 + src.normal(DIM, std=0.1)).to(param),
        pool=src.normal(slots, v_heads, DIM, DIM, std=0.02),
        out=torch.zeros(tokens, v_heads, DIM, dtype=torch.bfloat16, device="cuda"),
    )


def prepare(case, seed):
    src = _Source(seed)
    return {"decode": _prepare_decode, "conv": _prepare_decode, "copies": _prepare_copies,
            "prefill": _prepare_prefill}[case["kind"]](case, src)


def _prepare_decode(case, src):
    batch, width = case["batch"], case["width"]
    slots = batch * width + 1
    # each request: 1 .. width tokens, its accepted length, and slots of its own
    lengths = src.uniform(batch).mul(width).int().clamp_(max=width - 1) + 1
    cu = torch.zeros(batch + 1, dtype=torch.int32, device="cuda")
    cu[1:] = torch.cumsum(lengths, 0)
    indices = (src.perm(slots - 1) + 1).int().view(batch, width)
    accepted = (src.uniform(batch) * width).int().clamp_(max=width - 1) + 1
    if case["kind"] == "conv":  # the state columns of a conv step hold what was accepted
        accepted = torch.minimum(accepted, lengths)
    if case["padding"]:
        indices[-case["padding"]:] = 0
    # a captured batch has rows for every token it may hold
    layers = [_layer(src, case, batch * width, slots) for _ in range(case["layers"])]
    state = dict(case=case, layers=layers, indices=indices, cu=cu, accepted=accepted.int())
    if case["kind"] == "conv":
        conv_dim = (2 * case["heads"] + case["v_heads"]) * DIM
        for layer in layers:
            layer["conv_state"] = src.normal(slots, conv_dim, 2 + width, dtype=torch.bfloat16)
            layer["conv_weight"] = src.normal(conv_dim, 4, std=0.5, dtype=torch.bfloat16)
    else:
        state["backend"] = GDNBackend(BackendConfig(compute="cuda_fused", state_io="indexed"))
    if case["commit"]:
        state["commit"] = torch.minimum(accepted, lengths).int()
        chosen = indices.gather(1, (state["commit"] - 1)[:, None].long()).flatten()
        state["source"], state["home"] = chosen.contiguous(), indices[:, 0].contiguous()
    return state


def _prepare_copies(case, src):
    rows, v_heads = case["rows"], case["v_heads"]
    slots = 4 * rows + 1
    ids = (src.perm(slots - 1) + 1).int()
    valid = torch.ones(rows, dtype=torch.bool, device="cuda")
    old, new, twin, freed = (ids[i * rows:(i + 1) * rows].clone() for i in range(4))
    if rows > 4:
        old[rows // 2], new[rows // 3], valid[rows // 4] = 0, -1, False
    conv_dim = 2 * v_heads * DIM
    return dict(
        case=case, old=old, new=new, twin=twin, freed=freed, valid=valid,
        pool=src.normal(slots, v_heads, DIM, DIM, std=0.02),
        packed=torch.zeros(rows, v_heads, DIM, DIM, device="cuda"),
        conv=src.normal(slots, conv_dim, 4, dtype=torch.bfloat16),
        conv_packed=torch.zeros(rows, conv_dim, 4, dtype=torch.bfloat16, device="cuda"),
    )


def _prepare_prefill(case, src):
    lengths = _lengths(case)
    n = len(lengths)
    cu = torch.zeros(n + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(lengths), 0)
    state = _layer(src, case, sum(lengths), n + 1)
    state.update(case=case, cu=cu.to("cuda"), slots=(src.perm(n) + 1).int(),
                 has_initial=src.uniform(n) < case["initial"])
    return state


# ---- one pass ----------------------------------------------------------------------------


def run(state):
    kind = state["case"]["kind"]
    lightdelta = torch.ops.lightdelta
    if kind == "prefill":
        lightdelta.prefill(state["qkv"], state["a"], state["b"], state["a_log"],
                           state["dt_bias"], state["slots"], state["has_initial"], state["cu"],
                           state["pool"], state["gate"], state["weight"], state["out"], EPS)
        return {"out": state["out"], "pool": state["pool"]}
    if kind == "copies":
        lightdelta.gather_state(state["pool"], state["old"], state["valid"], state["packed"])
        lightdelta.gather_slots(state["conv"], state["old"], state["valid"],
                                state["conv_packed"])
        lightdelta.scatter_state(state["packed"], state["new"], state["pool"])
        lightdelta.scatter_slots(state["conv_packed"], state["new"], state["conv"])
        lightdelta.copy_state(state["pool"], state["new"], state["twin"])
        lightdelta.zero_slots(state["pool"], state["freed"])
        return {k: state[k] for k in ("pool", "packed", "conv", "conv_packed")}
    metadata = (state["indices"], state["cu"], state["accepted"])
    outputs = {}
    for i, layer in enumerate(state["layers"]):
        rest = (layer["a"], layer["b"], layer["a_log"], layer["dt_bias"], *metadata,
                layer["pool"], layer["gate"], layer["weight"], layer["out"], EPS)
        if kind == "conv":
            lightdelta.decode_conv(layer["qkv"], layer["conv_state"], layer["conv_weight"], None,
                                   *rest)
            outputs[f"conv_state{i}"] = layer["conv_state"]
        else:
            state["backend"](layer["qkv"], *rest)
        if state["case"]["commit"]:
            lightdelta.copy_state(layer["pool"], state["source"], state["home"])
        outputs[f"out{i}"], outputs[f"pool{i}"] = layer["out"], layer["pool"]
    return outputs


# ---- what a pass cannot do without ---------------------------------------------------------


def work(case):
    v_heads = case["v_heads"]
    tile = v_heads * DIM * DIM * 4
    if case["kind"] == "copies":
        conv_row = 2 * v_heads * DIM * 4 * 2
        # gather, scatter: read and write; copy: read and write; clear: write
        return {"bytes": case["rows"] * (7 * tile + 4 * conv_row), "flops": 0}
    heads = case["heads"]
    cols = (2 * heads + v_heads) * DIM
    token = 2 * (cols + 2 * v_heads * DIM + 2 * v_heads)  # qkv, gate in, out; a, b
    step = 6 * v_heads * DIM * DIM                        # S k, the update, S q
    if case["kind"] == "prefill":
        tokens, n = sum(_lengths(case)), case["prompts"]
        return {"bytes": int(tokens * token + n * (1 + case["initial"]) * tile),
                "flops": tokens * step}
    batch, width, layers = case["batch"] - case["padding"], case["width"], case["layers"]
    tokens = batch * (width + 1) / 2
    total = tokens * token + (batch + tokens) * tile
    if case["kind"] == "conv":
        total += 2 * batch * cols * (2 + width) * 2 + cols * 8
    if case["commit"]:
        total += 2 * batch * tile * (width - 1) / (2 * width)
    return {"bytes": int(layers * total), "flops": int(layers * tokens * step)}


def tolerance(case):
    """Copies move bytes.  Elsewhere the bf16 outputs set the limit: two correct programs
    round a raw output next to a bf16 midpoint to either side, and it then carries through
    the norm (measured between the token-serial and the chunked forms, and against `exact`)."""
    if case["kind"] == "copies":
        return "exact"
    return {"rel": 7e-3, "max": 0.04}


# ---- the same in 64 bits -------------------------------------------------------------------


def exact(case, seed):
    """The recurrence token by token in 64 bits on the same inputs.  Values that the calls
    define as bf16 on the way (the conv output, the raw output ahead of the norm) are rounded
    there."""
    if case["kind"] == "copies":
        return None
    state = prepare(case, seed)
    if case["kind"] == "prefill":
        cu = state["cu"].tolist()
        spans = [list(range(cu[i], cu[i + 1])) for i in range(len(cu) - 1)]
        pool = state["pool"].double()
        slots = state["slots"].long()
        start = pool[slots] * state["has_initial"].double()[:, None, None, None]
        out = torch.zeros(state["out"].shape, dtype=torch.float64, device="cuda")
        pool[slots] = _recur(state, state["qkv"].double(), spans, start, out, None)
        return {"out": out, "pool": pool}
    outputs = {}
    cu, accepted = state["cu"].tolist(), state["accepted"].tolist()
    indices = state["indices"].tolist()
    live = [r for r in range(case["batch"]) if indices[r][0] > 0]
    spans = [list(range(cu[r], cu[r + 1])) for r in live]
    for i, layer in enumerate(state["layers"]):
        pool = layer["pool"].double()
        out = torch.zeros(layer["out"].shape, dtype=torch.float64, device="cuda")
        qkv = layer["qkv"].double()
        if case["kind"] == "conv":
            conv_state, qkv = _conv(layer, state, qkv, live, spans, indices, accepted)
            outputs[f"conv_state{i}"] = conv_state
        start = pool[[indices[r][accepted[r] - 1] for r in live]]
        _recur(layer, qkv, spans, start, out,
               lambda t, rows, s: pool.index_copy_(
                   0, torch.tensor([indices[live[n]][t] for n in rows], device="cuda"), s))
        if case["commit"]:
            pool[state["home"].long()] = pool[state["source"].long()].clone()
        outputs[f"out{i}"], outputs[f"pool{i}"] = out, pool
    return outputs


def _bf16(x):
    """64-bit values rounded to the nearest bf16, ties to even, in 64 bits."""
    bits = x.contiguous().view(torch.int64)  # 52 bits of mantissa, of which 7 stay
    bits = bits + ((1 << 44) - 1) + ((bits >> 45) & 1)
    return (bits & -(1 << 45)).view(torch.float64)


def _conv(layer, state, x, live, spans, indices, accepted):
    """Depthwise causal conv of width 4 with SiLU over each request's tokens, and the conv
    state after them."""
    conv_state, weight = layer["conv_state"].double(), layer["conv_weight"].double()
    columns = conv_state.shape[2]
    y = x.clone()
    for r, span in zip(live, spans):
        slot, offset, n = indices[r][0], accepted[r] - 1, len(span)
        held = conv_state[slot].clone()
        sequence = torch.cat([held[:, offset:offset + 3], x[span].T], 1)
        acc = sum(weight[:, j, None] * sequence[:, j:j + n] for j in range(4))
        y[span] = _bf16(acc * torch.sigmoid(acc)).T
        kept = max(columns - n, 0)
        conv_state[slot] = torch.cat([held[:, offset + 1:offset + 1 + kept],
                                      x[span].T[:, n - (columns - kept):]], 1)
    return conv_state, y


def _recur(layer, qkv, spans, states, out, store):
    """Steps `states` [sequences, v_heads, V, K] through their rows; returns the last states.
    The longest sequences come first, so that those with a token left are a prefix."""
    v_heads = states.shape[1]
    heads = (qkv.shape[1] // DIM - v_heads) // 2
    group = v_heads // heads
    gate, a, b = (layer[k].double() for k in ("gate", "a", "b"))
    rate = torch.exp(layer["a_log"].double())
    dt_bias, weight = layer["dt_bias"].double(), layer["weight"].double()
    order = sorted(range(len(spans)), key=lambda n: -len(spans[n]))
    s = states[order].clone()
    for t in range(len(spans[order[0]]) if order else 0):
        rows = [n for n in order if len(spans[n]) > t]
        at = torch.tensor([spans[n][t] for n in rows], device="cuda")
        now = s[:len(rows)]
        x = qkv[at]
        q, k = (x[:, i * heads * DIM:(i + 1) * heads * DIM].view(-1, heads, DIM)
                for i in range(2))
        q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * DIM**-0.5
        k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        q, k = (y.repeat_interleave(group, 1) for y in (q, k))
        v = x[:, 2 * heads * DIM:].view(-1, v_heads, DIM)
        decay = torch.exp(-rate * torch.nn.functional.softplus(a[at] + dt_bias))
        now *= decay[..., None, None]
        delta = (v - (now * k[:, :, None, :]).sum(-1)) * torch.sigmoid(b[at])[..., None]
        now += delta[..., None] * k[:, :, None, :]
        raw = _bf16((now * q[:, :, None, :]).sum(-1))
        g = gate[at]
        out[at] = (raw * torch.rsqrt((raw * raw).mean(-1, keepdim=True) + EPS) * weight
                   * g * torch.sigmoid(g))
        if store is not None:
            store(t, rows, now)
    final = torch.empty_like(states)
    final[order] = s
    return final
