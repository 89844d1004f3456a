"""The work this library is used for, as calls of its public Python binding (qattn.py) that can be
timed and compared: whole embedding forwards, the attention operator, the Q4_0 projections, the
feed-forward block and the QK-norm + RoPE producer, from one short query to the largest batches.

A case is a dict of plain values.  `kind` names the call, `lengths` the packed sequences
("15", "500*16", "37,150*2"), `rows` the token rows of a projection.

  forward     one qattn_model_plan_run over 28 layers, as the Node engine plans it (prefix + local
              mask, batch-invariant): token ids in, one L2-normalised embedding per request out
  attention   one planned attention launch (run.encode) over packed Q, K, V
  projection  qattn_q4_matmul: y = x W^T for a tile32-compact Q4_0 weight [n, k]
  gate_up     qattn_q4_matmul_swiglu: the FFN's fused gate/up projection
  mlp         RMSNorm, gate_up and the down projection in a row: the feed-forward block
  rope        qattn_qk_norm_rope_qkv: qkvRaw rows to compact, normalised, rotated Q and K
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIDDEN, INTER, QKV, HEADS, KV_HEADS, DIM = 1024, 3072, 4096, 16, 8, 128
LAYERS, VOCAB = 28, 151669  # Qwen3-Embedding-0.6B
PREFIX, WINDOW = 176, 432  # the model's sparse mask
EPS, THETA = 1e-6, 1e6
# The model's plain projections: QKV, attention output, FFN down (k -> n).
SHAPES = ((1024, 4096), (2048, 1024), (3072, 1024))
MOST_TOKENS = 8000


def _binding():
    if "qattn" not in sys.modules:
        path = os.path.join(ROOT, "qwen3-embedding-webgpu-prepacked_amd", "qattn.py")
        spec = importlib.util.spec_from_file_location("qattn", path)
        sys.modules["qattn"] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules["qattn"])
    return sys.modules["qattn"]


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = _binding().Context(0)
    return _ctx


def lengths_of(case):
    out = []
    for part in case["lengths"].split(","):
        length, _, times = part.partition("*")
        out += [int(length)] * int(times or 1)
    return out


def _offsets(case):
    return np.concatenate([[0], np.cumsum(lengths_of(case))]).astype(np.int32)


def listed():
    return [
        # One short search query through the whole model: the smallest call of the engine.
        {"name": "forward_1x15", "kind": "forward", "lengths": "15"},
        # A full micro-batch of 16 concurrent documents: the engine's throughput case.
        {"name": "forward_16x500", "kind": "forward", "lengths": "500*16"},
        # Attention of one short query.
        {"name": "attention_1x50", "kind": "attention", "lengths": "50", "mask": "prefix_local", "invariant": True,
         "last": False, "v_in_qkv": False},
        # 16 concurrent short requests of mixed lengths, with the last-token rows that the pool
        # takes and V read in place from qkvRaw, as the runtimes call it.
        {"name": "attention_16_ragged", "kind": "attention",
         "lengths": "36,84,150,10,121,67,139,95,52,143,18,110,78,129,101,86", "mask": "prefix_local",
         "invariant": True, "last": True, "v_in_qkv": True},
        # The operator's two headline workloads: a full batch under the causal mask ...
        {"name": "attention_16x500", "kind": "attention", "lengths": "500*16", "mask": "causal", "invariant": False,
         "last": False, "v_in_qkv": False},
        # ... and one long document under the prefix + local mask.
        {"name": "attention_1x5000", "kind": "attention", "lengths": "5000", "mask": "prefix_local",
         "invariant": False, "last": False, "v_in_qkv": False},
        # The FFN down projection of one 50-token request.
        {"name": "down_50", "kind": "projection", "k": 3072, "n": 1024, "rows": 50},
        # The attention output projection of 16 ragged requests of 10 to 150 tokens.
        {"name": "output_1419", "kind": "projection", "k": 2048, "n": 1024, "rows": 1419},
        # The QKV projection of 16 x 500 tokens.
        {"name": "qkv_8000", "kind": "projection", "k": 1024, "n": 4096, "rows": 8000},
        # The fused gate/up projection of four 5,000-token documents: the largest batch.
        {"name": "gate_up_20000", "kind": "gate_up", "rows": 20000},
        # The feed-forward block of one 1,500-token document.
        {"name": "mlp_1500", "kind": "mlp", "rows": 1500},
        # The attention path's producer for 16 x 500 tokens.
        {"name": "rope_16x500", "kind": "rope", "lengths": "500*16"},
    ]


def _log_int(rng, low, high):
    return min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _packing(rng, most):
    """1 to 16 requests of 1 to 5,000 tokens, at most `most` together: alike or ragged."""
    requests = rng.choice((1, 1, 2, 3, 4, 8, 13, 16, 16))
    top = _log_int(rng, 10, min(5000, most // requests))
    if rng.random() < 0.4:
        return "%d*%d" % (top, requests)
    return ",".join(str(rng.randint(max(1, top // 8), top)) for _ in range(requests))


def draw(rng):
    kind = rng.choice(("forward", "attention", "attention", "projection", "projection", "gate_up", "mlp", "rope"))
    if kind == "forward":
        return {"kind": kind, "lengths": _packing(rng, MOST_TOKENS)}
    if kind == "attention":
        return {"kind": kind, "lengths": _packing(rng, 20000), "mask": rng.choice(("causal", "prefix_local")),
                "invariant": rng.random() < 0.5, "last": rng.random() < 0.5, "v_in_qkv": rng.random() < 0.5}
    if kind == "rope":
        return {"kind": kind, "lengths": _packing(rng, MOST_TOKENS)}
    rows = _log_int(rng, 1, 20000)
    if kind == "projection":
        k, n = rng.choice(SHAPES)
        return {"kind": kind, "k": k, "n": n, "rows": rows}
    return {"kind": kind, "rows": rows}


# ---- inputs ---------------------------------------------------------------------------------


class State:
    """What a program holds between calls; the library's handles are released with it."""

    def __init__(self, **parts):
        self.handles = []
        self.__dict__.update(parts)

    def __del__(self):
        for handle in self.handles:
            handle.destroy()


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).half()


def _gain(g, n):
    return 1.0 + 0.1 * torch.randn(n, generator=g, device="cuda", dtype=torch.float32)


def _q4(g, k, n):
    """A Q4_0 weight [n, k] in the tile32-compact layout: 20-byte records (f16 scale, two zero
    bytes, 16 bytes of nibbles), codes distributed as those of normal weights."""
    records = torch.zeros(n * k // 32, 20, dtype=torch.uint8, device="cuda")
    scale = 0.0045 * (0.75 + 0.5 * torch.rand(n * k // 32, 1, generator=g, device="cuda"))
    records[:, 0:2] = scale.half().view(torch.uint8).view(-1, 2)
    codes = torch.randn(n * k // 32, 32, generator=g, device="cuda").mul_(2.8).add_(8.0).round_().clamp_(0, 15)
    codes = codes.to(torch.uint8)
    records[:, 4:] = codes[:, :16] | (codes[:, 16:] << 4)
    return records.view(-1)


def _q6k_table(g):
    """A Q6_K table [VOCAB, HIDDEN]: 210-byte blocks of 256 values."""
    blocks = torch.randint(0, 256, (VOCAB * HIDDEN // 256, 210), generator=g, device="cuda", dtype=torch.uint8)
    sign = torch.randint(0, 2, (len(blocks), 16), generator=g, device="cuda", dtype=torch.int8) * 2 - 1
    scales = torch.randint(1, 16, (len(blocks), 16), generator=g, device="cuda", dtype=torch.int8) * sign
    blocks[:, 192:208] = scales.view(torch.uint8)
    d = 0.006 * (0.5 + torch.rand(len(blocks), 1, generator=g, device="cuda"))
    blocks[:, 208:210] = d.half().view(torch.uint8).view(-1, 2)
    return blocks.view(-1)


def _model_tensors(seed):
    g = _generator(seed)
    layers = [{"attn_norm": _gain(g, HIDDEN), "attn_qkv": _q4(g, HIDDEN, QKV), "attn_q_norm": _gain(g, DIM),
               "attn_k_norm": _gain(g, DIM), "attn_output": _q4(g, HEADS * DIM, HIDDEN), "ffn_norm": _gain(g, HIDDEN),
               "ffn_gate_up": _q4(g, HIDDEN, 2 * INTER), "ffn_down": _q4(g, INTER, HIDDEN)} for _ in range(LAYERS)]
    return {"table": _q6k_table(g), "output_norm": _gain(g, HIDDEN), "layers": layers}


def _token_ids(case, seed):
    return np.random.RandomState(seed % (1 << 32)).randint(0, VOCAB, sum(lengths_of(case))).astype(np.int32)


def _rope_rows(x, offsets):
    """Rotary positions of [tokens, heads, 128] rows, restarting at every sequence (float64)."""
    positions = torch.cat([torch.arange(b - a) for a, b in zip(offsets[:-1], offsets[1:])]).to(x)
    angle = positions[:, None] * THETA ** (-torch.arange(64, device=x.device, dtype=x.dtype) / 64)
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    low, high = x[..., :64], x[..., 64:]
    return torch.cat([low * cos - high * sin, high * cos + low * sin], dim=-1)


def _norm_rows(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain


def _attention_inputs(case, seed):
    """Q and K as the producer leaves them (unit-RMS heads, gains, rotated), V as projected."""
    g, offsets = _generator(seed), _offsets(case)
    tokens = int(offsets[-1])
    q, k = (_rope_rows(_norm_rows(_normal(g, tokens, h, DIM).float(), _gain(g, DIM)), offsets).half().reshape(tokens, -1)
            for h in (HEADS, KV_HEADS))
    v = _normal(g, tokens, QKV if case["v_in_qkv"] else KV_HEADS * DIM)
    return q, k, v


def prepare(case, seed):
    qattn, ctx, kind = _binding(), _context(), case["kind"]
    if kind == "forward":
        w, offsets = _model_tensors(seed), _offsets(case)
        compact = ("attn_qkv", "attn_output", "ffn_gate_up", "ffn_down")
        layers = [{n: (t.data_ptr(), t.numel()) if n in compact else t.data_ptr() for n, t in layer.items()}
                  for layer in w["layers"]]
        torch.cuda.current_stream().synchronize()  # the weights are on the device before the model is made
        model = ctx.model((w["table"].data_ptr(), w["table"].numel()), w["output_norm"].data_ptr(), layers,
                          flags=qattn.FLAG_BATCH_INVARIANT)
        plan = model.plan(int(offsets[-1]), len(offsets) - 1)
        out = torch.zeros(len(offsets) - 1, HIDDEN, device="cuda")
        return State(kind=kind, weights=w, plan=plan, ids=_token_ids(case, seed), offsets=offsets, out=out,
                     handles=[plan, model])
    if kind == "attention":
        offsets = _offsets(case)
        q, k, v = _attention_inputs(case, seed)
        o = torch.zeros_like(q)
        last = torch.zeros(len(offsets) - 1, HEADS * DIM, device="cuda", dtype=torch.float16) if case["last"] else None
        desc = qattn.make_desc(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), offsets,
            mask=qattn.MASK_CAUSAL if case["mask"] == "causal" else qattn.MASK_PREFIX_LOCAL, prefix=PREFIX,
            window=WINDOW, v_row_stride=v.shape[1], v_offset=3072 if case["v_in_qkv"] else 0,
            o_last=last.data_ptr() if case["last"] else None,
            flags=qattn.FLAG_BATCH_INVARIANT if case["invariant"] else 0)
        run_ = ctx.run(desc)
        return State(kind=kind, q=q, k=k, v=v, o=o, last=last, run=run_, handles=[run_])
    g = _generator(seed)
    if kind == "rope":
        offsets = _offsets(case)
        tokens = int(offsets[-1])
        return State(kind=kind, ctx=ctx, offsets=offsets, qkv=_normal(g, tokens, QKV), q_gain=_gain(g, DIM),
                     k_gain=_gain(g, DIM), q=torch.zeros(tokens, HEADS * DIM, device="cuda", dtype=torch.float16),
                     k=torch.zeros(tokens, KV_HEADS * DIM, device="cuda", dtype=torch.float16))
    rows = case["rows"]
    half = lambda width: torch.zeros(rows, width, device="cuda", dtype=torch.float16)  # noqa: E731
    if kind == "projection":
        return State(kind=kind, ctx=ctx, x=_normal(g, rows, case["k"]), w=_q4(g, case["k"], case["n"]), y=half(case["n"]),
                     k=case["k"], n=case["n"], rows=rows)
    state = State(kind=kind, ctx=ctx, x=_normal(g, rows, HIDDEN), gate_up=_q4(g, HIDDEN, 2 * INTER), ffn=half(INTER),
                  rows=rows)
    if kind == "mlp":
        state.gain, state.down = _gain(g, HIDDEN), _q4(g, INTER, HIDDEN)
        state.normalized, state.y = half(HIDDEN), half(HIDDEN)
    return state


def run(state):
    kind = state.kind
    if kind == "forward":
        state.plan.run(state.ids, state.offsets, state.out.data_ptr())
        return state.out
    if kind == "attention":
        state.run.encode()
        return state.o if state.last is None else (state.o, state.last)
    ctx = state.ctx
    if kind == "rope":
        ctx.qk_norm_rope_qkv(state.qkv.data_ptr(), state.q.data_ptr(), state.k.data_ptr(), state.offsets,
                             q_weight_ptr=state.q_gain.data_ptr(), k_weight_ptr=state.k_gain.data_ptr())
        return state.q, state.k
    if kind == "projection":
        ctx.q4_matmul(state.x.data_ptr(), state.rows, state.k, state.w.data_ptr(), state.w.numel(), state.n,
                      state.y.data_ptr())
        return state.y
    x = state.x
    if kind == "mlp":
        ctx.rmsnorm(state.x.data_ptr(), state.gain.data_ptr(), state.normalized.data_ptr(), state.rows)
        x = state.normalized
    ctx.q4_matmul_swiglu(x.data_ptr(), state.rows, HIDDEN, state.gate_up.data_ptr(), state.gate_up.numel(), INTER,
                         state.ffn.data_ptr())
    if kind == "gate_up":
        return state.ffn
    ctx.q4_matmul(state.ffn.data_ptr(), state.rows, INTER, state.down.data_ptr(), state.down.numel(), HIDDEN,
                  state.y.data_ptr())
    return state.normalized, state.ffn, state.y


# ---- what a pass cannot do without ----------------------------------------------------------


def _pairs(length, mask):
    """Retained (query, key) pairs of one sequence."""
    full = length * (length + 1) // 2
    if mask == "causal":
        return full
    beyond = length - PREFIX - WINDOW  # queries whose prefix and window leave keys out
    return full - (beyond * (beyond + 1) // 2 if beyond > 0 else 0)


def _q4_bytes(k, n):
    return n * k // 32 * 20


def work(case):
    kind = case["kind"]
    if kind in ("forward", "attention", "rope"):
        lengths = lengths_of(case)
        tokens = sum(lengths)
    if kind == "forward":
        shapes = ((HIDDEN, QKV), (HEADS * DIM, HIDDEN), (HIDDEN, 2 * INTER), (INTER, HIDDEN))
        per_token = 2 * sum(k * n for k, n in shapes)
        pairs = sum(_pairs(n, "prefix_local") for n in lengths)
        return {"bytes": LAYERS * (sum(_q4_bytes(k, n) for k, n in shapes) + 4 * (2 * HIDDEN + 2 * DIM)) +
                tokens * (4 + HIDDEN // 256 * 210) + len(lengths) * HIDDEN * 4,
                "flops": LAYERS * (tokens * per_token + 4 * DIM * HEADS * pairs)}
    if kind == "attention":
        return {"bytes": tokens * 2 * DIM * (2 * HEADS + 2 * KV_HEADS) +
                (len(lengths) * 2 * HEADS * DIM if case["last"] else 0),
                "flops": 4 * DIM * HEADS * sum(_pairs(n, case["mask"]) for n in lengths)}
    if kind == "rope":
        return {"bytes": tokens * 2 * 2 * (HEADS + KV_HEADS) * DIM, "flops": tokens * 7 * (HEADS + KV_HEADS) * DIM}
    rows = case["rows"]
    if kind == "projection":
        k, n = case["k"], case["n"]
        return {"bytes": 2 * rows * (k + n) + _q4_bytes(k, n), "flops": 2 * rows * k * n}
    gate_up = {"bytes": 2 * rows * (HIDDEN + INTER) + _q4_bytes(HIDDEN, 2 * INTER),
               "flops": 4 * rows * HIDDEN * INTER}
    if kind == "gate_up":
        return gate_up
    # The block's three results are returned; ffn and normalized are not read back from memory here.
    return {"bytes": gate_up["bytes"] + 2 * rows * 2 * HIDDEN + _q4_bytes(INTER, HIDDEN),
            "flops": gate_up["flops"] + 2 * rows * INTER * HIDDEN}


def tolerance(case):
    """About four times what the outputs differ by from the same call in 64 bits (fp16 storage and
    fp16 probabilities with fp32 sums; the forward carries its roundings through 28 layers)."""
    return {"forward": {"rel": 8e-3, "max": 0.05}, "attention": {"rel": 1.1e-3, "max": 2e-2},
            "projection": {"rel": 8.5e-4, "max": 4e-3}, "gate_up": {"rel": 1.5e-3, "max": 8e-3},
            "mlp": {"rel": 2.2e-3, "max": 1.2e-2}, "rope": {"rel": 8.5e-4, "max": 4e-3}}[case["kind"]]


# ---- the same calls in 64 bits --------------------------------------------------------------


def _q4_dense(records, k, n):
    """The float64 weights f16(scale * (code - 8)) [n, k] of a tile32-compact tensor."""
    rec = records.view(n // 32, k // 32, 32, 20)
    scale = rec[..., 0:2].contiguous().view(torch.float16).double()
    codes = torch.cat([rec[..., 4:] & 15, rec[..., 4:] >> 4], dim=-1).double() - 8.0
    return (scale * codes).half().double().permute(0, 2, 1, 3).reshape(n, k)


def _attend(q, k, v, offsets, mask):
    """softmax(mask(q k^T) / sqrt(128)) v per sequence and query head, in float64."""
    out = torch.empty_like(q)
    for a, b in zip(offsets[:-1].tolist(), offsets[1:].tolist()):
        rows = torch.arange(b - a, device=q.device)
        keep = rows[None, :] <= rows[:, None]
        if mask == "prefix_local":
            keep &= (rows[None, :] < PREFIX) | (rows[None, :] + WINDOW > rows[:, None])
        for h in range(HEADS):
            scores = q[a:b, h] @ k[a:b, h // 2].T / math.sqrt(DIM)
            out[a:b, h] = torch.softmax(scores.masked_fill(~keep, -math.inf), dim=-1) @ v[a:b, h // 2]
    return out


def _swiglu(x, w):
    gate, up = (x @ w.T).chunk(2, dim=-1)
    return torch.nn.functional.silu(gate) * up


def _q6k_rows(table, ids):
    """Float64 rows of the Q6_K table: value 128 h + 32 quad + l of a 256-value block has its low
    nibble in ql[64 h + 32 (quad & 1) + l], its high bits in qh[32 h + l]."""
    blocks = table.view(VOCAB, HIDDEN // 256, 210)[ids]
    low = blocks[..., :128].reshape(*blocks.shape[:-1], 2, 2, 32)
    low = torch.stack([low & 15, low >> 4], dim=-3)  # half, quad >> 1, quad & 1, l
    high = blocks[..., 128:192].reshape(*blocks.shape[:-1], 2, 1, 1, 32)
    shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=table.device).view(2, 2, 1)
    codes = (low | ((high >> shift) & 3) << 4).double() - 32.0
    codes = codes.reshape(*blocks.shape[:-1], 2, 4, 2, 16)
    scales = blocks[..., 192:208].contiguous().view(torch.int8).double().reshape(*blocks.shape[:-1], 2, 4, 2, 1)
    d = blocks[..., 208:210].contiguous().view(torch.float16).double()
    return (codes * scales * d[..., None, None, None]).reshape(len(ids), HIDDEN)


def _exact_forward(case, seed):
    w, offsets = _model_tensors(seed), _offsets(case)
    x = _q6k_rows(w["table"], torch.from_numpy(_token_ids(case, seed)).cuda().long())
    tokens = len(x)
    for layer in w["layers"]:
        qkv = _norm_rows(x, layer["attn_norm"].double()) @ _q4_dense(layer["attn_qkv"], HIDDEN, QKV).T
        qkv = qkv.view(tokens, HEADS + 2 * KV_HEADS, DIM)
        q = _rope_rows(_norm_rows(qkv[:, :HEADS], layer["attn_q_norm"].double()), offsets)
        k = _rope_rows(_norm_rows(qkv[:, HEADS:HEADS + KV_HEADS], layer["attn_k_norm"].double()), offsets)
        a = _attend(q, k, qkv[:, HEADS + KV_HEADS:], offsets, "prefix_local").view(tokens, -1)
        x = x + a @ _q4_dense(layer["attn_output"], HEADS * DIM, HIDDEN).T
        f = _swiglu(_norm_rows(x, layer["ffn_norm"].double()), _q4_dense(layer["ffn_gate_up"], HIDDEN, 2 * INTER))
        x = x + f @ _q4_dense(layer["ffn_down"], INTER, HIDDEN).T
    last = _norm_rows(x[torch.from_numpy(offsets[1:] - 1).cuda().long()], w["output_norm"].double())
    return last / last.norm(dim=-1, keepdim=True)


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        return _exact_forward(case, seed)
    if kind == "attention":
        offsets, (q, k, v) = _offsets(case), _attention_inputs(case, seed)
        tokens = len(q)
        v = v[:, 3072:] if case["v_in_qkv"] else v
        heads = [t.double().view(tokens, -1, DIM) for t in (q, k, v)]
        o = _attend(*heads, offsets, case["mask"]).view(tokens, -1)
        return (o, o[torch.from_numpy(offsets[1:] - 1).cuda().long()]) if case["last"] else o
    g = _generator(seed)
    if kind == "rope":
        offsets = _offsets(case)
        x = _normal(g, int(offsets[-1]), QKV).double().view(int(offsets[-1]), -1, DIM)
        q = _rope_rows(_norm_rows(x[:, :HEADS], _gain(g, DIM).double()), offsets)
        k = _rope_rows(_norm_rows(x[:, HEADS:HEADS + KV_HEADS], _gain(g, DIM).double()), offsets)
        return q.reshape(len(x), -1), k.reshape(len(x), -1)
    x = _normal(g, case["rows"], case["k"] if kind == "projection" else HIDDEN).double()
    if kind == "projection":
        return x @ _q4_dense(_q4(g, case["k"], case["n"]), case["k"], case["n"]).T
    w = _q4_dense(_q4(g, HIDDEN, 2 * INTER), HIDDEN, 2 * INTER)
    if kind == "gate_up":
        return _swiglu(x, w)
    x = _norm_rows(x, _gain(g, HIDDEN).double())
    f = _swiglu(x, w)
    return x, f, f @ _q4_dense(_q4(g, INTER, HIDDEN), INTER, HIDDEN).T
