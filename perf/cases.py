"""Timed cases of the token loop: what a program that uses the library has it
do, through the public Python binding (gemma_amd.capi, the C-ABI of gg.h).

Whole calls on the two Gemma-3 shapes of gemma_amd.synth (270M and 1B, seeded
random Q8_0 weights): decode steps queued one ahead as the JavaScript host's
generate() queues them, and prompt prefills up to the first token. Single
kernels through the kernel-level entry points: the Q8_0 GEMV, the vocabulary
selector and the Q8_0 dequantisation.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "webgpu-gemma_amd"))
from gemma_amd import capi, synth  # noqa: E402

SHAPES = {"270m": synth.GEMMA3_270M, "1b": synth.GEMMA3_1B}
VOCAB = 262144
DEV = "cuda"
NORM_STD, WEIGHT_STD = 0.1, 0.02


def listed():
    return [
        # the fused QKV projection of the 1B model as a call of its own: the
        # smallest piece of work that a program asks for, where launching counts
        {"name": "gemv_qkv_1b", "kind": "gemv", "k": 1152, "rows": 1536},
        # the FFN's down projection: few rows, long sums
        {"name": "gemv_down_1b", "kind": "gemv", "k": 6912, "rows": 1152},
        # the tied LM head: the largest matrix, a stream from memory
        {"name": "gemv_lm_head_1b", "kind": "gemv", "k": 1152, "rows": VOCAB},
        # one sampled selection over logits that the caller computed, at the
        # options of a chat (temperature 0.7, top-p 0.9, penalty 1.2)
        {"name": "select_sampled", "kind": "select", "n": VOCAB, "temperature": 0.7, "top_p": 0.9, "rep": 1.2},
        # a weight tensor (an FFN matrix of the 1B model) expanded to f32
        {"name": "dequant_ffn_1b", "kind": "dequant", "n": 1152 * 6912},
        # a chat answer on the small model: greedy decode after a 64-id prompt
        {"name": "decode_270m_chat", "kind": "decode", "model": "270m", "pos": 64, "steps": 32,
         "temperature": 0.0, "top_p": 0.9, "rep": 1.0},
        # greedy decode of the 1B model at 2048 positions: the headline figure
        {"name": "decode_1b_2k", "kind": "decode", "model": "1b", "pos": 2048, "steps": 32,
         "temperature": 0.0, "top_p": 0.9, "rep": 1.0},
        # sampled decode late in a long conversation
        {"name": "decode_1b_32k_sampled", "kind": "decode", "model": "1b", "pos": 32700, "steps": 32,
         "temperature": 0.7, "top_p": 0.9, "rep": 1.2},
        # time to the first token of a short chat prompt
        {"name": "prefill_270m_64", "kind": "prefill", "model": "270m", "start": 0, "n": 64},
        # the next user turn of a conversation: a ragged prompt on reused KV
        {"name": "prefill_1b_turn", "kind": "prefill", "model": "1b", "start": 1309, "n": 187},
        # time to the first token of a 2048-id prompt: the headline prefill
        {"name": "prefill_1b_2048", "kind": "prefill", "model": "1b", "start": 0, "n": 2048},
        # a long document up to its first token
        {"name": "prefill_1b_32k", "kind": "prefill", "model": "1b", "start": 0, "n": 32749},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemv", "select", "dequant", "decode", "decode", "prefill", "prefill"])
    if kind == "gemv":
        k = 64 * _log_int(rng, 1, 128)
        rows = 64 * _log_int(rng, 1, max(1, min(4096, 1152 * VOCAB // (64 * k))))
        return {"kind": kind, "k": k, "rows": rows}
    if kind == "select":
        t, rep = rng.choice([(0.0, 1.0), (0.7, 1.2), (1.0, 1.0), (0.0, 1.3), (1.4, 1.1)])
        return {"kind": kind, "n": _log_int(rng, 1000, VOCAB), "temperature": t, "top_p": rng.choice([0.5, 0.9, 0.95, 1.0]),
                "rep": rep}
    if kind == "dequant":
        return {"kind": kind, "n": 32 * _log_int(rng, 36, 1152 * VOCAB // 32)}
    model = rng.choice(["270m", "1b"])
    if kind == "decode":
        t, rep = rng.choice([(0.0, 1.0), (0.0, 1.0), (0.7, 1.2), (1.0, 1.0)])
        return {"kind": kind, "model": model, "pos": _log_int(rng, 2, 32700), "steps": rng.randint(4, 32),
                "temperature": t, "top_p": rng.choice([0.9, 0.95]), "rep": rep}
    n = _log_int(rng, 2, 32000)
    return {"kind": kind, "model": model, "n": n, "start": rng.choice([0, rng.randint(1, 32000 - n) if n < 32000 else 0])}


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _q8(gen, rows, k, std=WEIGHT_STD):
    """Q8_0 blocks of N(0, std): uint8 [rows * k / 32, 34] on the GPU."""
    w = torch.randn(rows * k // 32, 32, generator=gen, device=DEV) * std
    d = (w.abs().amax(1, keepdim=True) / 127).half()
    q = torch.round(w / d.float()).clamp_(-127, 127).to(torch.int8)
    return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1)


def _q8_wide(gen, rows, k):
    """Isolated operands: q uniform in [-127, 127], |d| lognormal, both signs."""
    nb = rows * k // 32
    q = torch.randint(-127, 128, (nb, 32), generator=gen, device=DEV, dtype=torch.int8)
    d = torch.exp(torch.randn(nb, 1, generator=gen, device=DEV) * 0.5 - 6)
    d = (d * (torch.randint(0, 2, (nb, 1), generator=gen, device=DEV) * 2 - 1)).half()
    return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1)


def _q8_f64(blocks, rows, k):
    """The blocks' exact values as f64 [rows, k]."""
    d = blocks[:, :2].contiguous().view(torch.float16).double()
    return (blocks[:, 2:].contiguous().view(torch.int8).double() * d).view(rows, k)


def _model(shape, seed):
    """(name, ggml type, dims, tensor on the GPU) of every tensor, in upload order."""
    gen = _generator(seed)
    H, I, Q, KV = shape.hidden, shape.inter, shape.q_dim, shape.kv_dim
    yield "token_embd.weight", capi.GG_TYPE_Q8_0, [H, shape.vocab], _q8(gen, shape.vocab, H)
    dims = {"attn_q": (H, Q), "attn_k": (H, KV), "attn_v": (H, KV), "attn_output": (Q, H),
            "ffn_gate": (H, I), "ffn_up": (H, I), "ffn_down": (I, H)}

    def norm(n):
        return 1 + NORM_STD * torch.randn(n, generator=gen, device=DEV)

    yield "output_norm.weight", capi.GG_TYPE_F32, [H], norm(H)
    for l in range(shape.layers):
        for n in synth.Q8_NAMES:
            k, rows = dims[n]
            yield f"blk.{l}.{n}.weight", capi.GG_TYPE_Q8_0, [k, rows], _q8(gen, rows, k)
        for n in synth.NORM_NAMES:
            size = shape.head_dim if n in ("attn_q_norm", "attn_k_norm") else H
            yield f"blk.{l}.{n}.weight", capi.GG_TYPE_F32, [size], norm(size)


def _shape(case):
    last = case["pos"] + case["steps"] if case["kind"] == "decode" else case["start"] + case["n"]
    ctx = 2048
    while ctx <= last:
        ctx *= 2
    return SHAPES[case["model"]].gemma3_mode().with_ctx(min(ctx, 32768 if last < 32768 else ctx))


def _ids(case, seed):
    """Ids already in the KV cache, then the ids of the timed call's own turn."""
    before, n = (case["pos"], 0) if case["kind"] == "decode" else (case["start"], case["n"])
    ids = np.random.default_rng(seed).integers(0, VOCAB, before + n).astype(np.int32)
    return ids[:before], ids[before:]


def _draws(case, seed):
    return [float(u) for u in np.random.default_rng([int(seed), 1]).random(case["steps"])]


def _seen(ids):
    """The decode cases' penalty set at the start: the turn's last ids, as generate() fills it."""
    return ids[-256:]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "select", "dequant"):
        gen = _generator(seed)
        stream = torch.cuda.current_stream().cuda_stream
        if kind == "gemv":
            k, rows = case["k"], case["rows"]
            src, x = _q8_wide(gen, rows, k), torch.randn(k, generator=gen, device=DEV)
            w = torch.empty(capi.q8_0_packed_size(rows, k), dtype=torch.uint8, device=DEV)
            capi.q8_0_repack(src.data_ptr(), w.data_ptr(), rows, k, stream)
            return {"case": case, "w": w, "x": x, "y": torch.empty(rows, device=DEV), "src": src, "stream": stream}
        if kind == "dequant":
            return {"case": case, "src": _q8_wide(gen, 1, case["n"]), "y": torch.empty(case["n"], device=DEV), "stream": stream}
        n = case["n"]
        logits = torch.randn(n, generator=gen, device=DEV) * 2
        seen = torch.zeros((n + 31) // 32, dtype=torch.int32, device=DEV)
        at = torch.randint(0, seen.numel(), (256,), generator=gen, device=DEV)
        seen[at] = torch.randint(-2**31, 2**31, (256,), generator=gen, device=DEV, dtype=torch.int64).to(torch.int32)
        return {"case": case, "logits": logits, "seen": seen, "u": random.Random(int(seed)).random(),
                "ws": torch.empty(capi.select_workspace_size(n), dtype=torch.uint8, device=DEV),
                "topk": torch.zeros(256, 2, dtype=torch.int32, device=DEV), "stream": stream}
    shape = _shape(case)
    e = capi.Engine(shape.gg_config(prefill_batch=min(4096, shape.ctx)))
    for name, t, dims, data in _model(shape, seed):
        e.upload(name, t, dims, data.cpu().numpy())
    e.finalize()
    before, ids = _ids(case, seed)
    state = {"case": case, "engine": e, "ids": ids}
    if len(before):
        e.prefill(before, 0)
    if kind == "decode":
        state.update(first=e.select(), seen=_seen(before), u=_draws(case, seed))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        capi.q8_0_gemv(state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(), case["rows"], case["k"],
                       state["stream"])
        return state["y"]
    if kind == "dequant":
        capi.q8_0_dequant(state["src"].data_ptr(), state["y"].data_ptr(), case["n"], state["stream"])
        return state["y"]
    if kind == "select":
        token = capi.select_logits(state["logits"].data_ptr(), case["n"], state["seen"].data_ptr(), case["temperature"],
                                   case["top_p"], case["rep"], state["u"], state["ws"].data_ptr(), state["topk"].data_ptr(),
                                   state["stream"])
        return {"token": token, "values": state["topk"][:, 0].view(torch.float32), "ids": state["topk"][:, 1]}
    e = state["engine"]
    if kind == "prefill":
        e.prefill(state["ids"], case["start"])
        return {"tokens": np.array([e.select()]), "logits": e.read(capi.READ_LOGITS)}
    # one step queued ahead, each taking the previous id on the device
    opt = (case["temperature"], case["top_p"], case["rep"])
    pos, steps, u = case["pos"], case["steps"], state["u"]
    e.penalty_reset()
    e.penalty_add(state["seen"])
    tokens = []
    e.step_submit(state["first"], pos, *opt, u[0])
    for i in range(steps):
        if i + 1 < steps:
            e.step_submit(-1, pos + i + 1, *opt, u[i + 1])
        tokens.append(e.step_collect())
    return {"tokens": np.array(tokens), "logits": e.read(capi.READ_LOGITS)}


def _span(pos, window):
    return pos + 1 if not window else min(pos + 1, window)


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        k, rows = case["k"], case["rows"]
        return {"bytes": rows * k // 32 * 34 + 4 * (k + rows), "flops": 2 * rows * k}
    if kind == "dequant":
        return {"bytes": case["n"] // 32 * 34 + 4 * case["n"], "flops": case["n"]}
    if kind == "select":
        return {"bytes": 4 * case["n"] + case["n"] // 8, "flops": case["n"]}
    s = _shape(case)
    layers = s.q8_bytes() - s.vocab * s.hidden // 32 * 34
    norms = 4 * (s.layers * (4 * s.hidden + 2 * s.head_dim) + s.hidden)
    head = s.vocab * s.hidden // 32 * 34 + 8 * s.vocab
    per_layer = (layers // 34 * 32) // s.layers
    kv_row, total, flops = 2 * 4 * s.head_dim, 0, 0
    windows = [s.window if l % s.swa_period < s.swa_period - 1 else 0 for l in range(s.layers)]
    if kind == "decode":
        for i in range(case["steps"]):
            spans = sum(_span(case["pos"] + i, w) for w in windows)
            total += layers + norms + head + kv_row * (spans + s.layers)
            flops += 2 * (per_layer * s.layers + s.vocab * s.hidden) + 4 * s.q_dim * spans
        return {"bytes": total, "flops": flops}
    n, start = case["n"], case["start"]
    spans = {w: sum(_span(p, w) for p in range(start, start + n)) for w in set(windows)}
    kv = sum(min(start, w) if w else start for w in windows)   # rows of earlier turns that are read
    total = layers + norms + head + kv_row * (kv + n * s.layers) + n * (4 + s.hidden // 32 * 34)
    flops = 2 * n * per_layer * s.layers + sum(4 * s.q_dim * spans[w] for w in windows) + 2 * s.vocab * s.hidden
    return {"bytes": total, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("select", "dequant"):
        return "exact"
    if kind == "gemv":
        # f32 sums over k: 1.3e-7 off the 64-bit product
        return {"rel": 6e-7, "max": 6e-6}
    # f32 sums and the products of bf16 hi + lo pairs through every layer: the
    # logits are 6e-6 to 1.6e-5 off the 64-bit model
    return {"rel": 6e-5, "max": 6e-4, "differ": 0.0}


# ---- the same in 64 bits, plain torch ---------------------------------------

def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope64(x, pos, theta):
    """NEOX rotation; the angle is f32(pos) * f32 frequency, as the model defines it."""
    half = x.shape[-1] // 2
    e = (np.arange(half) * 2).astype(np.float32) / np.float32(x.shape[-1])
    freq = np.float32(1) / (np.float64(theta) ** e.astype(np.float64)).astype(np.float32)
    a = torch.from_numpy((pos.astype(np.float32)[:, None] * freq).astype(np.float64)).to(DEV)
    c, s = torch.cos(a), torch.sin(a)
    if x.dim() == 3:
        c, s = c[:, None], s[:, None]
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], -1)


class _Model64:
    def __init__(self, shape, seed):
        self.s = shape
        self.w = {}
        for name, t, dims, data in _model(shape, seed):
            self.w[name[:-7]] = _q8_f64(data, dims[1], dims[0]) if t == capi.GG_TYPE_Q8_0 else data.double()
        self.kv = [[torch.empty(0, shape.head_dim, dtype=torch.float64, device=DEV)] * 2 for _ in range(shape.layers)]

    def forward(self, ids, start):
        """Rows of ids at positions start..; the last row's output-normed hidden."""
        s, w, n = self.s, self.w, len(ids)
        pos = np.arange(start, start + n)
        p = torch.from_numpy(pos).to(DEV)
        x = w["token_embd"][torch.from_numpy(np.asarray(ids, np.int64)).to(DEV)] * math.sqrt(s.hidden)
        for l in range(s.layers):
            b, local = f"blk.{l}.", l % s.swa_period < s.swa_period - 1
            theta = s.theta_local if local else s.theta_global
            h = _rms64(x, w[b + "attn_norm"], s.eps)
            q = (h @ w[b + "attn_q"].T).view(n, s.n_q, s.head_dim)
            k, v = h @ w[b + "attn_k"].T, h @ w[b + "attn_v"].T
            q = _rope64(_rms64(q, w[b + "attn_q_norm"], s.eps), pos, theta)
            k = _rope64(_rms64(k, w[b + "attn_k_norm"], s.eps), pos, theta)
            self.kv[l] = [torch.cat([self.kv[l][0], k]), torch.cat([self.kv[l][1], v])]
            lo = max(0, start - s.window + 1) if local and s.window else 0
            K, V = self.kv[l][0][lo:], self.kv[l][1][lo:]
            keys = torch.arange(lo, start + n, device=DEV)
            out = (keys[None] > p[:, None])
            if local and s.window:
                out |= keys[None] <= p[:, None] - s.window
            o = torch.empty(n, s.n_q, s.head_dim, dtype=torch.float64, device=DEV)
            for hd in range(s.n_q):
                sc = (q[:, hd] @ K.T) / math.sqrt(s.head_dim)
                o[:, hd] = torch.softmax(sc.masked_fill_(out, -math.inf), -1) @ V
            x = x + _rms64(o.view(n, -1) @ w[b + "attn_output"].T, w[b + "post_attention_norm"], s.eps)
            h = _rms64(x, w[b + "ffn_norm"], s.eps)
            g = h @ w[b + "ffn_gate"].T
            g = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
            x = x + _rms64((g * (h @ w[b + "ffn_up"].T)) @ w[b + "ffn_down"].T, w[b + "post_ffw_norm"], s.eps)
        return _rms64(x[-1], w["output_norm"], s.eps)

    def prompt(self, ids, start=0):
        h = None
        for i in range(0, len(ids), 1024):
            h = self.forward(ids[i:i + 1024], start + i)
        return h

    def logits(self, h):
        return w_matvec(self.w["token_embd"], h)


def w_matvec(w, x):
    return (w @ x[:, None])[:, 0]


def _pick64(logits, seen, t, top_p, rep, u):
    """The selection: the largest value of each class id % 256, penalty, temperature, top-p walk."""
    if t == 0 and rep <= 1:
        return int(logits.argmax())
    n = len(logits)
    rows = np.full(-(-n // 256) * 256, -np.inf)
    rows[:n] = logits
    rows = rows.reshape(-1, 256)
    ids = rows.argmax(0) * 256 + np.arange(256)
    v = logits[ids].copy()
    hit = np.isin(ids, list(seen))
    if rep > 1:
        v[hit] = np.where(v[hit] > 0, v[hit] / rep, v[hit] * rep)
    order = np.argsort(-v, kind="stable")
    ids, v = ids[order], v[order]
    if t == 0:
        return int(ids[0])
    p = np.exp((v - v[0]) / t)
    reach = np.nonzero(np.cumsum(p / p.sum()) >= top_p)[0]
    cut = int(reach[0]) + 1 if len(reach) else 256
    past = np.nonzero(u * p[:cut].sum() - np.cumsum(p[:cut]) <= 0)[0]
    return int(ids[int(past[0]) if len(past) else cut - 1])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "dequant"):
        gen = _generator(seed)
        k, rows = (case["k"], case["rows"]) if kind == "gemv" else (case["n"], 1)
        blocks = _q8_wide(gen, rows, k)
        if kind == "dequant":
            return _q8_f64(blocks, 1, k)[0]
        x = torch.randn(k, generator=gen, device=DEV).double()
        return torch.cat([w_matvec(_q8_f64(blocks[i * k // 32:(i + 16384) * k // 32], -1, k), x)
                          for i in range(0, rows, 16384)])
    if kind == "select":
        return None   # a choice among the given values: compared exactly
    m = _Model64(_shape(case), seed)
    before, ids = _ids(case, seed)
    if kind == "prefill":
        if len(before):
            m.prompt(before)
        logits = m.logits(m.prompt(ids, case["start"])).cpu().numpy()
        return {"tokens": None, "logits": logits}
    tok = int(m.logits(m.prompt(before)).argmax())
    seen, logits = set(int(i) for i in _seen(before)), None
    for i, u in enumerate(_draws(case, seed)):
        logits = m.logits(m.forward([tok], case["pos"] + i)).cpu().numpy()
        tok = _pick64(logits, seen, case["temperature"], case["top_p"], case["rep"], u)
        seen.add(tok)
    return {"tokens": None, "logits": logits}
