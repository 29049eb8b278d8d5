"""The calls whose speed this library is judged by, as data and as runnable passes.

Five paths, each through the entry point a program calls:
  projection  HipSession.run_device: W x for packed weights on the device, one
              token (decode) or a chunk of a prompt (prefill)
  boundary    HipSession.run_batch_into: the same from and to host arrays, as
              llambda's own descriptor calls it
  moe         HipMoeSession.run_device: a whole routed feed-forward layer
  step        HipLlamaSession.step_device: one decode step, logits out
  sample      HipSampler.sample: the next token from a row of logits

Weights follow llambda_amd/synthetic.py's distributions (uniform codes, fp16
scales in [1e-4, 1e-3]); activations are N(0, 1).
"""
import math

import numpy as np
import torch

from llambda_amd import ggml
from llambda_amd.hip_backend import make_hip_session_packed
from llambda_amd.llama import HipLlamaSession, LlamaConfig, synthetic_llama_device
from llambda_amd.moe import NEMOTRON_H, QWEN3NEXT, HipMoeSession, MoeLayer
from llambda_amd.sampling import HipSampler

TYPES = {"F32": ggml.F32, "Q5_0": ggml.Q5_0, "Q8_0": ggml.Q8_0, "Q4_K": ggml.Q4_K, "Q6_K": ggml.Q6_K}
GEOMETRY = {"F32": (1, 4), "Q5_0": (32, 22), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210)}

QWEN = dict(variant="qwen3next", hidden=2048, experts=512, top_k=10, ffn=512, shared_ffn=512,
            up="Q4_K", down="Q6_K")
NEMOTRON = dict(variant="nemotron_h", hidden=2688, experts=128, top_k=6, ffn=1856, shared_ffn=3712,
                up="Q5_0", down="Q5_0")


def listed():
    return [
        # attn_k of one decoded token: the smallest projection of a decode step
        {"name": "attn_k_1", "path": "projection", "type": "Q4_K", "rows": 1024, "columns": 4096, "tokens": 1},
        # the output head of one decoded token: the largest matrix a step reads
        {"name": "head_1", "path": "projection", "type": "Q6_K", "rows": 128256, "columns": 4096, "tokens": 1},
        # ffn_down from and to host arrays: the reference's run-session call
        {"name": "host_ffn_down_1", "path": "boundary", "type": "Q6_K", "rows": 4096, "columns": 14336, "tokens": 1},
        # a few sequences decoded together (or a few drafted tokens checked)
        {"name": "ffn_up_7", "path": "projection", "type": "Q4_K", "rows": 14336, "columns": 4096, "tokens": 7},
        # a short prompt through an 8-bit projection whose width is no multiple of 256
        {"name": "latent_down_129", "path": "projection", "type": "Q8_0", "rows": 1024, "columns": 2688, "tokens": 129},
        # a prompt of ragged length through ffn_down
        {"name": "ffn_down_1000", "path": "projection", "type": "Q6_K", "rows": 4096, "columns": 14336, "tokens": 1000},
        # a long prompt's chunk through ffn_gate: the largest call
        {"name": "ffn_gate_2048", "path": "projection", "type": "Q4_K", "rows": 14336, "columns": 4096, "tokens": 2048},
        # MoE layers: one decoded token, and prompts
        {"name": "moe_qwen3next_1", "path": "moe", "tokens": 1, **QWEN},
        {"name": "moe_qwen3next_256", "path": "moe", "tokens": 256, **QWEN},
        {"name": "moe_nemotron_h_1024", "path": "moe", "tokens": 1024, **NEMOTRON},
        # decode step of eight layers and the head, 4095 tokens in the cache
        {"name": "step_4095", "path": "step", "hidden": 4096, "layers": 8, "heads": 32, "kv_heads": 8,
         "ffn": 14336, "vocab": 128256, "position": 4095},
        # the next token, with the reference's default filters
        {"name": "sample_128256", "path": "sample", "vocab": 128256, "top_k": 40, "top_p": 0.95,
         "history": 256},
    ]


MOST_PRODUCTS = 14336 * 4096 * 2048 // 2  # of a drawn projection


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["projection", "projection", "projection", "moe", "moe", "boundary", "step", "sample"])
    if path in ("projection", "boundary"):
        kind = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q6_K", "Q8_0", "Q5_0", "F32"])
        rows = rng.choice([rng.choice([512, 1024, 2048, 4096, 5120, 14336]), _log(rng, 33, 16000)])
        if kind in ("Q4_K", "Q6_K"):
            columns = 256 * _log(rng, 2, 64)
        elif kind == "F32":
            columns = 4 * _log(rng, 64, 1024)
            rows = min(rows, 2048)
        else:
            columns = rng.choice([rng.choice([1024, 1856, 2688, 3712]), 32 * _log(rng, 8, 128)])
        most = min(2048, max(1, MOST_PRODUCTS // (rows * columns)))
        if path == "boundary":
            most = min(most, 64)
        if kind == "F32":
            most = min(most, 512)
        tokens = 1 if rng.random() < 0.3 else _log(rng, 1, most)
        return {"path": path, "type": kind, "rows": rows, "columns": columns, "tokens": tokens}
    if path == "moe":
        if rng.random() < 0.5:
            return {"path": "moe", "tokens": _log(rng, 1, 512), **QWEN}
        case = {"path": "moe", "tokens": _log(rng, 1, 1024), **NEMOTRON}
        case["up"], case["down"] = rng.choice([("Q5_0", "Q5_0"), ("Q8_0", "Q8_0"), ("Q5_0", "Q8_0")])
        return case
    if path == "step":
        case = rng.choice([
            dict(hidden=4096, layers=rng.randint(1, 8), heads=32, kv_heads=8, ffn=14336, vocab=128256),
            dict(hidden=2048, layers=rng.randint(2, 8), heads=32, kv_heads=8, ffn=5632, vocab=32000)])
        return {"path": "step", **case, "position": _log(rng, 1, 8000)}
    return {"path": "sample", "vocab": rng.choice([32000, 128256, _log(rng, 8000, 150000)]),
            "top_k": rng.choice([0, 1, 40, 40, 64, 200]), "top_p": rng.choice([0.5, 0.9, 0.95, 1.0]),
            "history": _log(rng, 1, 4096)}


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _bytes(g, kind, rows, columns):
    """rows * row_bytes packed bytes on the device."""
    if kind == "F32":
        return (torch.randn(rows * columns, device="cuda", generator=g) * 0.02).view(torch.uint8)
    elements, size = GEOMETRY[kind]
    n = rows * (columns // elements)
    b = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=g)

    def d16():
        return (torch.rand((n, 1), device="cuda", generator=g) * 9e-4 + 1e-4).half().view(torch.uint8)

    if kind == "Q6_K":
        b[:, 192:208] = torch.randint(-64, 64, (n, 16), dtype=torch.int8, device="cuda",
                                      generator=g).view(torch.uint8)
        b[:, 208:210] = d16()
    else:
        b[:, 0:2] = d16()
        if kind == "Q4_K":
            b[:, 2:4] = d16()
    return b.reshape(-1)


def _projection(case, seed):
    g = _generator(seed)
    w = _bytes(g, case["type"], case["rows"], case["columns"])
    x = torch.randn((case["tokens"], case["columns"]), device="cuda", generator=g)
    return w, x


def _moe(case, seed):
    """The layer's tensors on the device, by MoeLayer's field names, and x."""
    g = _generator(seed)
    h, e, f, fs = case["hidden"], case["experts"], case["ffn"], case["shared_ffn"]
    up, down = case["up"], case["down"]
    t = {"router": torch.randn((e, h), device="cuda", generator=g) * 0.02}
    t["up"] = _bytes(g, up, e * f, h)
    t["down"] = _bytes(g, down, e * h, f)
    t["shared_up"] = _bytes(g, up, fs, h)
    t["shared_down"] = _bytes(g, down, h, fs)
    if case["variant"] == "qwen3next":
        t["gate"] = _bytes(g, up, e * f, h)
        t["shared_gate"] = _bytes(g, up, fs, h)
        t["shared_gate_inp"] = torch.randn(h, device="cuda", generator=g) * 0.02
    else:  # Zipf-distributed popularity of the experts
        rank = torch.randperm(e, device="cuda", generator=g) + 1
        p = rank.double() ** -1.1
        t["router_bias"] = (0.5 * torch.log(p / p.sum())).float()
    x = torch.randn((case["tokens"], h), device="cuda", generator=g)
    return t, x


def _moe_layer(case, t):
    def host(name):
        return t[name].cpu().numpy() if name in t else None

    def packed(name, kind):
        return (TYPES[kind], host(name)) if name in t else None

    return MoeLayer(
        variant=QWEN3NEXT if case["variant"] == "qwen3next" else NEMOTRON_H,
        hidden=case["hidden"], expert_count=case["experts"], top_k=case["top_k"],
        expert_ffn=case["ffn"], shared_ffn=case["shared_ffn"], router=host("router"),
        up=packed("up", case["up"]), down=packed("down", case["down"]),
        gate=packed("gate", case["up"]), shared_gate_inp=host("shared_gate_inp"),
        router_bias=host("router_bias"), expert_weights_scale=1.0, expert_weights_norm=True,
        shared_gate=packed("shared_gate", case["up"]), shared_up=packed("shared_up", case["up"]),
        shared_down=packed("shared_down", case["down"]))


def _model(case, seed):
    """Weights (device tensors), the token, and the cache's keys and values."""
    c = LlamaConfig(hidden=case["hidden"], layer_count=case["layers"], head_count=case["heads"],
                    kv_head_count=case["kv_heads"], ffn=case["ffn"], vocab=case["vocab"],
                    rope_dimension=case["hidden"] // case["heads"], context=case["position"] + 1)
    rng = np.random.default_rng(seed)
    w = synthetic_llama_device(seed, c, rng)
    g = _generator(seed + 1)
    shape = (c.kv_head_count, case["position"], c.head_dim)
    kv = [(torch.randn(shape, device="cuda", generator=g), torch.randn(shape, device="cuda", generator=g))
          for _ in range(c.layer_count)]
    torch.cuda.synchronize()  # the session copies on a stream of its own
    return c, w, int(rng.integers(0, c.vocab)), kv


def _logits(case, seed):
    g = _generator(seed)
    logits = torch.randn(case["vocab"], device="cuda", generator=g) * 3.0
    rng = np.random.default_rng(seed)
    return logits, rng.integers(0, case["vocab"], size=case["history"]), float(rng.random())


_STREAM = []


def _stream():
    """The one stream that a program's passes follow each other on."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0].cuda_stream


def prepare(case, seed):
    path = case["path"]
    if path in ("projection", "boundary"):
        w, x = _projection(case, seed)
        session = make_hip_session_packed(w.cpu().numpy(), TYPES[case["type"]], case["rows"], case["columns"])
        if path == "boundary":
            return {"path": path, "session": session, "x": x.cpu().numpy(), "tokens": case["tokens"],
                    "y": np.empty((case["tokens"], case["rows"]), dtype=np.float32)}
        y = torch.empty((case["tokens"], case["rows"]), device="cuda")
        state = {"session": session, "x": x, "y": y, "tokens": case["tokens"], "stream": _stream()}
    elif path == "moe":
        t, x = _moe(case, seed)
        state = {"session": HipMoeSession(_moe_layer(case, t)), "x": x, "y": torch.empty_like(x),
                 "tokens": case["tokens"], "stream": _stream()}
    elif path == "step":
        c, w, token, kv = _model(case, seed)
        session = HipLlamaSession(w)
        for i, (k, v) in enumerate(kv):
            session.write_kv_device(i, 0, case["position"], k.data_ptr(), v.data_ptr())
        state = {"session": session, "weights": w, "token": token, "position": case["position"],
                 "logits": torch.empty(c.vocab, device="cuda"), "stream": _stream()}
    else:
        logits, history, roll = _logits(case, seed)
        state = {"session": HipSampler(case["vocab"]), "logits": logits, "roll": roll, "history": history,
                 "top_k": case["top_k"], "top_p": case["top_p"]}
    torch.cuda.synchronize()
    return {"path": path, **state}


def run(state):
    path, session = state["path"], state["session"]
    if path == "boundary":
        return session.run_batch_into(state["y"], state["x"], state["tokens"])
    if path == "projection":
        session.run_device(state["x"].data_ptr(), state["y"].data_ptr(), state["tokens"], state["stream"])
        return state["y"]
    if path == "moe":
        session.run_device(state["x"].data_ptr(), state["y"].data_ptr(), state["tokens"], state["stream"])
        return state["y"]
    if path == "step":
        session.step_device(state["token"], state["position"], state["logits"].data_ptr(), state["stream"])
        return state["logits"]
    return session.sample(state["logits"].data_ptr(), device_count=state["logits"].numel(),
                          random_value=state["roll"], history=state["history"], top_k=state["top_k"],
                          top_p=state["top_p"])


# ------------------------------------------------------------------ work

def _size(kind, rows, columns):
    elements, size = GEOMETRY[kind]
    return rows * columns // elements * size


def work(case):
    path = case["path"]
    if path in ("projection", "boundary"):
        n, k, t = case["rows"], case["columns"], case["tokens"]
        return {"bytes": _size(case["type"], n, k) + 4 * t * (n + k), "flops": 2 * n * k * t}
    if path == "moe":
        h, e, k, f, fs, t = (case[n] for n in ("hidden", "experts", "top_k", "ffn", "shared_ffn", "tokens"))
        ups = 2 if case["variant"] == "qwen3next" else 1
        expert = ups * _size(case["up"], f, h) + _size(case["down"], h, f)
        shared = ups * _size(case["up"], fs, h) + _size(case["down"], h, fs)
        touched = e * (1 - (1 - k / e) ** t)  # distinct experts, if all are as popular
        return {"bytes": int(touched * expert) + shared + 4 * e * h + 8 * t * h,
                "flops": 2 * t * (e * h + (ups + 1) * h * (k * f + fs))}
    if path == "step":
        h, f, v = case["hidden"], case["ffn"], case["vocab"]
        kv = h // case["heads"] * case["kv_heads"]
        layer = (_size("Q4_K", h + kv, h) + _size("Q6_K", kv, h) + _size("Q4_K", h, h)
                 + _size("Q4_K", 2 * f, h) + _size("Q6_K", h, f) + 8 * kv * (case["position"] + 1))
        products = case["layers"] * (h * (2 * h + 2 * kv + 3 * f) + 2 * h * (case["position"] + 1)) + v * h
        return {"bytes": case["layers"] * layer + _size("Q6_K", v, h) + 4 * v, "flops": 2 * products}
    return {"bytes": 4 * case["vocab"], "flops": 10 * case["vocab"]}


# ------------------------------------------------------------------ outputs

def tolerance(case):
    """About four times the error against exact() that was measured: one token's
    activations enter the products as two bf16 (2.8e-6), several tokens' as
    fp32 (2.4e-7); a MoE layer chains two such products (5.7e-6)."""
    path = case["path"]
    if path in ("projection", "boundary"):
        return {"rel": 1e-5 if case["tokens"] == 1 else 1e-6}
    if path == "moe":
        return {"rel": 2.5e-5}
    if path == "step":
        return {"rel": 5e-5}
    return "exact"


def _weights(b, kind, rows, columns):
    """The packed rows' values in 64 bits, [rows][columns]."""
    if kind == "F32":
        return b.view(torch.float32).reshape(rows, columns).double()
    elements, size = GEOMETRY[kind]
    b = b.reshape(-1, size)
    n = b.shape[0]

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if kind == "Q8_0":
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif kind == "Q5_0":
        bits = (b[:, 2:6, None] >> torch.arange(8, dtype=torch.uint8, device=b.device)) & 1
        bits = bits.reshape(n, 32)
        q = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], dim=1) | (bits << 4)
        w = half(0) * (q.double() - 16)
    elif kind == "Q4_K":
        s = b[:, 4:16]
        scale = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], dim=1)
        low = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], dim=1)
        p = b[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat([p & 15, p >> 4], dim=2).reshape(n, 8, 32)
        w = ((half(0) * scale.double())[:, :, None] * q.double()
             - (half(2) * low.double())[:, :, None])
    else:  # Q6_K: halves of 128, each four runs of 32
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).reshape(1, 1, 4, 1)
        q = torch.cat([ql & 15, ql >> 4], dim=2) | (((qh >> shift) & 3) << 4)
        scale = half(208) * b[:, 192:208].contiguous().view(torch.int8).double()
        w = scale.reshape(n, 16, 1) * (q.reshape(n, 16, 16).double() - 32)
    return w.reshape(rows, columns)


def _silu(v):
    return v * torch.sigmoid(v)


def _exact_moe(case, seed):
    t, x = _moe(case, seed)
    h, e, f, fs = case["hidden"], case["experts"], case["ffn"], case["shared_ffn"]
    up, down = case["up"], case["down"]
    x = x.double()

    def layer(names, i, width):
        u = x_i @ _weights(t[names[0]][i], up, width, h).T
        if case["variant"] == "qwen3next":
            u = u * _silu(x_i @ _weights(t[names[1]][i], up, width, h).T)
        else:
            u = torch.relu(u) ** 2
        return u @ _weights(t[names[2]][i], down, h, width).T

    logits = x @ t["router"].double().T
    if "router_bias" in t:
        logits = logits + t["router_bias"].double()
    top, chosen = logits.topk(case["top_k"], dim=1)
    weight = torch.sigmoid(top)
    weight = weight / weight.sum(dim=1, keepdim=True)
    for name in ("gate", "up", "down"):
        if name in t:
            t[name] = t[name].reshape(e, -1)
    y = torch.zeros_like(x)
    for i in range(e):
        token, rank = torch.nonzero(chosen == i, as_tuple=True)
        if token.numel():
            x_i = x[token]
            y.index_add_(0, token, weight[token, rank][:, None] * layer(("up", "gate", "down"), i, f))
    x_i = x
    shared = layer(("shared_up", "shared_gate", "shared_down"), slice(None), fs)
    if "shared_gate_inp" in t:
        shared = torch.sigmoid(x @ t["shared_gate_inp"].double())[:, None] * shared
    return y + shared


def _exact_step(case, seed):
    c, w, token, kv = _model(case, seed)
    names = {v: k for k, v in TYPES.items()}
    d, p = c.head_dim, case["position"]

    def rows(t, n, k):
        return _weights(t.owner.reshape(-1), names[t.type], n, k)

    def vector(a):
        return torch.from_numpy(np.asarray(a)).cuda().double()

    def norm(v, scale):
        return v / torch.sqrt((v * v).mean() + float(np.float32(c.norm_epsilon))) * vector(scale)

    # the power is a single float, as the path's definition has it
    power = (float(np.float32(c.rope_base)) ** (np.arange(0, d, 2) / d)).astype(np.float32).astype(np.float64)
    angle = torch.from_numpy(p / (np.asarray(w.rope_factors, dtype=np.float64) * power)).cuda()
    cos, sin = torch.cos(angle), torch.sin(angle)

    def rotated(v):
        a, b = v[:, 0::2], v[:, 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], dim=2).reshape(-1, d)

    e = w.token_embd.owner[token * (c.hidden // 256):(token + 1) * (c.hidden // 256)].reshape(-1)
    x = _weights(e, names[w.token_embd.type], 1, c.hidden)[0]
    share = c.head_count // c.kv_head_count
    for at, (keys, values) in zip(w.layers, kv):
        v = norm(x, at.attn_norm)
        q = rotated((rows(at.attn_q, c.head_count * d, c.hidden) @ v).reshape(-1, d)) / math.sqrt(d)
        k = rotated((rows(at.attn_k, c.kv_head_count * d, c.hidden) @ v).reshape(-1, d))
        u = (rows(at.attn_v, c.kv_head_count * d, c.hidden) @ v).reshape(-1, d)
        keys = torch.cat([keys.double(), k[:, None]], dim=1)
        values = torch.cat([values.double(), u[:, None]], dim=1)
        score = torch.softmax(q.reshape(-1, share, d) @ keys.transpose(1, 2).contiguous(), dim=2)
        x = x + rows(at.attn_output, c.hidden, c.hidden) @ (score @ values).reshape(-1)
        v = norm(x, at.ffn_norm)
        v = _silu(rows(at.ffn_gate, c.ffn, c.hidden) @ v) * (rows(at.ffn_up, c.ffn, c.hidden) @ v)
        x = x + rows(at.ffn_down, c.hidden, c.ffn) @ v
    return rows(w.output, c.vocab, c.hidden) @ norm(x, w.output_norm)


def exact(case, seed):
    """What run() returns, in 64 bits (None for the drawn token, a whole number)."""
    path = case["path"]
    if path == "moe":
        return _exact_moe(case, seed)
    if path == "step":
        return _exact_step(case, seed)
    if path == "sample":
        return None
    w, x = _projection(case, seed)
    n, k = case["rows"], case["columns"]
    size = _size(case["type"], 1, k)
    y = torch.empty((case["tokens"], n), dtype=torch.float64, device="cuda")
    for r in range(0, n, 16384):
        m = min(16384, n - r)
        y[:, r:r + m] = x.double() @ _weights(w[r * size:(r + m) * size], case["type"], m, k).T
    return y
