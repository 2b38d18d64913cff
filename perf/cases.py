"""The work that a user of this library has it do, as cases whose time and outputs can be measured.

Kinds of case (the sizes are Qwen3's, those of the benchmark's linear layers and MoE stack, and odd ones between):
  host      Linear.forward on host arrays: the drop-in call of a program that keeps its activations on the CPU.
  linear    Linear.forward_device, input and output in device memory: m = 1 is the decode GEMV (W8A32), m > 1 the
            prefill GEMM (W8A8, the activation rows quantized inside the call).
  prefill   Qwen3ForCausalLM.forward of a prompt, whole or in chunks, on loaded Q8_0 weights: logits.
  generate  a whole chat turn: prompt, new tokens (greedy or sampled), then the logits that follow the last of them.
  moe       one decode step of a Qwen3-30B-A3B-style stack of layers for T sequences at their positions.

`exact` restates the numerics that the calls promise (include/lq8.h) in 64 bits with plain torch: Q8_0 blocks, RMSNorm's
bf16 roundings, the activation quantization of W8A8.  Everything between those roundings is float64.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-omni-inference-rs_amd"))
import lq8  # noqa: E402

SHAPES = {
    "0.6b": lq8.qwen3_0_6b,
    "1.7b": lq8.qwen3_1_7b,
    "4b": lq8.qwen3_4b,
}
LARGEST_FLOPS = 2.0 * 4096 * 19456 * 2560  # the largest listed linear


def listed():
    return [
        # a crate that calls Linear::forward with host vectors, token by token (the smallest call)
        {"name": "host_m1_q", "kind": "host", "m": 1, "n": 2048, "k": 1024},
        # one decode linear on device memory: the benchmark's single GEMV, and the lm_head of every token
        {"name": "m1_gate", "kind": "linear", "m": 1, "n": 3072, "k": 1024},
        {"name": "m1_lm_head", "kind": "linear", "m": 1, "n": 151936, "k": 1024},
        # a handful of sequences or a prompt's tail: rows, columns and block count off every tile
        {"name": "m37_ragged", "kind": "linear", "m": 37, "n": 5003, "k": 2080},
        # the benchmark's prefill GEMM (down), and a long prompt through the widest layer (Qwen3-4B gate|up)
        {"name": "m512_down", "kind": "linear", "m": 512, "n": 1024, "k": 3072},
        {"name": "m4096_gate_up", "kind": "linear", "m": 4096, "n": 19456, "k": 2560},
        # time to the first token of a short prompt, whole Qwen3-0.6B
        {"name": "prefill_0.6b_128", "kind": "prefill", "shape": "0.6b", "layers": 28, "vocab": 151936, "tokens": 128, "chunk": 128},
        # a long document through decoder layers of Qwen3-1.7B, in chunks as a server feeds it (the last one ragged)
        {"name": "prefill_1.7b_2999", "kind": "prefill", "shape": "1.7b", "layers": 4, "vocab": 4096, "tokens": 2999, "chunk": 1024},
        # a chat turn, greedy, Qwen3-0.6B: the benchmark's decode
        {"name": "greedy_0.6b", "kind": "generate", "shape": "0.6b", "prompt": 128, "new": 64, "sampled": False},
        # a sampled answer to a page of text, Qwen3-1.7B
        {"name": "sampled_1.7b", "kind": "generate", "shape": "1.7b", "prompt": 700, "new": 32, "sampled": True},
        # decode of a MoE stack: one sequence, and a full batch
        {"name": "moe_t1", "kind": "moe", "layers": 2, "t": 1, "pos": 128},
        {"name": "moe_t32", "kind": "moe", "layers": 2, "t": 32, "pos": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "linear", "linear", "linear", "prefill", "prefill", "generate", "generate", "moe", "moe"])
    if kind in ("host", "linear"):
        while True:
            k = 32 * _log(rng, 2, 304)
            n = _log(rng, 48, 20000) if kind == "linear" else _log(rng, 48, 12000)
            if kind == "linear" and rng.random() < 0.15:
                n = 151936
            m = 1 if rng.random() < 0.35 else _log(rng, 2, 4096 if kind == "linear" else 256)
            if 2.0 * m * n * k <= LARGEST_FLOPS and m * n <= 1 << 27 and n * k <= 151936 * 2560:
                return {"kind": kind, "m": m, "n": n, "k": k}
    if kind == "prefill":
        shape = rng.choice(sorted(SHAPES))
        tokens = _log(rng, 2, 3000)
        chunk = rng.choice([tokens, tokens, 256, 512, 1024])
        if tokens % chunk == 1:
            tokens += 1  # every chunk has at least two rows
        return {"kind": kind, "shape": shape, "layers": rng.randint(1, 4), "vocab": 4096, "tokens": tokens, "chunk": chunk}
    if kind == "generate":
        shape = rng.choice(["0.6b", "0.6b", "1.7b", "4b"])
        return {"kind": kind, "shape": shape, "prompt": _log(rng, 1, 1500), "new": _log(rng, 8, 64), "sampled": rng.random() < 0.4}
    return {"kind": "moe", "layers": rng.randint(1, 2), "t": _log(rng, 1, 32), "pos": _log(rng, 8, 600)}


# ---- inputs ------------------------------------------------------------------------------------------------------

def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + what * 7919 + 17) % (1 << 62))
    return g


def _normal(seed, what, shape, std=1.0):
    return torch.randn(shape, generator=_gen(seed, what), device="cuda", dtype=torch.float32) * std


def _quantize(x):
    """Q8_0 of float32 rows: (codes int8 [..., nb, 32], stored float16 scales [..., nb])."""
    b = x.reshape(*x.shape[:-1], x.shape[-1] // 32, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    v = b * inv
    q = torch.sign(v) * torch.floor(v.abs().double() + 0.5).float()
    return q.clamp(-128, 127).to(torch.int8), d.squeeze(-1).to(torch.float16)


def _weight(seed, what, n, k):
    return _quantize(_normal(seed, what, (n, k), 0.02))


def _blocks(w):
    """GGUF block_q8_0 bytes (scale, 32 codes) on the host."""
    q, d = w
    raw = torch.cat([d.reshape(-1, 1).view(torch.uint8).reshape(-1, 2), q.reshape(-1, 32).view(torch.uint8)], 1)
    return raw.reshape(-1).cpu().numpy()


def _values(w):
    """The 64-bit matrix that Q8_0 blocks stand for."""
    q, d = w
    return (q.double() * d.double().unsqueeze(-1)).reshape(q.shape[0], -1)


class _Memory:
    """A torch tensor where the library's device calls want a buffer."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


class _State:
    """Inputs and the handles that a program keeps; the handles are given back with it."""

    def __init__(self, case):
        self.case, self.handles = case, []

    def __del__(self):
        for h in self.handles:
            try:
                h.free()
            except Exception:
                pass


_context = []


def _ctx():
    if not _context:
        torch.zeros(1, device="cuda")
        _context.append(lq8.Context(0))
    return _context[0]


def _norms(seed, what, n):
    return 1.0 + _normal(seed, what, (n,), 0.1)


def _dense_config(case):
    cfg = SHAPES[case["shape"]](max_positions=(case["tokens"] + 63) // 64 * 64)
    cfg.num_hidden_layers, cfg.vocab_size = case["layers"], case["vocab"]
    return cfg


def _dense_tensors(case, seed):
    """Q8_0 matrices and float32 norms in the library's table order, on the GPU."""
    cfg = _dense_config(case)
    for i in range(cfg.tensor_count()):
        kind, shape = cfg.tensor_shape(i)
        yield _norms(seed, i, shape[0]) if kind == "f32" else _weight(seed, i, *shape)


def _ids(seed, n, vocab):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, n]).integers(0, vocab, n).astype(np.uint32)


def _moe_config(case):
    c = lq8.qwen3_30b_a3b_layers(num_layers=case["layers"], max_positions=(case["pos"] + 64) // 64 * 64, max_batch=case["t"])
    return c


def _moe_tensor(cfg, seed, i):
    kind, shape = cfg.tensor_shape(i)
    return _norms(seed, i, shape[0]) if kind == "f32" else _weight(seed, i, *shape)


def _moe_inputs(case, seed):
    """Hidden rows and router scores: [pos + 1][t][...], the last entry the measured step; and its positions."""
    cfg, P, T = _moe_config(case), case["pos"], case["t"]
    hid = _normal(seed, 900001, (P + 1, T, cfg.hidden_size))
    sc = _normal(seed, 900002, (P + 1, cfg.num_layers, T, cfg.num_experts))
    pos = torch.tensor([P - t % 5 for t in range(T)], dtype=torch.int32, device="cuda")
    return hid, sc, pos


def prepare(case, seed):
    ctx, s = _ctx(), _State(case)
    kind = case["kind"]
    if kind in ("host", "linear"):
        m, n, k = case["m"], case["n"], case["k"]
        w = lq8.Q8Weight.from_blocks(ctx, _blocks(_weight(seed, 1, n, k)), n, k)
        s.handles.append(w)
        s.linear = lq8.Linear.new(w)
        x = _normal(seed, 2, (m, k))
        if kind == "host":
            s.x = x.cpu().numpy()
        else:
            s.x = _Memory(x)
            s.y = _Memory(torch.empty((m, n), dtype=torch.float32, device="cuda"))
    elif kind == "prefill":
        host = [t.cpu().numpy() if isinstance(t, torch.Tensor) else _blocks(t) for t in _dense_tensors(case, seed)]
        s.model = lq8.Qwen3ForCausalLM.load(ctx, _dense_config(case), host)
        s.handles.append(s.model)
        s.ids = _ids(seed, case["tokens"], case["vocab"])
    elif kind == "generate":
        cfg = SHAPES[case["shape"]](max_positions=4096)
        s.model = lq8.Qwen3ForCausalLM.random(ctx, cfg, seed=int(seed) & 0xFFFFFFFF)
        s.handles.append(s.model)
        s.ids = _ids(seed, case["prompt"], cfg.vocab_size)
        s.config = lq8.GenerationConfig.new(case["new"], 0.8, 50, 0.95, 1.1)
        s.seed = int(seed) & 0xFFFF
    else:
        cfg = _moe_config(case)
        host = []
        for i in range(cfg.tensor_count()):
            t = _moe_tensor(cfg, seed, i)
            host.append(t.cpu().numpy() if isinstance(t, torch.Tensor) else _blocks(t))
        s.model = lq8.Qwen3MoeLayers.load(ctx, cfg, host)
        s.handles.append(s.model)
        hid, sc, pos = _moe_inputs(case, seed)
        T = case["t"]
        s.hidden = _Memory(hid[-1].clone())
        s.scores = _Memory(sc[-1].clone())
        s.pos = _Memory(pos)
        s.out = _Memory(torch.empty_like(s.hidden.t))
        # the tokens before this one: the sequences decoded up to their positions
        torch.cuda.synchronize()
        steps = torch.arange(case["pos"], dtype=torch.int32, device="cuda").reshape(-1, 1).repeat(1, T).contiguous()
        sc = sc.contiguous()
        for p in range(case["pos"]):
            s.model.forward_device(_Memory(hid[p]), _Memory(sc[p]), _Memory(steps[p]), T)
        ctx.synchronize()
    torch.cuda.synchronize()
    return s


def run(s):
    kind, case = s.case["kind"], s.case
    if kind == "host":
        return s.linear.forward(s.x)
    if kind == "linear":
        s.linear.forward_device(s.x, case["m"], s.y)
        return s.y.t
    if kind == "prefill":
        s.model.clear_kv_cache()
        return [s.model.forward(s.ids[at:at + case["chunk"]], at) for at in range(0, case["tokens"], case["chunk"])]
    if kind == "generate":
        if case["sampled"]:
            tokens, _ = s.model.generate(s.ids, s.config, seed=s.seed)
        else:
            tokens, _ = s.model.generate_greedy(s.ids, case["new"])
        logits = s.model.forward(tokens[-1:], len(s.ids) + len(tokens) - 1)
        return {"tokens": tokens.astype(np.int64), "logits": logits}
    # the step works in place: the incoming hidden rows (the last layer before, or the embedding) are put there first
    lib, h = lq8.lib(), s.out.t
    if lib.lq8_copy_device(s.model.ctx.handle, s.out.ptr, s.hidden.ptr, h.numel() * 4):
        raise RuntimeError("copy")
    s.model.forward_device(s.out, s.scores, s.pos, case["t"])
    return h


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _q8_bytes(n, k):
    return n * (k // 32) * 34


def work(case):
    kind = case["kind"]
    if kind in ("host", "linear"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _q8_bytes(n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "moe":
        c, T, P = _moe_config(case), case["t"], case["pos"]
        QD, KD, H, I = c.num_heads * 128, c.num_kv_heads * 128, c.hidden_size, c.expert_intermediate_size
        experts = c.num_experts * (1 - (1 - c.top_k / c.num_experts) ** T)  # expected distinct ones
        attn = _q8_bytes(QD + 2 * KD, H) + _q8_bytes(H, QD)
        one = 2 * _q8_bytes(I, H) + _q8_bytes(H, I)
        return {"bytes": c.num_layers * (attn + experts * one + T * P * 2 * KD * 4),
                "flops": c.num_layers * T * 2 * ((QD + 2 * KD) * H + H * QD + c.top_k * 3 * I * H + 2 * P * QD)}
    if kind == "prefill":
        c, n, new = _dense_config(case), case["tokens"], 0
    else:
        c, n, new = SHAPES[case["shape"]](), case["prompt"], case["new"]
    QD, KD, H, I, L = c.num_attention_heads * 128, c.num_key_value_heads * 128, c.hidden_size, c.intermediate_size, c.num_hidden_layers
    lin = (QD + 2 * KD) * H + H * QD + 3 * I * H
    weights = L * (lin // 32 * 34)
    head = _q8_bytes(c.vocab_size, H)
    passes = 1 + new  # the prompt, then one per generated token that is forwarded
    cached = n + (n + new / 2) * new  # positions whose keys and values are read
    return {"bytes": passes * (weights + head) + L * cached * 2 * KD * 4,
            "flops": 2 * (n + new) * L * lin + 2 * passes * c.vocab_size * H + 4 * L * QD * (n * (n + 1) / 2 + new * (n + new / 2))}


def tolerance(case):
    # About four times the error seen against 64 bits.  The GEMV adds float32 products (1e-7).  In W8A8 the last bit of
    # an activation can move it to the next code, one value in ten millions (6e-6 at m = 4096).  In whole layers a
    # last-bit difference also meets bf16 roundings, and travels (2e-3 after two MoE layers, 1e-2 and more in prefill).
    kind = case["kind"]
    if kind in ("host", "linear"):
        return {"rel": 5e-7, "max": 1e-5} if case["m"] == 1 else {"rel": 2.5e-5, "max": 1e-2}
    if kind == "moe":
        return {"rel": 8e-3, "max": 0.2}
    return {"rel": 3e-2, "max": 0.5, "differ": 0.01}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------

def _bf16(x):
    return x.float().to(torch.bfloat16).double()


def _act(x):
    """Activation rows as W8A8 sees them."""
    return _values(_quantize(x.float().reshape(-1, x.shape[-1]))).reshape(x.shape)


def _rms(x, w, eps):
    v = _bf16(x)
    return _bf16(v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps) * _bf16(w))


def _rope(x, pos, theta):
    """x [..., tokens, heads, 128] at positions pos [..., tokens]."""
    i = torch.arange(32, device=x.device, dtype=torch.float64)
    f = pos.double().unsqueeze(-1) * (1.0 / theta ** (2 * i / 64))
    c = torch.cos(f).float().double().repeat_interleave(2, -1).unsqueeze(-2)
    s = torch.sin(f).float().double().repeat_interleave(2, -1).unsqueeze(-2)
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, allowed):
    """q [T, n, H, 128], k and v [T, m, G, 128], allowed [T, n, m] -> [T, n, H * 128], a head at a time."""
    T, n, H, _ = q.shape
    out = torch.empty((T, n, H, 128), dtype=torch.float64, device=q.device)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(128.0)))
    for h in range(H):
        g = h // (H // k.shape[2])
        kt = k[:, :, g].transpose(1, 2).contiguous()
        s = torch.bmm(q[:, :, h].contiguous(), kt) * scale
        s.masked_fill_(~allowed, -math.inf)
        out[:, :, h] = torch.bmm(torch.softmax(s, -1), v[:, :, g].contiguous())
    return out.reshape(T, n, H * 128)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _exact_prefill(case, seed):
    c = _dense_config(case)
    ts = list(_dense_tensors(case, seed))
    H, nq, nk, n = c.hidden_size, c.num_attention_heads, c.num_key_value_heads, case["tokens"]
    ids = torch.from_numpy(_ids(seed, n, case["vocab"]).astype(np.int64)).cuda()
    table = ts[0]
    h = _values((table[0][ids], table[1][ids])).reshape(1, n, H)
    pos = torch.arange(n, device="cuda").reshape(1, n)
    causal = pos.unsqueeze(-1) >= pos.unsqueeze(-2)
    eps = c.rms_norm_eps
    for l in range(c.num_hidden_layers):
        n_in, n_post, qn, kn, wq, wk, wv, wo, wg, wu, wd = ts[2 + 11 * l:13 + 11 * l]
        x = _act(_rms(h, n_in, eps))
        q = _rope(_rms((x @ _values(wq).T).reshape(1, n, nq, 128), qn, eps), pos, c.rope_theta)
        k = _rope(_rms((x @ _values(wk).T).reshape(1, n, nk, 128), kn, eps), pos, c.rope_theta)
        v = (x @ _values(wv).T).reshape(1, n, nk, 128)
        h = h + _act(_attend(q, k, v, causal)) @ _values(wo).T
        x = _act(_rms(h, n_post, eps))
        h = h + _act(_silu(x @ _values(wg).T) * (x @ _values(wu).T)) @ _values(wd).T
    ends = [min(a + case["chunk"], n) - 1 for a in range(0, n, case["chunk"])]
    last = _rms(h[0, ends], ts[1], eps)
    y = torch.cat([last @ _values((q, d)).T for q, d in zip(table[0].split(16384), table[1].split(16384))], 1)
    return [r.cpu().numpy() for r in y]


def _exact_moe(case, seed):
    c, T, P = _moe_config(case), case["t"], case["pos"]
    hid, sc, pos = _moe_inputs(case, seed)
    H, nq, nk, E, K, eps = c.hidden_size, c.num_heads, c.num_kv_heads, c.num_experts, c.top_k, c.rms_norm_eps
    h = hid.double().transpose(0, 1).contiguous()  # [T, P + 1, H]: the history, then the step
    at = torch.arange(P + 1, device="cuda").reshape(1, -1).repeat(T, 1)
    at[:, -1] = pos.long()
    own = torch.arange(P + 1, device="cuda")
    # the history is causal; the step sees the history before its position, and itself
    allowed = (own.reshape(1, 1, -1) <= own.reshape(1, -1, 1)).repeat(T, 1, 1)
    allowed[:, -1, :] = own.reshape(1, -1) < pos.reshape(-1, 1)
    allowed[:, -1, -1] = True
    act = _act if T > 1 else (lambda x: x)
    for l in range(c.num_layers):
        base = l * c.per_layer()
        n_in, n_post, qn, kn, wq, wk, wv, wo = (_moe_tensor(c, seed, base + i) for i in range(8))
        x = act(_rms(h, n_in, eps))
        q = _rope(_rms((x @ _values(wq).T).reshape(T, P + 1, nq, 128), qn, eps), at, c.rope_theta)
        k = _rope(_rms((x @ _values(wk).T).reshape(T, P + 1, nk, 128), kn, eps), at, c.rope_theta)
        v = (x @ _values(wv).T).reshape(T, P + 1, nk, 128)
        h = h + act(_attend(q, k, v, allowed)) @ _values(wo).T
        x = _rms(h, n_post, eps).reshape(-1, H)
        p = torch.softmax(sc[:, l].double().transpose(0, 1).reshape(-1, E), -1)
        top, ids = torch.topk(p, K, -1)
        top = top / top.sum(-1, keepdim=True)
        out = torch.zeros_like(x)
        for e in range(E):
            row, rank = (ids == e).nonzero(as_tuple=True)
            if not len(row):
                continue
            g, u, d = (_values(_moe_tensor(c, seed, base + 8 + j * E + e)) for j in range(3))
            xe = x[row]
            y = (_silu(xe @ g.T) * (xe @ u.T)) @ d.T
            out.index_add_(0, row, y * top[row, rank].unsqueeze(-1))
        h = h + out.reshape(h.shape)
    return h[:, -1].contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "linear"):
        x = _normal(seed, 2, (case["m"], case["k"]))
        x = x.double() if case["m"] == 1 else _act(x)
        q, d = _weight(seed, 1, case["n"], case["k"])
        y = torch.cat([x @ _values((a, b)).T for a, b in zip(q.split(16384), d.split(16384))], 1)
        return y.cpu().numpy() if kind == "host" else y
    if kind == "prefill":
        return _exact_prefill(case, seed)
    if kind == "moe":
        return _exact_moe(case, seed)
    return None  # a token depends on all before it: the chain in 64 bits takes minutes
