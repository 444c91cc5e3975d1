"""What is timed: the framework's public entry points over the range that a chat program uses.

Two kinds of case:

matmul   y[n] = W x[n] on caller-owned device buffers (ops.matmul_ptr, chatnet_matmul): the projections of a
         model that a program drives itself, W in one of the weight types that checkpoints come in, 1 to 512
         columns (a decode step, a few sequences or draft tokens at once, a prompt).
model    HipLlamaModel on a checkpoint of one of the repository's shapes, cut to some layers where the
         weights would take long to make: `n` tokens forwarded at position `pos` (a prompt, the next turn of
         a chat, one token of a host-driven loop) and then `gen` tokens decoded greedily on the device.

Weights are drawn as the codes and scales that quantizing N(0, 0.02) leaves (bell-shaped codes, block scales
that vary a little), in the block layouts the library reads; activations are N(0, 1) with a few channels eight
times larger, as the inputs of a model's projections are.
"""
import math

import numpy as np
import torch

from chatnet_amd import LLAMA2_7B, QWEN2_0_5B, TINYLLAMA_1B, HipLlamaModel, _native, ops, synth

SIGMA = 0.02
TYPES = {
    "f16": _native.GGML_F16,
    "q4_0": _native.GGML_Q4_0,
    "q5_0": _native.GGML_Q5_0,
    "q8_0": _native.GGML_Q8_0,
    "q3_k": _native.GGML_Q3_K,
    "q4_k": _native.GGML_Q4_K,
    "q5_k": _native.GGML_Q5_K,
    "q6_k": _native.GGML_Q6_K,
    "iq4_xs": _native.GGML_IQ4_XS,
}
# attention, ffn gate/up, ffn down, LM head
MIXES = {
    "q4_0": ("q4_0", "q4_0", "q4_0", "q4_0"),
    "q5_0": ("q5_0", "q5_0", "q5_0", "q5_0"),
    "q8_0": ("q8_0", "q8_0", "q8_0", "q8_0"),
    "f16": ("f16", "f16", "f16", "f16"),
    "q4_k_m": ("q4_k", "q4_k", "q6_k", "q6_k"),
    "q5_k_m": ("q5_k", "q5_k", "q6_k", "q6_k"),
    "iq4_xs": ("iq4_xs", "iq4_xs", "iq4_xs", "q6_k"),
}
SHAPES = {"tinyllama": TINYLLAMA_1B, "llama2_7b": LLAMA2_7B, "qwen2_0_5b": QWEN2_0_5B}


def _matmul(name, type, M, K, N):
    return {"name": name, "kind": "matmul", "type": type, "M": M, "K": K, "N": N}


def _model(name, shape, layers, mix, pos, n, gen, kv="f32"):
    return {"name": name, "kind": "model", "shape": shape, "layers": layers, "mix": mix, "pos": pos, "n": n,
            "gen": gen, "kv": kv}


def listed():
    return [
        # one decode projection of a 1.1B model: launch latency and little else
        _matmul("q4_0 2048x2048 x1", "q4_0", 2048, 2048, 1),
        # the LM head of a Q4_K_M 7B model, the widest product of a decode step
        _matmul("q6_k 32000x4096 x1", "q6_k", 32000, 4096, 1),
        # a 7B down projection in a type that older checkpoints keep
        _matmul("q5_0 4096x11008 x1", "q5_0", 4096, 11008, 1),
        # a small model's gate for a few sequences at once
        _matmul("q8_0 4864x896 x5", "q8_0", 4864, 896, 5),
        # an unquantized projection for a batch of sequences
        _matmul("f16 4096x4096 x24", "f16", 4096, 4096, 24),
        # an attention projection over a ragged prompt
        _matmul("iq4_xs 4096x4096 x77", "iq4_xs", 4096, 4096, 77),
        # a 7B gate over a prompt of the span size
        _matmul("q4_k 11008x4096 x512", "q4_k", 11008, 4096, 512),
        # a whole 1.1B model reading a 512-token prompt
        _model("tinyllama q4_0 prompt 512", "tinyllama", 22, "q4_0", 0, 512, 0),
        # layers of a 7B Q4_K_M model reading an odd-sized prompt
        _model("7b q4_k_m prompt 333", "llama2_7b", 2, "q4_k_m", 0, 333, 0),
        # the next turn of a chat: a handful of tokens after a context
        _model("qwen2 q8_0 turn 6 at 700", "qwen2_0_5b", 6, "q8_0", 700, 6, 0),
        # layers of a 7B model decoding on the device
        _model("7b q4_0 decode 16 at 128", "llama2_7b", 4, "q4_0", 128, 1, 16),
        # one token of a host-driven loop deep in a context, 16-bit cache
        _model("7b q5_k_m token at 1900", "llama2_7b", 2, "q5_k_m", 1900, 1, 0, "f16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.6:
        type = rng.choice(sorted(TYPES))
        N = _log_int(rng, 1, 512)
        K = 256 * _log_int(rng, 1, 56)
        if type in ("q4_0", "q5_0", "q8_0", "f16") and rng.random() < 0.5:
            K += 64 * rng.randrange(1, 4)
        M = _log_int(rng, 64, min(32000, 131072000 // K))
        return {"kind": "matmul", "type": type, "M": M, "K": K, "N": N}
    shape = rng.choice(sorted(SHAPES))
    mixes = ["f16", "q4_0", "q5_0", "q8_0"] if shape == "qwen2_0_5b" else sorted(MIXES)
    c = {"kind": "model", "shape": shape, "layers": rng.randint(1, 4), "mix": rng.choice(mixes)}
    if rng.random() < 0.5:  # a prompt or a turn
        c["n"], c["gen"] = _log_int(rng, 2, 512), 0
        c["pos"] = 0 if rng.random() < 0.5 else _log_int(rng, 16, 1400)
    else:  # a token, or a decode on the device
        c["n"], c["gen"] = 1, rng.choice([0, _log_int(rng, 2, 24)])
        c["pos"] = _log_int(rng, 4, 2000)
    c["kv"] = rng.choice(["f32", "f32", "f16"])
    return c


# ---- weights ------------------------------------------------------------------------------------------------


def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + stream * 7919) & 0x7FFFFFFF)


def _codes(g, nb, n, spread, center, hi):
    z = torch.randn(nb, n, generator=g, device="cuda")
    return (z * spread + center).round_().clamp_(0, hi).to(torch.uint8)


def _halves(g, nb, value):
    """[nb] fp16 block scales around `value`, and their bytes [nb, 2]."""
    d = (value * (0.85 + 0.3 * torch.rand(nb, 1, generator=g, device="cuda"))).half()
    return d, d.view(torch.uint8).view(nb, 2)


def _nibbles(q):
    """Codes [.., 32 per group] as bytes [.., 16 per group]: element j low, 16 + j high."""
    q = q.view(q.shape[0], -1, 2, 16)
    return (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(q.shape[0], -1)


def _bits(b):
    """0/1 codes [nb, n] as bytes [nb, n / 8], bit e % 8 of byte e / 8."""
    w = (1 << torch.arange(8, device=b.device)).to(torch.uint8)
    return (b.view(b.shape[0], -1, 8) * w).sum(2, dtype=torch.int32).to(torch.uint8)


def _k_scales(sc, mn):
    """6-bit scales and minima [nb, 8] as Q4_K / Q5_K's 12 bytes."""
    lo = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    mid = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
    hi = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return torch.cat([lo, mid, hi], 1)


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _weights(type, rows, cols, g, exact=False):
    """A rows x cols matrix in `type`: its bytes on the GPU, or with `exact` its float64 values."""
    n = 256 if "_k" in type or type == "iq4_xs" else 32
    nb = rows * cols // n

    def values(q, scale, offset=None):  # q [nb, n], scale / offset per equal groups of a block
        v = q.double().view(nb, scale.shape[1], -1) * scale.double().unsqueeze(2)
        if offset is not None:
            v -= offset.double().unsqueeze(2)
        return v.view(rows, cols)

    if type == "f16":
        w = (torch.randn(rows, cols, generator=g, device="cuda") * SIGMA).half()
        return w.double() if exact else w.view(torch.uint8)
    if type == "q4_0":
        d, db = _halves(g, nb, SIGMA / 3.3)
        q = _codes(g, nb, 32, 3.3, 8, 15)
        return values(q.short() - 8, d) if exact else torch.cat([db, _nibbles(q)], 1)
    if type == "q5_0":
        d, db = _halves(g, nb, SIGMA / 6.6)
        q = _codes(g, nb, 32, 6.6, 16, 31)
        return values(q.short() - 16, d) if exact else torch.cat([db, _bits(q >> 4), _nibbles(q & 15)], 1)
    if type == "q8_0":
        d, db = _halves(g, nb, SIGMA / 50)
        q = _codes(g, nb, 32, 50, 128, 255)
        return values(q.short() - 128, d) if exact else torch.cat([db, q ^ 128], 1)
    if type == "q3_k":
        d, db = _halves(g, nb, SIGMA / 1.7 / 24)
        q = _codes(g, nb, 256, 1.7, 4, 7)
        s = _codes(g, nb, 16, 4, 56, 63)  # 6-bit scale + 32
        if exact:
            return values(q.short() - 4, d.double() * (s.double() - 32))
        lo = (s[:, :8] & 15) | ((s[:, 8:] & 15) << 4)
        h = (s >> 4).view(nb, 4, 4)  # [i >> 2][i & 3]
        hi = h[:, 0] | (h[:, 1] << 2) | (h[:, 2] << 4) | (h[:, 3] << 6)
        q2 = (q & 3).view(nb, 64, 4)
        qs = q2[:, :, 0] | (q2[:, :, 1] << 2) | (q2[:, :, 2] << 4) | (q2[:, :, 3] << 6)
        return torch.cat([_bits(q >> 2), qs, lo, hi, db], 1)
    if type in ("q4_k", "q5_k"):
        spread, center, hi = (3.3, 7.5, 15) if type == "q4_k" else (6.6, 15.5, 31)
        d, db = _halves(g, nb, SIGMA / spread / 48)
        m, mb = _halves(g, nb, SIGMA / spread / 48 * center)
        q = _codes(g, nb, 256, spread, center, hi)
        sc, mn = _codes(g, nb, 8, 6, 48, 63), _codes(g, nb, 8, 6, 48, 63)
        if exact:
            return values(q, d.double() * sc.double(), m.double() * mn.double())
        qh = [_bits(q >> 4)] if type == "q5_k" else []
        return torch.cat([db, mb, _k_scales(sc, mn)] + qh + [_nibbles(q & 15)], 1)
    if type == "q6_k":
        d, db = _halves(g, nb, SIGMA / 12 / 90)
        q = _codes(g, nb, 256, 12, 32, 63)
        s = _codes(g, nb, 16, 14, 90, 127) * (1 - 2 * (_codes(g, nb, 16, 1, 0.5, 1).char()))
        if exact:
            return values(q.short() - 32, d.double() * s.double())
        h = q.view(nb, 2, 4, 32)  # half, quarter, element
        ql = torch.cat([(h[:, :, 0] & 15) | ((h[:, :, 2] & 15) << 4), (h[:, :, 1] & 15) | ((h[:, :, 3] & 15) << 4)], 2)
        p = h >> 4
        qh = p[:, :, 0] | (p[:, :, 1] << 2) | (p[:, :, 2] << 4) | (p[:, :, 3] << 6)
        return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), s.to(torch.int8).view(torch.uint8), db], 1)
    if type == "iq4_xs":
        d, db = _halves(g, nb, SIGMA / 40 / 100)
        q = _codes(g, nb, 256, 2.6, 7.6, 15)
        head = torch.randint(0, 256, (nb, 6), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
        raw = torch.cat([db, head, _nibbles(q)], 1)
        if not exact:
            return raw
        # the reference takes the low scale bits of sub-block s from byte 4 + s, quants included
        sh = raw[:, 2].int() | (raw[:, 3].int() << 8)
        hi = torch.stack([(sh >> (2 * s)) & 3 for s in range(8)], 1)
        s = ((raw[:, 4:12].int() & 63) | (hi << 6)) - 32
        t = torch.tensor(_IQ4, device="cuda", dtype=torch.int16)
        return values(t[q.long()], d.double() * s.double())
    raise ValueError(type)


def _nbytes(type, n):
    return _native.tensor_nbytes(TYPES[type], n)


# ---- matmul ---------------------------------------------------------------------------------------------------


def _x(seed, N, K):
    g = _gen(seed, 1)
    x = torch.randn(N, K, generator=g, device="cuda")
    return x * torch.where(torch.rand(K, generator=g, device="cuda") < 0.004, 8.0, 1.0)


# ---- model ----------------------------------------------------------------------------------------------------


def _config(case):
    kv = _native.KV_F16 if case["kv"] == "f16" else _native.KV_F32
    return SHAPES[case["shape"]].replace(n_layers=case["layers"], kv_dtype=kv)


def _tensors(case):
    """(GGUF name, type, rows, columns) of every matrix, in a fixed order."""
    c = _config(case)
    attn, gate_up, down, out = MIXES[case["mix"]]
    emb = "f16" if case["mix"] == "f16" else "q8_0"
    t = [("token_embd.weight", emb, c.vocab_size, c.dim)]
    if c.arch != _native.ARCH_QWEN2:  # Qwen2's head is its embedding
        t.append(("output.weight", out, c.vocab_size, c.dim))
    for i in range(c.n_layers):
        p = "blk.%d." % i
        t += [(p + "attn_q.weight", attn, c.dim, c.dim), (p + "attn_k.weight", attn, c.kv_dim, c.dim),
              (p + "attn_v.weight", attn, c.kv_dim, c.dim), (p + "attn_output.weight", attn, c.dim, c.dim),
              (p + "ffn_gate.weight", gate_up, c.hidden_dim, c.dim), (p + "ffn_up.weight", gate_up, c.hidden_dim, c.dim),
              (p + "ffn_down.weight", down, c.dim, c.hidden_dim)]
    return t


def _vectors(case, seed):
    """Norm weights and Qwen2's biases."""
    c = _config(case)
    rng = np.random.default_rng([int(seed), 77])
    v = {"output_norm.weight": 1 + 0.1 * rng.standard_normal(c.dim)}
    for i in range(c.n_layers):
        p = "blk.%d." % i
        for name in ("attn_norm.weight", "ffn_norm.weight"):
            v[p + name] = 1 + 0.1 * rng.standard_normal(c.dim)
        if c.arch == _native.ARCH_QWEN2:
            for name, n in (("attn_q.bias", c.dim), ("attn_k.bias", c.kv_dim), ("attn_v.bias", c.kv_dim)):
                v[p + name] = 0.25 * rng.standard_normal(n)
    return {k: a.astype(np.float32) for k, a in v.items()}


def _tokens(case, seed):
    n = case["pos"] + case["n"]
    return np.random.default_rng([int(seed), 3]).integers(0, _config(case).vocab_size, n).astype(np.int32)


def prepare(case, seed):
    if case["kind"] == "matmul":
        M, K, N = case["M"], case["K"], case["N"]
        w = _weights(case["type"], M, K, _gen(seed, 0)).reshape(-1)
        return {"case": case, "w": w, "x": _x(seed, N, K), "y": torch.empty(N, M, device="cuda")}
    cfg = _config(case)
    weights = {}
    for i, (name, type, rows, cols) in enumerate(_tensors(case)):
        raw = _weights(type, rows, cols, _gen(seed, 10 + i)).cpu().numpy()
        weights[name] = synth.SynthTensor(TYPES[type], (cols, rows), raw.reshape(-1))
    for name, v in _vectors(case, seed).items():
        weights[name] = synth.SynthTensor(_native.GGML_F32, (v.size,), v.view(np.uint8))
    torch.cuda.synchronize()
    model = HipLlamaModel(cfg, weights)
    tokens = _tokens(case, seed)
    logits = np.empty(cfg.vocab_size, dtype=np.float32)
    if case["pos"]:
        model.forward(tokens[: case["pos"]], 0, logits)
    return {"case": case, "model": model, "tokens": tokens[case["pos"]:], "logits": logits}


def run(state):
    case = state["case"]
    if case["kind"] == "matmul":
        ops.matmul_ptr(TYPES[case["type"]], state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(),
                       case["M"], case["K"], case["N"], torch.cuda.current_stream().cuda_stream)
        return state["y"]
    model = state["model"]
    logits = model.forward(state["tokens"], case["pos"], state["logits"])
    if not case["gen"]:
        return logits
    tokens = model.decode_greedy(case["gen"])
    return model.get_logits(), tokens


def work(case):
    if case["kind"] == "matmul":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": _nbytes(case["type"], M * K) + 4 * K * N + 4 * M * N, "flops": 2 * M * K * N}
    c = _config(case)
    layers = sum(_nbytes(t, r * k) for name, t, r, k in _tensors(case) if name.startswith("blk."))
    per_token = sum(r * k for name, _, r, k in _tensors(case) if name.startswith("blk."))
    head_type = MIXES[case["mix"]][3] if c.arch != _native.ARCH_QWEN2 else _tensors(case)[0][1]
    head = _nbytes(head_type, c.vocab_size * c.dim)
    steps = 1 + case["gen"]  # passes over the weights: the span, then every decoded token
    kv_row = 2 * c.n_layers * c.kv_dim * (2 if case["kv"] == "f16" else 4)
    last = case["pos"] + case["n"]
    kv = kv_row * sum(last + i for i in range(steps))
    seen = sum(range(case["pos"] + 1, last + 1)) + sum(last + 1 + i for i in range(case["gen"]))
    flops = 2 * per_token * (case["n"] + case["gen"]) + 4 * c.n_layers * c.dim * seen
    flops += 2 * c.vocab_size * c.dim * steps
    return {"bytes": steps * (layers + head + 4 * c.vocab_size) + kv, "flops": flops}


def tolerance(case):
    # four times the error against 64 bits that was measured, rounded
    if case["kind"] == "matmul":
        if case["type"] == "f16":
            return {"rel": 1e-6}  # 32-bit products and sums: 1e-7
        if case["N"] >= 8:
            return {"rel": 1.2e-3}  # x and W meet in fp16: 2.9e-4
        # 32-bit for the types without an integer dot (2.5e-7), else x to 19 bits of its block (4.5e-6)
        return {"rel": 1e-6 if case["type"] in ("q5_0", "iq4_xs") else 2e-5}
    # x to 19 bits (one token) or 22 (a span) in every projection: 8e-6 to 2.3e-5; an fp16 cache: 9e-4
    return {"rel": 2e-3 if case["kv"] == "f16" else 1e-4}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------


def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * w


def _rope(v, pos, c):
    """Rotates [n, heads * head_dim] rows at positions `pos`: adjacent pairs, or split halves for Qwen2."""
    hd = c.head_dim
    v = v.view(v.shape[0], -1, hd)
    theta = pos.double()[:, None] * c.rope_freq_base ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    cs, sn = torch.cos(theta)[:, None], torch.sin(theta)[:, None]
    if c.arch == _native.ARCH_QWEN2:
        a, b = v[..., : hd // 2], v[..., hd // 2:]
        out = torch.cat([a * cs - b * sn, b * cs + a * sn], 2)
    else:
        a, b = v[..., 0::2], v[..., 1::2]
        out = torch.stack([a * cs - b * sn, a * sn + b * cs], 3)
    return out.reshape(v.shape[0], -1)


class _Exact:
    def __init__(self, case, seed):
        self.c = _config(case)
        names = _tensors(case)
        self.w = {name: _weights(t, r, k, _gen(seed, 10 + i), exact=True) for i, (name, t, r, k) in enumerate(names)}
        self.v = {k: torch.from_numpy(a).cuda().double() for k, a in _vectors(case, seed).items()}
        self.cache = [[] for _ in range(self.c.n_layers)]

    def forward(self, tokens, position):
        c = self.c
        n = len(tokens)
        pos = torch.arange(position, position + n, device="cuda")
        x = self.w["token_embd.weight"][torch.as_tensor(np.asarray(tokens), device="cuda").long()]
        for i in range(c.n_layers):
            w = {k: self.w.get("blk.%d.%s.weight" % (i, k)) for k in
                 ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")}
            b = {k: self.v.get("blk.%d.%s.bias" % (i, k), 0.0) for k in ("attn_q", "attn_k", "attn_v")}
            h = _norm(x, self.v["blk.%d.attn_norm.weight" % i], c.rms_norm_eps)
            q, k, v = (h @ w[m].T + b[m] for m in ("attn_q", "attn_k", "attn_v"))
            self.cache[i].append((_rope(k, pos, c), v))
            keys = torch.cat([p for p, _ in self.cache[i]]).view(-1, c.n_kv_heads, c.head_dim)
            vals = torch.cat([p for _, p in self.cache[i]]).view(-1, c.n_kv_heads, c.head_dim)
            q = _rope(q, pos, c).view(n, c.n_heads, c.head_dim)
            hidden = torch.arange(keys.shape[0], device="cuda")[None] > pos[:, None]
            att = []
            for head in range(c.n_heads):
                s = q[:, head] @ keys[:, head // c.kv_mul].T / math.sqrt(c.head_dim)
                att.append(torch.softmax(s.masked_fill(hidden, -math.inf), 1) @ vals[:, head // c.kv_mul])
            x = x + torch.cat(att, 1) @ w["attn_output"].T
            h = _norm(x, self.v["blk.%d.ffn_norm.weight" % i], c.rms_norm_eps)
            g = h @ w["ffn_gate"].T
            x = x + (g * torch.sigmoid(g) * (h @ w["ffn_up"].T)) @ w["ffn_down"].T
        head = self.w.get("output.weight", self.w["token_embd.weight"])
        return (_norm(x[-1:], self.v["output_norm.weight"], c.rms_norm_eps) @ head.T)[0]


def exact(case, seed):
    if case["kind"] == "matmul":
        w = _weights(case["type"], case["M"], case["K"], _gen(seed, 0), exact=True)
        return _x(seed, case["N"], case["K"]).double() @ w.T
    m = _Exact(case, seed)
    tokens = _tokens(case, seed)
    logits = m.forward(tokens, 0)
    if not case["gen"]:
        return logits.cpu().numpy()
    for i in range(case["gen"]):
        logits = m.forward([int(torch.argmax(logits))], len(tokens) + i)
    return logits.cpu().numpy(), None
