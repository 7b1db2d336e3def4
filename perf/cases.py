"""Performance cases of the quantized Llama / Mixtral runner (`mistralrs_amd.llama.Llama`): prompts and decode steps.

Models (the configurations of `LlamaConfig` and of the benchmark): "8b" = Llama-3-8B, 32 layers; "moe" = four layers of Mixtral-8x7B's shape (8 experts, top-2), the
depth at which three of them fit next to each other.  Weights: "q4_k_m" = the Q4_K_M type map (Q4_K, with Q6_K in lm_head and in half of the value / down projections),
"q8_0" = Q8_0 everywhere.  Checkpoints are not available offline: the tensors are random valid GGUF blocks of trained-like scale (projections into the residual stream
are smaller by the square root of twice the full model's depth, as in trained models, so that rounding noise does not grow from layer to layer).

One pass is one scheduler step of a serving loop, entered with fresh token ids:
  * "decode": `batch` sequences at their positions -> the next tokens, logits and K / V rows (`set_state` + `replay` of the captured step; "eager": `set_state` +
    `forward_logits`, what a program that samples by itself calls);
  * "prefill": `tokens` prompt tokens behind `ctx` tokens that are in the pages already -> the last token's logits and the prompt's K / V rows.
"""
import math

import torch

from mistralrs_amd.gguf.qtensor import GgmlDType, QTensor
from mistralrs_amd.llama import Llama, LlamaConfig

DEPTH = 32  # layers of both full models
MOE_LAYERS = 4


def listed():
    return [
        # one user, chat-length context: the benchmark's decode workload
        dict(name="decode 8b b1 ctx 512", kind="decode", model="8b", quant="q4_k_m", batch=1, ctx=512, eager=False),
        # one user at the end of a long document
        dict(name="decode 8b b1 ctx 7001", kind="decode", model="8b", quant="q4_k_m", batch=1, ctx=7001, eager=False),
        # two users, contexts of unlike length
        dict(name="decode 8b b2 ctx 1500", kind="decode", model="8b", quant="q4_k_m", batch=2, ctx=1500, eager=False),
        # the largest batch of a step; the program samples by itself
        dict(name="decode 8b b8 ctx 1000", kind="decode", model="8b", quant="q4_k_m", batch=8, ctx=1000, eager=True),
        # in-situ quantized model: twice the weight bytes
        dict(name="decode 8b q8_0 b1 ctx 777", kind="decode", model="8b", quant="q8_0", batch=1, ctx=777, eager=False),
        # routed experts, one user and a few
        dict(name="decode moe b1 ctx 512", kind="decode", model="moe", quant="q4_k_m", batch=1, ctx=512, eager=False),
        dict(name="decode moe b5 ctx 300", kind="decode", model="moe", quant="q4_k_m", batch=5, ctx=300, eager=False),
        # a short chat turn behind an earlier conversation
        dict(name="prefill 8b 37 at 300", kind="prefill", model="8b", quant="q4_k_m", tokens=37, ctx=300),
        # the benchmark's prompt
        dict(name="prefill 8b 512", kind="prefill", model="8b", quant="q4_k_m", tokens=512, ctx=0),
        # a long document, ragged
        dict(name="prefill 8b 1999", kind="prefill", model="8b", quant="q4_k_m", tokens=1999, ctx=0),
        dict(name="prefill 8b q8_0 700", kind="prefill", model="8b", quant="q8_0", tokens=700, ctx=0),
        dict(name="prefill moe 512", kind="prefill", model="moe", quant="q4_k_m", tokens=512, ctx=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = "moe" if rng.random() < 0.3 else "8b"
    quant = "q8_0" if rng.random() < 0.25 else "q4_k_m"
    if rng.random() < 0.5:
        batch = rng.randint(1, 8)
        return dict(kind="decode", model=model, quant=quant, batch=batch, ctx=_log_int(rng, 16, 7000 if batch < 4 else 2000), eager=rng.random() < 0.3)
    tokens = _log_int(rng, 4, 1900)
    ctx = 0 if rng.random() < 0.6 else _log_int(rng, 16, 1900)
    return dict(kind="prefill", model=model, quant=quant, tokens=tokens, ctx=min(ctx, 2000 - tokens))


# ---------------------------------------------------------------------------------------------------------- sizes
def _config(case):
    batch = case.get("batch", 1)
    last = case["ctx"] + case.get("tokens", 1)  # positions in use, the new ones included
    kw = dict(max_batch=batch, max_context_len=(last + 63) // 64 * 64, max_position_embeddings=8192)
    if case["model"] == "8b":
        return LlamaConfig.llama3_8b(**kw)
    cfg = LlamaConfig.mixtral_8x7b(**kw)
    cfg.num_layers = MOE_LAYERS
    return cfg


def _tensors(cfg, quant):
    """(name, type, rows, columns, standard deviation) of every quantized tensor, in loading order; expert stacks have their experts' rows one after the other."""
    d, ff, L, E = cfg.hidden_size, cfg.intermediate_size, cfg.num_layers, cfg.num_experts
    nq, nkv = cfg.num_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim
    small = 0.02 / math.sqrt(2 * DEPTH)
    big = {"q4_k_m": "Q6K", "q8_0": "Q8_0"}[quant]
    base = {"q4_k_m": "Q4K", "q8_0": "Q8_0"}[quant]
    out = [("token_embd.weight", base, cfg.vocab_size, d, 1.0), ("output.weight", big, cfg.vocab_size, d, 0.02)]
    for i in range(L):
        more = big if i < L // 8 or i >= 7 * L // 8 or (i - L // 8) % 3 == 2 else base
        ex, n = ("_exps", E) if E else ("", 1)
        out += [(f"blk.{i}.attn_q.weight", base, nq, d, 0.02), (f"blk.{i}.attn_k.weight", base, nkv, d, 0.02), (f"blk.{i}.attn_v.weight", more, nkv, d, 0.02),
                (f"blk.{i}.attn_output.weight", base, d, nq, small), (f"blk.{i}.ffn_gate{ex}.weight", base, n * ff, d, 0.02),
                (f"blk.{i}.ffn_up{ex}.weight", base, n * ff, d, 0.02), (f"blk.{i}.ffn_down{ex}.weight", more, n * d, ff, small)]
    return out


def _contexts(case):
    """Positions of a decode step's new tokens: the first sequence is at `ctx`, the others are spread down to half of it."""
    b, c = case["batch"], case["ctx"]
    return [c - (c // 2) * s // max(1, b - 1) for s in range(b)]


# ---------------------------------------------------------------------------------------------------------- inputs, all from the seed
def _gen(seed, index, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed) * 100003 + index)


def _blocks(kind, rows, cols, std, seed, index):
    """Random GGUF blocks as bytes [blocks][bytes of a block]: random quants and sub-block scales, super-block scales such that the weights have about this deviation."""
    g = _gen(seed, index)
    size, per = {"Q4K": (144, 256), "Q6K": (210, 256), "Q8_0": (34, 32)}[kind]
    nb = rows * (cols // per)
    words = torch.randint(-2 ** 63, 2 ** 63 - 1, ((nb * size + 7) // 8,), dtype=torch.int64, device="cuda", generator=g)
    raw = words.view(torch.uint8)[: nb * size].view(nb, size)
    scale = 0.75 + 0.5 * torch.rand(nb, device="cuda", generator=g)
    put = lambda at, v: raw[:, at: at + 2].copy_((scale * v).to(torch.float16).view(torch.uint8).view(nb, 2))  # noqa: E731
    if kind == "Q4K":
        put(0, std / 170.0)
        put(2, std / 170.0 * 7.5)
    elif kind == "Q6K":
        put(208, std / (74.0 * 18.5))
    else:
        put(0, std / 74.0)
    return raw


def _norms(cfg, seed):
    g = _gen(seed, 1)
    return 1.0 + 0.01 * torch.randn(2 * cfg.num_layers + 1, cfg.hidden_size, device="cuda", generator=g)


def _router(cfg, layer, seed):
    return 0.05 * torch.randn(cfg.num_experts, cfg.hidden_size, device="cuda", generator=_gen(seed, 10 + layer))


def _past(cfg, layer, rows, seed):
    """K and V [rows][kv heads][head_dim] bf16 of tokens that were processed earlier."""
    g = _gen(seed, 1000 + layer)
    k, v = (1.28 * torch.randn(rows, cfg.num_kv_heads, cfg.head_dim, device="cuda", generator=g) for _ in range(2))
    return k.to(torch.bfloat16), v.to(torch.bfloat16)


def _token_ids(case, cfg, seed):
    n = case["batch"] if case["kind"] == "decode" else case["tokens"]
    return torch.randint(0, cfg.vocab_size, (n,), generator=_gen(seed, 2, "cpu")).tolist()


def _to_pages(cfg, blocks, k, v):
    """Token rows [blocks * block_size][kv heads][head_dim] in the layouts of the key and value pages."""
    bs, h, hd = cfg.block_size, cfg.num_kv_heads, cfg.head_dim
    kp = k.view(blocks, bs, h, hd // 8, 8).permute(0, 2, 3, 1, 4)
    return kp.contiguous(), v.view(blocks, bs, h, hd).permute(0, 2, 3, 1).contiguous()


def _seen_layers(cfg):
    """Layers whose pages a pass returns: the pages of the layers between are read by the later ones."""
    return sorted({0, cfg.num_layers // 2, cfg.num_layers - 1})


def prepare(case, seed):
    cfg = _config(case)
    dev = torch.device("cuda")
    m = Llama(cfg, dev, max_new_tokens=64)
    for i, (name, kind, rows, cols, std) in enumerate(_tensors(cfg, case["quant"])):
        m.set_tensor(name, QTensor(GgmlDType[kind], (rows, cols), _blocks(kind, rows, cols, std, seed, 5000 + i).reshape(-1)))
    norms = _norms(cfg, seed)
    for i in range(cfg.num_layers):
        m.set_tensor(f"blk.{i}.attn_norm.weight", norms[2 * i])
        m.set_tensor(f"blk.{i}.ffn_norm.weight", norms[2 * i + 1])
        if cfg.num_experts:
            m.set_tensor(f"blk.{i}.ffn_gate_inp.weight", _router(cfg, i, seed))
        kp, vp = _to_pages(cfg, m.num_blocks, *_past(cfg, i, m.num_blocks * cfg.block_size, seed))
        m.key_caches[i].copy_(kp)
        m.value_caches[i].copy_(vp)
    m.set_tensor("output_norm.weight", norms[-1])
    ids = _token_ids(case, cfg, seed)
    if case["kind"] == "decode" and not case["eager"]:
        m.set_state(ids, _contexts(case))
        m.capture_decode_graph(case["batch"])
    return dict(case=case, model=m, ids=ids)


def run(state):
    case, m, ids = state["case"], state["model"], state["ids"]
    out = {}
    if case["kind"] == "prefill":
        out["logits"] = m.prefill(ids, case["ctx"])
    else:
        m.set_state(ids, _contexts(case))
        if case["eager"]:
            out["logits"] = m.forward_logits(case["batch"])
        else:
            m.step_counter.zero_()
            m.replay()
            out["logits"] = m.logits
            out["next"] = m.input_ids
    for i in _seen_layers(m.cfg):
        out[f"k{i}"], out[f"v{i}"] = m.key_caches[i], m.value_caches[i]
    return out


# ---------------------------------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    cfg = _config(case)
    n = case["batch"] if case["kind"] == "decode" else case["tokens"]
    bits = {"Q4K": 144 / 256, "Q6K": 210 / 256, "Q8_0": 34 / 32}
    E, top = cfg.num_experts, cfg.num_experts_per_tok
    hit = 1.0 - (1.0 - top / E) ** n if E else 1.0  # share of the experts that some token takes
    nbytes = flops = 0.0
    for name, kind, rows, cols, _ in _tensors(cfg, case["quant"]):
        if name == "token_embd.weight":
            nbytes += n * cols * bits[kind]
            continue
        exps = "_exps" in name
        nbytes += rows * cols * bits[kind] * (hit if exps else 1.0)
        last_only = case["kind"] == "prefill" and name == "output.weight"
        flops += 2.0 * rows * cols * (1 if last_only else n) * (top / E if exps else 1.0)
    row = cfg.num_layers * cfg.num_kv_heads * cfg.head_dim * 2 * 2  # K and V bytes of a token
    q = cfg.num_layers * cfg.num_heads * cfg.head_dim
    if case["kind"] == "decode":
        seen = [p + 1 for p in _contexts(case)]
        nbytes += sum(seen) * row + n * cfg.vocab_size * 4
        flops += sum(4.0 * c * q for c in seen)
    else:
        nbytes += (case["ctx"] + n) * row + cfg.vocab_size * 4
        flops += 4.0 * q * (n * case["ctx"] + n * (n + 1) / 2)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # int8 activations: two summation orders of the same arithmetic agree to f32 rounding until one int8 quant of one layer falls to the other side of a rounding step.
    return {"rel": 0.03, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------------------------------------------------- the same in 64 bits
def _f16(raw, at):
    return raw[:, at: at + 2].contiguous().view(torch.float16).to(torch.float64)


def _weights(kind, raw, rows, cols):
    """GGUF blocks -> [rows][cols] float64 (the block formats' definitions)."""
    nb = raw.shape[0]
    if kind == "Q8_0":
        w = _f16(raw, 0) * raw[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif kind == "Q4K":
        s = raw[:, 4:16].to(torch.int16)
        lo, hi = s[:, 0:4], s[:, 4:8]
        sc = torch.cat([lo & 63, (s[:, 8:12] & 15) | ((lo >> 6) << 4)], 1)
        mn = torch.cat([hi & 63, (s[:, 8:12] >> 4) | ((hi >> 6) << 4)], 1)
        q = raw[:, 16:].reshape(nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(nb, 8, 32)
        a, b = _f16(raw, 0) * sc, _f16(raw, 2) * mn
        w = a.unsqueeze(2) * q - b.unsqueeze(2)
    else:  # Q6_K: halves of 128 values, each 4 quarters of 32
        ql, qh = raw[:, :128].reshape(nb, 2, 2, 32), raw[:, 128:192].reshape(nb, 2, 32)
        quarters = [(ql[:, :, k % 2] & 15 if k < 2 else ql[:, :, k % 2] >> 4) | (((qh >> (2 * k)) & 3) << 4) for k in range(4)]
        q = torch.stack(quarters, 2).reshape(nb, 16, 16).to(torch.int16) - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8)
        w = (_f16(raw, 208) * sc).unsqueeze(2) * q
    return w.reshape(rows, cols)


def _rope(cfg, x, pos):
    """Adjacent pairs of [tokens][heads][head_dim] rotated, with the long-context stretching of the low frequencies where the configuration has it."""
    hd = cfg.head_dim
    inv = 1.0 / cfg.rope_theta ** (torch.arange(0, hd, 2, dtype=torch.float64, device="cuda") / hd)
    s = cfg.rope_scaling
    if s is not None:
        wave, orig = 2 * math.pi / inv, s.original_max_position_embeddings
        t = ((orig / wave - s.low_freq_factor) / (s.high_freq_factor - s.low_freq_factor)).clamp(0, 1)
        inv = (1 - t) * inv / s.factor + t * inv
    a = pos.to(torch.float64)[:, None, None] * inv
    c, n = torch.cos(a), torch.sin(a)
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * n, x0 * n + x1 * c], -1).flatten(-2)


def _attend(cfg, q, k, v, first):
    """Query t of [tokens][heads][dim] sees keys 0 .. first + t of [rows][kv heads][dim]."""
    T, H, hd = q.shape
    G = H // cfg.num_kv_heads
    out = torch.empty_like(q)
    k, v = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    for t0 in range(0, T, 256):
        t1 = min(T, t0 + 256)
        rows = first + t1
        qs = q[t0:t1].view(t1 - t0, -1, G, hd).permute(1, 2, 0, 3).reshape(k.shape[0], -1, hd).contiguous()
        s = torch.matmul(qs, k[:, :, :rows].contiguous()).view(k.shape[0], G, t1 - t0, rows) / math.sqrt(hd)
        mask = torch.arange(rows, device="cuda")[None] > first + torch.arange(t0, t1, device="cuda")[:, None]
        p = torch.softmax(s.masked_fill(mask, -math.inf), -1).view(k.shape[0], -1, rows)
        out[t0:t1] = torch.matmul(p, v[:, :rows].contiguous()).view(-1, G, t1 - t0, hd).permute(2, 0, 1, 3).reshape(t1 - t0, H, hd)
    return out


def exact(case, seed):
    cfg = _config(case)
    hd, kvh, bs = cfg.head_dim, cfg.num_kv_heads, cfg.block_size
    per = cfg.max_blocks_per_seq
    specs = {name: (i, kind, rows, cols, std) for i, (name, kind, rows, cols, std) in enumerate(_tensors(cfg, case["quant"]))}

    def tensor(name):
        i, kind, rows, cols, std = specs[name]
        return kind, _blocks(kind, rows, cols, std, seed, 5000 + i), rows, cols

    def dense(name):
        return _weights(*tensor(name))

    def rms(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + cfg.rms_eps) * w

    norms = _norms(cfg, seed).to(torch.float64)
    ids = torch.tensor(_token_ids(case, cfg, seed), device="cuda")
    decode = case["kind"] == "decode"
    pos = torch.tensor(_contexts(case) if decode else range(case["ctx"], case["ctx"] + case["tokens"]), device="cuda")
    base = torch.arange(len(ids), device="cuda") * (per * bs) if decode else 0
    x = dense("token_embd.weight")[ids]
    out = {}
    for i in range(cfg.num_layers):
        p = f"blk.{i}."
        y = rms(x, norms[2 * i])
        q, k, v = (torch.matmul(y, dense(p + f"attn_{c}.weight").T).view(len(ids), -1, hd) for c in "qkv")
        q, k = _rope(cfg, q, pos), _rope(cfg, k, pos)
        K, V = (t.to(torch.float64) for t in _past(cfg, i, cfg.max_batch * per * bs, seed))
        K[base + pos], V[base + pos] = k, v
        if decode:
            a = torch.cat([_attend(cfg, q[s: s + 1], K[s * per * bs: s * per * bs + c + 1], V[s * per * bs: s * per * bs + c + 1], c) for s, c in enumerate(_contexts(case))])
        else:
            a = _attend(cfg, q, K, V, case["ctx"])
        if i in _seen_layers(cfg):
            out[f"k{i}"], out[f"v{i}"] = _to_pages(cfg, cfg.max_batch * per, K, V)
        x = x + torch.matmul(a.flatten(1), dense(p + "attn_output.weight").T)
        y = rms(x, norms[2 * i + 1])
        glu = lambda g, u: torch.nn.functional.silu(g) * u  # noqa: E731
        if not cfg.num_experts:
            f = glu(torch.matmul(y, dense(p + "ffn_gate.weight").T), torch.matmul(y, dense(p + "ffn_up.weight").T))
            x = x + torch.matmul(f, dense(p + "ffn_down.weight").T)
            continue
        share, who = torch.topk(torch.softmax(torch.matmul(y, _router(cfg, i, seed).to(torch.float64).T), -1), cfg.num_experts_per_tok, -1)
        share = share / share.sum(-1, keepdim=True)
        gate, up, down = (tensor(p + f"ffn_{c}_exps.weight") for c in ("gate", "up", "down"))
        for e in range(cfg.num_experts):
            at, slot = torch.nonzero(who == e, as_tuple=True)
            if len(at):
                g, u, dn = (_weights(kind, raw.view(cfg.num_experts, -1, raw.shape[1])[e], rows // cfg.num_experts, cols) for kind, raw, rows, cols in (gate, up, down))
                f = glu(torch.matmul(y[at], g.T), torch.matmul(y[at], u.T))
                x = x.index_add(0, at, share[at, slot, None] * torch.matmul(f, dn.T))
    logits = torch.matmul(rms(x if decode else x[-1:], norms[-1]), dense("output.weight").T)
    out["logits"] = logits if decode else logits[0]
    if decode and not case["eager"]:
        out["next"] = None
    return out
