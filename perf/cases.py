"""The work that a user of this framework has it do, as cases that can be timed.

A case is one call (or two decode steps) of a model whose layers have the real
sizes of a preset and whose number is cut, so that a state is made in a second:
prompts go through ``RingExecutor.prefill_slots`` (serving) or the model's own
``prefill_window`` (equal prompts in one batch), decode steps through
``RingExecutor.slot_step_compute``, which replays a captured step.

Weights are random but the same through every load: what is quantized consists
of whole numbers times powers of two, which the loader's quantization gives
back exactly. Each projection has the scale of a trained one relative to the
residual stream (a layer adds a part of the residual's size to it), scores
spread over a few units, so that attention has favourites.
"""
import math

import torch

from dnet_amd.models import ModelConfig, PRESETS, QuantConfig
from dnet_amd.parallel.ring import RingExecutor

STEPS = 2       # decode steps of one pass


# ---------------------------------------------------------------- the cases

def _decode(name, model, layers, weights, batch, ctx_lo, ctx_hi, capacity,
            kv_bits=16):
    return {"name": name, "kind": "decode", "model": model, "layers": layers,
            "weights": weights, "batch": batch, "ctx_lo": ctx_lo,
            "ctx_hi": ctx_hi, "capacity": capacity, "kv_bits": kv_bits}


def _prefill(name, model, layers, weights, batch, tokens, start=0,
             ragged=False):
    return {"name": name, "kind": "prefill", "model": model, "layers": layers,
            "weights": weights, "batch": batch, "tokens": tokens,
            "start": start, "ragged": ragged}


def listed():
    return [
        # the smallest model, one user: launches and latency
        _decode("decode-small-1", "opt-125m-like", 12, "bf16", 1, 90, 90, 1024),
        # a chat with an 8B model on one GPU, one stream
        _decode("decode-8b-1", "llama-3-8b", 4, "bf16", 1, 700, 700, 4096),
        # the headline: a 32B model in 8 bits, 64 sequences, short context
        _decode("decode-32b-int8-64", "qwen-2.5-32b", 4, "int8", 64, 128, 160,
                1024),
        # eight serving slots, 4-bit weights, conversations of any length
        _decode("decode-32b-int4-8", "qwen-2.5-32b", 4, "int4", 8, 50, 1900,
                4096),
        # long documents: the cache is most of what is read
        _decode("decode-8b-long", "qwen3-8b", 2, "bf16", 32, 1500, 8000, 8192),
        # the same with an 8-bit cache and an odd number of sequences
        _decode("decode-32b-kv8-13", "qwen-2.5-32b", 2, "int8", 13, 900, 4000,
                4096, kv_bits=8),
        # experts, sinks, sliding windows; half-full batch
        _decode("decode-moe-20", "gpt-oss-20b", 2, "bf16", 20, 100, 1500,
                4096),
        # a short question to a chat
        _prefill("prefill-8b-37", "llama-3-8b", 4, "bf16", 1, 37),
        # the headline's time to first token: 64 prompts of 128 tokens
        _prefill("prefill-32b-int8-64x128", "qwen-2.5-32b", 2, "int8", 64,
                 128),
        # a document of 6000 tokens in the middle of a conversation
        _prefill("prefill-8b-6000", "llama-3-8b", 2, "bf16", 1, 6000, 1000),
        # a prompt through routed experts
        _prefill("prefill-moe-700", "mixtral-8x7b", 1, "int8", 1, 700),
        # prompts of unequal length admitted together, fp32 residual and
        # modified scores
        _prefill("prefill-posudra-ragged", "posudra-8b-like", 2, "bf16", 5,
                 1023, ragged=True),
    ]


# model, weights, layers
_DECODES = [("opt-125m-like", "bf16", 12), ("opt-125m-like", "int8", 12),
            ("llama-3-8b", "bf16", 3), ("llama-3-8b", "int8", 3),
            ("qwen3-8b", "bf16", 2), ("qwen3-8b", "int8", 2),
            ("qwen-2.5-32b", "int8", 3), ("qwen-2.5-32b", "int4", 3),
            ("qwen-2.5-32b", "int8", 2), ("gpt-oss-20b", "bf16", 2),
            ("mixtral-8x7b", "int8", 1), ("posudra-8b-like", "bf16", 2)]
_PREFILLS = [("opt-125m-like", "bf16", 12), ("llama-3-8b", "bf16", 2),
             ("llama-3-8b", "int8", 2), ("qwen3-8b", "bf16", 2),
             ("qwen-2.5-32b", "int8", 1), ("qwen-2.5-32b", "int4", 1),
             ("gpt-oss-20b", "bf16", 2), ("mixtral-8x7b", "int8", 1),
             ("posudra-8b-like", "bf16", 2)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Decode: 1 to 64 sequences, contexts of 16 to 8000 tokens. Prefill: one
    prompt of 8 to 6000 tokens, or up to 64 equal ones, 8000 tokens at most."""
    if rng.random() < 0.55:
        model, weights, layers = rng.choice(_DECODES)
        batch = _log(rng, 1, 64)
        hi = _log(rng, 16, min(8000, 200000 // batch))
        lo = rng.randint(max(8, hi // 8), hi)
        cap = 1 << max(10, (hi + STEPS).bit_length())
        dense = not any(m in model for m in ("posudra", "gpt-oss", "mixtral"))
        kv = 8 if dense and rng.random() < 0.25 else 16
        c = _decode("", model, layers, weights, batch, lo, hi, cap, kv)
    else:
        model, weights, layers = rng.choice(_PREFILLS)
        dense = not any(m in model for m in ("posudra", "gpt-oss", "mixtral"))
        if model.startswith("posudra"):
            batch = rng.randint(1, 6)
            tokens = _log(rng, 8, 1200)
            c = _prefill("", model, layers, weights, batch, tokens,
                         ragged=True)
        elif dense and rng.random() < 0.4:
            batch = _log(rng, 2, 64)
            c = _prefill("", model, layers, weights, batch,
                         _log(rng, 8, min(2048, 8000 // batch)))
        else:
            hi = 6000 if dense else 1500
            c = _prefill("", model, layers, weights, 1, _log(rng, 8, hi),
                         rng.choice([0, 0, _log(rng, 16, 2000)]))
    del c["name"]
    return c


# ---------------------------------------------------------------- the model

def _hf(case):
    p = dict(PRESETS[case["model"]])
    if "architecture" in p:
        p["layers"] = p["layers"][:case["layers"]]
    else:
        p["num_hidden_layers"] = case["layers"]
    return p


def _config(case):
    bits = {"bf16": 0, "int8": 8, "int4": 4}[case["weights"]]
    return ModelConfig.from_hf(_hf(case),
                               quant=QuantConfig(bits, 128) if bits else None)


def _posudra(case):
    return case["model"].startswith("posudra")


def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + part) & 0x7FFFFFFFFFFF)
    return g


def _weights(case, seed):
    """Checkpoint tensors by name, bf16 on the GPU."""
    cfg = _config(case)
    g = _gen(seed, 1)
    bits = {"bf16": 0, "int8": 8, "int4": 4}[case["weights"]]
    W = cfg.hidden_size

    def rn(*shape, std=1.0):
        t = torch.randn(*shape, generator=g, device="cuda",
                        dtype=torch.bfloat16)
        return t.mul_(std)

    def lin(n, k, gain=1.0, plain=False):
        std = gain * k ** -0.5
        if not bits or plain:
            return rn(n, k, std=std)
        top = 127 if bits == 8 else 7
        # whole numbers with a standard deviation of 0.3 of the largest, a
        # largest one in each group, times a power of two per group
        q = rn(n, k // 128, 128, std=0.3 * top).round_().clamp_(-top, top)
        q[:, :, 5] = torch.where(q[:, :, 5] < 0, -top, top).to(q.dtype)
        e = torch.randint(-1, 2, (n, k // 128, 1), generator=g, device="cuda")
        s = math.floor(math.log2(std / (0.3 * top)))
        return q.mul_(torch.exp2((e + s).to(torch.float32)).to(
            torch.bfloat16)).view(n, k)

    def near_one(n):
        return 1 + rn(n, std=0.1)

    sd = {}
    if _posudra(case):
        for i in range(case["layers"]):
            m = cfg.layer_specs[i]["mixer"]
            H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            F = cfg.layer_specs[i]["mlp"]["ff"]

            def ru(n, lo, hi):
                return torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo
            t = {"norm1": near_one(W), "mix.q": lin(H * D, W),
                 "mix.k": lin(G * D, W), "mix.v": lin(G * V, W),
                 "mix.q.norm": near_one(H * D), "mix.k.norm": near_one(G * D),
                 "mix.temp": ru(H, 0.5, 2.0), "mix.r1": ru(H, 0.0, 1.0),
                 "mix.r2": ru(H, 0.05, 1.0), "mix.sink": rn(H),
                 "mix.o": lin(W, H * V), "ls1": ru(W, 0.2, 1.0),
                 "mlp.up": lin(F, W), "mlp.down": lin(W, F),
                 "mlp.act": rn(2, std=0.5), "ls2": ru(W, 0.2, 1.0)}
            sd.update({f"l{i}.{n}": x.to(torch.bfloat16)
                       for n, x in t.items()})
        sd["embed"] = rn(cfg.vocab_size, W)
        sd["final.norm"] = near_one(W)
        sd["head"] = lin(cfg.vocab_size, W)
        return sd
    H, G, D = cfg.num_q_heads, cfg.num_kv_heads, cfg.head_dim
    oss = cfg.model_type == "gpt_oss"
    # a trained router decides clearly: tokens lie along its directions (the
    # layers have them in different orders), so that rounding turns few picks
    E = cfg.num_experts
    ways = rn(E, W, std=W ** -0.5) if E else None
    for i in range(case["layers"]):
        p = f"layers.{i}."
        a = p + "self_attn."
        sd[p + "input_layernorm.weight"] = near_one(W)
        sd[p + "post_attention_layernorm.weight"] = near_one(W)
        sd[a + "q_proj.weight"] = lin(H * D, W, 1.5)
        sd[a + "k_proj.weight"] = lin(G * D, W)
        sd[a + "v_proj.weight"] = lin(G * D, W)
        sd[a + "o_proj.weight"] = lin(W, H * D)
        if cfg.attention_bias or oss:
            sd[a + "q_proj.bias"] = rn(H * D, std=0.2)
            sd[a + "k_proj.bias"] = rn(G * D, std=0.2)
            sd[a + "v_proj.bias"] = rn(G * D, std=0.2)
        if cfg.qk_norm:
            sd[a + "q_norm.weight"] = 1.5 * near_one(D)
            sd[a + "k_norm.weight"] = near_one(D)
        F = cfg.moe_intermediate_size or cfg.intermediate_size
        router = 0.5 * ways[torch.randperm(E, generator=g, device="cuda")] \
            if E else None
        if oss:
            sd[a + "o_proj.bias"] = rn(W, std=0.02)
            sd[a + "sinks"] = rn(H)
            sd[p + "mlp.router.weight"] = router
            sd[p + "mlp.router.bias"] = rn(E, std=0.1)
            sd[p + "mlp.experts.gate_up_proj"] = rn(E, W, 2 * F,
                                                    std=W ** -0.5)
            sd[p + "mlp.experts.gate_up_proj_bias"] = rn(E, 2 * F, std=0.05)
            sd[p + "mlp.experts.down_proj"] = rn(E, F, W, std=0.2 * F ** -0.5)
            sd[p + "mlp.experts.down_proj_bias"] = rn(E, W, std=0.02)
        elif E:
            sd[p + "block_sparse_moe.gate.weight"] = router
            for e in range(E):
                x = f"{p}block_sparse_moe.experts.{e}."
                sd[x + "w1.weight"] = lin(F, W)
                sd[x + "w3.weight"] = lin(F, W)
                sd[x + "w2.weight"] = lin(W, F, 0.3)
        else:
            sd[p + "mlp.gate_proj.weight"] = lin(cfg.intermediate_size, W)
            sd[p + "mlp.up_proj.weight"] = lin(cfg.intermediate_size, W)
            sd[p + "mlp.down_proj.weight"] = lin(W, cfg.intermediate_size, 0.5)
    sd["embed_tokens.weight"] = rn(cfg.vocab_size, W)
    if E:
        sd["embed_tokens.weight"] += rn(cfg.vocab_size, E, std=6.0) @ ways
    sd["norm.weight"] = near_one(W)
    sd["lm_head.weight"] = lin(cfg.vocab_size, W, plain=bool(E))
    return sd


def _heads(case):
    """(kv heads, key size, value size)"""
    cfg = _config(case)
    if _posudra(case):
        m = cfg.layer_specs[0]["mixer"]
        return m["kv_heads"], m["dim"], m["vdim"]
    return cfg.num_kv_heads, cfg.head_dim, cfg.head_dim


def _capacity(case):
    if case["kind"] == "decode":
        return case["capacity"]
    return -(-(case["start"] + case["tokens"]) // 256) * 256


def _context(case, seed, layer):
    """What a layer's cache holds before the call: keys and values
    [B, heads, capacity, size], bf16 or (8-bit cache) codes and scales."""
    g = _gen(seed, 100 + layer)
    G, D, V = _heads(case)
    shape = (case["batch"], G, _capacity(case))
    if case.get("kv_bits", 16) == 8:
        out = []
        for d in (D, V):
            out.append(torch.randint(-127, 128, (*shape, d), generator=g,
                                     device="cuda", dtype=torch.int8))
            out.append((torch.rand(*shape, d // 64, generator=g,
                                   device="cuda") * 0.01 + 0.008).to(
                                       torch.bfloat16))
        return out
    return [torch.randn(*shape, d, generator=g, device="cuda",
                        dtype=torch.bfloat16) for d in (D, V)]


def _has_context(case):
    return case["kind"] == "decode" or case["start"] > 0


def _contexts(case):
    """Decode: how many tokens each sequence has, spread over the range."""
    B, lo, hi = case["batch"], case["ctx_lo"], case["ctx_hi"]
    return [hi - (hi - lo) * ((i * 7) % B) // max(1, B - 1) for i in range(B)]


def _lengths(case):
    """Prefill: the prompts' lengths."""
    B, T = case["batch"], case["tokens"]
    if not case["ragged"]:
        return [T] * B
    return [max(1, T - (T * 3 * i) // (4 * B)) for i in range(B)]


def _tokens(case, seed):
    g = _gen(seed, 7)
    n = STEPS if case["kind"] == "decode" else case["tokens"]
    return torch.randint(0, _config(case).vocab_size, (case["batch"], n),
                         generator=g, device="cuda")


# ---------------------------------------------------------------- the calls

def prepare(case, seed):
    cfg = _config(case)
    B = case["batch"]
    ex = RingExecutor(cfg, 0, 1, torch.device("cuda"), mb_size=B,
                      smax=_capacity(case), init_weights=False,
                      kv_bits=case.get("kv_bits", 16))
    ex.model.load_state_dict(_weights(case, seed))
    kv = ex.kvs[0]
    if _has_context(case):
        for l in range(case["layers"]):
            c = _context(case, seed, l)
            if case.get("kv_bits", 16) == 8:
                kv.k[l].copy_(c[0])
                kv.kscale[l].copy_(c[1])
                kv.v[l].copy_(c[2])
                kv.vscale[l].copy_(c[3])
            else:
                kv.k[l].copy_(c[0])
                kv.v[l].copy_(c[1])
    s = {"case": case, "ex": ex, "tokens": _tokens(case, seed)}
    if case["kind"] == "decode":
        s["pos"] = torch.tensor(_contexts(case), dtype=torch.int32,
                                device="cuda")
        s["none"] = torch.zeros(B, dtype=torch.bool, device="cuda")
        kv.pos.copy_(s["pos"])
        ex.slot_step_compute(park=s["none"])    # a server captures the step
    else:                                       # when it loads a model
        s["prompts"] = [s["tokens"][i, :n] for i, n in
                        enumerate(_lengths(case))]
    return s


def run(state):
    case, ex = state["case"], state["ex"]
    kv = ex.kvs[0]
    if case["kind"] == "decode":
        kv.pos.copy_(state["pos"])
        logits = []
        for i in range(STEPS):
            ex.tokbuf[0].copy_(state["tokens"][:, i])
            ex.slot_step_compute(park=state["none"])
            logits.append(ex.logits_buf[0].clone())
            ex.slot_advance(state["none"], state["none"])
        out = {"logits": logits}
        a, b = case["ctx_lo"], case["ctx_hi"] + STEPS
        for n, t in (("k", kv.k), ("v", kv.v), ("kscale", kv.kscale),
                     ("vscale", kv.vscale)):
            if t is not None:
                out[n] = [t[l][:, :, a:b] for l in range(case["layers"])]
        return out
    B, T, p0 = case["batch"], case["tokens"], case["start"]
    if B > 1 and not case["ragged"]:
        # equal prompts in one batch
        m = ex.model
        h = m.embed_tokens(state["tokens"]).clone()
        m.prefill_window(h, ex.my_layers, kv, p0)
        kv.pos.fill_(p0 + T)
        logits = [m.normalize_project(h[:, -1].contiguous())]
    else:
        logits = ex.prefill_slots(list(range(B)), state["prompts"],
                                  start=[p0] * B)
    return {"logits": logits,
            "k": [kv.k[l][:, :, p0:p0 + T] for l in range(case["layers"])],
            "v": [kv.v[l][:, :, p0:p0 + T] for l in range(case["layers"])]}


# ---------------------------------------------------------------- the work

def _sizes(case):
    """Values of a layer's projections (experts apart), of one expert, bytes
    a value of each."""
    cfg = _config(case)
    W = cfg.hidden_size
    per = {"bf16": 2.0, "int8": 1.0 + 2 / 128, "int4": 0.5 + 2 / 128}[
        case["weights"]]
    G, D, V = _heads(case)
    H = cfg.num_q_heads
    att = W * (H * D + G * D + G * V) + W * H * V
    if _posudra(case):
        return att + 2 * W * cfg.intermediate_size, 0, per, per
    F = cfg.moe_intermediate_size or cfg.intermediate_size
    if cfg.num_experts:
        return att + W * cfg.num_experts, 3 * W * F, per, 2.0
    return att + 3 * W * cfg.intermediate_size, 0, per, per


def work(case):
    cfg = _config(case)
    G, D, V = _heads(case)
    H = cfg.num_q_heads
    dense, expert, per, head_per = _sizes(case)
    L, W = case["layers"], cfg.hidden_size
    E, top = cfg.num_experts, cfg.num_experts_per_tok
    cell = G * (D + V) * (2 if case.get("kv_bits", 16) == 16 else 1 + 2 / 64)
    if case["kind"] == "decode":
        rows, times = case["batch"], STEPS
        ctx = _contexts(case)
        pairs = [sum(c + s + 1 for c in ctx) for s in range(STEPS)]
        seen = list(pairs)
        heads = rows
        if cfg.model_type == "gpt_oss":     # every second layer is windowed
            w = cfg.sliding_window
            near = [sum(min(w, c + s + 1) for c in ctx) for s in range(STEPS)]
            pairs = seen = [(a + b) / 2 for a, b in zip(pairs, near)]
    else:
        times, ls, p0 = 1, _lengths(case), case["start"]
        rows = sum(ls)
        pairs = [sum(n * p0 + n * (n + 1) / 2 for n in ls)]
        seen = [sum(n + p0 for n in ls)]
        heads = case["batch"]
        if cfg.model_type == "gpt_oss":
            w = cfg.sliding_window
            near = sum(min(w, p0 + t + 1) for t in range(ls[0]))
            pairs = [(pairs[0] + near) / 2]
    touched = E * (1 - (1 - top / E) ** rows) if E else 0
    weights = L * (dense + touched * expert) * per + \
        cfg.vocab_size * W * head_per
    nbytes = times * (weights + rows * W * 2 + heads * cfg.vocab_size * 2 +
                      L * rows * cell) + sum(seen) * L * cell
    flops = times * (2 * L * rows * (dense + top * expert) +
                     2 * heads * cfg.vocab_size * W) + \
        sum(pairs) * L * H * 2 * (D + V)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 activations, residual and cache: 0.4 to 1.4 % off 64 bits, up to
    # 0.8 % between two passes whose sums come in another order. An 8-bit
    # cache rounds a value near the middle of two codes either way.
    return {"rel": 0.03, "max": 0.5, "differ": 0.002}


# ---------------------------------------------------------------- 64 bits

def _mm(x, w):
    """x [..., K] @ w [N, K]^T in 64 bits, w bf16, in parts of its rows."""
    f = x.reshape(-1, x.shape[-1])
    step = max(1, (1 << 28) // w.shape[1])
    y = torch.cat([f @ w[i:i + step].double().t().contiguous()
                   for i in range(0, w.shape[0], step)], dim=1)
    return y.view(*x.shape[:-1], w.shape[0])


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, pos, theta):
    """x [B, T, H, D], pos [B, T]: halves turn against each other."""
    n = x.shape[-1] // 2
    f = theta ** (-torch.arange(n, device=x.device, dtype=torch.float64) / n)
    a = (pos.double().unsqueeze(-1) * f).unsqueeze(2)
    x1, x2 = x[..., :n], x[..., n:]
    return torch.cat([x1 * a.cos() - x2 * a.sin(),
                      x2 * a.cos() + x1 * a.sin()], -1)


def _attend(q, K, V, pos, scale, window=0, sinks=None, extra=None):
    """q [B, T, H, D]; K, V [B, G, S, D]; pos [B, T] -> [B, T, H, V]."""
    B, T, H, D = q.shape
    G, S = K.shape[1], K.shape[2]
    n = H // G
    Kt = K.transpose(-1, -2).contiguous()
    out = torch.empty(B, T, H, V.shape[-1], dtype=torch.float64,
                      device=q.device)
    j = torch.arange(S, device=q.device)
    step = max(1, (1 << 27) // (B * H * S))
    for t0 in range(0, T, step):
        qc = q[:, t0:t0 + step]
        t = qc.shape[1]
        pc = pos[:, t0:t0 + step]
        x = qc.view(B, t, G, n, D).permute(0, 2, 3, 1, 4)
        s = (x.reshape(B, G, n * t, D) @ Kt).view(B, H, t, S) * scale
        if extra is not None:
            s = extra(s, (pc.unsqueeze(-1) - j).clamp(min=0).double()
                      .unsqueeze(1))
        hide = j > pc.unsqueeze(-1)
        if window:
            hide |= j <= pc.unsqueeze(-1) - window
        s.masked_fill_(hide.unsqueeze(1), -math.inf)
        if sinks is not None:
            z = sinks.double().view(1, H, 1, 1).expand(B, H, t, 1)
            p = torch.softmax(torch.cat([s, z], -1), -1)[..., :-1]
        else:
            p = torch.softmax(s, -1)
        o = p.reshape(B, G, n * t, S) @ V
        out[:, t0:t0 + step] = o.view(B, G, n, t, -1).permute(
            0, 3, 1, 2, 4).reshape(B, t, H, -1)
    return out


def _experts(y, sd, p, cfg):
    f = y.reshape(-1, y.shape[-1])
    top, E = cfg.num_experts_per_tok, cfg.num_experts
    out = torch.zeros_like(f)
    oss = cfg.model_type == "gpt_oss"
    if oss:
        r = _mm(f, sd[p + "mlp.router.weight"]) + \
            sd[p + "mlp.router.bias"].double()
    else:
        r = _mm(f, sd[p + "block_sparse_moe.gate.weight"])
    w, idx = torch.topk(r, top, -1)
    w = torch.softmax(w, -1)
    for e in range(E):
        row, col = (idx == e).nonzero(as_tuple=True)
        if not row.numel():
            continue
        x = f[row]
        if oss:
            m = p + "mlp.experts."
            gu = x @ sd[m + "gate_up_proj"][e].double() + \
                sd[m + "gate_up_proj_bias"][e].double()
            a, b = gu[:, 0::2].clamp(max=7.0), gu[:, 1::2].clamp(-7.0, 7.0)
            d = ((b + 1) * a * torch.sigmoid(1.702 * a)) @ \
                sd[m + "down_proj"][e].double() + \
                sd[m + "down_proj_bias"][e].double()
        else:
            m = f"{p}block_sparse_moe.experts.{e}."
            a = torch.nn.functional.silu(_mm(x, sd[m + "w1.weight"]))
            d = _mm(a * _mm(x, sd[m + "w3.weight"]), sd[m + "w2.weight"])
        out.index_add_(0, row, d * w[row, col].unsqueeze(-1))
    return out.view_as(y)


def _forward(case, sd, cfg, tokens, start, cache):
    """Logits and residual of tokens [B, T] at positions start [B] + t; the
    caches (one (K, V) a layer, 64 bits) get the new rows."""
    B, T = tokens.shape
    pos = start.view(B, 1).long() + torch.arange(T, device=tokens.device)
    at = torch.arange(B, device=tokens.device).view(B, 1)
    eps = cfg.rms_eps
    G, D, V = _heads(case)
    H = cfg.num_q_heads
    pos_ = _posudra(case)
    x = sd["embed" if pos_ else "embed_tokens.weight"][tokens].double()
    for i in range(case["layers"]):
        K, Vc = cache[i]
        if pos_:
            m = {n[len(f"l{i}."):]: t for n, t in sd.items()
                 if n.startswith(f"l{i}.")}
            u = _rms(x, m["norm1"], eps)
            q = _rms(_mm(u, m["mix.q"]), m["mix.q.norm"], eps)
            k = _rms(_mm(u, m["mix.k"]), m["mix.k.norm"], eps)
            K[at, :, pos] = k.view(B, T, G, D)
            Vc[at, :, pos] = _mm(u, m["mix.v"]).view(B, T, G, V)
            mx = cfg.layer_specs[i]["mixer"]
            cap = mx["softcap"]

            def extra(s, dist, m=m, cap=cap):
                v = [m["mix." + n].double().view(1, H, 1, 1)
                     for n in ("temp", "r1", "r2")]
                s = cap * torch.tanh(s * v[0] / cap)
                return s - v[1] * torch.log1p(v[2] * dist)
            a = _attend(q.view(B, T, H, D), K, Vc, pos, mx["scale"],
                        sinks=m["mix.sink"], extra=extra)
            o = _mm(a.reshape(B, T, H * V), m["mix.o"])
            z = _mm(u, m["mlp.up"])
            pq = torch.nn.functional.softplus(m["mlp.act"].double())
            z = torch.where(z > 0, pq[0] * z * z + 0.5 * z, (0.5 + pq[1]) *
                            (torch.expm1(z.clamp(max=0)) - z) + 0.5 * z)
            x = x + m["ls1"].double() * o + \
                m["ls2"].double() * _mm(z, m["mlp.down"])
            continue
        p = f"layers.{i}."
        a = p + "self_attn."
        y = _rms(x, sd[p + "input_layernorm.weight"], eps)
        q, k, v = (_mm(y, sd[f"{a}{n}_proj.weight"]) for n in "qkv")
        if a + "q_proj.bias" in sd:
            q, k, v = (t + sd[f"{a}{n}_proj.bias"].double()
                       for t, n in ((q, "q"), (k, "k"), (v, "v")))
        q, k = q.view(B, T, H, D), k.view(B, T, G, D)
        if cfg.qk_norm:
            q = _rms(q, sd[a + "q_norm.weight"], eps)
            k = _rms(k, sd[a + "k_norm.weight"], eps)
        q, k = _rope(q, pos, cfg.rope_theta), _rope(k, pos, cfg.rope_theta)
        K[at, :, pos] = k
        Vc[at, :, pos] = v.view(B, T, G, V)
        slide = cfg.sliding_window if cfg.model_type == "gpt_oss" and \
            i % 2 == 0 else 0
        o = _attend(q, K, Vc, pos, D ** -0.5, slide, sd.get(a + "sinks"))
        o = _mm(o.reshape(B, T, H * D), sd[a + "o_proj.weight"])
        if a + "o_proj.bias" in sd:
            o = o + sd[a + "o_proj.bias"].double()
        x = x + o
        y = _rms(x, sd[p + "post_attention_layernorm.weight"], eps)
        if cfg.num_experts:
            x = x + _experts(y, sd, p, cfg)
        else:
            g = torch.nn.functional.silu(_mm(y, sd[p + "mlp.gate_proj.weight"]))
            x = x + _mm(g * _mm(y, sd[p + "mlp.up_proj.weight"]),
                        sd[p + "mlp.down_proj.weight"])
    return x


def _project(sd, cfg, x):
    y = _rms(x, sd["final.norm" if "final.norm" in sd else "norm.weight"],
             cfg.rms_eps)
    return _mm(y, sd["head" if "head" in sd else "lm_head.weight"])


def exact(case, seed):
    cfg, sd, tokens = _config(case), _weights(case, seed), _tokens(case, seed)
    B = case["batch"]
    G, D, V = _heads(case)
    cache = []
    for l in range(case["layers"]):
        if not _has_context(case):
            cache.append([torch.zeros(B, G, _capacity(case), d,
                                      dtype=torch.float64, device="cuda")
                          for d in (D, V)])
            continue
        c = _context(case, seed, l)
        if len(c) == 4:
            c = [(c[i].double().unflatten(-1, (-1, 64)) *
                  c[i + 1].double().unsqueeze(-1)).flatten(-2)
                 for i in (0, 2)]
        cache.append([t.double() for t in c])
    if case["kind"] == "decode":
        x = _forward(case, sd, cfg, tokens,
                     torch.tensor(_contexts(case), device="cuda"), cache)
        out = {"logits": list(_project(sd, cfg, x).unbind(1))}
        a, b = case["ctx_lo"], case["ctx_hi"] + STEPS
        if case["kv_bits"] == 8:    # codes and scales have no such values
            out.update({n: [None] * case["layers"]
                        for n in ("k", "v", "kscale", "vscale")})
        else:
            out["k"] = [c[0][:, :, a:b] for c in cache]
            out["v"] = [c[1][:, :, a:b] for c in cache]
        return out
    T, p0 = case["tokens"], case["start"]
    if not case["ragged"]:
        x = _forward(case, sd, cfg, tokens,
                     torch.full((B,), p0, device="cuda"), cache)
        logits = [_project(sd, cfg, x[:, -1])]
    else:
        logits = []
        for r, n in enumerate(_lengths(case)):
            x = _forward(case, sd, cfg, tokens[r:r + 1, :n],
                         torch.zeros(1, dtype=torch.long, device="cuda"),
                         [[t[r:r + 1] for t in c] for c in cache])
            logits.append(_project(sd, cfg, x[:, -1]))
    return {"logits": logits,
            "k": [c[0][:, :, p0:p0 + T] for c in cache],
            "v": [c[1][:, :, p0:p0 + T] for c in cache]}
