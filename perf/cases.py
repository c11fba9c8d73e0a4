"""The work that a user of litemind_amd has it do, as measurable cases.

A case is one call (or, for the decode step, one short sequence of calls)
through the package's public entry points, at the sizes of the repository's own
configurations: DeepSeek-V2-Lite (hidden 2048, 64 experts of 1408, top-6, 2
shared experts, 16 heads, latent 512, vocabulary 102400) and DeepSeek-V2's MoE
layer (hidden 5120, 160 experts of 1536 in 8 groups, 3 kept).  Weights are
BF16 N(0, 0.02) as the benchmark draws them, tokens RMS-normalised N(0, 1).

Kinds:
  moe        lm_moe_forward, path AUTO: router, experts, shared expert, combine
  dense      lm_dense_forward, path AUTO: the dense SwiGLU layer
  attention  lm_attention_forward after `cached` tokens, path AUTO or GEMV (bit-exact)
  head       lm_head_forward: final norm, logits and the greedy token
  decode     lm_decoder_forward over one dense and two MoE layers, then lm_head_forward
"""
import math

import torch

import litemind_amd as lm
from litemind_amd import workload as wl

V2_LITE, V2_FULL = wl.V2_LITE, wl.V2_FULL
MLA = wl.V2_LITE_MLA
VOCAB = 102400
DECODE_LAYERS = 3  # layer 0 dense, then MoE, as the model begins
PATHS = {"auto": lm.PATH_AUTO, "gemv": lm.PATH_GEMV}


def _case(kind, tokens, cached=0, path="auto", model="lite", skew=0.0):
    return {"kind": kind, "tokens": tokens, "cached": cached, "path": path, "model": model, "skew": skew}


def listed():
    def named(name, *args, **kw):
        return {"name": name, **_case(*args, **kw)}

    return [
        # one token of one sequence: the call that every decode step makes 26 times
        named("moe_decode_1", "moe", 1),
        # a batch of 32 sequences decoding together
        named("moe_batch_32", "moe", 32),
        # a prompt of ordinary length, an odd number of tokens
        named("moe_prompt_509", "moe", 509),
        # a long prompt chunk whose routing is uneven, as trained routers' is
        named("moe_prompt_2048", "moe", 2048, skew=1.0),
        # the larger model's layer, one token
        named("moe_v2_decode_1", "moe", 1, model="v2"),
        # the dense first layer over a long prompt
        named("dense_prompt_4096", "dense", 4096),
        # one token after a long conversation
        named("attention_decode_4000", "attention", 1, cached=4000),
        # a prompt of ordinary length into an empty cache
        named("attention_prompt_512", "attention", 512),
        # the longest prompt that the default context holds
        named("attention_prompt_4096", "attention", 4096),
        # a short prompt after a system prompt, on the path that keeps the CPU's bits
        named("attention_exact_77", "attention", 77, cached=301, path="gemv"),
        # the logits of a batch of 32 sequences
        named("head_batch_32", "head", 32),
        # a whole decode step: attention, dense and MoE layers, head and greedy token
        named("decode_step_1", "decode", 1, cached=1000),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "dense", "attention", "attention", "attention", "head", "decode"])
    if kind == "moe":
        tokens = _log_uniform(rng, 1, 2048)
        return _case("moe", tokens, skew=rng.choice([0.0, 0.5, 1.0]) if tokens >= 64 else 0.0)
    if kind == "dense":
        return _case("dense", _log_uniform(rng, 1, 4096))
    if kind == "head":
        return _case("head", _log_uniform(rng, 1, 32))
    if kind == "decode":
        return _case("decode", rng.choice([1, 1, 2, 3]), cached=_log_uniform(rng, 16, 1000))
    use = rng.choice(["decode", "prompt", "prompt", "chunk", "exact"])
    if use == "decode":
        return _case("attention", rng.choice([1, 1, 2, 5]), cached=_log_uniform(rng, 16, 4000))
    if use == "prompt":
        return _case("attention", _log_uniform(rng, 16, 4096))
    if use == "chunk":
        tokens = _log_uniform(rng, 16, 2048)
        return _case("attention", tokens, cached=_log_uniform(rng, 16, 4096 - tokens))
    return _case("attention", _log_uniform(rng, 2, 128), cached=_log_uniform(rng, 1, 1000), path="gemv")


# ---- inputs, from the seed alone ----

def _dims(case):
    return V2_FULL if case["model"] == "v2" else V2_LITE


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _normal(g, shape, sigma, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype).mul_(sigma)


def _tokens(g, count, hidden):
    x = torch.randn((count, hidden), generator=g, device="cuda")
    return (x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6)).contiguous()


def _moe_weights(g, d):
    H, I, E, S = d.hidden, d.inter, d.experts, d.shared_inter
    return {"router": _normal(g, (E, H), 0.02, torch.float32), "gate": _normal(g, (E, I, H), 0.02),
            "up": _normal(g, (E, I, H), 0.02), "down": _normal(g, (E, H, I), 0.02),
            "shared": [_normal(g, (S, H), 0.02), _normal(g, (S, H), 0.02), _normal(g, (H, S), 0.02)]}


def _dense_weights(g, d):
    H, D = d.hidden, d.dense_inter
    return [_normal(g, (D, H), 0.02), _normal(g, (D, H), 0.02), _normal(g, (H, D), 0.02)]


def _attention_weights(g, d):
    H, heads = d.hidden, d.heads
    return {"q_proj": _normal(g, (heads * d.qk_head, H), 0.02),
            "kv_a_proj": _normal(g, (d.kv_lora_rank + d.qk_rope, H), 0.02),
            "kv_a_layernorm": 1.0 + _normal(g, (d.kv_lora_rank,), 0.1, torch.float32),
            "kv_b_proj": _normal(g, (heads * (d.qk_nope + d.v_head), d.kv_lora_rank), 0.05),
            "o_proj": _normal(g, (H, heads * d.v_head), 0.02)}


def _cache_entries(g, d, cached):
    """Cached keys and values with the spread that kv_b and kv_a give them."""
    return [_normal(g, (cached, d.heads, d.qk_nope), 1.13, torch.float32),
            _normal(g, (cached, d.qk_rope), 0.9, torch.float32),
            _normal(g, (cached, d.heads, d.v_head), 1.13, torch.float32)]


def _norm_weight(g, n):
    return 1.0 + _normal(g, (n,), 0.1, torch.float32)


def _skew_bias(d, x, router, skew):
    """A logit bias under which 8 experts take most of the assignments and the rest fall off as the benchmark's do."""
    if not skew:
        return None
    target = torch.from_numpy(wl.skew_targets(d)).to(x.device) * (x.shape[0] * d.top_k)
    logits = x.double() @ router.double().T
    bias = torch.zeros(d.experts, dtype=torch.float64, device=x.device)
    for _ in range(60):
        top = (logits + bias).topk(d.top_k, dim=1).indices
        counts = torch.bincount(top.reshape(-1), minlength=d.experts).double()
        bias += 0.5 * (torch.log(target + 0.5) - torch.log(counts + 0.5))
        bias -= bias.mean()
    return (bias * skew).float().contiguous()


def _inputs(case, seed):
    """Everything the case draws, on the GPU: prepare() hands it to the library, exact() computes with it."""
    g, kind, T = _generator(seed), case["kind"], case["tokens"]
    d = _dims(case)
    p = {"x": _tokens(g, T, d.hidden)}
    if kind == "moe":
        p["moe"] = _moe_weights(g, d)
        p["bias"] = _skew_bias(d, p["x"], p["moe"]["router"], case["skew"])
    elif kind == "dense":
        p["dense"] = _dense_weights(g, d)
    elif kind == "attention":
        p["attention"] = _attention_weights(g, MLA)
        p["cache"] = _cache_entries(g, MLA, case["cached"])
    if kind == "decode":
        p["layers"] = [{"input_norm": _norm_weight(g, d.hidden), "attention": _attention_weights(g, MLA),
                        "cache": _cache_entries(g, MLA, case["cached"]), "norm": _norm_weight(g, d.hidden),
                        **({"dense": _dense_weights(g, d)} if i == 0 else {"moe": _moe_weights(g, d)})}
                       for i in range(DECODE_LAYERS)]
    if kind in ("head", "decode"):
        p["final_norm"], p["head"] = _norm_weight(g, d.hidden), _normal(g, (VOCAB, d.hidden), 0.02)
    return p


# ---- what a program holds before the call ----

def _host(t):
    """A tensor as a host array, BF16 as its bit patterns, through page-locked memory."""
    t = t.contiguous()
    t = t.view(torch.int16) if t.dtype == torch.bfloat16 else t
    h = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
    h.copy_(t)
    a = h.numpy()
    return a.view("uint16") if t.dtype == torch.int16 else a


def _upload_moe(ctx, layer, w, chunk=16):
    ctx.upload_router(layer, _host(w["router"]))
    experts = w["gate"].shape[0]
    for e0 in range(0, experts, chunk):
        gate, up, down = (_host(w[k][e0:e0 + chunk]) for k in ("gate", "up", "down"))
        for i in range(gate.shape[0]):
            ctx.upload_expert(layer, e0 + i, gate[i], up[i], down[i])
    ctx.upload_shared(layer, *[_host(t) for t in w["shared"]])


def _upload_attention(ctx, layer, w, cache):
    ctx.upload_attention(layer, **{k: _host(v) for k, v in w.items()})
    if cache[0].shape[0]:
        ctx.kv_cache_write(layer, 0, *[_host(t) for t in cache])


class State:
    """A context with its resident weights, the call's inputs and the buffers it writes."""

    def __init__(self, case, seed):
        self.case, d, T = case, _dims(case), case["tokens"]
        kind = case["kind"]
        self.ctx = lm.Context(d.moe_config(num_layers=DECODE_LAYERS if kind == "decode" else 1))
        p = _inputs(case, seed)
        self.x = p["x"]
        if kind in ("attention", "decode"):
            self.ctx.attention_configure(wl.mla_config(MLA))
        if kind == "moe":
            _upload_moe(self.ctx, 0, p["moe"])
            self.ctx.finalize_layer(0)
            self.bias = p["bias"]
            self.y = torch.zeros((T, d.hidden), device="cuda")
            self.idx = torch.zeros((T, d.top_k), device="cuda", dtype=torch.int32)
            self.w = torch.zeros((T, d.top_k), device="cuda")
        elif kind == "dense":
            self.ctx.upload_dense(0, *[_host(t) for t in p["dense"]])
            self.ctx.finalize_layer(0)
            self.y = torch.zeros((T, d.hidden), device="cuda")
        elif kind == "attention":
            _upload_attention(self.ctx, 0, p["attention"], p["cache"])
            self.ctx.attention_set_path(PATHS[case["path"]])
            self.y = torch.zeros((T, d.hidden), device="cuda")
        elif kind == "decode":
            for i, layer in enumerate(p["layers"]):
                _upload_attention(self.ctx, i, layer["attention"], layer["cache"])
                self.ctx.upload_input_norm(i, _host(layer["input_norm"]))
                self.ctx.upload_norm(i, _host(layer["norm"]))
                if "dense" in layer:
                    self.ctx.upload_dense(i, *[_host(t) for t in layer["dense"]])
                else:
                    _upload_moe(self.ctx, i, layer["moe"])
                self.ctx.finalize_layer(i)
            self.hidden = torch.zeros((T, d.hidden), device="cuda")
            self.stream = torch.cuda.ExternalStream(self.ctx.stream())
        if kind in ("head", "decode"):
            self.ctx.upload_head(_host(p["final_norm"]), _host(p["head"]))
            self.logits = torch.zeros((T, VOCAB), device="cuda")
            self.token = torch.zeros((T,), device="cuda", dtype=torch.int32)
        torch.cuda.synchronize()

    def __del__(self):
        ctx = getattr(self, "ctx", None)
        if ctx is not None and ctx.handle:
            ctx.synchronize()
            ctx.close()


def prepare(case, seed):
    return State(case, seed)


def _p(t):
    return None if t is None else t.data_ptr()


def run(s):
    kind, T, ctx = s.case["kind"], s.case["tokens"], s.ctx
    if kind == "moe":
        ctx.moe_forward(0, _p(s.x), T, _p(s.y), bias=_p(s.bias), idx=_p(s.idx), w=_p(s.w))
        return {"y": s.y, "experts": s.idx, "weights": s.w}
    if kind == "dense":
        ctx.dense_forward(0, _p(s.x), T, _p(s.y))
        return {"y": s.y}
    cached = s.case["cached"]
    if kind == "attention":
        ctx.kv_cache_truncate(0, cached)  # the conversation that the call continues
        ctx.attention_forward(0, _p(s.x), T, cached, _p(s.y))
        return {"y": s.y}
    if kind == "decode":
        for layer in range(DECODE_LAYERS):
            ctx.kv_cache_truncate(layer, cached)
        with torch.cuda.stream(s.stream):  # the embedding rows of the step's tokens
            s.hidden.copy_(s.x)
        ctx.decoder_forward(0, DECODE_LAYERS - 1, _p(s.hidden), T, cached)
        ctx.head_forward(_p(s.hidden), T, logits=_p(s.logits), token=_p(s.token))
        return {"hidden": s.hidden, "logits": s.logits, "token": s.token}
    ctx.head_forward(_p(s.x), T, logits=_p(s.logits), token=_p(s.token))
    return {"logits": s.logits, "token": s.token}


# ---- what a pass cannot do without ----

def _sum(*works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def _moe_work(d, T, skew):
    if skew:
        share = torch.from_numpy(wl.skew_targets(d)) * d.top_k
        hit = float((1.0 - (1.0 - share.clamp(max=1.0)) ** T).sum())
    else:
        hit = d.experts * (1.0 - (1.0 - d.top_k / d.experts) ** T)
    weights = (hit * d.inter + d.shared_inter) * 3 * d.hidden * 2 + d.experts * d.hidden * 4
    flops = 2.0 * T * d.hidden * (3 * (d.top_k * d.inter + d.shared_inter) + d.experts)
    return {"bytes": weights + T * d.hidden * 8 + T * d.top_k * 8, "flops": flops}


def _dense_work(d, T):
    n = 3 * d.hidden * d.dense_inter
    return {"bytes": 2.0 * n + T * d.hidden * 8, "flops": 2.0 * T * n}


def _attention_work(d, T, cached):
    n = d.hidden * (d.heads * d.qk_head + d.kv_lora_rank + d.qk_rope + d.heads * d.v_head)
    n += d.kv_lora_rank * d.heads * (d.qk_nope + d.v_head)
    entry = 4 * (d.heads * (d.qk_nope + d.v_head) + d.qk_rope)
    pairs = T * cached + T * (T + 1) / 2
    return {"bytes": 2.0 * n + (cached + T) * entry + T * d.hidden * 8,
            "flops": 2.0 * T * n + 2.0 * pairs * d.heads * (d.qk_head + d.v_head)}


def _head_work(d, T):
    return {"bytes": 2.0 * VOCAB * d.hidden + T * (4 * VOCAB + 4 * d.hidden + 4), "flops": 2.0 * T * VOCAB * d.hidden}


def work(case):
    kind, T, d = case["kind"], case["tokens"], _dims(case)
    if kind == "moe":
        return _moe_work(d, T, case["skew"])
    if kind == "dense":
        return _dense_work(d, T)
    if kind == "attention":
        return _attention_work(MLA, T, case["cached"])
    if kind == "head":
        return _head_work(d, T)
    return _sum(*[_attention_work(MLA, T, case["cached"])] * DECODE_LAYERS, _dense_work(d, T),
                *[_moe_work(d, T, 0.0)] * (DECODE_LAYERS - 1), _head_work(d, T))


def tolerance(case):
    kind, T = case["kind"], case["tokens"]
    # fp16 operands and 32-bit sums: four times the 3.6e-4 (one layer's GEMMs) and 7e-4 (projections
    # and the attention core) that the path shows against 64 bits
    if kind == "moe" and T > lm.DECODE_TOKENS or kind == "dense" and T > lm.MFMA_CROSSOVER:
        return {"rel": 1.5e-3}
    if kind == "attention" and T >= 16 and case["path"] == "auto":
        return {"rel": 3e-3}
    return {"rel": 1e-5}


# ---- the same in 64 bits ----

def _swiglu(x, gate, up, down):
    a = x @ gate.double().T
    return (a * torch.sigmoid(a) * (x @ up.double().T)) @ down.double().T


def _exact_moe(d, w, x, bias):
    logits = x @ w["router"].double().T
    if bias is not None:
        logits = logits + bias.double()
    scores = torch.softmax(logits, dim=1)
    ranked = scores
    if d.group_limited and d.n_group > 1:
        best = scores.view(x.shape[0], d.n_group, -1).max(dim=2).values
        keep = torch.zeros_like(best).scatter_(1, best.topk(d.topk_group, dim=1).indices, 1.0)
        ranked = torch.where(keep.repeat_interleave(d.experts // d.n_group, dim=1) > 0, scores, -1.0)
    idx = ranked.topk(d.top_k, dim=1).indices
    weights = scores.gather(1, idx) * d.routed_scaling_factor
    y = _swiglu(x, *w["shared"])
    for e in range(d.experts):
        token, rank = (idx == e).nonzero(as_tuple=True)
        if token.numel():
            part = _swiglu(x[token], w["gate"][e], w["up"][e], w["down"][e])
            y.index_add_(0, token, part * weights[token, rank, None])
    return y, idx, weights


def _yarn_magnitude(factor, mscale):
    return 1.0 if factor <= 1.0 else 0.1 * mscale * math.log(factor) + 1.0


def _rotary(d, positions):
    """YaRN's cos and sin [T, rope / 2] at the given positions, rounded to fp32 as the tables hold them."""
    half = d.qk_rope // 2
    i = torch.arange(half, dtype=torch.float64, device="cuda")
    plain = d.rope_theta ** (-2.0 * i / d.qk_rope)

    def turn(rotations):
        return d.qk_rope * math.log(d.original_max / (rotations * 2.0 * math.pi)) / (2.0 * math.log(d.rope_theta))

    low, high = max(math.floor(turn(d.beta_fast)), 0.0), min(math.ceil(turn(d.beta_slow)), d.qk_rope - 1.0)
    mask = 1.0 - ((i - low) / (high - low)).clamp(0.0, 1.0)
    inverse = plain / d.factor * (1.0 - mask) + plain * mask
    magnitude = _yarn_magnitude(d.factor, d.mscale) / _yarn_magnitude(d.factor, d.mscale_all_dim)
    angle = positions.double()[:, None] * inverse
    return (angle.cos() * magnitude).float().double(), (angle.sin() * magnitude).float().double()


def _rotate(v, cos, sin):
    even, odd = v[..., 0::2], v[..., 1::2]
    return torch.cat([even * cos - odd * sin, odd * cos + even * sin], dim=-1)


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _exact_attention(d, w, cache, x, cached):
    T = x.shape[0]
    cos, sin = _rotary(d, torch.arange(cached, cached + T, device="cuda"))
    q = (x @ w["q_proj"].double().T).view(T, d.heads, d.qk_head)
    q_rope = _rotate(q[..., d.qk_nope:], cos[:, None], sin[:, None])
    kv = x @ w["kv_a_proj"].double().T
    latent = _rms(kv[:, :d.kv_lora_rank], w["kv_a_layernorm"], d.rms_norm_eps)
    expanded = (latent @ w["kv_b_proj"].double().T).view(T, d.heads, d.qk_nope + d.v_head)
    k_nope = torch.cat([cache[0].double(), expanded[..., :d.qk_nope]])
    k_rope = torch.cat([cache[1].double(), _rotate(kv[:, d.kv_lora_rank:], cos, sin)])
    value = torch.cat([cache[2].double(), expanded[..., d.qk_nope:]])
    scale = _yarn_magnitude(d.factor, d.mscale_all_dim) ** 2 / math.sqrt(d.qk_head)
    hidden_from = torch.arange(cached + T, device="cuda")[None] > torch.arange(cached, cached + T, device="cuda")[:, None]
    context = torch.empty((T, d.heads, d.v_head), dtype=torch.float64, device="cuda")
    for h in range(d.heads):
        scores = scale * (q[:, h, :d.qk_nope] @ k_nope[:, h].T + q_rope[:, h] @ k_rope.T)
        context[:, h] = torch.softmax(scores.masked_fill(hidden_from, -math.inf), dim=1) @ value[:, h]
    return context.reshape(T, -1) @ w["o_proj"].double().T


def _exact_head(norm, head, hidden, eps):
    x = _rms(hidden, norm, eps)
    return torch.cat([x @ rows.double().T for rows in head.split(25600)], dim=1)


def exact(case, seed):
    p, d, kind = _inputs(case, seed), _dims(case), case["kind"]
    x = p["x"].double()
    if kind == "moe":
        y, idx, weights = _exact_moe(d, p["moe"], x, p["bias"])
        return {"y": y, "experts": idx, "weights": weights}
    if kind == "dense":
        return {"y": _swiglu(x, *p["dense"])}
    if kind == "attention":
        return {"y": _exact_attention(MLA, p["attention"], p["cache"], x, case["cached"])}
    if kind == "decode":
        for layer in p["layers"]:
            x = x + _exact_attention(MLA, layer["attention"], layer["cache"],
                                     _rms(x, layer["input_norm"], MLA.rms_norm_eps), case["cached"])
            n = _rms(x, layer["norm"], d.rms_norm_eps)
            x = x + (_swiglu(n, *layer["dense"]) if "dense" in layer else _exact_moe(d, layer["moe"], n, None)[0])
    logits = _exact_head(p["final_norm"], p["head"], x, d.rms_norm_eps)
    out = {"logits": logits, "token": logits.argmax(dim=1)}
    return {"hidden": x, **out} if kind == "decode" else out
