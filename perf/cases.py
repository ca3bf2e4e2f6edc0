"""What is timed: decoder serving and training as the preset models have it.

Every case is one call of a stage (the slice of a model that one GPU holds)
or of a trainer, at the presets' own widths and heads with few layers, since
all layers of a model do the same work. The kinds are

  decode   one new token per sequence on a contiguous or paged KV cache
  prefill  a prompt, or the next portion of one, into a KV cache
  moe      the same two with routed experts, in bf16 or with fp8 weights
  train    forward, backward and the AdamW update of a stage that is fed
           with its predecessor's activations and its successor's gradients
  trainer  a whole model's training step, from token ids to new weights
"""

import dataclasses
import math

import torch

from tensorlink_amd.models.configs import get_config
from tensorlink_amd.models.dense import build_stage
from tensorlink_amd.models.loader import init_random_stage
from tensorlink_amd.models.quant import quantize_experts_fp8
from tensorlink_amd.optim import FusedAdamW
from tensorlink_amd.parallel.pipeline import PipelineTrainer
from tensorlink_amd.parallel.planner import StageSpec, plan_for_world

QWEN = "Qwen/Qwen2.5-7B-Instruct"
QWEN3 = "Qwen/Qwen3-8B"
LLAMA = "meta-llama/Llama-3.1-8B"
MOE = "Qwen/Qwen3-30B-A3B"
PAGE = 128                      # positions per page of a paged cache
LR, BETAS, EPS, DECAY = 1e-4, (0.9, 0.999), 1e-8, 0.01


def listed():
    return [
        # a chat with one user: every token waits for one pass over the
        # weights, and small launches weigh most
        _decode("decode_one", QWEN, 4, 1, 512, 512),
        # the serving benchmark's decode step: 256 sequences in step
        _decode("decode_batch", QWEN, 2, 256, 576, 576),
        # continuous batching: slots of all ages on a paged cache
        _decode("decode_ragged", QWEN3, 2, 48, 17, 3900, paged=True),
        # two long contexts: the KV cache outweighs the weights
        _decode("decode_long", LLAMA, 2, 2, 32000, 32700),
        # the first token of a short chat prompt of odd length
        _prefill("prefill_one", QWEN, 4, 1, 333),
        # the serving benchmark's prompts, one micro-batch of them
        _prefill("prefill_batch", QWEN, 2, 32, 512),
        # a long document in one piece
        _prefill("prefill_long", LLAMA, 2, 1, 7001),
        # the next portion of a long prompt beside running decodes
        _prefill("prefill_portion", QWEN, 2, 1, 512, start=3456, paged=True),
        # sparse decoding with fp8 experts, the quantised serving mode
        _moe("moe_decode_fp8", 64, 1, 1000, fp8=True),
        # a prompt through sparse experts in bf16
        _moe("moe_prefill", 2, 1200, 0, fp8=False),
        # one rank's share of a training step
        _train("train_stage", QWEN, 2, 2, 2048),
        # a small model trained whole on one GPU
        _trainer("train_small", "gpt2-small", 4, 512),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "prefill", "prefill", "moe",
                       "train", "trainer"])
    model = rng.choice([QWEN, QWEN3, LLAMA])
    if kind == "decode":
        batch = size(1, 256)
        hi = size(40, min(32000, 400000 // batch))
        lo = rng.choice([hi, size(8, hi)])
        c = _decode("", model, rng.choice([1, 2]), batch, lo, hi,
                    paged=rng.random() < 0.5)
    elif kind == "prefill":
        tokens = size(20, 14000)
        start = rng.choice([0, 0, size(100, 6000)])
        paged = start > 0 or rng.random() < 0.3
        batch = 1 if start else min(rng.choice([1, 1, size(2, 32)]),
                                    max(1, tokens // 16))
        length = min(max(2, tokens // batch), 2048 if start else 7000)
        c = _prefill("", model, rng.choice([1, 2]), batch, length,
                     start=start, paged=paged)
    elif kind == "moe":
        fp8 = rng.random() < 0.5
        if rng.random() < 0.5:
            c = _moe("", size(1, 200), 1, size(30, 4000), fp8=fp8)
        else:
            batch = rng.choice([1, 2, 4])
            c = _moe("", batch, size(40, 2400 // batch), 0, fp8=False)
    elif kind == "train":
        length = size(60, 4000)
        batch = max(1, min(16, size(200, 4096) // length))
        c = _train("", model, rng.choice([1, 2]), batch, length)
    else:
        length = size(40, 1000)
        c = _trainer("", rng.choice(["gpt2-small", "tiny"]),
                     max(1, size(100, 2048) // length), min(length, 512))
    del c["name"]
    return c


def _decode(name, model, layers, batch, lo, hi, paged=False):
    return {"name": name, "kind": "decode", "model": model, "layers": layers,
            "batch": batch, "ctx_lo": lo, "ctx_hi": hi, "paged": paged}


def _prefill(name, model, layers, batch, length, start=0, paged=False):
    return {"name": name, "kind": "prefill", "model": model,
            "layers": layers, "batch": batch, "length": length,
            "start": start, "paged": paged}


def _moe(name, batch, length, ctx, fp8):
    return {"name": name, "kind": "moe", "model": MOE, "layers": 1,
            "batch": batch, "length": length, "ctx": ctx, "fp8": fp8}


def _train(name, model, layers, batch, length):
    return {"name": name, "kind": "train", "model": model, "layers": layers,
            "batch": batch, "length": length}


def _trainer(name, model, batch, length):
    return {"name": name, "kind": "trainer", "model": model, "batch": batch,
            "length": length}


# --------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _config(case):
    config = get_config(case["model"])
    if "layers" in case:
        config = dataclasses.replace(config,
                                     num_hidden_layers=case["layers"])
    return config


def _perturb(stage, g):
    """Norm weights and biases as a trained model has them, off 1 and 0."""
    with torch.no_grad():
        for p in stage.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn(p.shape, generator=g,
                                         device=p.device).to(p.dtype))


def _stage(case, ends, seed, g):
    """The stage of ``case``; ``ends``: with embedding and head."""
    config = _config(case)
    with torch.device("cuda"):
        stage = build_stage(config, StageSpec(
            rank=0, layer_start=0, layer_end=config.num_hidden_layers,
            has_embedding=ends, has_head=ends))
    init_random_stage(stage, device="cuda", dtype=torch.bfloat16, seed=seed)
    _perturb(stage, g)
    return stage


def _fill(cache, lens, g):
    """Keys and values of the tokens that a cache already holds."""
    last = int(lens.max())
    for layer in range(len(cache.k)):
        for pool in (cache.k[layer], cache.v[layer]):
            if hasattr(cache, "table"):
                pool.normal_(generator=g)
            else:
                pool[:, :, :last].normal_(generator=g)
    cache.seq_lens.copy_(lens)


def _hidden(stage, batch, length, g):
    """Activations of the stage before. The router of a trained model tells
    experts apart clearly, and some are busier than others."""
    dev = "cuda"
    H = stage.config.hidden_size
    x = torch.randn(batch * length, H, generator=g, device=dev)
    if stage.config.num_local_experts:
        E, k = stage.config.num_local_experts, stage.config.num_experts_per_tok
        use = 1.0 / torch.sqrt(torch.arange(E, device=dev) + 10.0)
        use = use[torch.randperm(E, generator=g, device=dev)]
        idx = torch.multinomial(use.expand(batch * length, E), k, generator=g)
        gate = stage.layers[0].mlp.gate.weight.float()
        gate = gate / stage.layers[0].post_attention_layernorm.float()
        gate = gate / gate.norm(dim=1, keepdim=True)
        for j in range(k):
            x += (8.0 + 0.25 * j) * gate[idx[:, j]]
    return x.view(batch, length, H).to(torch.bfloat16)


def prepare(case, seed):
    g = _gen(seed)
    dev = "cuda"
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "trainer":
        config = _config(case)
        with torch.device(dev):
            s["trainer"] = PipelineTrainer(
                plan_for_world(config, 1, batch_size=case["batch"],
                               seq_len=case["length"]), 0, 1, device=dev,
                dtype=torch.bfloat16, seed=seed, lr=LR, betas=BETAS, eps=EPS,
                weight_decay=DECAY)
        _perturb(s["trainer"].stage, g)
        s["ids"] = torch.randint(0, config.vocab_size,
                                 (case["batch"], case["length"]),
                                 generator=g, device=dev)
        return s
    B = case["batch"]
    stage = s["stage"] = _stage(case, kind in ("decode", "prefill"), seed, g)
    config = stage.config
    if kind == "train":
        stage.train()
        s["opt"] = FusedAdamW(stage.parameters(), lr=LR, betas=BETAS,
                              eps=EPS, weight_decay=DECAY)
        s["x"] = _hidden(stage, B, case["length"], g)
        s["dy"] = torch.randn(s["x"].shape, generator=g, device=dev).to(
            torch.bfloat16) / 64
        s["pos"] = torch.arange(case["length"], device=dev,
                                dtype=torch.int32).expand(B, -1).contiguous()
        return s
    stage.eval()
    if kind == "decode":
        new = 1
        lens = torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (B,),
                             generator=g, device=dev, dtype=torch.int32)
        top = case["ctx_hi"]
    else:
        new = case["length"]
        top = case["start"] if kind == "prefill" else case["ctx"]
        lens = torch.full((B,), top, device=dev, dtype=torch.int32)
    cache = s["cache"] = stage.make_kv_cache(
        B, top + new + 63, torch.device(dev), torch.bfloat16,
        kv_mode="paged" if case.get("paged") else "contiguous")
    if int(lens.max()):
        _fill(cache, lens, g)
    s["lens"] = lens
    s["pos"] = lens.unsqueeze(1) + torch.arange(new, device=dev,
                                                dtype=torch.int32)
    if kind == "moe":
        if case["fp8"]:
            quantize_experts_fp8(stage)
        s["x"] = _hidden(stage, B, new, g)
    else:
        s["x"] = torch.randint(0, config.vocab_size, (B, new), generator=g,
                               device=dev)
    return s


# ----------------------------------------------------------------- passes
def run(s):
    kind = s["kind"]
    if kind == "trainer":
        t = s["trainer"]
        loss = t.train_step(s["ids"], s["ids"])
        o = t.optimizer
        return {"loss": loss, "weights": o.flat_param, "m": o.exp_avg,
                "v": o.exp_avg_sq}
    stage = s["stage"]
    if kind == "train":
        x = s["x"].detach().requires_grad_(True)
        out = stage(x, s["pos"], training=True, return_logits=False)
        out.backward(s["dy"])
        o = s["opt"]
        o.step()
        o.zero_grad()
        return {"out": out.detach(), "dx": x.grad, "weights": o.flat_param,
                "m": o.exp_avg, "v": o.exp_avg_sq}
    cache = s["cache"]
    with torch.no_grad():
        cache.seq_lens.copy_(s["lens"])     # back to before the last pass
        if kind == "decode":
            r = {"logits": stage(s["x"], s["pos"], kv_cache=cache)}
        else:
            r = {"hidden": stage(s["x"], s["pos"], kv_cache=cache,
                                 return_logits=False)}
            if kind == "prefill":           # the first token's logits
                r["logits"] = stage.head(r["hidden"][:, -1:])
    r["k"], r["v"] = cache.k, cache.v
    return r


# ------------------------------------------------------------------- cost
def _weights(config):
    """(weights of a layer's projections that every token needs, of one
    expert)"""
    h = config.hidden_size
    attn = h * (config.q_size + 2 * config.kv_size) + config.q_size * h
    if config.num_local_experts:
        return (attn + h * config.num_local_experts,
                3 * h * config.expert_intermediate_size)
    mats = 2 if config.architecture == "gpt2" else 3
    return attn + mats * h * config.intermediate_size, 0


def work(case):
    config = _config(case)
    kind, B = case["kind"], case["batch"]
    L, H, V = config.num_hidden_layers, config.hidden_size, config.vocab_size
    dense, expert = _weights(config)
    new = case.get("length", 1)
    M = B * new
    if kind in ("train", "trainer"):
        params = L * dense
        pairs = B * new * (new + 1) // 2
        head = H * V if kind == "trainer" else 0
        n = params + head
        flops = 6 * M * n + 12 * L * pairs * config.q_size
        # gradients are written, weights and both moments read and written
        bytes_ = n * (2 + 2 + 4 + 16) + 3 * M * H * 2
        return {"bytes": bytes_, "flops": flops}
    if kind == "decode":
        ctx = (case["ctx_lo"] + case["ctx_hi"]) / 2
    else:
        ctx = case["start"] if kind == "prefill" else case["ctx"]
    pairs = B * (new * ctx + new * (new + 1) / 2)
    flops = 2 * M * L * dense + 4 * L * pairs * config.q_size
    kv = L * B * (ctx + 2 * new) * 2 * config.kv_size * 2
    bytes_ = L * dense * 2 + kv + 2 * M * H * 2
    if kind == "moe":
        E, k = config.num_local_experts, config.num_experts_per_tok
        seen = E * (1 - (1 - k / E) ** M)       # experts with a token
        flops += 2 * M * k * expert * L
        bytes_ += L * seen * expert * (1 if case["fp8"] else 2)
        return {"bytes": bytes_, "flops": flops}
    rows = B                                    # rows with logits
    flops += 2 * rows * H * V
    return {"bytes": bytes_ + H * V * 2 + rows * V * 2, "flops": flops}


def tolerance(case):
    """bf16 activations: against 64 bits the outputs are up to 0.013 off, the
    moments of a whole model's training step up to 0.024, and another order
    of sums lies as far off on its own side. Single values: passes whose
    attention sums ran in another order were up to 0.06 apart, squared
    gradients of a whole model up to 0.31."""
    if case["kind"] == "trainer":
        return {"rel": 0.03, "max": 0.99}
    return {"rel": 0.02, "max": 0.3}


# ------------------------------------------------------- the same in 64 bits
def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, inv):
    """x [B, S, heads, D], pos [B, S]"""
    a = pos.double()[..., None, None] * inv
    u, w = x.chunk(2, -1)
    return torch.cat([u * a.cos() - w * a.sin(),
                      w * a.cos() + u * a.sin()], -1)


def _attend(q, k, v, pos):
    """q [S, Hq, D] at positions pos, k and v [T, Hkv, D] from position 0"""
    S, Hq, D = q.shape
    T, Hkv, _ = k.shape
    out = []
    step = max(1, 400_000_000 // (Hq * T))
    kt = k.permute(1, 2, 0)[:, None]                      # [Hkv, 1, D, T]
    vt = v.transpose(0, 1)[:, None]                       # [Hkv, 1, T, D]
    far = torch.arange(T, device=q.device)
    for i in range(0, S, step):
        qi = q[i:i + step].reshape(-1, Hkv, Hq // Hkv, D).permute(1, 2, 0, 3)
        z = qi @ kt / math.sqrt(D)
        z = z.masked_fill(far > pos[i:i + step, None], -math.inf)
        o = z.softmax(-1) @ vt                            # [Hkv, G, s, D]
        out.append(o.permute(2, 0, 1, 3).reshape(-1, Hq * D))
    return torch.cat(out)


def _attention(config, P, x, pos, old=None):
    """``old(b)``: the keys and values [T, Hkv, D] that sequence b has."""
    B, S, _ = x.shape
    Hq, Hkv, D = (config.num_attention_heads, config.num_key_value_heads,
                  config.head_dim)
    qkv = x @ P["qkv_proj.weight"].t()
    if "qkv_proj.bias" in P:
        qkv = qkv + P["qkv_proj.bias"]
    q, k, v = qkv.split([Hq * D, Hkv * D, Hkv * D], -1)
    q, k, v = (t.reshape(B, S, -1, D) for t in (q, k, v))
    if "q_norm" in P:
        q = _rms(q, P["q_norm"], config.rms_norm_eps)
        k = _rms(k, P["k_norm"], config.rms_norm_eps)
    inv = P["inv_freq"]
    q, k = _rope(q, pos, inv), _rope(k, pos, inv)
    rows = []
    for b in range(B):
        kb, vb = k[b], v[b]
        if old is not None:
            k0, v0 = old(b)
            kb, vb = torch.cat([k0.double(), kb]), torch.cat([v0.double(), vb])
        rows.append(_attend(q[b], kb, vb, pos[b].long()))
    return torch.stack(rows) @ P["o_proj.weight"].t(), k, v


def _gated(x, gate_up, down):
    g, u = (x @ gate_up.t()).chunk(2, -1)
    return (g * torch.sigmoid(g) * u) @ down.t()


def _experts(config, mlp, x):
    z = x @ mlp.gate.weight.double().t()
    w, idx = z.softmax(-1).topk(config.num_experts_per_tok, -1)
    w = w / w.sum(-1, keepdim=True)
    out = torch.zeros_like(x)

    def full(lin):
        if hasattr(lin, "weight_fp8"):
            return lin.weight_fp8.double() * lin.scale.double()[:, None]
        return lin.weight.double()

    for e, m in enumerate(mlp.experts):
        at, slot = (idx == e).nonzero(as_tuple=True)
        if len(at):
            out.index_add_(0, at, w[at, slot, None] * _gated(
                x[at], full(m.gate_up_proj), full(m.down_proj)))
    return out


def _under(P, name):
    return {k[len(name):]: v for k, v in P.items() if k.startswith(name)}


def _layer(config, P, x, pos, old=None, mlp=None):
    eps = config.rms_norm_eps
    y, k, v = _attention(config, _under(P, "self_attn."),
                         _rms(x, P["input_layernorm"], eps), pos, old)
    x = x + y
    h = _rms(x, P["post_attention_layernorm"], eps)
    if mlp is not None:
        y = _experts(config, mlp, h.reshape(-1, h.shape[-1])).view_as(x)
    else:
        y = _gated(h, P["mlp.gate_up_proj.weight"], P["mlp.down_proj.weight"])
    return x + y, k, v


def _norm(x, P, name, eps):
    x = x - x.mean(-1, keepdim=True)
    return _rms(x, P[name + ".weight"], eps) + P[name + ".bias"]


def _gpt2_layer(config, P, x):
    B, S, H = x.shape
    D, eps = config.head_dim, config.rms_norm_eps

    def lin(t, name):
        return t @ P[name + ".weight"].t() + P[name + ".bias"]

    h = _norm(x, P, "ln_1", eps)
    q, k, v = (t.reshape(B, S, -1, D)
               for t in lin(h, "attn.c_attn").chunk(3, -1))
    pos = torch.arange(S, device=x.device)
    a = torch.stack([_attend(q[b], k[b], v[b], pos) for b in range(B)])
    x = x + lin(a, "attn.c_proj")
    u = lin(_norm(x, P, "ln_2", eps), "c_fc")
    u = 0.5 * u * (1 + torch.tanh(math.sqrt(2 / math.pi)
                                  * (u + 0.044715 * u ** 3)))
    return x + lin(u, "c_proj")


def _updated(named):
    """The flat weights and moments after a first AdamW step."""
    w = torch.cat([p.detach().reshape(-1) for p in named])
    g = torch.cat([(torch.zeros_like(p) if p.grad is None else p.grad)
                   .reshape(-1) for p in named])
    w = w * (1 - LR * DECAY) - LR * g / (g.abs() + EPS)
    return w, (1 - BETAS[0]) * g, (1 - BETAS[1]) * g * g


def _layers_of(P, stage):
    """Each layer's tensors; its rotation frequencies as the stage has them,
    which holds them in its own data type."""
    out = []
    for i, layer in enumerate(stage.layers):
        p = _under(P, "layers.%d." % i)
        if hasattr(layer, "self_attn"):
            p["self_attn.inv_freq"] = layer.self_attn.inv_freq.double()
        out.append(p)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("train", "trainer"):
        return _exact_training(case, s)
    stage, cache, config = s["stage"], s["cache"], s["stage"].config
    lens, pos = s["lens"].tolist(), s["pos"]
    table = getattr(cache, "table", None)
    with torch.no_grad():
        P = {n: p for n, p in stage.named_parameters() if ".experts." not in n}
        x = s["x"]
        x = x.double() if kind == "moe" else P["embed_tokens.weight"][
            x].double()
        r = {"k": [], "v": []}
        for i, p in enumerate(_layers_of(P, stage)):
            p = {n: t.double() for n, t in p.items()}
            pools = [c[i].double() for c in (cache.k, cache.v)]

            def old(b):
                if table is None:
                    return [c[b, :, :lens[b]].transpose(0, 1) for c in pools]
                got = (c[table[b].long()].transpose(1, 2).flatten(0, 1)
                       for c in pools)
                return [c[:lens[b]] for c in got]

            x, *new = _layer(config, p, x, pos, old,
                             stage.layers[i].mlp if kind == "moe" else None)
            for name, pool, t in zip("kv", pools, new):
                for b in range(case["batch"]):
                    at = pos[b].long()
                    if table is None:
                        pool[b][:, at] = t[b].transpose(0, 1)
                    else:
                        pool[table[b].long()[at // PAGE], :, at % PAGE] = t[b]
                r[name].append(pool)
        if kind == "decode":
            r["logits"] = _logits(config, P, x)
        else:
            r["hidden"] = x
            if kind == "prefill":
                r["logits"] = _logits(config, P, x[:, -1:])
    return r


def _logits(config, P, x):
    h = _rms(x, P["norm"].double(), config.rms_norm_eps)
    return torch.cat([h @ w.double().t()
                      for w in P["lm_head.weight"].split(16384)], -1)


def _exact_training(case, s):
    trainer = case["kind"] == "trainer"
    stage = s["trainer"].stage if trainer else s["stage"]
    config = stage.config
    P = {n: p.detach().double().requires_grad_(True)
         for n, p in stage.named_parameters()}
    eps = config.rms_norm_eps
    if not trainer:
        x = x0 = s["x"].double().requires_grad_(True)
        for p in _layers_of(P, stage):
            x, _, _ = _layer(config, p, x, s["pos"])
        x.backward(s["dy"].double())
        w, m, v = _updated(list(P.values()))
        return {"out": x.detach(), "dx": x0.grad, "weights": w, "m": m,
                "v": v}
    ids = s["ids"]
    B, S = ids.shape
    if config.architecture == "gpt2":
        x = P["wte.weight"][ids] + P["wpe.weight"][:S]
        for p in _layers_of(P, stage):
            x = _gpt2_layer(config, p, x)
        z = _norm(x, P, "ln_f", eps) @ P["wte.weight"].t()
    else:
        pos = torch.arange(S, device="cuda").expand(B, -1)
        x = P["embed_tokens.weight"][ids]
        for p in _layers_of(P, stage):
            x, _, _ = _layer(config, p, x, pos)
        z = _rms(x, P["norm"], eps) @ P["lm_head.weight"].t()
    loss = torch.nn.functional.cross_entropy(
        z[:, :-1].reshape(-1, z.shape[-1]), ids[:, 1:].reshape(-1))
    loss.backward()
    w, m, v = _updated(list(P.values()))
    return {"loss": loss.detach(), "weights": w, "m": m, "v": v}
