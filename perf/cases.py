"""The calls of this framework whose speed is followed, as its users make them.

A case is one pass of one public entry point, in the direction(s) a training
program runs it: the checkpointed decoder layer (forward, then backward with its
recompute) through ``ActivationCheckpointWrapper`` and ``fused_checkpoint``; the
parts that selective checkpointing leaves (``fuse_attention``'s attention, the
checkpointed MLP and RMSNorm); the loss head, the token embedding, the optimizer
step; and one whole model step.  Widths are those of the repository's
configurations (tests/helpers.py): "debug" (hidden 256, fp32), "tinyllama",
"llama3-8b" and "llama2-7b"; token counts run from one short sequence to the
longest configured one, most of them not multiples of anything.

Weights are N(0, 0.02) (norm weights 1 + N(0, 0.02)) and packed once, as
``pack_layer_weights`` does for a user; activations are N(0, 1); gradients coming
in are N(0, 0.01); token ids are Zipf-distributed like text, or uniform.
"""
from __future__ import annotations

import math
import types

import torch
import torch.nn.functional as F
from torch import nn
from transformers import LlamaConfig
from transformers.models.llama.modeling_llama import (LlamaDecoderLayer, LlamaRMSNorm,
                                                      LlamaRotaryEmbedding)

from femtotron_amd import fuse_attention, fuse_boundary_ops, fused_checkpoint, pack_layer_weights
from femtotron_amd.boundary_ops import FusedEmbedding
from femtotron_amd.fused_loss import fused_causal_lm_loss
from femtotron_amd.model import build_llama_model, init_llama_weights_
from femtotron_amd.optim import FusedAdamW, get_param_groups
from femtotron_amd.scripts.presets import get_ac_policy
from femtotron_amd.training import ActivationCheckpointWrapper, apply_activation_checkpointing

DEV = "cuda"
EPS = 1e-5
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}

WIDTHS = {
    "debug": dict(hidden=256, heads=8, kv=4, ffn=688, vocab=1024, theta=1e4),
    "tinyllama": dict(hidden=2048, heads=32, kv=4, ffn=5632, vocab=32000, theta=1e4),
    "llama3-8b": dict(hidden=4096, heads=32, kv=8, ffn=14336, vocab=128256, theta=5e5),
    "llama2-7b": dict(hidden=4096, heads=32, kv=32, ffn=11008, vocab=32000, theta=1e4),
}


def _case(kind, width, batch, seq, dtype="bf16", **more):
    return dict(kind=kind, batch=batch, seq=seq, dtype=dtype, **WIDTHS[width], **more)


def listed():
    return [
        # The smallest: a step of the two-layer fp32 debug model, where launches and host work are the time.
        dict(name="model_debug_fp32", **_case("model", "debug", 2, 128, "fp32", layers=2)),
        # An fp32 layer at real widths on one short sequence: parity and debugging runs.
        dict(name="layer_fp32", **_case("layer", "tinyllama", 1, 512, "fp32", grads="new")),
        # One short sequence (fine-tuning samples, tests): too few output tiles to fill the chip.
        dict(name="layer_short", **_case("layer", "tinyllama", 1, 256, grads="new")),
        # A ragged batch, its token count odd: variable-length training data, the last batch of an epoch.
        dict(name="layer_ragged", **_case("layer", "tinyllama", 3, 333, grads="new")),
        # The configured TinyLlama training step's layer, its gradients kept and accumulated into.
        dict(name="layer_train", **_case("layer", "tinyllama", 8, 2048, grads="kept")),
        # The 8B-wide layer at its configured 8192 tokens (head_dim 128, grouped kv heads).
        dict(name="layer_8b", **_case("layer", "llama3-8b", 1, 8192, grads="new")),
        # The largest: selective checkpointing's attention at the long-context configuration.
        dict(name="attn_long", **_case("attn", "llama2-7b", 1, 32768, grads="new")),
        # Selective checkpointing's MLP on a mid-sized ragged batch.
        dict(name="mlp_ragged", **_case("mlp", "llama3-8b", 2, 1001, grads="new")),
        # Selective checkpointing's (and the model's final) RMSNorm at the training step's size.
        dict(name="norm_train", **_case("norm", "tinyllama", 8, 2048)),
        # The loss head of the training step without materialised logits.
        dict(name="loss_train", **_case("loss", "tinyllama", 8, 2048)),
        # The token embedding of the training step on text-like ids.
        dict(name="embed_train", **_case("embed", "tinyllama", 8, 2048, ids="zipf")),
        # The optimizer step over one TinyLlama layer's parameters, with clipping.
        dict(name="adamw", **_case("adamw", "tinyllama", 1, 1)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer32", "attn", "attn", "mlp", "norm", "loss", "embed", "adamw",
                       "model"])
    if kind == "layer32":  # fp32: debugging sizes
        return _case("layer", rng.choice(["debug", "tinyllama"]), rng.randint(1, 2), _log_int(rng, 16, 512), "fp32",
                     grads=rng.choice(["new", "kept"]))
    if kind == "model":
        return _case("model", "debug", rng.randint(1, 4), _log_int(rng, 16, 300), rng.choice(["fp32", "bf16"]),
                     layers=rng.randint(1, 3))
    if kind == "adamw":
        return _case("adamw", rng.choice(["debug", "tinyllama", "llama3-8b"]), 1, 1, rng.choice(["bf16", "fp32"]))
    width = rng.choice(["debug", "tinyllama", "tinyllama", "llama3-8b", "llama2-7b"])
    batch = rng.choice([1, 1, 2, 3, 4, 8])
    most = 16384 if width in ("debug", "tinyllama") else 8192
    seq = _log_int(rng, 16, most // batch)
    if rng.random() < 0.3:  # the configured lengths are powers of two
        seq = 1 << (seq.bit_length() - 1)
    dtype = "fp32" if kind in ("norm", "embed") and rng.random() < 0.3 else "bf16"
    more = {}
    if kind in ("layer", "attn", "mlp"):
        more["grads"] = rng.choice(["new", "kept"])
    if kind == "embed":
        more["ids"] = rng.choice(["zipf", "uniform"])
        if width == "llama3-8b":
            width = "tinyllama"
    if kind == "loss" and width == "llama3-8b":
        width = "llama2-7b"
    return _case(kind, width, batch, seq, dtype, **more)


# ------------------------------------------------------------------ prepare
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _config(c, layers=1):
    cfg = LlamaConfig(hidden_size=c["hidden"], intermediate_size=c["ffn"], num_attention_heads=c["heads"],
                      num_key_value_heads=c["kv"], num_hidden_layers=layers, vocab_size=c["vocab"], rms_norm_eps=EPS,
                      hidden_act="silu", max_position_embeddings=max(2048, c["seq"]), tie_word_embeddings=False,
                      rope_theta=c["theta"], attention_dropout=0.0)
    cfg._attn_implementation = "sdpa"
    return cfg


def _fill(mod, g):
    """Every parameter ~ N(0, 0.02), norm weights 1 + N(0, 0.02)."""
    with torch.no_grad():
        for p in mod.parameters():
            p.normal_(0.0, 0.02, generator=g)
            if p.dim() == 1:
                p.add_(1.0)


def _make_layer(c, g):
    with torch.device("meta"):
        layer = LlamaDecoderLayer(_config(c), 0)
    layer = layer.to_empty(device=DEV).to(DTYPES[c["dtype"]])
    _fill(layer, g)
    pack_layer_weights(layer)
    layer.train()
    return layer


def _rope(c):
    """cos, sin [1, S, head_dim] as the model's rotary module gives them."""
    rot = LlamaRotaryEmbedding(config=_config(c)).to(DEV)
    pos = torch.arange(c["seq"], device=DEV).unsqueeze(0)
    return rot(torch.empty(1, device=DEV, dtype=DTYPES[c["dtype"]]), position_ids=pos)


def _ids(c, g):
    shape, V = (c["batch"], c["seq"]), c["vocab"]
    if c.get("ids", "uniform") == "uniform":
        return torch.randint(0, V, shape, generator=g, device=DEV)
    # Zipf's law: P(rank r) ~ 1/r, ranks scattered over the vocabulary
    u = torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)
    rank = torch.exp(u * math.log(V + 1.0)).long().clamp_(1, V) - 1
    return torch.randperm(V, generator=g, device=DEV)[rank]


def _inputs(c, seed):
    """Everything that both run() and exact() start from."""
    g = _gen(seed)
    dt = DTYPES[c["dtype"]]
    kind, B, S, H = c["kind"], c["batch"], c["seq"], c["hidden"]
    s = types.SimpleNamespace(case=c)
    if kind in ("layer", "attn", "mlp"):
        s.layer = _make_layer(c, g)
        s.cos, s.sin = _rope(c)
    if kind in ("layer", "attn", "mlp", "norm"):
        s.x = _randn(g, B, S, H, dtype=dt)
        s.dy = _randn(g, B, S, H, dtype=dt, std=0.01)
    if kind == "norm":
        s.norm = LlamaRMSNorm(H, eps=EPS).to(DEV, dt)
        _fill(s.norm, g)
    if kind == "loss":
        s.x = _randn(g, B, S, H, dtype=dt)
        s.weight = nn.Parameter(_randn(g, c["vocab"], H, dtype=dt, std=0.02))
        s.labels = _ids(c, g)
    if kind == "embed":
        s.weight = nn.Parameter(_randn(g, c["vocab"], H, dtype=dt, std=0.02))
        s.ids = _ids(c, g)
        s.dy = _randn(g, B, S, H, dtype=dt, std=0.01)
    if kind == "adamw":
        s.layer = _make_layer(c, g)
        for p in s.layer.parameters():
            p.grad = _randn(g, *p.shape, dtype=dt, std=0.01)
    if kind == "model":
        s.model = init_llama_weights_(build_llama_model(_config(c, c["layers"])), device=DEV, dtype=dt, seed=seed,
                                      generator_device="cuda")
        _fill(s.model, g)
        s.ids = _ids(c, g)
    return s


def _zero_grads(params):
    for p in params:
        p.grad = torch.zeros_like(p)


def _pack_grads(mod):
    """Gradients as a first backward leaves them: q/k/v and gate/up row blocks of one buffer."""
    a, m = mod.self_attn, mod.mlp
    for group in ((a.q_proj, a.k_proj, a.v_proj), (m.gate_proj, m.up_proj)):
        ws = [q.weight for q in group]
        buf = torch.zeros(sum(w.shape[0] for w in ws), ws[0].shape[1], dtype=ws[0].dtype, device=DEV)
        for w, part in zip(ws, buf.split([w.shape[0] for w in ws])):
            w.grad = part


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "layer":
        s.call = ActivationCheckpointWrapper(s.layer, checkpoint_fn=fused_checkpoint)
        s.params = dict(s.layer.named_parameters())
    elif kind == "attn":
        fuse_attention(s.layer)
        s.call = s.layer.self_attn
        s.params = dict(s.call.named_parameters())
    elif kind == "mlp":
        s.call = ActivationCheckpointWrapper(s.layer.mlp, checkpoint_fn=fused_checkpoint)
        s.params = dict(s.layer.mlp.named_parameters())
    elif kind == "norm":
        s.call = ActivationCheckpointWrapper(s.norm, checkpoint_fn=fused_checkpoint)
        s.params = dict(s.norm.named_parameters())
    elif kind == "loss":
        s.params = {"weight": s.weight}
    elif kind == "embed":
        s.call = FusedEmbedding(s.weight)
        s.params = {"weight": s.weight}
    elif kind == "adamw":
        s.opt = FusedAdamW(get_param_groups(s.layer, 0.1), lr=3e-4, max_grad_norm=1.0)
    elif kind == "model":
        pack_layer_weights(s.model)
        fuse_boundary_ops(s.model)
        apply_activation_checkpointing(s.model, get_ac_policy("llama_decoder_layer"), checkpoint_fn=fused_checkpoint)
        s.params = dict(s.model.named_parameters())
    if kind in ("layer", "attn", "mlp", "norm", "loss"):
        s.x.requires_grad_(True)
    s.kept = case.get("grads") == "kept"
    if s.kept:  # a training loop's gradient buffers, zeroed in place at every step
        _zero_grads(s.params.values())
        _pack_grads(s.layer)
        s.bufs = [p.grad for p in s.params.values()]
    return s


# ---------------------------------------------------------------------- run
def _start_step(s):
    if s.kept:
        torch._foreach_zero_(s.bufs)
    else:
        for p in s.params.values():
            p.grad = None
    if getattr(s, "x", None) is not None:
        s.x.grad = None


def run(s):
    kind = s.case["kind"]
    if kind == "adamw":
        s.opt.step()
        return {"norm": s.opt.grad_norm, "params": [e[0].detach() for e in s.opt.entries],
                "master": [e[2] for e in s.opt.entries], "m": [e[3] for e in s.opt.entries],
                "v": [e[4] for e in s.opt.entries]}
    _start_step(s)
    if kind == "model":
        out = s.model(s.ids, labels=s.ids)
        out["loss"].backward()
        return {"logits": out["logits"].detach(), "loss": out["loss"].detach(), "grads": _grads(s)}
    if kind == "loss":
        out = fused_causal_lm_loss(s.x, s.weight, s.labels)
        out.backward()
        return {"out": out.detach(), "dx": s.x.grad, "grads": _grads(s)}
    if kind == "embed":
        out = s.call(s.ids)
        out.backward(s.dy)
        return {"out": out.detach(), "grads": _grads(s)}
    if kind == "layer":
        out = s.call(s.x, attention_mask=None, position_embeddings=(s.cos, s.sin), past_key_values=None,
                     use_cache=False)
    elif kind == "attn":
        out, _ = s.call(hidden_states=s.x, position_embeddings=(s.cos, s.sin), attention_mask=None)
    else:
        out = s.call(s.x)
    out.backward(s.dy)
    return {"out": out.detach(), "dx": s.x.grad, "grads": _grads(s)}


def _name(n):
    return n.replace("_checkpoint_wrapped_module.", "")


def _grads(s):
    return {_name(n): p.grad for n, p in s.params.items()}


# --------------------------------------------------------------------- work
def _layer_params(c):
    H, hd = c["hidden"], c["hidden"] // c["heads"]
    attn = H * (H + 2 * c["kv"] * hd) + H * H
    return attn, 3 * H * c["ffn"]


def work(case):
    """One pass's products (multiply-adds as two) and, read or written once, its inputs and outputs.  The
    checkpointed layer and MLP store their input only, so the recompute (which needs no down projection)
    belongs to the path."""
    c, kind = case, case["kind"]
    e = 2 if c["dtype"] == "bf16" else 4
    B, S, H, V = c["batch"], c["seq"], c["hidden"], c["vocab"]
    T = B * S
    attn_p, mlp_p = _layer_params(c)
    down_p = H * c["ffn"]
    score = 4 * B * (S * S / 2) * H  # causal q k^T and p v of one forward
    layer_flops = 2 * T * (4 * (attn_p + mlp_p) - down_p) + (2 + 2.5) * score
    act = T * H * e
    if kind == "layer":
        return {"flops": layer_flops, "bytes": 2 * (attn_p + mlp_p + 2 * H) * e + 4 * act}
    if kind == "attn":
        return {"flops": 2 * T * 3 * attn_p + (1 + 2.5) * score, "bytes": 2 * attn_p * e + 4 * act}
    if kind == "mlp":
        return {"flops": 2 * T * (4 * mlp_p - down_p), "bytes": 2 * mlp_p * e + 4 * act}
    if kind == "norm":
        return {"flops": 0, "bytes": 4 * act + 2 * H * e}
    if kind == "loss":
        return {"flops": 2 * T * 3 * V * H, "bytes": 2 * V * H * e + 2 * act + 8 * T}
    if kind == "embed":
        return {"flops": 0, "bytes": 3 * act + V * H * e + 16 * T}
    if kind == "adamw":
        return {"flops": 0, "bytes": (attn_p + mlp_p + 2 * H) * (24 + 2 * e)}
    n = c["layers"] * (attn_p + mlp_p + 2 * H) + 2 * V * H + H  # model
    return {"flops": c["layers"] * layer_flops + 2 * T * 3 * V * H, "bytes": 2 * n * e + T * V * e + 16 * T}


# About four times the largest relative error of an output against exact(): bf16 layers 0.9-1.3e-2 (a rounding
# that falls the other way travels through every later step of the layer; 0.03 is the most this file allows),
# attention 0.85e-2, the MLP 0.39e-2, the norm 0.23e-2, the loss head 0.17e-2, the embedding's gradient 0.15e-2,
# the optimizer's bf16 parameters 0.19e-2; fp32 layers 2.7e-6, the debug model 1.3e-6, the others below 2e-7.
TOLERANCE = {
    "bf16": dict(layer=0.03, model=0.03, attn=0.03, mlp=0.016, norm=0.01, loss=0.007, embed=0.006, adamw=0.0075),
    "fp32": dict(layer=1e-5, model=6e-6, norm=1e-6, embed=1e-6, adamw=1e-6),
}


def tolerance(case):
    return {"rel": TOLERANCE[case["dtype"]][case["kind"]]}


# -------------------------------------------------------------------- exact
class _Attention64(torch.autograd.Function):
    """Causal attention of one head in float64, a block of queries at a time: q, k, v [S, hd]."""

    ROWS = 4096

    @staticmethod
    def _blocks(q, k, scale):
        S = q.shape[0]
        for r0 in range(0, S, _Attention64.ROWS):
            r1 = min(S, r0 + _Attention64.ROWS)
            x = torch.mm(q[r0:r1], k[:r1].t().contiguous()).mul_(scale)
            x.masked_fill_(torch.ones(r1 - r0, r1, dtype=torch.bool, device=x.device).triu_(r0 + 1), -math.inf)
            yield r0, r1, torch.softmax(x, -1)

    @staticmethod
    def forward(ctx, q, k, v, scale):
        ctx.save_for_backward(q, k, v)
        ctx.scale = scale
        return torch.cat([torch.mm(p, v[:r1]) for _, r1, p in _Attention64._blocks(q, k, scale)])

    @staticmethod
    def backward(ctx, do):
        q, k, v = ctx.saved_tensors
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
        do = do.contiguous()
        for r0, r1, p in _Attention64._blocks(q, k, ctx.scale):
            g = do[r0:r1]
            dv[:r1] += torch.mm(p.t().contiguous(), g)
            dp = torch.mm(g, v[:r1].t().contiguous())
            ds = p.mul_(dp.sub_((dp * p).sum(-1, keepdim=True))).mul_(ctx.scale)
            dq[r0:r1] = torch.mm(ds, k[:r1])
            dk[:r1] += torch.mm(ds.t().contiguous(), q[r0:r1])
        return dq, dk, dv, None


def _norm64(x, w):
    return w * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS))


def _rotate64(x, cos, sin):
    h = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., h:], x[..., :h]), -1) * sin


def _attn64(c, w, y, cos, sin, pre):
    B, S, H = y.shape
    nh, kv, hd = c["heads"], c["kv"], H // c["heads"]
    q, k, v = (F.linear(y, w[pre + n + "_proj.weight"]).view(B, S, -1, hd) for n in "qkv")
    q, k = _rotate64(q, cos.unsqueeze(2), sin.unsqueeze(2)), _rotate64(k, cos.unsqueeze(2), sin.unsqueeze(2))
    o = [torch.stack([_Attention64.apply(q[b, :, h].contiguous(), k[b, :, h * kv // nh].contiguous(),
                                         v[b, :, h * kv // nh].contiguous(), hd ** -0.5) for h in range(nh)], 1)
         for b in range(B)]
    return F.linear(torch.stack(o).reshape(B, S, H), w[pre + "o_proj.weight"])


def _mlp64(w, z, pre):
    p = F.silu(F.linear(z, w[pre + "gate_proj.weight"])) * F.linear(z, w[pre + "up_proj.weight"])
    return F.linear(p, w[pre + "down_proj.weight"])


def _layer64(c, w, x, cos, sin, pre=""):
    h = x + _attn64(c, w, _norm64(x, w[pre + "input_layernorm.weight"]), cos, sin, pre + "self_attn.")
    return h + _mlp64(w, _norm64(h, w[pre + "post_attention_layernorm.weight"]), pre + "mlp.")


def _next_token_loss64(logits, labels):
    V = logits.shape[-1]
    return F.cross_entropy(logits[:, :-1].reshape(-1, V), labels[:, 1:].reshape(-1))


def exact(case, seed):
    """run()'s results for the same inputs, computed in float64 by plain torch."""
    c, kind = case, case["kind"]
    s = _inputs(case, seed)
    if kind == "adamw":
        return _adamw64(s)
    mod = {"layer": lambda: s.layer, "attn": lambda: s.layer.self_attn, "mlp": lambda: s.layer.mlp,
           "norm": lambda: s.norm, "model": lambda: s.model}.get(kind)
    if mod is None:
        w = {"weight": s.weight}
    else:
        w = dict(mod().named_parameters())
    w = {n: p.detach().double().requires_grad_(True) for n, p in w.items()}
    x = s.x.detach().double().requires_grad_(True) if hasattr(s, "x") else None
    if kind == "model":
        cos, sin = (t.double() for t in _rope(c))
        h = F.embedding(s.ids, w["model.embed_tokens.weight"])
        for i in range(c["layers"]):
            h = _layer64(c, w, h, cos, sin, "model.layers.%d." % i)
        logits = F.linear(_norm64(h, w["model.norm.weight"]), w["lm_head.weight"])
        loss = _next_token_loss64(logits, s.ids)
        loss.backward()
        return {"logits": logits.detach(), "loss": loss.detach(), "grads": {n: p.grad for n, p in w.items()}}
    if kind == "loss":
        out = _next_token_loss64(F.linear(x, w["weight"]), s.labels)
        out.backward()
    elif kind == "embed":
        out = F.embedding(s.ids, w["weight"])
        out.backward(s.dy.double())
        return {"out": out.detach(), "grads": {"weight": w["weight"].grad}}
    else:
        if kind == "layer":
            out = _layer64(c, w, x, s.cos.double(), s.sin.double())
        elif kind == "attn":
            out = _attn64(c, w, x, s.cos.double(), s.sin.double(), "")
        elif kind == "mlp":
            out = _mlp64(w, x, "")
        else:
            out = _norm64(x, w["weight"])
        out.backward(s.dy.double())
    return {"out": out.detach(), "dx": x.grad, "grads": {n: p.grad for n, p in w.items()}}


def _adamw64(s):
    lr, b1, b2, eps, max_norm = 3e-4, 0.9, 0.95, 1e-8, 1.0
    groups = get_param_groups(s.layer, 0.1)
    ps = [(p.detach().double(), p.grad.double(), g["weight_decay"]) for g in groups for p in g["params"]]
    norm = torch.sqrt(sum(g.pow(2).sum() for _, g, _ in ps))
    coef = torch.clamp(max_norm / (norm + 1e-6), max=1.0)
    master, first, second = [], [], []
    for p, g, wd in ps:
        g = g * coef
        m = (1 - b1) * g
        v = (1 - b2) * g * g
        master.append(p * (1 - lr * wd) - lr / (1 - b1) * m / (v.sqrt() / math.sqrt(1 - b2) + eps))
        first.append(m)
        second.append(v)
    return {"norm": norm, "params": master, "master": master, "m": first, "v": second}
