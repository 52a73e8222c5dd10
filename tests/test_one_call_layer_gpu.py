"""The decoder layer as one call per direction (fh_layer_fwd / fh_layer_bwd) against the same layer run op by op
(femtotron_amd/fused_layer.py's layer_forward / layer_backward, checked elsewhere against the oracle): the same
launches in the same order, so the same bits in bf16; in fp32 other products (fh_gemm_f32 throughout)."""
from __future__ import annotations

import pytest
import torch
from transformers.models.llama.modeling_llama import LlamaDecoderLayer

from femtotron_amd import fused_checkpoint, fused_layer, pack_layer_weights
from femtotron_amd.training import ActivationCheckpointWrapper
from oracle import torch_llama as ot
from tests.helpers import CFG1, CFG3, hf_layer_grads, layer_weights, llama_config, load_into_hf_layer, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(c, B, S, dtype, packed, per_token, passes):
    hd = c["hidden"] // c["heads"]
    layer = LlamaDecoderLayer(llama_config(c, layers=1), 0)
    load_into_hf_layer(layer, layer_weights(c, seed=5, norm_mean=1.0))
    layer = layer.to(DEV, dtype)
    if packed:
        pack_layer_weights(layer)
    cos, sin = (t.to(DEV) for t in ot.rope_cos_sin(S, hd, c["theta"], dtype))
    if per_token:
        cos, sin = cos.expand(B, S, hd).contiguous(), sin.expand(B, S, hd).contiguous()
    wrapped = ActivationCheckpointWrapper(layer, checkpoint_fn=fused_checkpoint)
    outs = []
    for i in range(passes):  # later passes accumulate into the gradients of the first
        x = randn((B, S, c["hidden"]), 7 + i).to(DEV, dtype).requires_grad_(True)
        dy = randn((B, S, c["hidden"]), 17 + i).to(DEV, dtype)
        out = wrapped(x, attention_mask=None, position_embeddings=(cos, sin), past_key_values=None, use_cache=False)
        out.backward(dy)
        outs += [out.detach(), x.grad]
    return outs + [g.clone() for g in hf_layer_grads(layer).values()]


def _count_calls(monkeypatch):
    calls = []
    for name in ("layer_fwd", "layer_bwd"):
        fn = getattr(fused_layer.ops, name)
        monkeypatch.setattr(fused_layer.ops, name, lambda *a, _f=fn, _n=name: (calls.append(_n), _f(*a))[1])
    return calls


@pytest.mark.parametrize("packed", [True, False], ids=["packed", "unpacked"])
@pytest.mark.parametrize("c,B,S,per_token", [(CFG3, 1, 64, False), (CFG3, 3, 333, True), (CFG1, 2, 128, False),
                                             (CFG1, 1, 65, False), (CFG1, 5, 700, True)])
def test_one_call_bf16_is_the_op_by_op_layer_bitwise(monkeypatch, c, B, S, per_token, packed):
    calls = _count_calls(monkeypatch)
    got = _run(c, B, S, torch.bfloat16, packed, per_token, 2)
    assert calls == ["layer_fwd", "layer_bwd"] * 2
    monkeypatch.setattr(fused_layer, "ONE_CALL_MAX_BYTES", 0)
    want = _run(c, B, S, torch.bfloat16, packed, per_token, 2)
    assert calls == ["layer_fwd", "layer_bwd"] * 2
    for a, b in zip(got, want):
        assert torch.equal(a, b)


# S = 2 is the least: the softmax over one key has no gradient, so at S = 1 dq and dk are what rounding leaves of
# dP - delta (two orders of one 64-term dot product: up to 64 * 2^-24 of it), and nothing bounds their relative error.
@pytest.mark.parametrize("B,S", [(1, 2), (2, 128), (1, 37)])
def test_one_call_fp32_matches_the_op_by_op_layer(monkeypatch, B, S):
    calls = _count_calls(monkeypatch)
    got = _run(CFG1, B, S, torch.float32, True, False, 1)
    assert calls == ["layer_fwd", "layer_bwd"]
    monkeypatch.setattr(fused_layer, "ONE_CALL_MAX_BYTES", 0)
    for a, b in zip(got, _run(CFG1, B, S, torch.float32, True, False, 1)):
        # two fp32 orders of sums of at most 688 terms through the layer's five products
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max()) + 1e-9


def test_one_call_is_left_to_the_settings_it_implements(monkeypatch):
    from femtotron_amd import projections
    calls = _count_calls(monkeypatch)
    _run(CFG1, 1, 48, torch.bfloat16, True, False, 1)  # fewer tokens than a weight gradient's least k
    for on, off in ((lambda: projections.set_gemm_policy("library"), lambda: projections.set_gemm_policy("hand")),
                    (lambda: fused_layer.set_wgrad_side_stream(True), lambda: fused_layer.set_wgrad_side_stream(False))):
        on()
        try:
            _run(CFG1, 2, 128, torch.bfloat16, True, False, 1)
        finally:
            off()
    assert calls == []


def _operands(c, B, S):
    hd = c["hidden"] // c["heads"]
    layer = LlamaDecoderLayer(llama_config(c, layers=1), 0)
    load_into_hf_layer(layer, layer_weights(c, seed=5, norm_mean=1.0))
    layer = layer.to(DEV, torch.bfloat16)
    pack_layer_weights(layer)
    cos, sin = (t.to(DEV) for t in ot.rope_cos_sin(S, hd, c["theta"], torch.bfloat16))
    x = randn((B, S, c["hidden"]), 7).to(DEV, torch.bfloat16)
    w = tuple(p.detach() for p in (layer.self_attn.q_proj.weight, layer.self_attn.k_proj.weight,
                                   layer.self_attn.v_proj.weight, layer.self_attn.o_proj.weight,
                                   layer.mlp.gate_proj.weight, layer.mlp.up_proj.weight, layer.mlp.down_proj.weight,
                                   layer.input_layernorm.weight, layer.post_attention_layernorm.weight))
    shp = fused_layer.LayerShape(c["hidden"], c["heads"], c["kv"], hd, c["ffn"], 1e-5, 1e-5, hd ** -0.5)
    return x, cos, sin, shp, w


def test_operands_that_the_call_does_not_take():
    x, cos, sin, shp, w = _operands(CFG1, 1, 128)

    def moved(t, shift):  # t's values at an address `shift` elements past an aligned one
        return torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)[shift:shift + t.numel()].view(t.shape).copy_(t)

    call = fused_layer._one_call
    assert call(x, cos, sin, shp, w) is not None and call(x, cos, sin, shp, w, x) is not None
    assert call(moved(x, 1), cos, sin, shp, w) is None and call(x, cos, sin, shp, w, moved(x, 1)) is None
    assert call(x, cos, sin, shp, w, x.float()) is None
    for i in (3, 6, 7):  # wo, wd, w1
        for bad in (moved(w[i], 1), w[i].float(), w[i].cpu(), w[i].t().contiguous().t() if w[i].dim() == 2 else w[i][:-8]):
            assert call(x, cos, sin, shp, (*w[:i], bad, *w[i + 1:])) is None


def test_one_call_replays_in_a_graph():
    """Captured and replayed, with eager work in between: every replay gives the eager bits."""
    x, cos, sin, shp, w = _operands(CFG3, 1, 256)

    def step():
        args, nbytes, alive = fused_layer._one_call(x, cos, sin, shp, w)
        y = fused_layer.ops.layer_fwd(args, nbytes, x)
        bwd = fused_layer._one_call(x, cos, sin, shp, w, y)
        dx, dws = fused_layer._one_call_backward(bwd, x, y, shp, w)
        return [y, dx, *dws]

    want = [t.clone() for t in step()]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        step()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
