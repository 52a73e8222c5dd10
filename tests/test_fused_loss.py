"""Fused lm_head + chunked cross-entropy (femtotron_amd/fused_loss.py, fh_ce_fwd_bwd).

Checkers: the reference's loss head itself (femtotron/model/llama.py:91-111:
shifted logits, .float(), F.cross_entropy with ignore_index -100) in fp64 on
the CPU for the label shift and the kernel's per-row losses and gradients; the
CPU fp32 oracle model (config 1, 1e-5) end to end; the stock loss head of the
same model on the GPU (bf16, the north star's tensor-level metric).
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from femtotron_amd.fused_loss import IGNORE_INDEX, shift_labels
from tests.helpers import BF16_ATOL, BF16_RTOL, CFG1, CFG3, llama_config, rel_err

DEV = "cuda:0"


def _labels(B, S, V, seed, ignore_frac=0.1):
    g = torch.Generator().manual_seed(seed)
    lab = torch.randint(0, V, (B, S), generator=g)
    lab[torch.rand(B, S, generator=g) < ignore_frac] = IGNORE_INDEX
    return lab


def test_label_shift_pairs_like_the_reference():
    """CE over all rows with shifted labels == the reference's CE over shifted
    logits (same pairs, same valid count), loss and gradient, fp64."""
    B, S, V = 3, 17, 50
    logits = torch.randn(B, S, V, dtype=torch.float64, generator=torch.Generator().manual_seed(1))
    labels = _labels(B, S, V, 2)
    a = logits.clone().requires_grad_(True)
    ref = F.cross_entropy(a[..., :-1, :].reshape(-1, V), labels[..., 1:].reshape(-1), ignore_index=-100)
    ref.backward()
    b = logits.clone().requires_grad_(True)
    got = F.cross_entropy(b.reshape(-1, V), shift_labels(labels), ignore_index=-100)
    got.backward()
    assert torch.allclose(got, ref, rtol=1e-14, atol=0)
    assert torch.allclose(b.grad, a.grad, rtol=1e-12, atol=1e-16)


def test_materialize_flag_keeps_reference_behaviour_off_device():
    from femtotron_amd.model import build_llama_model, init_llama_weights_
    model = init_llama_weights_(build_llama_model(llama_config(CFG1)), device="cpu", dtype=torch.float32)
    ids = torch.randint(0, CFG1["vocab"], (2, 16), generator=torch.Generator().manual_seed(0))
    a = model(ids, labels=ids)
    b = model(ids, labels=ids, materialize_logits=False)
    assert b["logits"] is not None and torch.equal(a["loss"], b["loss"])


def _ce_truth(x64, labels, inv):
    """Per-row loss and gradient of the reference's CE in fp64."""
    valid = labels != IGNORE_INDEX
    lse = torch.logsumexp(x64, dim=1)
    safe = labels.clamp(min=0)
    loss = torch.where(valid, lse - x64.gather(1, safe[:, None])[:, 0], torch.zeros_like(lse))
    p = torch.softmax(x64, dim=1)
    p[torch.arange(len(labels)), safe] -= 1.0
    grad = torch.where(valid[:, None], p * inv, torch.zeros_like(p))
    return loss, grad


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,V", [(37, 1024), (64, 32000), (9, 70016)])
def test_ce_kernel_matches_fp64(dtype, rows, V):
    """Row losses and the in-place gradient vs the fp64 reference: fp32 within
    1e-5 (relative, per tensor); bf16 gradient = the fp64 value rounded to bf16
    up to one bf16 ulp.  V = 70016 takes the streaming path (> 65536)."""
    from femtotron_amd import ops
    g = torch.Generator().manual_seed(rows + V)
    x = (torch.randn(rows, V, generator=g) * 3).to(dtype)
    labels = _labels(1, rows, V, rows)[0]
    n_valid = int((labels != IGNORE_INDEX).sum())
    inv = 1.0 / n_valid
    loss_t, grad_t = _ce_truth(x.double(), labels, inv)
    xd = x.to(DEV)
    loss_rows = ops.ce_fwd_bwd_(xd, labels.to(DEV), torch.tensor([inv], dtype=torch.float32, device=DEV))
    assert rel_err(loss_rows.double().cpu(), loss_t) < 1e-5
    got = xd.cpu()
    if dtype == torch.float32:
        assert rel_err(got.double(), grad_t) < 1e-5
    else:
        want = grad_t.to(torch.bfloat16)
        ulp = (want.float().abs() * 2.0 ** -7).clamp(min=2.0 ** -126)
        assert bool(((got.float() - want.float()).abs() <= ulp).all())
        assert torch.equal(got[labels == IGNORE_INDEX], torch.zeros_like(got[labels == IGNORE_INDEX]))


@pytest.mark.gpu
def test_ce_kernel_out_of_range_label_gives_nan_row():
    """A label outside [0, V) (torch raises) yields a NaN loss and gradient row;
    the kernel never addresses memory with it."""
    from femtotron_amd import ops
    x = torch.randn(4, 1024, device=DEV)
    labels = torch.tensor([3, 1024, -100, -5], device=DEV)
    loss = ops.ce_fwd_bwd_(x, labels, torch.tensor([0.5], device=DEV))
    assert torch.isfinite(loss[0]) and torch.isnan(loss[1]) and loss[2] == 0 and torch.isnan(loss[3])
    assert torch.isnan(x[1]).all() and (x[2] == 0).all() and torch.isfinite(x[0]).all()


def _model(c, layers, dtype, seed=42):
    from femtotron_amd.model import build_llama_model, init_llama_weights_
    return init_llama_weights_(build_llama_model(llama_config(c, layers=layers)), device=DEV,
                               dtype=dtype, seed=seed)


@pytest.mark.gpu
def test_fused_loss_cfg1_fp32_vs_cpu_oracle():
    """Config 1 end to end with fused layers and the fused loss head: loss and
    all 21 gradients within 1e-5 of the CPU fp32 oracle."""
    from femtotron_amd import fused_checkpoint
    from femtotron_amd.scripts.presets import get_ac_policy
    from femtotron_amd.training import apply_activation_checkpointing
    from oracle import torch_llama as ot
    c = CFG1
    model = _model(c, c["layers"], torch.float32)
    apply_activation_checkpointing(model, get_ac_policy("llama_decoder_layer"), checkpoint_fn=fused_checkpoint)
    ids = torch.randint(0, c["vocab"], (c["batch"], c["seq"]), generator=torch.Generator().manual_seed(2000))
    out = model(ids.to(DEV), labels=ids.to(DEV), materialize_logits=False)
    assert out["logits"] is None
    out["loss"].backward()
    grads = {n.replace("._checkpoint_wrapped_module", ""): p.grad for n, p in model.named_parameters()}
    orc = ot.OracleLlama(vocab=c["vocab"], hidden=c["hidden"], n_layers=c["layers"], n_heads=c["heads"],
                         n_kv=c["kv"], ffn=c["ffn"], theta=c["theta"])
    _, oloss = orc.forward(ids, ids)
    oloss.backward()
    assert abs(out["loss"].item() - oloss.item()) <= 1e-5 * abs(oloss.item())
    for n, t in orc.named_params():
        assert rel_err(grads[n], t.grad) < 1e-5, f"{n}: rel {rel_err(grads[n], t.grad):.3e}"


@pytest.mark.gpu
def test_fused_loss_bf16_matches_stock_loss_head():
    """2-layer TinyLlama-shaped bf16 model, B=2, S=1024 (two chunks of logits):
    fused loss head vs the stock one, same model and weights; loss within 1e-3
    relative, every gradient within the tensor-level bf16 metric."""
    from femtotron_amd import fused_checkpoint
    from femtotron_amd.scripts.presets import get_ac_policy
    from femtotron_amd.training import apply_activation_checkpointing
    import femtotron_amd.fused_loss as fl
    model = _model(CFG3, 2, torch.bfloat16)
    apply_activation_checkpointing(model, get_ac_policy("llama_decoder_layer"), checkpoint_fn=fused_checkpoint)
    ids = torch.randint(0, CFG3["vocab"], (2, 1024), generator=torch.Generator().manual_seed(7)).to(DEV)
    res = []
    old = fl._chunk_rows
    fl._chunk_rows = lambda *a: 1024  # exercise chunking
    try:
        for fused in (True, False):
            for p in model.parameters():
                p.grad = None
            loss = model(ids, labels=ids, materialize_logits=not fused)["loss"]
            loss.backward()
            res.append((loss.detach().float(), {n: p.grad.float() for n, p in model.named_parameters()}))
    finally:
        fl._chunk_rows = old
    (lf, gf), (lr, gr) = res
    assert abs(lf.item() - lr.item()) <= 1e-3 * abs(lr.item())
    for n in gr:
        err = float((gf[n] - gr[n]).abs().max())
        lim = BF16_ATOL + BF16_RTOL * float(gr[n].abs().max())
        assert err <= lim, f"{n}: {err:.3e} > {lim:.3e}"


@pytest.mark.gpu
def test_fused_loss_lowers_peak_activation_memory():
    """Peak memory of one fwd+bwd of a 2-layer TinyLlama-shaped model (B=4, S=2048):
    the fused loss head needs less than half of the stock one's (no [T, V] fp32 logits)."""
    from femtotron_amd import fused_checkpoint
    from femtotron_amd.scripts.presets import get_ac_policy
    from femtotron_amd.training import apply_activation_checkpointing
    model = _model(CFG3, 2, torch.bfloat16)
    apply_activation_checkpointing(model, get_ac_policy("llama_decoder_layer"), checkpoint_fn=fused_checkpoint)
    ids = torch.randint(0, CFG3["vocab"], (4, 2048), generator=torch.Generator().manual_seed(3)).to(DEV)

    def peak(fused):
        for _ in range(2):
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            base = torch.cuda.memory_allocated()
            model(ids, labels=ids, materialize_logits=not fused)["loss"].backward()
            torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - base

    p_stock = peak(False)
    p_fused = peak(True)
    assert p_fused < 0.5 * p_stock, f"fused {p_fused / 2**20:.0f} MiB vs stock {p_stock / 2**20:.0f} MiB"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,H,V,rows", [(512, 256, 1024, 512),   # one chunk
                                        (700, 256, 1024, 256),   # three, the last of 188 rows
                                        (530, 264, 1000, 256),   # the last of 18: fewer than a hand-written product takes
                                        (520, 100, 1000, 256),   # a width that the hand-written products do not take
                                        (40, 2056, 1024, 256)])  # a wide one, and few rows
@pytest.mark.parametrize("by_hand", [True, False])
def test_loss_head_in_chunks_matches_fp64(monkeypatch, dtype, N, H, V, rows, by_hand):
    """Loss and both gradients against fp64 with the logits and their gradient rounded where the head rounds them:
    every product sums in fp32 and rounds once, so only those roundings and the output's are left (bf16 2^-8 each)."""
    import femtotron_amd.fused_loss as fl
    monkeypatch.setattr(fl, "_chunk_rows", lambda *a: rows)
    assert not fl._acc_by_hand(V, H)  # so small a vocabulary's sum is the library's
    monkeypatch.setattr(fl, "_acc_by_hand", lambda *a: by_hand)
    g = torch.Generator().manual_seed(N + H)
    x = torch.randn(N, H, generator=g).to(dtype).to(DEV).requires_grad_(True)
    w = (torch.randn(V, H, generator=g) * H ** -0.5).to(dtype).to(DEV).requires_grad_(True)
    labels = _labels(1, N, V, 3)[0].to(DEV)
    loss = fl.FusedLinearCrossEntropy.apply(x, w, labels)
    loss.backward()
    x64, w64 = (t.detach().double().requires_grad_(True) for t in (x, w))
    want = F.cross_entropy(x64 @ w64.t(), labels, ignore_index=IGNORE_INDEX)
    want.backward()
    # relative to the tensor's norm: roundings are independent, so their sums grow no faster than the norm
    tol = 1e-5 if dtype == torch.float32 else 3 * 2.0 ** -8
    assert abs(loss.item() - want.item()) <= tol * abs(want.item())
    for got, ref in ((x.grad, x64.grad), (w.grad, w64.grad)):
        assert float((got.double() - ref).norm() / ref.norm()) < tol


def test_a_chunk_is_added_by_hand_where_its_tiles_fill_the_chip():
    """One tile of 256 x 256 per workgroup and no k split: a small vocabulary over many tokens (4 tiles over 131072
    tokens: twice the head's time) stays with the library."""
    import femtotron_amd.fused_loss as fl
    assert fl._acc_by_hand(32000, 2048) and fl._acc_by_hand(128256, 256)
    assert not fl._acc_by_hand(1024, 256) and not fl._acc_by_hand(32000, 256)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("need_dw", [True, False])
def test_chunks_stay_within_their_room(dtype, need_dw):
    """Logits beside the fp32 sum (or, in one chunk, the gradient alone): no more than 256 MB beside the sum, or than
    rounding the sum; whole 256s of rows, at least 256; the fp32 head and one without a weight gradient as ever."""
    import femtotron_amd.fused_loss as fl
    for V in (1000, 1024, 32000, 128256, 1 << 20):
        for H in (100, 256, 2048, 4096):
            w = torch.empty(V, H, dtype=dtype, device="meta")
            plain = max(256, (256 << 20) // (V * w.element_size()) // 256 * 256)
            for N in (1, 63, 64, 300, 4096, 8192, 16385, 200000):
                rows = fl._chunk_rows(torch.empty(N, H, dtype=dtype, device="meta"), w, need_dw)
                W, L = V * H * 2, min(rows, N) * V * w.element_size()
                if dtype == torch.float32 or not need_dw:
                    assert rows == plain
                elif rows == N and (N % 256 or rows != plain):  # all in one: no sum
                    assert W + L <= max(2 * W + (256 << 20), 3 * W)
                else:
                    assert rows % 256 == 0 and rows >= plain
                    assert 2 * W + L <= max(2 * W + (256 << 20), 3 * W) or rows == 256


@pytest.mark.gpu
@pytest.mark.parametrize("N,H,V", [(16384, 256, 32000),   # the logits, 1000 MiB, are the larger part
                                   (9000, 2048, 32000),   # two chunks and a remainder
                                   (8192, 1024, 32000),   # all rows in one chunk would not fit, by little
                                   (1100, 1024, 128256)])  # one chunk, no sum
def test_loss_head_peak_memory(N, H, V):
    """Peak of the bf16 head over its inputs: the input gradient, the fp32 sum of the weight gradient and 256 MB of
    logits, or the sum and the gradient it is rounded to where those are more, and the K slices of a product."""
    import femtotron_amd.fused_loss as fl
    g = torch.Generator(device=DEV).manual_seed(N)
    x = torch.randn(1, N, H, device=DEV, generator=g).bfloat16().requires_grad_(True)
    w = (torch.randn(V, H, device=DEV, generator=g) * 0.02).bfloat16().requires_grad_(True)
    labels = torch.randint(0, V, (1, N), device=DEV, generator=g)
    for _ in range(2):  # the second step finds the library's own workspace there
        x.grad = w.grad = None
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        fl.fused_causal_lm_loss(x, w, labels).backward()
    peak = torch.cuda.max_memory_allocated() - base
    room = 2 * N * H + max(4 * V * H + (256 << 20), 6 * V * H) + (64 << 20)
    assert peak <= room + (4 << 20), f"{peak / 2**20:.0f} MiB, {room / 2**20:.0f} MiB expected"
