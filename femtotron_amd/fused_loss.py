"""Fused lm_head + chunked cross-entropy: the loss head without full logits.

Reference loss head (femtotron/model/llama.py:91-111, femtotron/model/base.py:20-31):

    logits = lm_head(hidden)                                    # [B, S, V], model dtype
    loss = F.cross_entropy(logits[..., :-1, :].float().view(-1, V),
                           labels[..., 1:].view(-1), ignore_index=-100)

It materialises the logits in the model dtype and twice more in fp32 (the
``.float()`` copy and the log-softmax), ~0.38 MB per token at V = 32000, which
is the largest activation term of a checkpointed step.  Here the rows are
processed in chunks of 256 MB of logits (more where that needs no more memory,
CHUNK_BYTES below): per chunk one GEMM forms the logits, ``fh_ce_fwd_bwd``
computes the fp32 row losses and overwrites the chunk with its gradient (softmax - onehot) / n_valid in the model dtype (the
rounding point of the reference's ``.float()`` backward), and two GEMMs turn it
into the chunk's input gradient (dlogits @ W, in the model dtype like the
reference) and its weight-gradient contribution (dlogits^T @ hidden,
accumulated in fp32, across chunks too, and rounded once).  Both gradients are
computed in the forward and scaled by the incoming gradient in the backward, so
nothing of size [tokens, V] outlives a chunk.

The next-token shift needs no copy: the labels are shifted instead
(``shift_labels``: position s takes label s+1, the last position of each
sequence is ignore_index), which pairs exactly the same (logits row, label)
pairs and counts the same number of valid labels as the reference.
"""
from __future__ import annotations

import torch

from . import ops
from .projections import _choose_hand, gemm_policy

IGNORE_INDEX = -100
# Logits bytes per chunk, at least.  Beside them lies the fp32 sum of the weight
# gradient (twice W, the bf16 gradient's bytes), from the first chunk to the last: the
# head takes 2 W + CHUNK_BYTES, or the 3 W of rounding the sum where that is more, and
# the products' K slices (64 MB at most here).  In that room (_chunk_rows) a chunk
# grows to W for a large vocabulary, and one chunk takes all rows where their logits
# and the gradient alone, with no sum, fit: each chunk past the first reads and each
# before the last writes the sum, a third to half of that product's own time at 256
# MB.  Forward and backward, and the peak over the inputs: 16384 x 2048 hidden states
# and a vocabulary of 32000 5.71 ms and 628 MiB (in one chunk 5.06 and 1189; library
# products in 256 MB chunks 6.21 and 564), 4096 x 2048 and 32000 1.46 and 391 (library
# 1.73 and 516), 8192 x 4096 and 128256 19.4 and 3070, in one chunk (library 34.3 and
# 3070; in 1 GiB chunks with the sum 20.3 and 4072).
CHUNK_BYTES = 256 << 20
# The logits run hand-written up to this width, where a tile is few stages long:
# 16384 x 32000 352 us against the library's 426 at 256 wide, 508 against 613 at
# 512, 848 against 842 at 1024, and 1544 against 1497 at 2048.
LOGITS_HAND_MAX_HIDDEN = 1024


def shift_labels(labels: torch.Tensor, ignore_index: int = IGNORE_INDEX) -> torch.Tensor:
    """[B, S] labels -> [B*S] next-token targets: out[b, s] = labels[b, s+1],
    ignore_index at s = S-1 (femtotron/model/llama.py:97-98 shifts the logits instead)."""
    out = torch.full_like(labels, ignore_index)
    out[:, :-1] = labels[:, 1:]
    return out.reshape(-1).contiguous()


def supported(hidden: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether the fused loss can run: HIP device, bf16/fp32, matching dtypes."""
    return (hidden.is_cuda and weight.is_cuda and hidden.device == weight.device
            and hidden.dtype in (torch.bfloat16, torch.float32) and weight.dtype == hidden.dtype
            and weight.dim() == 2 and weight.shape[1] == hidden.shape[-1]
            and weight.shape[0] % 8 == 0 and not torch.is_autocast_enabled())


def _logits(x_c: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    if x_c.size(1) <= LOGITS_HAND_MAX_HIDDEN and _choose_hand("nt", x_c, weight):
        return ops.gemm("nt", x_c, weight, any_k=True)
    return torch.mm(x_c, weight.t())


def _input_grad(dlogits: torch.Tensor, weight: torch.Tensor, out: torch.Tensor) -> None:
    """out = dlogits @ weight.  Hand-written where supported: 4096 x 2048 x 32000 392
    us against the library's 439, 1024 x 2048 x 32000 119 against 298."""
    if _choose_hand("nn", dlogits, weight) and out.is_contiguous() and out.data_ptr() % 16 == 0:
        ops.gemm("nn", dlogits, weight, out=out, any_k=True)
    else:
        torch.mm(dlogits, weight, out=out)


def _peak_bytes(weight: torch.Tensor) -> int:
    """Bytes that the logits, the fp32 sum and the bf16 gradient may take together."""
    w = weight.numel() * weight.element_size()
    return max(2 * w + CHUNK_BYTES, 3 * w)


def _chunk_rows(hidden2: torch.Tensor, weight: torch.Tensor, need_dw: bool) -> int:
    """Rows per chunk (CHUNK_BYTES above)."""
    N, H = hidden2.shape
    row = weight.size(0) * weight.element_size()
    w = row * H
    sums = need_dw and weight.dtype == torch.bfloat16  # fp32: the sum is the gradient itself
    # One chunk needs no sum if its product runs hand-written.
    if (sums and gemm_policy() == "hand" and N >= 64 and H % 8 == 0 and hidden2.data_ptr() % 16 == 0
            and w + N * row <= _peak_bytes(weight)):
        return N
    return max(256, max(CHUNK_BYTES, w if sums else 0) // row // 256 * 256)


def _acc_by_hand(V: int, H: int) -> bool:
    """Whether a chunk's product is added to the fp32 sum by fh_gemm_bf16_acc: from 192
    tiles of 256 x 256 on, as it splits no k and fewer leave CUs idle.  Hand-written and
    library: 4096 x 32000 x 2048 481 and 575 us, x 512 level, x 256 103 and 83; 8192 x
    1024 x 256 151 and 49 (the head of 140000 tokens 3.35 and 1.5 ms)."""
    return V * H >= 192 * 256 * 256


def _weight_grad(dlogits: torch.Tensor, x_c: torch.Tensor, dw32: torch.Tensor | None, first: bool, last: bool,
                 peak: int):
    """(dw or None, the running fp32 sum or None) after this chunk: dw appears
    with the last one.  A last chunk whose product is not added by hand (fp32, a
    width that is no multiple of 8, fewer than 64 rows, few tiles), or that leaves no room for
    dw beside its logits, leaves the rounding to the caller."""
    V, H = dlogits.size(1), x_c.size(1)
    if _choose_hand("tn", dlogits, x_c):
        if first and last:
            return ops.gemm("tn", dlogits, x_c, any_k=True), None
        if _acc_by_hand(V, H):
            dw = None
            if first:
                dw32 = torch.empty(V, H, dtype=torch.float32, device=x_c.device)
            elif last and 6 * dw32.numel() + 2 * dlogits.numel() <= peak:
                dw = torch.empty(V, H, dtype=x_c.dtype, device=x_c.device)
            ops.gemm_acc(dlogits, x_c, dw32, add=not first, out=dw)
            return dw, dw32
    if first:
        dw32 = torch.zeros(V, H, dtype=torch.float32, device=x_c.device)
    if x_c.dtype == torch.float32:
        dw32.addmm_(dlogits.t(), x_c)
    else:
        torch.addmm(dw32, dlogits.t(), x_c, out_dtype=torch.float32, out=dw32)
    return None, dw32


class FusedLinearCrossEntropy(torch.autograd.Function):
    """loss = mean over non-ignored rows of CE(hidden2 @ weight^T, targets).
    Saved for backward: the input gradient [N, H] and the weight gradient."""

    @staticmethod
    def forward(ctx, hidden2, weight, targets):
        N, H = hidden2.shape
        V = weight.shape[0]
        dev = hidden2.device
        n_valid = (targets != IGNORE_INDEX).sum().to(torch.float32)
        inv_count = (1.0 / n_valid).reshape(1)  # inf when nothing is valid -> NaN loss, as torch
        need_dx, need_dw = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        dx = torch.empty_like(hidden2) if need_dx else None
        dw = dw32 = None
        loss_sum = torch.zeros((), dtype=torch.float32, device=dev)
        chunk = _chunk_rows(hidden2, weight, need_dw)
        for r0 in range(0, N, chunk):
            r1 = min(N, r0 + chunk)
            x_c = hidden2[r0:r1]
            logits = _logits(x_c, weight)
            loss_rows = ops.ce_fwd_bwd_(logits, targets[r0:r1], inv_count, IGNORE_INDEX)
            loss_sum += loss_rows.sum()
            if need_dx:
                _input_grad(logits, weight, dx[r0:r1])
            if need_dw:
                dw, dw32 = _weight_grad(logits, x_c, dw32, r0 == 0, r1 == N, _peak_bytes(weight))
            del logits
        if need_dw and dw is None:  # no rows, or the library's last chunk
            dw = torch.zeros_like(weight) if dw32 is None else dw32.to(weight.dtype)
        ctx.save_for_backward(dx, dw)
        return loss_sum * inv_count[0]

    @staticmethod
    def backward(ctx, grad):
        dx, dw = ctx.saved_tensors
        g = grad.to(torch.float32)

        def scaled(t):  # (t * g).to(t.dtype): fh_scale, one streaming pass
            if t is None:
                return None
            if t.numel() % 8 == 0 and t.data_ptr() % 16 == 0 and t.is_contiguous():
                return ops.scale(t, g)
            return (t * g).to(t.dtype)
        return scaled(dx), scaled(dw), None


def fused_causal_lm_loss(hidden: torch.Tensor, weight: torch.Tensor,
                         labels: torch.Tensor) -> torch.Tensor:
    """The reference's shifted next-token cross-entropy of ``hidden @ weight^T``
    (hidden [B, S, H], weight [V, H], labels [B, S], ignore_index -100)."""
    B, S, H = hidden.shape
    return FusedLinearCrossEntropy.apply(hidden.reshape(B * S, H).contiguous(), weight,
                                         shift_labels(labels))
