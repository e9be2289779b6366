"""LM-head loss on operands that the vector loaders refuse, with vocabularies off multiples of
8 and enough rows for a transposed weight: every mode agrees with 64-bit arithmetic, and the
one-pass and two-pass gradients with each other bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d,vocab,pad,modes", [
    (1030, 100, 2047, 0, ("two", "fused")), (1100, 128, 1031, 1, ("two", "fused")),
    (1100, 128, 1028, 0, ("two", "fused", "stored")), (1030, 100, 1032, 0, ("two", "fused"))])
def test_gradients(rows, d, vocab, pad, modes):
    from ops.benchmark_configs import lm_head_inputs
    from ops.fused_execution import (CrossEntropyState, linear_cross_entropy_backward,
                                     linear_cross_entropy_forward)

    inp = lm_head_inputs(m=rows, d=d, vocab=vocab, seed=9)
    h, w, t = (inp[k].cuda() for k in ("hidden", "weight", "targets"))
    if pad:
        wide = torch.empty((rows, d + pad), dtype=h.dtype, device="cuda")
        wide[:, :d] = h
        h = wide[:, :d]
    logits = h.double() @ w.double().T
    valid = t != -100
    g = torch.exp(logits - torch.logsumexp(logits, -1)[:, None])
    g.scatter_add_(1, t.clamp_min(0)[:, None], -torch.ones_like(g[:, :1]))
    g *= (valid / valid.sum().clamp_min(1))[:, None]
    wants = (g @ w.double(), g.T @ h.double())
    one, results = torch.ones((), device="cuda"), {}
    for mode in modes:
        print(f"{rows}x{d} over {vocab} pad={pad} {mode}", flush=True)
        state = CrossEntropyState(rows, vocab, h.device, 512, d=d, fused=mode == "fused",
                                  weight_grad=mode == "fused", store_logits=mode == "stored")
        linear_cross_entropy_forward(h, w, t, state)
        dw = torch.full((vocab, d), float("nan"), device="cuda")
        dh = linear_cross_entropy_backward(h, w, t, state, one, weight_grad=dw, accumulate=False)
        results[mode] = (dh, dw)
        # Logits, gradients and dHidden are rounded to BF16 (2^-9 each).
        for got, want in zip((dh, dw), wants):
            assert (got.double() - want).norm() <= 4 * 2 ** -9 * want.norm()
    for mode in modes[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[modes[0]], results[mode]))
