"""The head weight's gradient written instead of accumulated: into a buffer of NaNs it gives
the bits of accumulating into zeros, in every mode and for every kind of upstream gradient."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("rows,d,vocab,chunk", [(512, 256, 1024, 8192), (1001, 128, 2048, 256),
                                                (700, 100, 1030, 512)])
def test_written_weight_gradient_matches_accumulating_into_zeros(rows, d, vocab, chunk, fused):
    from ops.benchmark_configs import lm_head_inputs
    from ops.fused_execution import (CrossEntropyState, linear_cross_entropy_backward,
                                     linear_cross_entropy_forward)

    inp = lm_head_inputs(m=rows, d=d, vocab=vocab, seed=6)
    h, w, t = (inp[k].cuda() for k in ("hidden", "weight", "targets"))
    for grad in (1.0, -0.25, 1.0 / 3.0):
        state = CrossEntropyState(rows, vocab, h.device, chunk, d=d, fused=fused,
                                  weight_grad=fused)
        if fused:
            state.dweight_unit.fill_(float("nan"))
        linear_cross_entropy_forward(h, w, t, state)
        g = torch.full((), grad, device="cuda")
        results = []
        for start, accumulate in ((0.0, True), (float("nan"), False)):
            dw = torch.full((vocab, d), start, device="cuda")
            dh = linear_cross_entropy_backward(h, w, t, state, g, weight_grad=dw,
                                               accumulate=accumulate)
            results.append((dh, dw))
        (dh0, dw0), (dh1, dw1) = results
        print(f"rows={rows} fused={fused} grad={grad}", flush=True)
        assert torch.equal(dh0, dh1) and torch.equal(dw0, dw1)
        assert not dw1.isnan().any()


@pytest.mark.parametrize("rows,d,vocab,chunk", [(300, 64, 1, 512), (513, 264, 4099, 200),
                                                (1030, 128, 2047, 1024), (64, 2048, 517, 64),
                                                (700, 136, 1028, 300)])
def test_vocabulary_that_is_no_multiple_of_8(rows, d, vocab, chunk):
    """The chunk's gradient rows are padded: both modes agree bit for bit and with 64-bit
    arithmetic, with a workspace full of NaNs and guard values around the outputs."""
    from ops.benchmark_configs import lm_head_inputs
    from ops.fused_execution import (CrossEntropyState, linear_cross_entropy_backward,
                                     linear_cross_entropy_forward)

    inp = lm_head_inputs(m=rows, d=d, vocab=vocab, seed=7)
    h, w, t = (inp[k].cuda() for k in ("hidden", "weight", "targets"))
    one, results = torch.ones((), device="cuda"), []
    for fused in (True, False):
        state = CrossEntropyState(rows, vocab, h.device, chunk, d=d, fused=fused,
                                  weight_grad=fused)
        ws = state.workspace
        ws.view(torch.uint8)[: ws.numel() // 4 * 4].view(torch.float32).fill_(float("nan"))
        linear_cross_entropy_forward(h, w, t, state)
        dw = torch.full((vocab + 1, d), 3.0, device="cuda")
        dh = linear_cross_entropy_backward(h, w, t, state, one, weight_grad=dw[:vocab],
                                           accumulate=False)
        assert (dw[vocab] == 3).all()
        results.append((state.loss, dh, dw[:vocab]))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    logits = h.double() @ w.double().T
    valid = t != -100
    lse = torch.logsumexp(logits, -1)
    g = torch.exp(logits - lse[:, None])
    g.scatter_add_(1, t.clamp_min(0)[:, None], -torch.ones_like(g[:, :1]))
    g *= (valid / valid.sum().clamp_min(1))[:, None]
    loss, dh, dw = results[0]
    # Logits, gradients and dHidden are rounded to BF16 (2^-9 each); with a vocabulary of one
    # the gradient is a difference of equal numbers.
    if vocab > 1:
        for got, want in ((dh, g @ w.double()), (dw, g.T @ h.double())):
            assert (got.double() - want).norm() <= 4 * 2 ** -9 * want.norm()
    else:
        assert not dh.any() and not dw.any()
