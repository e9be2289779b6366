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
