"""RMSNorm backward on either side of each change of rows per block: against 64-bit sums, and
the static-scratch call against the workspace call, with ragged last blocks and both widths of
row kernel (vector and generic)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,d", [(63, 512), (64, 512), (65, 100), (513, 1280), (4097, 2048),
                                    (4633, 1810), (8192, 1024), (8193, 1024), (2047, 8)])
@pytest.mark.parametrize("eager", [True, False])
def test_backward_matches_64_bit_sums(rows, d, eager):
    from ops import _hip
    from ops.activation_execution import _rms_backward

    gen = torch.Generator("cuda").manual_seed(rows + d)
    x = torch.randn((rows, d), generator=gen, device="cuda").bfloat16()
    g = torch.randn((rows, d), generator=gen, device="cuda").bfloat16()
    w = 1 + 0.1 * torch.randn((d,), generator=gen, device="cuda")
    r = torch.rsqrt(x.double().square().mean(-1) + 1e-6).float()
    dx, dw = _rms_backward(x, w, r, g, eager)
    xd, gd, rd = x.double(), g.double(), r.double()[:, None]
    dz = gd * w.double()
    want_dx = dz * rd - xd * rd ** 3 * (dz * xd).mean(-1, keepdim=True)
    want_dw = (gd * xd * rd).sum(0)
    # Up to four BF16 roundings (2^-9 each) per dX element; the weight gradient's terms carry
    # two and the sum one.
    assert (dx.double() - want_dx).norm() / want_dx.norm() < 4 * 2 ** -9
    assert (dw.double() - want_dw).norm() / want_dw.norm() < 3 * 2 ** -9
    sx, sw = torch.empty_like(dx), torch.empty_like(dw)
    _hip.call("ws_rmsnorm_backward_static", x.data_ptr(), w.data_ptr(), r.data_ptr(),
              g.data_ptr(), sx.data_ptr(), sw.data_ptr(), rows, d, int(eager), _hip.stream(x))
    assert torch.equal(sx, dx) and torch.equal(sw, dw)
