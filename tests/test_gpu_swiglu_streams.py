"""Standalone SwiGLU on either side of the size where it passes the caches by: the same bits
as the same rows in pieces below that size."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 256 MB is moved at 10922.7 rows of 4096 forward (6 bytes an element) and 6553.6 backward (10).
@pytest.mark.parametrize("rows,h", [(6553, 4096), (6554, 4096), (10922, 4096), (10923, 4096),
                                    (33333, 1816)])
@pytest.mark.parametrize("eager", [0, 1])
def test_pieces_agree(rows, h, eager):
    from ops import _hip

    gen = torch.Generator("cuda").manual_seed(rows + h)
    x = torch.randn((rows, 2 * h), generator=gen, device="cuda", dtype=torch.bfloat16)
    g = torch.randn((rows, h), generator=gen, device="cuda", dtype=torch.bfloat16)

    def run(x, g):
        y, dx = torch.empty_like(g), torch.empty_like(x)
        _hip.call("ws_swiglu_forward", x.data_ptr(), y.data_ptr(), len(x), h, eager, _hip.stream(x))
        _hip.call("ws_swiglu_backward", x.data_ptr(), g.data_ptr(), dx.data_ptr(), len(x), h,
                  eager, _hip.stream(x))
        return y, dx

    pieces = [run(a, b) for a, b in zip(x.split(4096), g.split(4096))]
    for whole, part in zip(run(x, g), zip(*pieces)):
        assert torch.equal(whole, torch.cat(part))
