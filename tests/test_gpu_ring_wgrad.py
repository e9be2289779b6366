"""FP32 weight gradients on the smaller macro-tiles, bit for bit on integer products: single
calls with every split the caller allows, stored and accumulated, and groups whose members
run apart. The shapes have few 256 x 256 tiles, ragged edges and short and long reductions."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, 72), (1288, 4488, 512), (6408, 1288, 1000), (520, 264, 16384),
          (2056, 520, 4104), (136, 8200, 256)]


def _ints(gen, rows, cols):
    return torch.randint(-3, 4, (rows, cols), generator=gen, device="cuda").bfloat16()


@pytest.mark.parametrize("n_out,n_in,tokens", SHAPES)
@pytest.mark.parametrize("splits", [None, 1, 2, 4])
def test_single_gradient_is_exact(n_out, n_in, tokens, splits):
    from ops.fused_execution import mm_accumulate_, mm_f32

    gen = torch.Generator("cuda").manual_seed(n_out + tokens)
    dy, x = _ints(gen, tokens, n_out), _ints(gen, tokens, n_in)
    product = (dy.double().T @ x.double()).float()
    for round_bf16 in (True, False):
        want = product.bfloat16().float() if round_bf16 else product
        print(f"{n_out}x{n_in}x{tokens} splits={splits} round={round_bf16}", flush=True)
        out = torch.full((n_out, n_in), float("nan"), device="cuda")
        mm_f32(dy.T, x, round_bf16, out=out, splits=splits)
        assert torch.equal(out, want)
        g = torch.full((n_out, n_in + 4), 5.0, device="cuda")
        mm_accumulate_(g[:, :n_in], dy.T, x, round_bf16, splits)
        assert torch.equal(g[:, :n_in], want + 5) and (g[:, n_in:] == 5).all()


@pytest.mark.parametrize("tokens", [72, 512, 2000])
def test_group_is_exact(tokens):
    from ops.fused_execution import mm_f32_group

    gen = torch.Generator("cuda").manual_seed(tokens)
    dy, act = _ints(gen, tokens, 1280), _ints(gen, tokens, 4480)
    dp, x = _ints(gen, tokens, 8960), _ints(gen, tokens, 1280)
    got = mm_f32_group([(dy.T, act), (dp.T, x)])
    for g, (a, b) in zip(got, ((dy, act), (dp, x))):
        assert torch.equal(g, (a.double().T @ b.double()).float().bfloat16().float())
