"""The smaller macro-tiles of the vector GEMM at their edges, bit for bit.

Integer-valued BF16 operands make every FP32 partial sum exact, so each tile, layout and
epilogue must give the exactly rounded product. The shapes put one row or column past a
tile, fewer k-tiles than LDS stages, a ragged last k-tile, and more tiles than compute units
in front of the dispatch, whatever macro-tile it picks (test_gpu_tiles.py asks for each one).
"""
import pytest
import torch

from ops import _hip

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 8, 8), (64, 64, 64), (65, 72, 136), (130, 200, 2056),
    (1001, 2056, 1032), (712, 2568, 584),
    (520, 4488, 264), (2040, 2056, 520),
    (520, 8968, 328), (4104, 1288, 648),
    (8200, 2056, 200), (5128, 4104, 72),
]


def _ints(gen, rows, cols):
    return torch.randint(-3, 4, (rows, cols), generator=gen, device="cuda").bfloat16()


def _product(a, b):
    return (a.double() @ b.double()).float()


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_every_layout_is_exact(m, n, k):
    """ws_mm and the FP32 store with A and B each K- and M/N-contiguous; the M/N-contiguous
    layouts take rows padded to a multiple of 8, as the vector loader asks."""
    gen = torch.Generator("cuda").manual_seed(m * 7 + n)
    a, b = _ints(gen, m, k), _ints(gen, k, n)
    want = _product(a, b)
    for a_mn in (False, True):
        if a_mn and m % 8:
            continue
        for b_mn in (False, True):
            ga = a.T.contiguous().T if a_mn else a
            gb = b if b_mn else b.T.contiguous().T
            print(f"m={m} n={n} k={k} a_mn={a_mn} b_mn={b_mn}", flush=True)
            guard = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device="cuda")
            _hip.call("ws_mm", ga.data_ptr(), ga.stride(0), ga.stride(1), gb.data_ptr(),
                      gb.stride(0), gb.stride(1), guard.data_ptr(), m, n, k, 1, 0, _hip.stream(ga))
            assert torch.equal(guard[:m], want.bfloat16())
            assert (guard[m] == 7).all()
            g = torch.full((m, n + 4), 3.0, device="cuda")
            _hip.call("ws_mm_accumulate_f32", ga.data_ptr(), ga.stride(0), ga.stride(1),
                      gb.data_ptr(), gb.stride(0), gb.stride(1), g.data_ptr(), g.stride(0), m, n,
                      k, 0, None, 1, _hip.stream(ga))
            assert torch.equal(g[:, :n], want + 3) and (g[:, n:] == 3).all()


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("weight_rows", [True, False])
def test_residual_epilogue_is_exact(m, n, k, weight_rows):
    """The residual epilogue, on a weight stored [N, K] and one stored [K, N]."""
    from ops.fused_execution import residual_mm

    gen = torch.Generator("cuda").manual_seed(m + 3 * n)
    h, w = _ints(gen, m, k), _ints(gen, n, k)
    r = torch.randint(-300, 301, (m, n), generator=gen, device="cuda").bfloat16()
    want = (r.float() + _product(h, w.T).bfloat16().float()).bfloat16()
    weight = w if weight_rows else w.T.contiguous().T
    print(f"m={m} n={n} k={k} rows={weight_rows}", flush=True)
    assert torch.equal(residual_mm(h, weight, r), want)
