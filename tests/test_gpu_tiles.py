"""Every macro-tile, epilogue and operand layout of the vector GEMMs, bit for bit, at the
reductions their pipelines treat specially.

Integer-valued BF16 operands make every FP32 partial sum exact, so the product must be the
exactly rounded one, and the SwiGLU epilogues must give what the standalone kernels give on it.
tile_shapes.py finds, for each macro-tile, shapes whose launch picks it,
with rows, columns and reduction off the tiles' edges; test_tile_choice.py keeps it in reach.
Each output has a guard row behind it.
"""
import pytest
import torch

from ops import _hip
from tile_shapes import (LONG, RESIDUAL, SHORT, SIGMOID, STORE, SWIGLU, SWIGLU_BACKWARD, TILES,
                         gemm_shape, gradient_shape)

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _ints(gen, rows, cols, low=-3, high=3):
    return torch.randint(low, high + 1, (rows, cols), generator=gen, device="cuda").to(BF16)


def _operands(gen, m, n, k, a_mn, b_n):
    a, b = _ints(gen, m, k), _ints(gen, k, n)
    want = (a.double() @ b.double()).float()
    return (a.T.contiguous().T if a_mn else a, b if b_n else b.T.contiguous().T, want)


def _guarded(m, n, dtype=BF16):
    full = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
    return full, full[:m]


def _strides(t):
    return t.data_ptr(), t.stride(0), t.stride(1)


def _near(got, want):
    # One BF16 rounding apart (2^-8); values below the smallest normal number flush to zero.
    torch.testing.assert_close(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -126)


def _run(epilogue, m, n, k, a_mn, b_n):
    gen = torch.Generator("cuda").manual_seed(m + 3 * n + 5 * k)
    if epilogue == SIGMOID:
        # Rows of +-1 have an RMS of one, so the normalized operand is the norm weight's
        # integers with signs.
        x = 2 * _ints(gen, m, k, 0, 1) - 1
        weight = torch.randint(1, 3, (k,), generator=gen, device="cuda").float()
        b = _ints(gen, k, n)
        want = ((x.double() * weight.double()) @ b.double()).float().to(BF16)
        gate = (n // 16 * 8, n // 16 * 8 + 24)
        b = b if b_n else b.T.contiguous().T
        full, out = _guarded(m, n)
        rstd = torch.empty(m, device="cuda")
        normed = torch.empty_like(x)
        _hip.call("ws_rmsnorm_gate_mm", x.data_ptr(), x.stride(0), weight.data_ptr(), 0.0,
                  rstd.data_ptr(), normed.data_ptr(), *_strides(b), out.data_ptr(), m, n, k, *gate,
                  _hip.stream(x))
        assert torch.equal(out[:, :gate[0]], want[:, :gate[0]])
        assert torch.equal(out[:, gate[1]:], want[:, gate[1]:])
        _near(out[:, gate[0]:gate[1]], torch.sigmoid(want[:, gate[0]:gate[1]].float()).to(BF16))
        return full
    cols = 2 * n if epilogue == SWIGLU else n
    a, b, product = _operands(gen, m, cols, k, a_mn, b_n)
    want = product.to(BF16)
    full, out = _guarded(m, 2 * n if epilogue in (SWIGLU, SWIGLU_BACKWARD) else n)
    if epilogue == STORE:
        _hip.call("ws_mm", *_strides(a), *_strides(b), out.data_ptr(), m, n, k, 1, 0, _hip.stream(a))
        assert torch.equal(out, want)
    elif epilogue == RESIDUAL:
        residual = _ints(gen, m, n, -300, 300)
        _hip.call("ws_residual_mm", *_strides(a), *_strides(b), residual.data_ptr(), n,
                  out.data_ptr(), m, n, k, _hip.stream(a))
        assert torch.equal(out, (residual.float() + want.float()).to(BF16))
    elif epilogue == SWIGLU:
        act_full, act = _guarded(m, n)
        _hip.call("ws_swiglu_mm", *_strides(a), *_strides(b), out.data_ptr(), act.data_ptr(), m, n,
                  k, 1, 1, 0, _hip.stream(a))
        assert torch.equal(out, want)
        alone = torch.empty((m, n), dtype=BF16, device="cuda")
        _hip.call("ws_swiglu_forward", want.data_ptr(), alone.data_ptr(), m, n, 1, _hip.stream(a))
        assert torch.equal(act, alone)
        assert (act_full[m] == 7).all()
    else:
        packed = torch.randn((m, 2 * n), generator=gen, device="cuda").to(BF16)
        _hip.call("ws_swiglu_backward_mm", *_strides(a), *_strides(b), packed.data_ptr(),
                  out.data_ptr(), m, n, k, 1, _hip.stream(a))
        alone = torch.empty_like(packed)
        _hip.call("ws_swiglu_backward", packed.data_ptr(), want.data_ptr(), alone.data_ptr(), m, n,
                  1, _hip.stream(a))
        assert torch.equal(out, alone)
    return full


# The gated projection's normalized operand is always row by row; a token-major A beside another
# epilogue than the plain store runs on 256 x 256 tiles only.
CASES = [(e, tile, a_mn) for e in (STORE, RESIDUAL, SIGMOID, SWIGLU, SWIGLU_BACKWARD)
         for tile in TILES for a_mn in (0, 1)
         if not a_mn or e == STORE or (tile == 0 and e != SIGMOID)]


@pytest.mark.parametrize("b_n", [0, 1])
@pytest.mark.parametrize("epilogue,tile,a_mn", CASES)
def test_products_are_exact(epilogue, tile, a_mn, b_n):
    ran = 0
    for k in SHORT + LONG:
        shape = gemm_shape(epilogue, a_mn, b_n, tile, k)
        if shape is None:
            continue
        m, n = shape
        # Rows of A that are no multiple of 8 where its loader takes any count.
        for rows in ((m,) if a_mn else (m, m - 3)):
            cols = 2 * n if epilogue == SWIGLU else n
            if _hip.query("ws_gemm_tile", rows, cols, k, a_mn, b_n, epilogue) != tile:
                continue
            print(f"{TILES[tile]} epilogue={epilogue} {rows}x{n}x{k} a_mn={a_mn} b_n={b_n}",
                  flush=True)
            full = _run(epilogue, rows, n, k, a_mn, b_n)
            assert (full[rows] == 7).all()
            ran += 1
    # There is no paired 64 x 64 tile, and none of these shapes is one for 128 x 128 alone under
    # the SwiGLU backward.
    assert ran or (epilogue, tile) in ((SWIGLU, 4), (SWIGLU_BACKWARD, 2))


@pytest.mark.parametrize("store", [0, 1])
@pytest.mark.parametrize("splits", [1, 2, 4])
@pytest.mark.parametrize("tile", list(TILES))
def test_gradients_are_exact(tile, splits, store):
    """FP32 gradients of token-major operands on every tile, with every number of slices."""
    for k in SHORT + LONG + (8200,):
        for slices in range(1, splits + 1):
            shape = gradient_shape(tile, slices, splits, store, k)
            if shape is None:
                continue
            m, n = shape
            gen = torch.Generator("cuda").manual_seed(m + 3 * n + 5 * k)
            a, b, product = _operands(gen, m, n, k, 1, 1)
            print(f"{TILES[tile]} slices={slices}/{splits} store={store} {m}x{n}x{k}", flush=True)
            full, g = _guarded(m, n, torch.float32)
            g.fill_(float("nan") if store else 5.0)
            floats = _hip.query("ws_mm_accumulate_workspace_floats", m, n, k, splits)
            workspace = torch.full((floats + 4,), 9.0, device="cuda")
            _hip.call("ws_mm_store_f32" if store else "ws_mm_accumulate_f32", *_strides(a),
                      *_strides(b), g.data_ptr(), n, m, n, k, 1, workspace.data_ptr(), splits,
                      _hip.stream(a))
            want = product.to(BF16).float()
            assert torch.equal(g, want if store else want + 5)
            assert (full[m] == 7).all() and (workspace[floats:] == 9).all()
