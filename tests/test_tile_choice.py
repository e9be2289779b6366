"""Every macro-tile of the GEMM dispatch stays within reach of the GPU tests' shapes (CPU only;
the queries answer for 256 compute units where there is no GPU)."""
import ctypes

import pytest

from ops import _hip
from tile_shapes import (LONG, RESIDUAL, SHORT, SIGMOID, STORE, SWIGLU, SWIGLU_BACKWARD, TILES,
                         gemm_shape, gradient_shape)

EPILOGUES = [STORE, RESIDUAL, SIGMOID, SWIGLU, SWIGLU_BACKWARD]


@pytest.mark.parametrize("b_n", [0, 1])
@pytest.mark.parametrize("a_mn", [0, 1])
@pytest.mark.parametrize("epilogue", EPILOGUES)
def test_each_tile_is_reached(epilogue, a_mn, b_n):
    for tile in TILES:
        # The smaller tiles are built for a token-major A with the plain store only, and there
        # is no paired 64 x 64 tile.
        built = tile == 0 or ((epilogue == STORE or not a_mn)
                              and not (epilogue == SWIGLU and tile == 4))
        short = [k for k in SHORT if gemm_shape(epilogue, a_mn, b_n, tile, k)]
        long = [k for k in LONG if gemm_shape(epilogue, a_mn, b_n, tile, k)]
        if not built:
            assert not short and not long
        elif tile == 2:  # 128 x 128 alone: worth its idle second workgroup on long reductions
            assert short or long or epilogue == SWIGLU_BACKWARD, (epilogue, a_mn, b_n)
        else:
            assert short == list(SHORT) and long, (epilogue, a_mn, b_n, tile, short, long)


@pytest.mark.parametrize("store", [0, 1])
def test_each_gradient_tile_is_reached(store):
    for tile in TILES:
        assert all(gradient_shape(tile, 1, 1, store, k) for k in (SHORT if tile != 2 else LONG))
        assert gradient_shape(tile, 1, 1, store, 8200)
        for splits in (2, 4):
            assert gradient_shape(tile, splits, splits, store, 8200), (tile, splits)


# Gradients whose last round on a smaller tile holds a pair on a few compute units only, with
# the time of that tile and of the 256 x 256 schemes, us.
@pytest.mark.parametrize("m,n,k,splits,store,slow,us", [
    (1400, 1632, 6601, 4, 0, (3, 1), (79, 59)), (592, 3816, 5622, 4, 0, (3, 1), (72, 47)),
    (3184, 856, 4363, 4, 1, (3, 1), (55, 45)), (4376, 1048, 8414, 2, 1, (1, 1), (121, 107)),
    (6312, 680, 8448, 2, 1, (1, 1), (123, 106))])
def test_a_few_pairs_do_not_end_the_launch_late(m, n, k, splits, store, slow, us):
    got = ctypes.c_int()
    tile = _hip.query("ws_mm_f32_tile", m, n, k, splits, store, ctypes.byref(got))
    assert (tile, got.value) != slow


def test_invalid_sizes():
    assert _hip.query("ws_gemm_tile", 0, 8, 8, 0, 0, 0) == -1
    assert _hip.query("ws_gemm_tile", 8, 8, 8, 0, 0, 5) == -1
    assert _hip.query("ws_gemm_tile", 8, 8, 8, 0, 0, -1) == -1
    assert _hip.query("ws_mm_f32_tile", 8, 8, 8, 0, 0, None) == -1
    assert _hip.query("ws_mm_f32_tile", 8, 8, 8, 1, 0, None) in TILES
