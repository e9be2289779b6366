"""Every macro-tile of the GEMM dispatch stays within reach of the GPU tests' shapes (CPU only;
the queries answer for 256 compute units where there is no GPU)."""
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


def test_invalid_sizes():
    assert _hip.query("ws_gemm_tile", 0, 8, 8, 0, 0, 0) == -1
    assert _hip.query("ws_gemm_tile", 8, 8, 8, 0, 0, 5) == -1
    assert _hip.query("ws_gemm_tile", 8, 8, 8, 0, 0, -1) == -1
    assert _hip.query("ws_mm_f32_tile", 8, 8, 8, 0, 0, None) == -1
    assert _hip.query("ws_mm_f32_tile", 8, 8, 8, 1, 0, None) in TILES
