"""Shapes that reach each macro-tile of the GEMM dispatch, found through its own queries.

For an epilogue, an operand layout, a macro-tile and a number of 64-wide k-tiles, the smallest
output of a fixed list whose rows, columns and reduction lie off the tiles' edges and whose
launch picks that macro-tile. What no shape of the list reaches is None, so that a change of
the cost rule that takes a tile out of reach shows in the tests that count on it."""
import ctypes
import functools

from ops import _hip

TILES = {0: "256x256", 1: "128x128 two per CU", 2: "128x128 alone", 3: "64x128", 4: "64x64"}
STORE, RESIDUAL, SIGMOID, SWIGLU, SWIGLU_BACKWARD = range(5)
# Reduction lengths of one to five 64-wide k-tiles (fewer than any pipeline's stages, and one or
# two more), with and without a ragged last one, and of enough for every stage to wrap often.
SHORT = (40, 64, 72, 128, 136, 192, 200, 256, 264, 320)
LONG = (2056,)
_ROWS = (40, 72, 136, 264, 520, 712, 1016, 1032, 2056, 2568, 4104, 5128, 8200, 12296)
_COLS = (72, 136, 264, 520, 1032, 1288, 2056, 2568, 4088, 4104, 5128, 8200)


@functools.cache
def gemm_shape(epilogue, a_token_major, b_n_contiguous, tile, k):
    best = None
    for m in _ROWS:
        for n in _COLS:
            cols = 2 * n if epilogue == SWIGLU else n
            if best is None or m * n < best[0] * best[1]:
                if _hip.query("ws_gemm_tile", m, cols, k, a_token_major, b_n_contiguous,
                              epilogue) == tile:
                    best = (m, n)
    return best


@functools.cache
def gradient_shape(tile, slices, splits, store, k):
    best, got = None, ctypes.c_int()
    for m in _ROWS:
        for n in _COLS:
            if best is None or m * n < best[0] * best[1]:
                if (_hip.query("ws_mm_f32_tile", m, n, k, splits, store, ctypes.byref(got)) == tile
                        and got.value == slices):
                    best = (m, n)
    return best
