"""Which form the expert GEMMs of a batch take, on both sides of the rules' lines (host code of the
library; no GPU needed)."""
import pytest

from pisceslx_amd import _lib
from helpers import few_forms, tile_rows

UP, DOWN = 1, 2
I8, I4, F8, B16, F32 = _lib.W_INT8, _lib.W_INT4, _lib.W_FP8, _lib.W_BF16, _lib.W_F32


@pytest.mark.parametrize("tokens,k,E,S,H,F,fmt,want", [
    # few work-groups on the streaming form: both GEMMs; then gate/up alone; then neither
    (1, 6, 64, 2, 4096, 1408, I8, UP | DOWN), (3, 6, 64, 2, 4096, 1408, I8, UP), (3, 6, 64, 2, 4096, 1408, F8, UP | DOWN),
    (4, 6, 64, 2, 4096, 1408, I8, UP), (16, 6, 64, 2, 4096, 1408, I8, UP), (32, 6, 64, 2, 4096, 1408, I8, 0),
    (16, 6, 64, 2, 4096, 1408, B16, UP | DOWN), (41, 6, 64, 2, 4096, 1408, B16, UP),
    (43, 6, 64, 2, 4096, 1408, B16, 0), (64, 6, 64, 2, 4096, 1408, I8, 0),
    (31, 2, 8, 1, 1024, 2816, I8, UP | DOWN), (31, 2, 8, 1, 1024, 2816, I4, UP | DOWN),
    # a down projection of four k-steps leaves the form early
    (2, 8, 128, 1, 2048, 256, I8, UP | DOWN), (10, 8, 128, 1, 2048, 256, I8, UP),
    (20, 1, 64, 2, 4096, 1408, I8, UP),
    # many shared rows, which it would read once per 16: not beyond the first lines
    (15, 1, 256, 2, 2048, 1024, I8, UP | DOWN), (100, 1, 256, 2, 2048, 1024, I8, 0),
    (400, 1, 64, 2, 4096, 512, I8, 0), (64, 1, 64, 2, 4096, 1408, B16, 0), (250, 1, 256, 2, 2048, 1024, F8, 0),
    (5, 4, 32, 2, 7168, 1024, F8, UP | DOWN), (24, 4, 32, 2, 7168, 1024, F8, UP),
    (3, 16, 8, 0, 1024, 512, I8, UP | DOWN),  # a dispatch of more slots than experts
])
def test_few_token_form(tokens, k, E, S, H, F, fmt, want):
    assert few_forms(tokens, k, E, S, H, F, fmt) == want


MID, SMALL = (6, 64, 2, 4096, 1408), (2, 8, 1, 1024, 2816)  # k, E, S, H, F


@pytest.mark.parametrize("layer,fmt,tokens,rows", [
    # fp32
    (SMALL, F32, 191, 64), (SMALL, F32, 192, 128), ((8, 128, 1, 5120, 1536), F32, 114, 64), ((8, 128, 1, 5120, 1536), F32, 115, 128),
    ((6, 64, 2, 4096, 1408), F32, 148, 64), ((6, 64, 2, 4096, 1408), F32, 149, 128),
])
def test_rows_per_tile(layer, fmt, tokens, rows):
    k, E, S, H, F = layer
    assert tile_rows(tokens, k, E, S, H, F, fmt) == rows
