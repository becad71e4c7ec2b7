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


MID, CFG5, SMALL = (6, 64, 2, 4096, 1408), (8, 256, 0, 7168, 2048), (2, 8, 1, 1024, 2816)  # k, E, S, H, F


@pytest.mark.parametrize("layer,fmt,tokens,rows", [
    # streaming to mid-sized: 9 rows of a segment with shared experts, 8 without, int4 4 or 7
    (MID, I8, 74, 16), (MID, I8, 75, 128), (MID, B16, 74, 16), (MID, F8, 75, 128), (MID, I4, 32, 16), (MID, I4, 33, 64),
    ((8, 256, 0, 7168, 2048), I8, 255, 16), ((8, 256, 0, 7168, 2048), I8, 256, 128),
    ((4, 64, 0, 4224, 1024), I4, 111, 16), ((4, 64, 0, 4224, 1024), I4, 112, 64),
    # many experts on a part-filled mid grid: 12, int4 14; a few experts on the few-token form: 14
    ((4, 64, 1, 1024, 640), I8, 155, 16), ((4, 64, 1, 1024, 640), I8, 156, 64), ((6, 64, 2, 2688, 640), I4, 115, 16),
    ((6, 64, 2, 2688, 640), I4, 116, 64), (SMALL, I8, 32, 16), (SMALL, I8, 33, 64),
    # 64 to 128 rows per tile: 48 rows of an expert in int4 and where the down grid is small
    (MID, I4, 512, 64), (MID, I4, 513, 128), (SMALL, B16, 192, 64), (SMALL, B16, 193, 128),
    # mid-sized to the 256-row tiles: int8 and int4 150 rows, fp8 125, bf16 112; many experts fp8 112, bf16 96
    (MID, I8, 1599, 128), (MID, I8, 1600, 256), (MID, I4, 1600, 256), (MID, F8, 1333, 128), (MID, F8, 1334, 256),
    (MID, B16, 1194, 128), (MID, B16, 1195, 256), (CFG5, F8, 3583, 128), (CFG5, F8, 3584, 256),
    (CFG5, B16, 3071, 128), (CFG5, B16, 3072, 256), ((1, 64, 2, 4096, 512), B16, 5119, 128), ((1, 64, 2, 4096, 512), B16, 5120, 256),
    # ... earlier for shared experts and a narrow F
    ((1, 64, 2, 4096, 1408), B16, 4671, 128), ((1, 64, 2, 4096, 1408), B16, 4672, 256),
    ((1, 64, 2, 3840, 640), I8, 6143, 128), ((1, 64, 2, 3840, 640), I8, 6144, 256), ((1, 64, 2, 3840, 640), I8, 11520, 256),
    ((1, 64, 2, 3840, 640), B16, 3199, 128), ((1, 64, 2, 3840, 640), B16, 3200, 256),
    ((2, 64, 1, 3840, 640), I8, 4095, 128), ((2, 64, 1, 3840, 640), I8, 4096, 256), ((2, 64, 1, 3840, 640), I4, 3839, 128),
    ((2, 64, 1, 3840, 640), I4, 3840, 256), ((2, 64, 1, 3840, 640), B16, 2559, 128), ((2, 64, 1, 3840, 640), B16, 2560, 256),
    ((1, 64, 2, 3840, 640), F8, 6143, 128), ((1, 64, 2, 3840, 640), F8, 6144, 256),
    # ... not where those would leave much of the chip idle
    (SMALL, I8, 1000, 128), (SMALL, B16, 1000, 128), (SMALL, B16, 1600, 256), ((4, 32, 2, 7168, 1024), B16, 1000, 128),
    ((4, 32, 2, 7168, 1024), B16, 1200, 256), ((2, 64, 0, 4096, 512), I8, 4800, 256), (SMALL, I8, 2000, 256),
    # ... nor where their scale tables do not hold K
    ((6, 64, 0, 8320, 1408), F8, 4000, 128), ((6, 64, 0, 4096, 8320), I4, 4000, 128), ((6, 64, 0, 8320, 1408), I8, 4000, 256),
    # fp32
    (SMALL, F32, 191, 64), (SMALL, F32, 192, 128), ((8, 128, 1, 5120, 1536), F32, 114, 64), ((8, 128, 1, 5120, 1536), F32, 115, 128),
    ((6, 64, 2, 4096, 1408), F32, 148, 64), ((6, 64, 2, 4096, 1408), F32, 149, 128),
])
def test_rows_per_tile(layer, fmt, tokens, rows):
    k, E, S, H, F = layer
    assert tile_rows(tokens, k, E, S, H, F, fmt) == rows


@pytest.mark.parametrize("fmt", [I8, I4, F8, B16])
@pytest.mark.parametrize("layer", [MID, CFG5, SMALL, (8, 128, 1, 5120, 1536), (2, 40, 1, 1024, 1024), (4, 32, 2, 7168, 1024),
                                   (2, 64, 0, 4096, 512), (6, 64, 2, 2688, 640)])
def test_rows_per_tile_grow_with_the_batch(layer, fmt):
    """A larger batch never goes back to smaller tiles on layers of these sizes. (Much smaller ones may:
    their 256-row work-groups fill one round on the chip or just start a second.)"""
    k, E, S, H, F = layer
    rows = [tile_rows(n, k, E, S, H, F, fmt) for n in range(1, 20000, 7)]
    assert rows == sorted(rows)
