"""The mid-sized expert GEMM form (64- and 128-row tiles, a few to about a hundred rows per
expert) where it can go wrong: segment lengths at the edges of its row-block variants and
tiles, K of fewer k-steps than its weight ring, partial last column groups, and scale tables
refilled every 8192 of K."""
import numpy as np
import pytest
import torch

from helpers import ends_of_segments, few_forms_of, forced_rows, tile_rows_of
from test_gpu_layer import _run_and_check
from pisceslx_amd.workloads import LayerSpec, make_workload

pytestmark = pytest.mark.gpu

# rows per expert: the edges of the 32-, 64-, 96- and 128-row variants, an empty expert and an
# expert of two tiles; the first list has 56 rows on average (128-row tiles), the second 30 (64-row
# tiles on these small layers, but for fp8 at hidden 8320)
WIDE = [0, 1, 15, 17, 32, 33, 63, 65, 96, 97, 128, 129]
NARROW = [1, 16, 31, 33, 64, 65, 0, 30]


@pytest.mark.parametrize("counts", [WIDE, NARROW], ids=["rows128", "rows64"])
@pytest.mark.parametrize("fmt,hidden,ffn", [
    ("int8", 192, 320),    # 3 and 5 k-steps; 1.5 down column groups
    ("bf16", 64, 192),     # a single k-step
    ("int8", 1024, 1088),  # 16 and 17 k-steps (ring remainders 0 and 1), 17 gate/up groups
    ("int4", 128, 384),
    ("fp8", 384, 128),
    ("int4", 8320, 128),   # K past one scale table
    ("fp8", 8320, 128),
])
def test_segment_edges(cuda, oracle, fmt, hidden, ffn, counts):
    from pisceslx_amd import _lib
    spec = LayerSpec("mid", hidden, ffn, len(counts), 1, 1, getattr(_lib, "W_" + fmt.upper()),
                     torch.bfloat16, fixed_shape_mode=True)
    w = forced_rows(spec, counts)
    assert tile_rows_of(w) == (128 if counts is WIDE or (fmt, hidden) == ("fp8", 8320) else 64)
    _, _, routing = _run_and_check(oracle, w, label=f"mid {fmt} H={hidden} F={ffn} N={sum(counts)}")
    assert routing.counts.cpu().tolist() == counts


@pytest.mark.parametrize("layer,fmt,n", [
    ((6, 8, 256), "int8", 18), ((6, 8, 256), "int4", 18),    # few-token form to 64-row tiles
    ((6, 8, 256), "int8", 65), ((6, 8, 256), "bf16", 65),    # 64- to 128-row tiles
    ((2, 40, 1024), "int8", 21), ((2, 40, 1024), "bf16", 21),  # gate/up leaves the few-token form
    ((2, 40, 1024), "fp8", 164), ((2, 40, 1024), "int4", 192),
    ((2, 40, 1024), "int8", 961), ((2, 40, 1024), "int4", 961),
    ((2, 40, 1024), "bf16", 2817), ((2, 40, 1024), "int8", 5121), ((2, 40, 1024), "fp8", 5121),  # to 256 rows
])
def test_form_boundaries(cuda, oracle, layer, fmt, n):
    """The last token count of one form and the first of the next (hidden 512, one shared expert)."""
    from pisceslx_amd import _lib
    k, E, F = layer
    spec = LayerSpec("line", 512, F, E, k, 1, getattr(_lib, "W_" + fmt.upper()), torch.bfloat16)
    forms = []
    for m in (n - 1, n):
        w = make_workload(spec, device="cuda", lengths=[m])
        forms.append((tile_rows_of(w), few_forms_of(w) if tile_rows_of(w) == 16 else 0))
        tokens = None if m <= 1000 else np.linspace(0, m - 1, 256).astype(np.int64)
        _run_and_check(oracle, w, tokens=tokens, label=f"form line {fmt} F={F} N={m}")
    assert forms[0] != forms[1]


@pytest.mark.parametrize("fmt,light", [("int8", 64), ("int8", 63), ("int4", 64), ("fp8", 64), ("bf16", 64)])
def test_light_remainders_of_many_experts(cuda, oracle, fmt, light):
    """Prefill-sized skewed batches of many experts: remainders of 1 .. 96 rows leave the 256-row
    tiles for the mid-sized form when there are enough of them (64 at ffn 512; the tile table's
    kernel decides), whole experts and tails after full tiles alike; 97 rows keep a tile. (int4
    takes up to 64 rows, so here too few and only those of up to 32, as with bf16 at this ffn.)"""
    from pisceslx_amd import _lib
    counts = [1 + (e * 37) % 96 for e in range(light - 8)] + [256 + 96, 512 + 1] * 4
    counts += [97, 0, 256, 700, 3 * 256 + 200] * 7
    counts.append((128 - sum(counts)) % 256 + 512)  # the shared segment ends in 128 rows: not light
    counts[-1] += 97 if 0 < counts[-1] % 256 <= 96 else 0
    assert sum(0 < c % 256 <= 96 for c in counts) == light and not 0 < sum(counts) % 256 <= 96
    spec = LayerSpec("manylight", 256, 512, len(counts), 1, 1, getattr(_lib, "W_" + fmt.upper()),
                     torch.bfloat16, fixed_shape_mode=True)
    w = forced_rows(spec, counts)
    assert tile_rows_of(w) == 256
    _, _, routing = _run_and_check(oracle, w, tokens=ends_of_segments(counts, last=100),
                                   label=f"many light {fmt} N={sum(counts)} E={len(counts)}")
    assert routing.counts.cpu().tolist() == counts


# a mean of 283 rows per expert on grids large enough for the 256-row form; each list entry is six
# experts: remainders of none, 1 .. 32 (folded), 33 .. 96, more, and an expert under one tile
MANY = [256, 257, 272, 273, 288, 289, 320, 321, 544, 16] * 6


@pytest.mark.parametrize("fmt,hidden,ffn", [
    ("int8", 256, 512), ("int4", 256, 512), ("fp8", 256, 512), ("bf16", 256, 512),  # folded rows
    ("int8", 320, 448), ("bf16", 320, 448),   # partial column blocks (64 of 128, 64 of 256): no folding
    ("int8", 64, 576), ("bf16", 448, 512),    # one k-step; gate/up whole, down partial
    ("int4", 384, 640), ("fp8", 384, 640),    # down partial (128 of 256)
])
def test_tiled_forms(cuda, oracle, fmt, hidden, ffn):
    from pisceslx_amd import _lib
    spec = LayerSpec("tiled", hidden, ffn, len(MANY), 1, 1, getattr(_lib, "W_" + fmt.upper()),
                     torch.bfloat16, fixed_shape_mode=True)
    w = forced_rows(spec, MANY)
    assert tile_rows_of(w) == 256
    _, _, routing = _run_and_check(oracle, w, label=f"tiled {fmt} H={hidden} F={ffn} N={sum(MANY)}")
    assert routing.counts.cpu().tolist() == MANY


@pytest.mark.parametrize("fmt,hidden,ffn", [
    ("int8", 64, 64),      # one k-step: three wavefronts without a chunk
    ("int8", 192, 320),    # 3 and 5 k-steps: a partial chunk, one or two wavefronts
    ("int8", 1024, 1088),  # 16 and 17 k-steps: a chunk each, and one left over
    ("bf16", 64, 192), ("bf16", 1152, 640),
    ("int4", 128, 384), ("int4", 1152, 640), ("fp8", 384, 128), ("fp8", 2432, 640),
])
def test_a_few_rows(cuda, oracle, fmt, hidden, ffn):
    """The few-token form (K dealt out to the wavefronts): tiles of 1, 2, 16 and 16 + 1 rows, empty
    experts, a shared segment of several tiles, and a single token."""
    from pisceslx_amd import _lib
    counts = [0, 1, 2, 16, 17, 3, 1, 0]
    spec = LayerSpec("few", hidden, ffn, len(counts), 1, 1, getattr(_lib, "W_" + fmt.upper()),
                     torch.bfloat16, fixed_shape_mode=True)
    w = forced_rows(spec, counts)
    assert tile_rows_of(w) == 16 and few_forms_of(w) == 3
    _, _, routing = _run_and_check(oracle, w, label=f"few {fmt} H={hidden} F={ffn} N={sum(counts)}")
    assert routing.counts.cpu().tolist() == counts
    _run_and_check(oracle, make_workload(spec, device="cuda", lengths=[1]), label=f"few {fmt} N=1")
