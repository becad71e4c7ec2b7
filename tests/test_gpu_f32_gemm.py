"""The fp32 expert GEMMs: the K-split form for few rows per expert and the split-operand form on
the bf16 MFMAs, at the edges of their tiles and row blocks and of K, against the CPU oracle;
infinities, NaN and values next to fp32's largest come out as plain fp32 arithmetic gives them."""
import pytest
import torch

from pisceslx_amd import _lib
from pisceslx_amd import functional as yvf
from pisceslx_amd.quant import pack_experts
from pisceslx_amd.workloads import LayerSpec, make_workload
from helpers import forced_rows, tile_rows_of
from test_gpu_layer import _run_and_check

pytestmark = pytest.mark.gpu


FEW, FEWER = [0, 1, 15, 16, 17, 33, 48, 49, 64, 65], [0, 1, 15, 16, 17, 33]
MANY = [0, 1, 16, 63, 64, 65, 80, 127, 128, 129, 200]


@pytest.mark.parametrize("hidden,ffn,counts,rows", [
    (64, 64, FEW, 64), (192, 320, FEW, 64), (1024, 1088, FEW, 64), (4160, 192, FEWER, 64), (4160, 192, FEW, 128),
    (64, 64, MANY, 128), (192, 320, MANY, 128), (1024, 1088, MANY, 128), (4160, 192, MANY, 128)])
def test_segment_edges(cuda, oracle, hidden, ffn, counts, rows):
    spec = LayerSpec("f32", hidden, ffn, len(counts), 1, 1, _lib.W_F32, torch.float32, fixed_shape_mode=True)
    w = forced_rows(spec, counts)
    assert tile_rows_of(w) == rows
    _, _, routing = _run_and_check(oracle, w, label=f"f32 H={hidden} F={ffn} N={sum(counts)}")
    assert routing.counts.cpu().tolist() == counts


def _positive_experts(g, E, F, H, up_scale):
    return [tuple(torch.rand(o, i, device="cuda", generator=g).clamp(min=0.1) * s
                  for o, i, s in ((F, H, up_scale), (F, H, up_scale), (H, F, 1.0))) for _ in range(E)]


@pytest.mark.parametrize("tokens", [40, 400])  # per expert: both forms
def test_non_finite_and_largest_values(cuda, tokens):
    """Positive weights, so a row with +inf gives +inf and one with NaN gives NaN in every output;
    a row whose largest element rounds past bf16's range stays finite. Each poisons no other row."""
    H, F, E = 128, 192, 2
    g = torch.Generator(device="cuda").manual_seed(3)
    ws = _positive_experts(g, E, F, H, 1.0)
    for w in ws:
        for m in w[:2]:
            m[:, 5] = 1e-38
    N = tokens * E
    x = torch.rand(N, H, device="cuda", generator=g)
    x[3, 7], x[60 % N, 9] = float("inf"), float("nan")
    x[10, 5] = torch.finfo(torch.float32).max
    idx = (torch.arange(N, device="cuda") % E).view(N, 1)
    out = yvf.dispatch(x, torch.ones(N, 1, device="cuda"), idx, pack_experts(ws, E, _lib.W_F32))[0]
    want = torch.empty(N, H, dtype=torch.float64, device="cuda")
    for e, w in enumerate(ws):
        a, b, d = (m.double() for m in w)
        xs = x[e::E].double()
        want[e::E] = (torch.nn.functional.silu(xs @ a.t()) * (xs @ b.t())) @ d.t()
    assert torch.isposinf(out[3]).all() and torch.isnan(out[60 % N]).all()
    keep = torch.ones(N, dtype=torch.bool, device="cuda")
    keep[3] = keep[60 % N] = False
    assert torch.isfinite(out[keep]).all()
    # positive terms only: relative error of an fp32 sum of K terms is below K * 2^-24; three sums
    # and the product of two of them
    bound = (2 * H + F + 8) * 2.0 ** -24
    assert float(((out[keep].double() - want[keep]).abs() / want[keep]).max()) < bound


@pytest.mark.parametrize("tokens", [40, 400])
@pytest.mark.parametrize("x_exp,w_exp", [(-122, 100), (100, -122), (-60, 40)])
def test_operands_at_the_ends_of_the_range(cuda, tokens, x_exp, w_exp):
    """Operands next to fp32's smallest normal number keep all of their bits: positive terms only, so
    the relative error of a sum of K is below K * 2^-24."""
    H, F, E = 128, 192, 2
    g = torch.Generator(device="cuda").manual_seed(5)
    ws = _positive_experts(g, E, F, H, 2.0 ** w_exp)
    N = tokens * E
    x = torch.rand(N, H, device="cuda", generator=g).clamp(min=0.1) * 2.0 ** x_exp
    idx = (torch.arange(N, device="cuda") % E).view(N, 1)
    out = yvf.dispatch(x, torch.ones(N, 1, device="cuda"), idx, pack_experts(ws, E, _lib.W_F32))[0]
    for e, w in enumerate(ws):
        a, b, d = (m.double() for m in w)
        xs = x[e::E].double()
        want = (torch.nn.functional.silu(xs @ a.t()) * (xs @ b.t())) @ d.t()
        assert float(((out[e::E].double() - want).abs() / want).max()) < (2 * H + F + 8) * 2.0 ** -24


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3e38])
def test_a_row_depends_on_no_other_row(cuda, bad):
    """A row that is computed again because its sums are not finite changes no bit of the others."""
    H, F, E, N = 128, 192, 2, 800
    g = torch.Generator(device="cuda").manual_seed(6)
    experts = pack_experts([tuple(torch.randn(o, i, device="cuda", generator=g) * 0.05
                                  for o, i in ((F, H), (F, H), (H, F))) for _ in range(E)], E, _lib.W_F32)
    x = torch.randn(N, H, device="cuda", generator=g)
    idx = (torch.arange(N, device="cuda") % E).view(N, 1)
    w = torch.ones(N, 1, device="cuda")
    clean = yvf.dispatch(x, w, idx, experts)[0]
    rows = [0, 7, 130, 799]
    y = x.clone()
    y[rows, 11] = bad
    out = yvf.dispatch(y, w, idx, experts)[0]
    keep = torch.ones(N, dtype=torch.bool, device="cuda")
    keep[rows] = False
    assert torch.equal(out[keep], clean[keep])
