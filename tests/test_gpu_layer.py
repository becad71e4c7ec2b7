"""Yv MoE layer forward on the GPU against the CPU oracle.

For every configuration (full size where the CPU oracle finishes in seconds, reduced N /
expert count otherwise) the GPU gate logits are checked against float64, the device
capacity against the oracle's, the routing bit for bit given the GPU's fp32 logits, and
the outputs against the oracle's reference forward: bf16 max-abs <= 2e-2 and cosine >=
0.9999; fp32 max-abs <= 1e-4 and cosine >= 0.999999.

bf16 tolerance (tests/helpers.py bf16_allowance): every element within 2e-2 of the oracle,
except where |want| >= 2: two bf16 steps (0.03125) in [2, 4), where the reference's own bf16
chain lands two steps from the correctly rounded oracle (pinned on the CPU by
tests/test_oracle_bf16_envelope.py at cfg4, 384 tokens), and the adjacent bf16 value from 4 up;
at most 1e-5 of the elements above 2e-2; cosine >= 0.9999. The raw max-abs is printed.
"""
import numpy as np
import pytest
import torch

from pisceslx_amd import functional as yvf
from pisceslx_amd.workloads import make_workload, mix_weights, router_state

from helpers import check_close, ends_of_segments, few_forms_of, forced_rows, oracle_params, tile_rows_of

pytestmark = pytest.mark.gpu

def _run_and_check(oracle, w, skip=None, tokens=None, label=None):
    spec = w.spec
    print(f"layer {spec.name} N={w.n_tokens} H={spec.hidden} E={spec.num_experts} "
          f"F={spec.ffn} fmt={spec.fmt}", flush=True)
    st = router_state(w)
    mix = mix_weights(w)
    x = w.x
    logits = yvf.router_logits(x, st)
    out, shared, routing = yvf.moe_forward(x, st, w.experts, mix, skip)
    torch.cuda.synchronize()
    E, k = spec.num_experts, spec.top_k
    lg = logits[:, :E].cpu().numpy()
    xc = x.cpu()
    ref_lg = oracle.router_logits(xc, w.gate_weight.cpu())
    np.testing.assert_allclose(lg, ref_lg, rtol=0, atol=2e-4 * max(1.0, np.abs(ref_lg).max()))
    params = oracle_params(w)
    cap = int(routing.capacity.item())
    if spec.fixed_shape_mode:
        assert cap == -1
    else:
        assert cap == oracle.layer_capacity(params, xc)
    o = oracle.layer_forward(xc, params, logits=lg, cap=cap,
                             skip=None if skip is None else skip.cpu(), tokens=tokens)
    r = o["routing"]
    assert np.array_equal(routing.indices.cpu().numpy(), r.indices.astype(np.int64))
    assert np.array_equal(routing.weights.cpu().numpy().view(np.uint32), r.weights.view(np.uint32))
    assert np.array_equal(routing.perm.cpu().numpy(), r.perm)
    assert np.array_equal(routing.counts.cpu().numpy(), r.counts)
    got = out.cpu()
    want = o["out"]
    if tokens is not None:
        got, want = got[tokens], want[tokens]
    if label is None:
        label = f"layer {spec.name} N={w.n_tokens} E={spec.num_experts}" + (
            "" if tokens is None else f" ({len(tokens)} sampled tokens)")
    check_close(got, want, label)
    if spec.num_shared > 0:
        gs, ws = shared.cpu(), o["shared"]
        if tokens is not None:
            gs, ws = gs[tokens], ws[tokens]
        check_close(gs, ws, label + " shared")
    return out, shared, routing


@pytest.mark.parametrize("name,kw", [
    ("cfg1", {}),
    ("cfg2", {}),
    ("cfg3", {"n_tokens": 512}),
    ("cfg4", {"n_tokens": 384}),
    ("cfg5", {"n_tokens": 384, "num_experts": 32}),
    ("cfg5", {"n_tokens": 64, "num_experts": 32}),       # fp8 weights, 16 rows of an expert: mid-sized form
    ("cfg2", {"n_tokens": 1}),                             # one token: six one-row experts
    ("cfg2", {"n_tokens": 200}),                           # the small-batch routing at 200 tokens
])
def test_layer_matches_oracle(cuda, oracle, name, kw):
    w = make_workload(name, device="cuda", **kw)
    _run_and_check(oracle, w)


def test_layer_with_skip_buffer(cuda, oracle):
    w = make_workload("cfg2", device="cuda", n_tokens=40)
    g = torch.Generator(device="cuda").manual_seed(3)
    skip = torch.randn(40, w.spec.hidden, device="cuda", generator=g).to(torch.bfloat16)
    _run_and_check(oracle, w, skip=skip)


def test_cfg3_full_size_sampled_tokens(cuda, oracle):
    w = make_workload("cfg3", device="cuda")
    rng = np.random.default_rng(0)
    tokens = np.sort(rng.choice(w.n_tokens, 96, replace=False))
    _run_and_check(oracle, w, tokens=tokens)


def test_cfg5_full_size_sampled_tokens(cuda, oracle):
    """cfg5 at its full size: 8192 tokens, 256 fp8 experts (128x128 block scales), top-8,
    fixed-shape routing with the Zipf(1.2) expert bias and 16 experts that receive no tokens,
    so the skewed tile table of the LDS-tiled form (tiles of every fill, empty experts) is the
    one the kernels run; checked on sampled tokens."""
    w = make_workload("cfg5", device="cuda")
    assert w.n_tokens == 8192 and w.spec.num_experts == 256
    rng = np.random.default_rng(2)
    tokens = np.sort(rng.choice(w.n_tokens, 64, replace=False))
    _, _, routing = _run_and_check(oracle, w, tokens=tokens)
    counts = routing.counts.cpu().numpy()
    assert int((counts == 0).sum()) >= 16
    assert counts.max() > 8 * counts[counts > 0].min()  # the load is skewed


def test_cfg4_full_size_tiled_int4_sampled_tokens(cuda, oracle):
    """cfg4 at its full size (4344 tokens, 271 rows per expert): the LDS-tiled form with int4 weights
    (group scales staged in LDS, 512-byte weight blocks), checked on sampled tokens."""
    w = make_workload("cfg4", device="cuda")
    rng = np.random.default_rng(1)
    tokens = np.sort(rng.choice(w.n_tokens, 64, replace=False))
    _run_and_check(oracle, w, tokens=tokens)


def test_bf16_and_small_shapes(cuda, oracle):
    # unquantized bf16 experts on a small layer, ragged odd lengths
    from pisceslx_amd import _lib
    from pisceslx_amd.workloads import LayerSpec
    spec = LayerSpec("tiny_bf16", 256, 384, 12, 3, 1, _lib.W_BF16, torch.bfloat16)
    w = make_workload(spec, device="cuda", lengths=[37, 1, 90])
    _run_and_check(oracle, w)


def test_bf16_tiled_prefill_shapes(cuda, oracle):
    # unquantized bf16 experts with many rows per expert (the mid-sized form's 128-row tiles), segment
    # ends inside tiles
    from pisceslx_amd import _lib
    from pisceslx_amd.workloads import LayerSpec
    spec = LayerSpec("tiled_bf16", 256, 384, 4, 2, 1, _lib.W_BF16, torch.bfloat16)
    w = make_workload(spec, device="cuda", lengths=[200, 77, 3])
    assert tile_rows_of(w) == 128
    _run_and_check(oracle, w)


@pytest.mark.parametrize("fmt,hidden", [("int8", 256), ("int4", 256), ("fp8", 256), ("bf16", 256),
                                        ("int4", 6144)])
def test_tiled_folded_remainders(cuda, oracle, fmt, hidden):
    """Expert segments of 256, 257, 272, 273, 288, 289, 320, 321, 544 and 16 rows, seven of each,
    and a shared segment of 19852 rows (77 x 256 + 140), forced through one-hot gate rows: the
    LDS-tiled form folds a remainder of 1 .. 32 rows into the segment's last full tile (a second
    launch runs those tiles; 17+ rows reach the second wavefront row's block), sends remainders of
    33 .. 64 rows and a segment of 16 rows to the mid-sized form's light tiles, and keeps 65 rows as
    a tile of its own. int4 at hidden 6144 takes the gate/up form for K > 5120 (2-stage ring beside
    the 64-group scale table); its ffn of 256 leaves no light tiles."""
    from pisceslx_amd import _lib
    from pisceslx_amd.workloads import LayerSpec
    counts = [256, 257, 272, 273, 288, 289, 320, 321, 544, 16] * 7
    spec = LayerSpec("folds", hidden, 512 if hidden == 256 else 256, len(counts), 1, 1, getattr(_lib, "W_" + fmt.upper()),
                     torch.bfloat16, fixed_shape_mode=True)
    w = forced_rows(spec, counts)
    assert tile_rows_of(w) == 256
    _, _, routing = _run_and_check(oracle, w, tokens=ends_of_segments(counts, last=66),
                                   label=f"layer folded tiles {fmt} H={hidden} N={sum(counts)}")
    assert routing.counts.cpu().tolist() == counts


@pytest.mark.parametrize("fmt,hidden", [("int8", 1024), ("int4", 1024), ("fp8", 1024), ("bf16", 1024),
                                        ("fp8", 896)])
def test_tiled_light_remainders(cuda, oracle, fmt, hidden):
    """Skewed prefill-sized batches (mean under two 256-row tiles per expert, no folding) with too few
    light remainders for all of them to leave the tiles: one of at most 32 rows runs on the
    mid-sized form after the LDS-tiled launch (segments of 10, 32, 256 + 24 and 256 + 32 rows), a
    longer remainder keeps its 256-row tile (33, 57, 512 + 88, and the shared segment's 48 x 256 +
    60), and a segment of exactly 256 rows has no remainder; forced through one-hot gate rows."""
    from pisceslx_amd import _lib
    from pisceslx_amd.workloads import LayerSpec
    counts = [10, 32, 33, 256, 280, 288, 600, 57] * 3 + [256] * 30
    spec = LayerSpec("light", hidden, 768, len(counts), 1, 1, getattr(_lib, "W_" + fmt.upper()), torch.bfloat16,
                     fixed_shape_mode=True)
    w = forced_rows(spec, counts)
    assert w.n_tokens == 48 * 256 + 60 and tile_rows_of(w) == 256
    _, _, routing = _run_and_check(oracle, w, tokens=ends_of_segments(counts),
                                   label=f"layer light remainders {fmt} H={hidden} N={w.n_tokens}")
    assert routing.counts.cpu().tolist() == counts


def _shared_spec(fmt_name, S):
    from pisceslx_amd import _lib
    from pisceslx_amd.workloads import LayerSpec
    fmt = {"int8": _lib.W_INT8, "int4": _lib.W_INT4, "fp8": _lib.W_FP8, "bf16": _lib.W_BF16}[fmt_name]
    return LayerSpec(f"shared_{fmt_name}_s{S}", 1024, 512, 16, 4, S, fmt, torch.bfloat16)


@pytest.mark.parametrize("fmt,S,n", [("int8", 2, 23), ("fp8", 3, 5), ("int4", 1, 64),
                                     ("bf16", 2, 17)])
def test_decode_shared_expert_segments(cuda, oracle, fmt, S, n):
    """Decode sizes of a small layer (the few-token form; int4's 64 tokens the mid-sized one): the
    shared experts' segments of the tile table (rows N*k + s*N, tiles cut at each segment end) for
    every weight format, 1-3 shared experts and batches that end inside a 16-row tile."""
    w = make_workload(_shared_spec(fmt, S), device="cuda", lengths=[n])
    assert (tile_rows_of(w), few_forms_of(w)) == (64 if n == 64 else 16, 3)
    _run_and_check(oracle, w, label=f"shared segments {fmt} S={S} N={n}")


@pytest.mark.parametrize("fmt,S,n,few", [("int8", 2, 33, 0), ("int4", 1, 33, 0), ("fp8", 3, 24, 0), ("fp8", 1, 49, 0),
                                         ("bf16", 2, 40, 0), ("int8", 0, 33, 2), ("bf16", 0, 40, 2)])
def test_decode_on_the_streaming_form(cuda, oracle, fmt, S, n, few):
    """Decode sizes of a layer large enough for the streaming form, in both GEMMs or in gate/up alone
    (few: the GEMMs on the few-token form): 16-row tiles of 3 to 6 rows, the shared experts' 64-row
    items, batches that end inside either, none to three shared experts."""
    from pisceslx_amd import _lib
    from pisceslx_amd.workloads import LayerSpec
    spec = LayerSpec("streaming", 1536, 2048, 32, 4, S, getattr(_lib, "W_" + fmt.upper()), torch.bfloat16)
    w = make_workload(spec, device="cuda", lengths=[n])
    assert (tile_rows_of(w), few_forms_of(w)) == (16, few)
    _run_and_check(oracle, w, label=f"streaming {fmt} S={S} N={n}")


def test_forward_is_deterministic(cuda, oracle):
    w = make_workload("cfg3", device="cuda", n_tokens=700)
    st = router_state(w)
    mix = mix_weights(w)
    a = yvf.moe_forward(w.x, st, w.experts, mix, None)[0]
    b = yvf.moe_forward(w.x, st, w.experts, mix, None)[0]
    assert torch.equal(a, b)


def test_misaligned_pointers_rejected(cuda):
    """x, y / out and the workspace are accessed in 16-byte vectors: the FFN entry points
    reject pointers that are not 16-byte aligned before launching anything."""
    import ctypes

    from pisceslx_amd import _lib
    w = make_workload("cfg2", device=cuda, n_tokens=8)
    st, mix = router_state(w), mix_weights(w)
    N, H = w.x.shape
    ws = torch.empty(yvf.workspace_bytes(N, _lib.ACT_BF16, st, w.experts) + 64, dtype=torch.uint8,
                     device=cuda)
    out, _, routing = yvf.moe_forward(w.x, st, w.experts, mix, None, workspace=ws)
    y = torch.empty(N * (w.spec.top_k + w.spec.num_shared) + 1, H, dtype=torch.bfloat16, device=cuda)
    e, o, r = w.experts.struct(), routing.struct(), st.struct()
    stream = torch.cuda.current_stream().cuda_stream
    lib = _lib.lib()
    for xp, yp, wp in ((w.x.data_ptr() + 2, y.data_ptr(), ws.data_ptr()),
                       (w.x.data_ptr(), y.data_ptr() + 8, ws.data_ptr()),
                       (w.x.data_ptr(), y.data_ptr(), ws.data_ptr() + 4)):
        rc = lib.yvmoe_expert_ffn(xp, _lib.ACT_BF16, N, w.spec.top_k, ctypes.byref(e), ctypes.byref(o),
                                  yp, wp, ws.numel() - 8, stream)
        assert rc == _lib.YVMOE_ERR_ARG and b"16-byte" in lib.yvmoe_last_error()
        rc = lib.yvmoe_forward(xp, _lib.ACT_BF16, N, ctypes.byref(r), ctypes.byref(e), mix.data_ptr(),
                               None, yp, None, ctypes.byref(o), wp, ws.numel() - 8, stream)
        assert rc == _lib.YVMOE_ERR_ARG and b"16-byte" in lib.yvmoe_last_error()
    torch.cuda.synchronize()
    ref, _, _ = yvf.moe_forward(w.x, st, w.experts, mix, None, workspace=ws)
    assert torch.equal(ref, out)
