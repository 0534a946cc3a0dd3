"""Segmented chains of the bf16 GDN and KDA forwards (few long chains): against the fp64 oracle where the segments
divide the chain and where the last one is shorter, with and without a gate and an initial state,
against the same call on a workspace too small for segments (which runs whole chains), in both layouts of
the map kernel and at every slice width of the scan, with rising and steep gates, inside a captured
graph, without a final state, and with a NaN in one value column.  Bound of the forward tests: max abs
2e-2 on o and the final state."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import announce, record_error
from oracle.gdn_oracle import gdn_reference, kda_reference
from pto_fuser_amd import _hip, gdn_chunk_forward, kda_chunk_forward, ops
from pto_fuser_amd.forwards import as_oracle_inputs, make_delta_inputs

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
D = 128


def _base_bytes(chunks):
    """T (bf16, 64 x 64) and G (fp32) of every chunk and the scale: what whole chains need."""
    return chunks * (64 * 64 * 2 + 64 * 4) + 256


def _segmented(B, H, T):
    return _hip.load().pf_gdn_workspace_bytes(B, H, T, 64, D, D, _hip.PF_DTYPE_BF16) > _base_bytes(B * H * T // 64)


@pytest.mark.parametrize("B,H,T,kind,h0_std", [
    (1, 1, 8192, "gdn", 0.02), (1, 2, 64 * 67, "gdn", None), (1, 3, 64 * 59, "deltanet", 0.02),
    (2, 4, 4096, "deltanet", None), (1, 9, 64 * 97, "gdn", 0.02)])
def test_segmented_forward(B, H, T, kind, h0_std):
    announce(f"segmented {kind} B{B} H{H} T{T} h0={h0_std}")
    assert _segmented(B, H, T), "the shape is meant to run in segments"
    inp = make_delta_inputs(B, H, T, kind=kind, dtype=torch.bfloat16, seed=T + H, h0_std=h0_std)
    d = {n: (None if t is None else t.to(DEV)) for n, t in inp.items()}
    o, h = gdn_chunk_forward(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"])
    o2, h2 = gdn_chunk_forward(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"])
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(h, h2)
    x = as_oracle_inputs(inp)
    g = x["g"] if x["g"] is not None else np.zeros_like(x["beta"])
    ro, rh = gdn_reference(x["q"], x["k"], x["v"], x["beta"], g, h0=x["h0"], C=64, dtype=np.float64)
    for name, got, ref in (("o", o, ro), ("h", h, rh)):
        e = record_error(f"segments {kind} B{B} H{H} T{T}", name, got.cpu().numpy(), ref, "max abs <= 0.02")
        assert e["abs"] <= 2e-2, (name, e)


@pytest.mark.parametrize("B,H,T,gate_scale,h0_std", [
    (1, 1, 4096, 0.05, 0.02), (1, 2, 64 * 67, 0.3, None), (1, 3, 64 * 59, 0.002, 0.02)])
def test_segmented_kda_forward(B, H, T, gate_scale, h0_std):
    announce(f"segmented kda B{B} H{H} T{T} gate {gate_scale} h0={h0_std}")
    lib = _hip.load()
    chunks = B * H * T // 64                               # W, QE, KB, T diag(beta) and the decay
    base = chunks * (3 * 64 * D * 2 + 64 * 64 * 2 + D * 4)
    assert lib.pf_kda_workspace_bytes(B, H, T, 64, D, D, _hip.PF_DTYPE_BF16) > base + 4 * 256
    inp = make_delta_inputs(B, H, T, kind="kda", dtype=torch.bfloat16, seed=T + H, h0_std=h0_std,
                            gate_scale=gate_scale)
    d = {n: (None if t is None else t.to(DEV)) for n, t in inp.items()}
    o, h = kda_chunk_forward(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"])
    o2, h2 = kda_chunk_forward(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"])
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(h, h2)
    x = as_oracle_inputs(inp)
    ro, rh = kda_reference(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"], C=64, dtype=np.float64)
    for name, got, ref in (("o", o, ro), ("h", h, rh)):
        e = record_error(f"segments kda B{B} H{H} T{T}", name, got.cpu().numpy(), ref, "max abs <= 0.02")
        assert e["abs"] <= 2e-2, (name, e)


def test_small_workspace_runs_whole_chains():
    """A handle that holds what whole chains need (reserved for another shape of as many chunks) still
    serves the call; both routes agree within their bf16 rounding."""
    B, H, T = 1, 2, 8192
    announce(f"whole chains on a small workspace B{B} H{H} T{T}")
    lib = _hip.load()
    assert _segmented(B, H, T) and not _segmented(16, 16, T // 128)
    d = make_delta_inputs(B, H, T, kind="gdn", dtype=torch.bfloat16, seed=5, h0_std=0.02, device=DEV)
    seg = gdn_chunk_forward(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"])
    ws = ctypes.c_void_p(lib.pf_gdn_create())
    try:
        assert lib.pf_gdn_reserve(ws, 16, 16, T // 128, 64, D, D, _hip.PF_DTYPE_BF16) == _hip.PF_OK
        o, h = torch.empty_like(seg[0]), torch.empty_like(seg[1])
        st = lib.pf_gdn_exec(*(_hip.ptr(t) for t in (d["q"], d["k"], d["v"], d["beta"], d["g"], d["h0"], o, h)),
                             B, H, T, 64, D, D, _hip.PF_DTYPE_BF16, D ** -0.5, ws, _hip.current_stream_handle(DEV))
        _hip.check("pf_gdn_exec", st)
        torch.cuda.synchronize()
    finally:
        lib.pf_gdn_teardown(ws)
    for a, b in zip(seg, (o, h)):
        assert not torch.equal(a, b)                     # the other route ran
        # two correct bf16 forwards lie 2.9e-3 from float64 each: sqrt(2) of that apart, times two
        assert float((a - b).norm() / b.norm()) <= 8.2e-3


def test_nan_stays_in_its_column_and_behind_its_token():
    B, H, T, tok, col = 1, 2, 8192, 5000, 17
    announce(f"segmented NaN containment B{B} H{H} T{T}")
    d = make_delta_inputs(B, H, T, kind="gdn", dtype=torch.bfloat16, seed=6, device=DEV)
    d["v"][0, 0, tok, col] = float("nan")
    o, h = gdn_chunk_forward(d["q"], d["k"], d["v"], d["beta"], d["g"])
    torch.cuda.synchronize()
    bad = torch.isnan(o)
    assert bad[0, 0, tok:, col].all() and bool(torch.isnan(h)[0, 0, :, col].all())
    assert not bad[0, 1].any() and not bad[0, 0, :tok // 64 * 64].any()
    others = [c for c in range(D) if c != col]
    assert not bad[0, 0][:, others].any() and not torch.isnan(h)[0, 0][:, others].any()


@pytest.mark.parametrize("op,B,H,T", [
    ("gdn", 1, 9, 64 * 97), ("gdn", 4, 5, 64 * 107), ("kda", 1, 2, 64 * 67), ("kda", 1, 10, 64 * 65)])
def test_state_updated_in_place(op, B, H, T):
    """final_out is h0 itself: the first segment starts from h0 in one workgroup while the last segment's
    writes the final state over it, so the call keeps a copy of h0.  The same bits as with two tensors, in
    both map layouts (9 and 20 chains) and at both KDA slice widths."""
    announce(f"in-place state, segmented {op} B{B} H{H} T{T}")
    d = make_delta_inputs(B, H, T, kind=op, dtype=torch.bfloat16, seed=T + H, h0_std=0.5, device=DEV)
    fn = gdn_chunk_forward if op == "gdn" else kda_chunk_forward
    o, h = fn(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"])
    state = d["h0"].clone()
    o2, h2 = fn(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=state, final_out=state)
    torch.cuda.synchronize()
    assert h2.data_ptr() == state.data_ptr()
    assert torch.equal(o, o2) and torch.equal(h, h2)


def _forward(op, d, whole=False, **kw):
    """The forward; ``whole`` runs it on a workspace made for as many one-chunk chains, which has no
    room for segments."""
    fn, cls = (gdn_chunk_forward, ops.GdnWorkspace) if op == "gdn" else (kda_chunk_forward, ops.KdaWorkspace)
    B, H, T, _ = d["q"].shape
    ws = cls(B, H * T // 64, 64, 64, D, D, _hip.PF_DTYPE_BF16, DEV) if whole else None
    out = fn(d["q"], d["k"], d["v"], d["beta"], d["g"], h0=d["h0"], workspace=ws, **kw)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("op,B,H,T", [("gdn", 1, 2, 64 * 256), ("kda", 1, 2, 64 * 64), ("kda", 1, 10, 64 * 65)])
def test_maps_outside_fp32_range(op, B, H, T):
    """A segment's map overflows (long keys make the recurrence grow by about e^15 per chunk; KDA: gates
    that rise by e^16 per chunk) while the state it is applied to is exactly zero: v is zero up to the
    last two chunks.  The chain is then run whole: finite, and the whole chain's bits."""
    announce(f"segment maps outside fp32 range {op} B{B} H{H} T{T}")
    d = make_delta_inputs(B, H, T, kind=op, dtype=torch.bfloat16, seed=T, device=DEV)
    d["v"][:, :, :T - 128] = 0
    if op == "gdn":
        d["k"] = (d["k"].float() * 5).bfloat16()
    else:
        d["g"].fill_(0.25)
    assert d["h0"] is None
    o, h = _forward(op, d)
    assert bool(torch.isfinite(o).all() and torch.isfinite(h).all())
    assert bool((o[:, :, :T - 128] == 0).all()) and float(o.abs().max()) > 0
    wo, wh = _forward(op, d, whole=True)
    assert torch.equal(o, wo) and torch.equal(h, wh)


def _against_oracle(case, op, inp, o, h):
    x = as_oracle_inputs(inp)
    if op == "kda":
        ro, rh = kda_reference(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"], C=64, dtype=np.float64)
    else:
        g = x["g"] if x["g"] is not None else np.zeros_like(x["beta"])
        ro, rh = gdn_reference(x["q"], x["k"], x["v"], x["beta"], g, h0=x["h0"], C=64, dtype=np.float64)
    for name, got, ref in (("o", o, ro), ("h", h, rh)):
        got = got.cpu().numpy()
        assert np.isfinite(got).all(), (case, name)
        e = record_error(case, name, got, ref, "max abs <= 0.02")
        assert e["abs"] <= 2e-2, (case, name, e)


def _segments(op, B, H, T):
    """How many segments a chain of the shape has room for in its own workspace (1: none)."""
    size = getattr(_hip.load(), f"pf_{op}_workspace_bytes")
    args = (64, D, D, _hip.PF_DTYPE_BF16)
    extra = size(B, H, T, *args) - size(B, H * T // 64, 64, *args)   # as many one-chunk chains
    return 1 + extra // (B * H * 2 * D * D * 4)


@pytest.mark.parametrize("B,H,nc,kind,h0_std,count", [
    (4, 5, 107, "gdn", 0.02, 12), (2, 9, 107, "deltanet", None, 14),   # nine chunks, the last of eight; 8 and 3
    (1, 17, 85, "gdn", None, 15), (1, 22, 113, "deltanet", 0.02, 10)])  # six and one; twelve and five
def test_segmented_forward_with_both_maps_in_a_workgroup(B, H, nc, kind, h0_std, count):
    """More than one generation of maps: D and M of a segment share a workgroup."""
    announce(f"segmented {kind}, maps together B{B} H{H} nc{nc} h0={h0_std}")
    seg = _segments("gdn", B, H, 64 * nc)
    assert seg == count and B * H * (2 * seg - 3) > 256
    inp = make_delta_inputs(B, H, 64 * nc, kind=kind, dtype=torch.bfloat16, seed=nc + H, h0_std=h0_std)
    d = {n: (None if t is None else t.to(DEV)) for n, t in inp.items()}
    o, h = _forward("gdn", d)
    _against_oracle(f"segments {kind} B{B} H{H} nc{nc}", "gdn", inp, o, h)


@pytest.mark.parametrize("B,H,nc", [(1, 2, 67), (1, 17, 85)])          # maps apart, maps together
@pytest.mark.parametrize("gate", ["rising", "steep"])
def test_segmented_forward_gates(gate, B, H, nc):
    """Gates that rise in places (g > 0), and over 80 of decay inside a 16-token block."""
    announce(f"segmented gdn {gate} gate B{B} H{H} nc{nc}")
    assert _segments("gdn", B, H, 64 * nc) > 1
    inp = make_delta_inputs(B, H, 64 * nc, kind="gdn", dtype=torch.bfloat16, seed=nc, h0_std=0.02)
    x = torch.randn(B, H, 64 * nc, generator=torch.Generator().manual_seed(nc))
    inp["g"] = x * 0.05 - 0.03 if gate == "rising" else -torch.nn.functional.softplus(x) * 12.0
    o, h = _forward("gdn", {n: (None if t is None else t.to(DEV)) for n, t in inp.items()})
    _against_oracle(f"segments gdn {gate} B{B} H{H} nc{nc}", "gdn", inp, o, h)


@pytest.mark.parametrize("B,H,nc,gate_scale,h0_std,units", [
    (2, 5, 65, 0.05, 0.02, 110), (1, 12, 65, 0.3, None, 120),          # 64-column scan, last segment shorter
    (1, 2, 40, 1.0, 0.02, 16)])                                        # a chunk decays by up to e^-65
def test_segmented_kda_forward_edges(B, H, nc, gate_scale, h0_std, units):
    announce(f"segmented kda B{B} H{H} nc{nc} gate {gate_scale} h0={h0_std}")
    assert B * H * _segments("kda", B, H, 64 * nc) == units
    inp = make_delta_inputs(B, H, 64 * nc, kind="kda", dtype=torch.bfloat16, seed=nc + H, h0_std=h0_std,
                            gate_scale=gate_scale)
    o, h = _forward("kda", {n: (None if t is None else t.to(DEV)) for n, t in inp.items()})
    _against_oracle(f"segments kda B{B} H{H} nc{nc} gate {gate_scale}", "kda", inp, o, h)


def test_small_workspace_runs_whole_kda_chains():
    B, H, T = 1, 2, 64 * 67
    announce(f"whole KDA chains on a small workspace B{B} H{H} T{T}")
    assert _segments("kda", B, H, T) > 1
    inp = make_delta_inputs(B, H, T, kind="kda", dtype=torch.bfloat16, seed=5, h0_std=0.02)
    d = {n: t.to(DEV) for n, t in inp.items()}
    seg, (o, h) = _forward("kda", d), _forward("kda", d, whole=True)
    assert not torch.equal(seg[0], o) and not torch.equal(seg[1], h)   # the other route ran
    _against_oracle(f"whole kda B{B} H{H} T{T}", "kda", inp, o, h)


@pytest.mark.parametrize("op", ["gdn", "kda"])
def test_segmented_forward_without_final_state(op):
    B, H, T = 1, 3, 64 * 59
    announce(f"segmented {op} without a final state B{B} H{H} T{T}")
    assert _segments(op, B, H, T) > 1
    d = make_delta_inputs(B, H, T, kind=op, dtype=torch.bfloat16, seed=8, h0_std=0.02, device=DEV)
    o, h = _forward(op, d)
    o2, none = _forward(op, d, output_final_state=False)
    assert none is None and h is not None and torch.equal(o, o2)


@pytest.mark.parametrize("op,B,H,nc", [("gdn", 1, 2, 67), ("gdn", 1, 17, 85), ("kda", 1, 2, 67)])
def test_segmented_forward_in_a_graph(op, B, H, nc):
    """Captured with the state carried in place and replayed on new operands, with eager calls between the
    replays: every replay gives the eager bits."""
    announce(f"segmented {op} in a graph B{B} H{H} nc{nc}")
    assert _segments(op, B, H, 64 * nc) > 1
    fn = gdn_chunk_forward if op == "gdn" else kda_chunk_forward

    def draw(seed):
        return make_delta_inputs(B, H, 64 * nc, kind=op, dtype=torch.bfloat16, seed=seed, h0_std=0.02, device=DEV)

    x = draw(0)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    args = [x[n] for n in ("q", "k", "v", "beta", "g")]
    out = torch.empty(B, H, 64 * nc, D, device=DEV)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        fn(*args, h0=x["h0"], out=out)                   # the stream's workspace
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            fn(*args, h0=x["h0"], out=out, final_out=x["h0"])
    for seed in (1, 2, 3):
        d = draw(seed)
        o, h = _forward(op, d)
        for n in x:
            x[n].copy_(d[n])
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, o) and torch.equal(x["h0"], h), seed
