"""GPU parity of the resident-state scan at the edges of its dispatch: every (C, D) tile, the
32-column slices (few chains) and the 64-column ones (at least one workgroup per CU), chain counts
that do and do not divide over the XCDs, one chunk and several, both snapshot types, scalar and
per-row decay.  Bounds of the stage tests: max rel 1e-4 for fp32 operands, 2e-2 for bf16 (the state
is rounded to 8 bits as a product operand every chunk); bf16 snapshots of fp32 operands add their own
rounding: 8 significant bits, so half a unit is at most 2^-8 of the value."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle.gdn_oracle import max_rel, scan_reference
from pto_fuser_amd.ops import chunk_scan

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

SHAPES = [(32, 64, 2, 3, 3), (64, 64, 1, 8, 2), (128, 64, 1, 1, 1), (32, 128, 1, 5, 4),
          (64, 128, 3, 8, 2), (128, 128, 1, 8, 3), (128, 128, 1, 1, 1),      # 32-column slices
          (32, 64, 3, 87, 2), (128, 64, 2, 128, 2), (32, 128, 2, 64, 3), (64, 128, 2, 65, 2),
          (128, 128, 2, 64, 2)]                                                # 64-column slices


CASES = [(torch.float32, *x) for x in SHAPES + [(16, 64, 1, 3, 3), (16, 128, 2, 65, 2)]] + \
        [(torch.bfloat16, *x) for x in SHAPES]           # bf16 stages take C >= 32


@pytest.mark.parametrize("dtype,C,D,B,H,nc", CASES)
def test_chunk_scan_dispatch_edges(dtype, C, D, B, H, nc):
    perdim, out16, with_h0 = (B + H + nc) % 2 == 0, H % 2 == 1, nc != 2
    announce(f"chunk_scan C={C} D={D} B={B} H={H} nc={nc} {dtype} perdim={perdim} out16={out16}")
    rng = np.random.default_rng(C + D + B * H + nc)

    def t(x, dt=torch.float32):
        return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dt)

    w = t(rng.standard_normal((B, nc, C, H, D)) * 0.02, dtype)
    u = t(rng.standard_normal((B, nc, C, H, D)) * 0.5, dtype)
    k = t(rng.standard_normal((B, nc, C, H, D)) * 0.05, dtype)
    decay = np.exp(-rng.random((B, H, nc, D) if perdim else (B, H, nc)) * 0.5).astype(np.float32)
    h0 = (rng.standard_normal((B, H, D, D)) * 0.1).astype(np.float32) if with_h0 else None
    h_out, final = chunk_scan(w.to(DEV), u.to(DEV), k.to(DEV), t(decay).to(DEV),
                              None if h0 is None else t(h0).to(DEV),
                              out_dtype=torch.bfloat16 if out16 else torch.float32)
    torch.cuda.synchronize()

    def f(x):
        return x.float().cpu().numpy().astype(np.float64)

    ref_h, ref_f = scan_reference(f(w), f(u), f(k), decay, h0=h0, dtype=np.float64)
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    assert h_out.dtype == (torch.bfloat16 if out16 else torch.float32)
    e = max_rel(f(h_out), ref_h) if np.abs(ref_h).max() > 0 else float(np.abs(f(h_out)).max())
    assert e <= tol + (2 ** -8 if out16 else 0), e
    assert max_rel(f(final), ref_f) <= tol, max_rel(f(final), ref_f)
