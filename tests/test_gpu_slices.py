"""The bf16 scan's column slices: 16, 32 and 64 columns, chosen by how many chains a call has.  A state
column is computed the same way in all three, so while chains run whole a chain's outputs do not
depend on how many run beside it: the first 40 and the first 8 of 72 chains give the same bits as
within the 72, with every score-gate path, one chunk to five, and 72 and 69 chains (grouped by XCD
and not).  KDA likewise with its 32- and 64-column slices.  (Long chains that are few run in segments,
and how many segments depends on how many chains there are: there the same chain alone and in a batch
differs by its bf16 rounding; test_gpu_segments.py has them.)"""
import pytest
import torch

from conftest import announce
from pto_fuser_amd import _hip, gdn_chunk_forward, kda_chunk_forward, ops
from pto_fuser_amd.forwards import make_delta_inputs

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _gate(name, shape, seed):
    x = torch.randn(*shape, generator=torch.Generator().manual_seed(seed))
    sp = torch.nn.functional.softplus
    if name == "rising":                  # g > 0 in places
        return x * 0.05 - 0.03
    if name == "steep":                   # over 80 of decay inside a 16-token block
        return -sp(x) * 12.0
    return -sp(x) * 0.1


@pytest.mark.parametrize("gate", ["gentle", "rising", "steep"])
@pytest.mark.parametrize("H,T", [(72, 64), (72, 192), (69, 320)])
def test_a_chain_does_not_depend_on_its_neighbours(gate, H, T):
    announce(f"GDN bf16 slices {gate} H{H} T{T}")
    d = make_delta_inputs(1, H, T, kind="gdn", dtype=torch.bfloat16, seed=H + T, h0_std=0.02)
    d["g"] = _gate(gate, (1, H, T), T).float()
    d = {n: t.to(DEV) for n, t in d.items()}

    def run(n):
        x = {k: t[:, :n].contiguous() for k, t in d.items()}
        return gdn_chunk_forward(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"])

    o, h = run(H)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(o).all() and torch.isfinite(h).all())
    for n in (40, 8):
        on, hn = run(n)
        torch.cuda.synchronize()
        assert torch.equal(on, o[:, :n]) and torch.equal(hn, h[:, :n])


@pytest.mark.parametrize("H,T", [(72, 64), (72, 192), (69, 320)])
def test_a_kda_chain_does_not_depend_on_its_neighbours(H, T):
    announce(f"KDA bf16 slices H{H} T{T}")
    d = make_delta_inputs(1, H, T, kind="kda", dtype=torch.bfloat16, seed=H + T, h0_std=0.02, device=DEV)

    def run(n):
        x = {k: t[:, :n].contiguous() for k, t in d.items()}
        return kda_chunk_forward(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"])

    o, h = run(H)
    on, hn = run(40)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(o).all() and torch.isfinite(h).all())
    assert torch.equal(on, o[:, :40]) and torch.equal(hn, h[:, :40])


@pytest.mark.parametrize("op", ["gdn", "kda"])
def test_long_chains_on_a_workspace_without_segments(op):
    """Where few chains would run in segments, a workspace made for as many one-chunk chains keeps them whole:
    again the bits they have in a batch."""
    H, T = 72, 64 * 45
    announce(f"{op} whole long chains H{H} T{T}")
    fn, cls = (gdn_chunk_forward, ops.GdnWorkspace) if op == "gdn" else (kda_chunk_forward, ops.KdaWorkspace)
    d = make_delta_inputs(1, H, T, kind=op, dtype=torch.bfloat16, seed=H + T, h0_std=0.02, device=DEV)

    def run(n, whole):
        x = {k: t[:, :n].contiguous() for k, t in d.items()}
        ws = cls(1, n * T // 64, 64, 64, 128, 128, _hip.PF_DTYPE_BF16, DEV) if whole else None
        out = fn(x["q"], x["k"], x["v"], x["beta"], x["g"], h0=x["h0"], workspace=ws)
        torch.cuda.synchronize()
        return out

    o, h = run(H, False)                                 # 72 chains run whole
    on, hn = run(8, True)
    assert torch.equal(on, o[:, :8]) and torch.equal(hn, h[:, :8])
    assert not torch.equal(run(8, False)[0], on)         # in segments otherwise
