"""Operands that are contiguous views starting inside a larger buffer, one element past its 16-byte
boundary: the vector loads of a caller's fp32 operands need an element's alignment only.  The same bits
as with aligned copies."""
import pytest
import torch

from conftest import announce
from pto_fuser_amd import tri_inv
from pto_fuser_amd.ops import chunk_scan, gated_qk

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _randn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def _inside(t):
    """The same values, one element into a buffer."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    view = buf[1:].view(t.shape)
    view.copy_(t)
    assert view.is_contiguous() and view.data_ptr() % 16 == 4
    return view


@pytest.mark.parametrize("C", [64, 128])
def test_tri_inv_of_a_view(C):
    announce(f"tri_inv of a view C={C}")
    A = _randn(C, 5, C, C) * 0.1
    a, b = tri_inv(A), tri_inv(_inside(A))
    torch.cuda.synchronize()
    assert torch.equal(a, b)


@pytest.mark.parametrize("C,D", [(32, 64), (128, 128)])
def test_chunk_scan_of_views(C, D):
    announce(f"chunk_scan of views C={C} D={D}")
    w, u, k = (_randn(i, 1, 3, C, 2, D) * 0.05 for i in range(3))
    decay = torch.rand(1, 2, 3, D, generator=torch.Generator().manual_seed(4)).to(DEV)
    a = chunk_scan(w, u, k, decay)
    b = chunk_scan(w, _inside(u), k, _inside(decay))
    torch.cuda.synchronize()
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("C", [16, 32, 64, 128])
def test_gated_qk_with_a_mask_view(C):
    announce(f"gated_qk with a mask view C={C}")
    x, mask = _randn(1, 3 * C, 128), _randn(2, C, C)
    a = gated_qk(x, x, mask=mask, chunk_size=C)
    b = gated_qk(x, x, mask=_inside(mask), chunk_size=C)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
