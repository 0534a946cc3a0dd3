"""The opaque inverse at its edges: one block, more blocks than fit one generation of workgroups, and
what lies on and above the diagonal of A (infinities and NaN included) never read; T is exactly zero
above its diagonal and one on it.  fp32 bound of the inverse tests, max rel 1e-4."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle.gdn_oracle import max_rel, tri_inv_reference
from pto_fuser_amd import tri_inv

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("C,M", [(64, 1), (64, 2600), (128, 1), (128, 900), (48, 3), (16, 5)])
def test_tri_inv_edges(C, M):
    announce(f"tri_inv C={C} M={M}")
    rng = np.random.default_rng(C + M)
    A = (rng.standard_normal((M, C, C)) * 0.1).astype(np.float32)
    low = np.tril(A, -1)
    junk = np.where(rng.random((M, C, C)) < 0.5, np.float32("nan"), np.float32("inf"))
    A = np.where(np.tril(np.ones((C, C), bool), -1), A, junk).astype(np.float32)
    T = tri_inv(torch.from_numpy(A).to(DEV)).cpu().numpy()
    keep = np.tril(np.ones((C, C), bool), -1)
    assert np.all(T[:, np.triu(np.ones((C, C), bool), 1)] == 0)
    assert np.all(T[:, np.arange(C), np.arange(C)] == 1)
    pick = sorted({0, M // 2, M - 1})
    ref = tri_inv_reference(low[pick])
    assert max_rel(T[pick][:, keep], ref[:, keep]) <= 1e-4
