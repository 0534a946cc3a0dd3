"""GPU parity of the two score stages over every (C, D) tile, both layouts, both output types, with and
without gates, prescales and an explicit mask, and one chunk: a wave owns whole query blocks (fewer
blocks than waves at C = 16 and 32, two per wave at C = 128), bf16 scores leave as pairs of tiles.
Bounds of the stage tests: max rel 1e-4 for fp32 operands, 1e-2 for bf16; bf16 scores of fp32 operands
add their own rounding, 2^-8 of the value (8 significant bits)."""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle.gdn_oracle import gated_qk_reference, max_rel
from pto_fuser_amd.ops import gated_qk, qkv_flash

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = [(torch.float32, C, D) for C in (16, 32, 64, 128) for D in (64, 128)] + \
        [(torch.bfloat16, C, D) for C in (32, 64, 128) for D in (64, 128)]


def _rows(rng, shape, dtype, scale=0.2):
    return torch.from_numpy((rng.standard_normal(shape) * scale).astype(np.float32)).to(dtype)


def _np(t):
    return t.float().cpu().numpy().astype(np.float64)


def _dev(x):
    return None if x is None else torch.as_tensor(x, dtype=torch.float32).to(DEV)


@pytest.mark.parametrize("form", ["plain", "gated", "scaled", "mask", "heads"])
@pytest.mark.parametrize("dtype,C,D", TILES)
def test_gated_qk_tiles(dtype, C, D, form):
    rng = np.random.default_rng(C * D + len(form))
    H, nc, causal = (3 if form == "heads" else 1), (5 if form != "plain" else 1), form != "gated"
    out16 = form in ("gated", "heads")
    announce(f"gated_qk {form} C={C} D={D} {dtype} out16={out16}")
    n = nc * C * H
    a = _rows(rng, (n, D), dtype)
    b = a if form == "gated" else _rows(rng, (n, D), dtype)
    G = beta = sa = sb = mask = None
    if form in ("gated", "heads"):
        g = -np.log1p(np.exp(rng.standard_normal((nc, C, H)))) * 0.1
        G = np.cumsum(g, axis=1).astype(np.float32).reshape(n)
        beta = (1 / (1 + np.exp(-rng.standard_normal(n)))).astype(np.float32)
    if form == "scaled":
        sa, sb = (rng.random((n, D)).astype(np.float32) + 0.5 for _ in range(2))
    if form == "mask":
        mask = ((rng.random((C, C)) < 0.5) * rng.random((C, C))).astype(np.float32)
    L = gated_qk(a.to(DEV), b.to(DEV), _dev(G), _dev(beta), chunk_size=C, heads=H, causal=causal,
                 mask=_dev(mask), a_scale=_dev(sa), b_scale=_dev(sb),
                 out_dtype=torch.bfloat16 if out16 else torch.float32)
    torch.cuda.synchronize()

    def chunks(x):                          # rows (c*C + i)*H + h -> [c*H + h, i]
        return x.reshape(nc, C, H, -1).transpose(0, 2, 1, 3).reshape(nc * H, C, -1)

    ad = chunks(_np(a) * (1 if sa is None else sa))
    bd = chunks(_np(b) * (1 if sb is None else sb))
    gz = np.zeros((nc * H, C)) if G is None else chunks(G.astype(np.float64))[..., 0]
    bz = np.ones((nc * H, C)) if beta is None else chunks(beta.astype(np.float64))[..., 0]
    if mask is not None:
        ref = np.einsum("mid,mjd->mij", ad, bd) * mask
    else:
        ref = gated_qk_reference(ad, bd, gz, bz, causal=causal, dtype=np.float64)
    got = chunks(_np(L).reshape(n, C))
    tol = (1e-4 if dtype == torch.float32 else 1e-2) + (2 ** -8 if out16 else 0)
    assert max_rel(got, ref) <= tol, max_rel(got, ref)
    if mask is None:
        keep = np.tril(np.ones((C, C)), 0 if causal else -1).astype(bool)
        assert np.all(got[:, ~keep] == 0)


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("dtype,C,D", TILES)
def test_qkv_flash_tiles(dtype, C, D, scaled):
    M = 1 if scaled and C == 128 else 7
    announce(f"qkv_flash C={C} D={D} {dtype} M={M} scaled={scaled}")
    rng = np.random.default_rng(C * D + scaled)
    q, k, v = (_rows(rng, (M, C, D), dtype, s) for s in (0.2, 0.2, 1.0))
    g = beta = sq = sk = None
    if scaled:
        sq, sk = (rng.random((M, C, D)).astype(np.float32) + 0.5 for _ in range(2))
    else:
        g = np.cumsum(-np.log1p(np.exp(rng.standard_normal((M, C)))) * 0.1, axis=1).astype(np.float32)
        beta = (1 / (1 + np.exp(-rng.standard_normal((M, C))))).astype(np.float32)
    o = qkv_flash(q.to(DEV), k.to(DEV), v.to(DEV), _dev(g), _dev(beta), chunk_size=C,
                  q_scale=_dev(sq), k_scale=_dev(sk))
    torch.cuda.synchronize()
    if scaled:
        ref = np.tril(np.einsum("mid,mjd->mij", _np(q) * sq, _np(k) * sk)) @ _np(v)
    else:
        ref = gated_qk_reference(_np(q), _np(k), g, beta, causal=True, dtype=np.float64) @ _np(v)
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    assert max_rel(_np(o), ref) <= tol, max_rel(_np(o), ref)


SMALL = [(torch.float32, 16), (torch.float32, 32), (torch.bfloat16, 32)]


@pytest.mark.parametrize("M", [1, 2, 259])
@pytest.mark.parametrize("dtype,C", SMALL)
def test_small_chunks(dtype, C, M):
    """Chunks of 16 and 32 tokens have one or two query blocks, whose work the four waves share: key blocks of
    the score (gated, and with prescales and an explicit mask; both output types), columns of o."""
    D, tol = (64 if M % 2 else 128), (1e-4 if dtype == torch.float32 else 1e-2)
    announce(f"small chunks C={C} D={D} M={M} {dtype}")
    rng = np.random.default_rng(C + M)
    a, b, v = (_rows(rng, (M, C, D), dtype, s) for s in (0.2, 0.2, 1.0))
    G = np.cumsum(-np.log1p(np.exp(rng.standard_normal((M, C)))) * 0.1, axis=1).astype(np.float32)
    beta = (1 / (1 + np.exp(-rng.standard_normal((M, C))))).astype(np.float32)
    sa, sb = (rng.random((M, C, D)).astype(np.float32) + 0.5 for _ in range(2))
    mask = ((rng.random((C, C)) < 0.5) * rng.random((C, C))).astype(np.float32)
    ad, bd = a.to(DEV), b.to(DEV)
    for out16 in (False, True):
        od = torch.bfloat16 if out16 else torch.float32
        gated = gated_qk(ad, bd, _dev(G), _dev(beta), chunk_size=C, causal=True, out_dtype=od)
        masked = gated_qk(ad, bd, chunk_size=C, mask=_dev(mask), a_scale=_dev(sa), b_scale=_dev(sb), out_dtype=od)
        torch.cuda.synchronize()
        ref = gated_qk_reference(_np(a), _np(b), G, beta, causal=True, dtype=np.float64)
        bound = tol + (2 ** -8 if out16 else 0)
        assert max_rel(_np(gated).reshape(ref.shape), ref) <= bound
        mref = np.matmul(_np(a) * sa, (_np(b) * sb).transpose(0, 2, 1)) * mask
        assert max_rel(_np(masked).reshape(mref.shape), mref) <= bound
    o = qkv_flash(ad, bd, v.to(DEV), _dev(G), _dev(beta), chunk_size=C)
    scaled = qkv_flash(ad, bd, v.to(DEV), chunk_size=C, q_scale=_dev(sa), k_scale=_dev(sb))
    torch.cuda.synchronize()
    assert max_rel(_np(o), ref @ _np(v)) <= tol
    sref = np.tril(np.matmul(_np(a) * sa, (_np(b) * sb).transpose(0, 2, 1))) @ _np(v)
    assert max_rel(_np(scaled), sref) <= tol


@pytest.mark.parametrize("nc,H", [(1, 3), (65, 4)])
def test_small_chunks_of_interleaved_heads(nc, H):
    """Small chunks in the token layout: the staged query and key rows lie H rows apart."""
    C, D = 16, 128
    announce(f"small chunks C={C} nc={nc} H={H} heads interleaved")
    rng = np.random.default_rng(nc)
    a, b = (_rows(rng, (nc * C * H, D), torch.float32) for _ in range(2))
    g = (-np.cumsum(rng.random((nc, C, H)), axis=1) * 0.1).astype(np.float32)
    L = gated_qk(a.to(DEV), b.to(DEV), _dev(g.reshape(-1)), chunk_size=C, heads=H, causal=False)
    torch.cuda.synchronize()

    def chunks(x):
        return x.reshape(nc, C, H, -1).transpose(0, 2, 1, 3).reshape(nc * H, C, -1)

    ref = gated_qk_reference(chunks(_np(a)), chunks(_np(b)), chunks(g)[..., 0], np.ones((nc * H, C)), causal=False,
                             dtype=np.float64)
    assert max_rel(chunks(_np(L)), ref) <= 1e-4
