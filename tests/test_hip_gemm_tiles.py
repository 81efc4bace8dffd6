"""Prefill GEMM at every tile shape's edges (GPU): row, column and K remainders,
fewer K-steps than pipeline stages, and the same rows bit-identical whichever
shape serves them; that the sizes reach every tile shape is checked on the CPU.
Bar: bf16 allclose(atol 2e-2, rtol 1e-2) of the fp32 product
(W of exact powers scaled so that outputs are O(1))."""

import pytest
import torch

from ezops import _hip

gpu = pytest.mark.gpu
DEV = "cuda"


def _gemm(X, W, R=None):
    M, K, N = X.shape[0], X.shape[1], W.shape[0]
    Y = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device=DEV)
    _hip.call("ezops_gemm_bf16", X.data_ptr(), X.stride(0), W.data_ptr(), Y.data_ptr(), N, _hip.ptr(R), M, N, K, None, 0,
              _hip.stream())
    torch.cuda.synchronize()
    assert (Y[M] == 7.0).all()
    return Y[:M]


def _data(M, N, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    X = torch.randn(M, K, generator=g, device=DEV, dtype=torch.bfloat16)
    W = torch.randn(N, K, generator=g, device=DEV, dtype=torch.bfloat16) * 2.0 ** -6
    return X, W


CUS = 256  # MI355X
# (M, N) chosen so that each tile shape of the table is picked: 256x256, 256x192, 256x128,
# 128x128 (two per CU), 128x128 (K-steps of 128), 64x128 (three times), 192x256
SHAPES = [(4000, 4090), (2040, 6136), (2040, 4090), (700, 6136), (1020, 4090), (200, 6136), (1, 130), (65, 72),
          (3000, 4090)]
# gate/up (M, IS): 256x256, 192x256, 256x256, 128x128 (two per CU), 128x128 (K-steps of 128, three
# times), 256x128 twice
SWIGLU_SHAPES = [(500, 12288), (740, 12288), (4000, 2048), (600, 12288), (120, 12288), (1, 128), (130, 384), (499, 6144),
                 (1000, 3072)]


def _tile(M, N, swiglu):
    return _hip.lib().ezops_gemm_tile(M, N, swiglu, CUS)


@pytest.mark.parametrize("swiglu", [0, 1])
def test_shapes_reach_every_tile(swiglu):
    """Every tile shape the rule picks anywhere in a sweep of prompt lengths and projection sizes is one that a size
    below picks (CPU)."""
    tested = {_tile(M, 2 * N if swiglu else N, swiglu) for M, N in (SWIGLU_SHAPES if swiglu else SHAPES)}
    picked = {_tile(M, N, swiglu) for M in range(1, 6000, 37) for N in range(256, 26000, 256)}
    assert picked <= tested and len(tested) == (5 if swiglu else 7)


@gpu
@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("K", [8, 72, 128, 192, 264, 520, 1032])
@pytest.mark.parametrize("resid", [False, True])
def test_gemm_tile_edges(M, N, K, resid):
    X, W = _data(M, N, K)
    R = torch.randn(M, N, device=DEV, dtype=torch.bfloat16) if resid else None
    ref = (X.float() @ W.float().T).bfloat16().float()
    if resid:
        ref = (ref + R.float()).bfloat16().float()
    torch.testing.assert_close(_gemm(X, W, R).float(), ref, rtol=1e-2, atol=2e-2)


@gpu
@pytest.mark.parametrize("K", [520, 4096])
def test_gemm_tile_shapes_bit_identical(K):
    X, W = _data(4000, 6136, K, seed=1)
    full = _gemm(X, W)
    for M, N in [(4000, 4090), (2040, 6136), (2040, 4090), (700, 6136), (1020, 4090), (200, 6136), (5, 40), (3000, 4090)]:
        assert torch.equal(_gemm(X[:M], W[:N]), full[:M, :N]), (M, N)


@gpu
@pytest.mark.parametrize("M,IS", SWIGLU_SHAPES)
@pytest.mark.parametrize("K", [40, 128, 520])
def test_gemm_swiglu_tiles_match_plain(M, IS, K):
    X, W = _data(M, 2 * IS, K, seed=2)
    Y = torch.full((M + 1, IS), 7.0, dtype=torch.bfloat16, device=DEV)
    _hip.call("ezops_gemm_swiglu_bf16", X.data_ptr(), K, W.data_ptr(), Y.data_ptr(), IS, M, IS, K, _hip.stream())
    torch.cuda.synchronize()
    assert (Y[M] == 7.0).all()
    gu = _gemm(X, W).float()
    act = torch.nn.functional.silu(gu[:, :IS]).bfloat16().float()
    torch.testing.assert_close(Y[:M].float(), act * gu[:, IS:], rtol=1e-2, atol=1e-2)
