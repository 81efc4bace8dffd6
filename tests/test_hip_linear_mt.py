"""Linear stages of 5 and more batch rows against the oracle, on both sides of the line
between the tiles of 16 by 16 rows (above 16 batch rows: matrices of few weight
rows) and the kernel that reads W once per 64 rows.

Sizes at the edges of the kernels: batch blocks of 16 (1 to 4 per block,
two 64-row groups), weight-row remainders of a 16-row tile, K with fewer
chunks than waves and a masked last chunk, one tile per CU / two blocks per
CU / two-tile blocks.  Bar: bf16 allclose(atol 2e-2, rtol 1e-2) against the
fp32-accumulated oracle, as for the other linear stages.
"""

import numpy as np
import pytest
import torch

import oracle
from ezops import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


def g(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(torch.bfloat16).to(DEV)


def _run(M, N, K, epi, norm, pad=0, seed=0):
    rng = np.random.default_rng(seed)
    bf = lambda *s: oracle.bf16(rng.standard_normal(s, dtype=np.float32))  # noqa: E731
    X, R = bf(M, K + pad), bf(M, N)
    W, W2 = bf(N, K) * np.float32(2.0 ** -6), bf(N, K) * np.float32(2.0 ** -6)  # exact in bf16
    w = oracle.bf16(rng.standard_normal(K).astype(np.float32) * 0.1 + 1)
    Xn = oracle.rmsnorm_bf16(X[:, :K], w) if norm else X[:, :K]
    ref = oracle.linear_bf16(Xn, W)
    if epi == 1:
        ref = oracle.bf16(R + ref)
    elif epi == 2:
        u = oracle.linear_bf16(Xn, W2)
        ref = oracle.bf16(oracle.bf16(ref / (1 + np.exp(-ref.astype(np.float64)))) * u)
    elif epi == 3:
        ref = Xn @ W.T
    tX, tW, tW2, tR, tw = g(X), g(W), g(W2), g(R), g(w)
    # a guard row behind Y: nothing is written past row M
    Y = torch.full((M + 1, N), 7.0, dtype=torch.float32 if epi == 3 else torch.bfloat16, device=DEV)
    ws = torch.zeros(max(256, _hip.size("ezops_linear_stage_workspace_size", M, K, norm)), dtype=torch.uint8, device=DEV)
    _hip.call("ezops_linear_stage_bf16", tX.data_ptr(), K + pad, tW.data_ptr(), tW2.data_ptr(), Y.data_ptr(), N,
              tR.data_ptr(), N, tw.data_ptr(), norm, 1e-6, epi, M, N, K, ws.data_ptr(), ws.numel(), _hip.stream())
    torch.cuda.synchronize()
    out = Y.float().cpu().numpy()
    assert (out[M] == 7.0).all()
    np.testing.assert_allclose(out[:M], ref, rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("M", [5, 16, 17, 32, 33, 48, 49, 64, 65, 100])
@pytest.mark.parametrize("epi,norm", [(0, 0), (1, 0), (2, 1), (3, 0)])
@pytest.mark.parametrize("N,K", [(48, 512), (37, 1032), (16, 40), (250, 2048)])
def test_linear_mt_edges(M, epi, norm, N, K):
    _run(M, N, K, epi, norm, pad=0 if norm else 8 * (N % 2))


# the same edges where the matrix is wide enough for one read of W per 64 rows
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64, 65, 96, 97, 100])
@pytest.mark.parametrize("epi,norm", [(0, 0), (1, 0), (2, 1), (3, 0)])
@pytest.mark.parametrize("N,K", [(4133, 40), (4112, 1032)])
def test_linear_mt_edges_wide(M, epi, norm, N, K):
    _run(M, N, K, epi, norm, pad=0 if norm else 8 * (N % 2))


def _tiles(n):
    """Weight rows of n 16-row tiles, n in tiles per CU."""
    return 16 * int(n * torch.cuda.get_device_properties(0).multi_processor_count)


# the line itself: (tiles per CU of the matrix, batch rows) with the last shape of the 16 x 16 tiles and the first
# beyond it -- one tile per CU; two for plain stages of more than 32 rows and for SwiGLU of K <= 1024; the norm
# inside the kernel (K = 4096) up to one
@pytest.mark.parametrize("over", [0, 16])
@pytest.mark.parametrize("tiles,M,K,epi,norm", [(1 / 2, 32, 512, 1, 0), (1 / 2, 64, 256, 1, 0), (1 / 4, 64, 768, 0, 1),
                                                (1 / 4, 64, 4096, 0, 1), (1 / 2, 20, 4096, 2, 1), (1 / 4, 64, 2048, 2, 1),
                                                (1 / 2, 64, 1024, 2, 1), (1 / 4, 128, 512, 3, 0)])
def test_linear_narrow_line(tiles, M, K, epi, norm, over):
    _run(M, _tiles(tiles) + over, K, epi, norm, seed=2)


# 4104 rows: two blocks per CU and a remainder; 5200 and 16400: two-tile blocks,
# odd tile count; 4096 x 4096: one tile per CU.
@pytest.mark.parametrize("M,N,K,epi,norm", [(33, 4104, 256, 1, 0), (40, 5200, 520, 0, 0), (8, 20000, 1024, 1, 0), (64, 16400, 512, 0, 1), (20, 16424, 256, 3, 0),
                                            (64, 4096, 4096, 1, 0), (40, 4112, 1024, 2, 1)])
def test_linear_mt_tilings(M, N, K, epi, norm):
    _run(M, N, K, epi, norm, seed=1)


# per_cu: 16-row weight tiles per CU -- the streaming, multi-tile and one-tile launches
@pytest.mark.parametrize("per_cu,K,epi", [(4, 4096, 0), (3, 512, 1), (3, 4096, 2), (2, 4096, 2), (1, 520, 2), (1 / 4, 40, 3)])
def test_linear_rows_far_apart(per_cu, K, epi):
    """20 batch rows at a stride of 2^23 elements and more, beyond the 32-bit extents of a 64-row block of X: two batch
    blocks of the 16-row kernels.  Against fp32 torch on the same GPU, the bar above."""
    M, N, ldx = 20, _tiles(per_cu) + 8, (1 << 23) + 8
    if per_cu in (2, 3):
        N -= 8  # the multi-tile launches need whole tiles
    gen = torch.Generator(device=DEV).manual_seed(N + K)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)  # noqa: E731
    buf = torch.zeros(M * ldx, dtype=torch.bfloat16, device=DEV)
    X = buf.view(M, ldx)[:, :K]
    X.copy_(r(M, K))
    W, W2, R = r(N, K) * 2.0 ** -6, r(N, K) * 2.0 ** -6, r(M, N)
    Xf = X.float()
    ref = Xf @ W.float().T
    if epi != 3:
        ref = ref.bfloat16().float()
    if epi == 1:
        ref = (R.float() + ref).bfloat16().float()
    elif epi == 2:
        ref = torch.nn.functional.silu(ref).bfloat16().float() * (Xf @ W2.float().T).bfloat16().float()
    Y = torch.full((M + 1, N), 7.0, dtype=torch.float32 if epi == 3 else torch.bfloat16, device=DEV)
    _hip.call("ezops_linear_stage_bf16", X.data_ptr(), ldx, W.data_ptr(), W2.data_ptr(), Y.data_ptr(), N, R.data_ptr(), N,
              None, 0, 1e-6, epi, M, N, K, None, 0, _hip.stream())
    torch.cuda.synchronize()
    assert (Y[M] == 7.0).all()
    torch.testing.assert_close(Y[:M].float(), ref, rtol=1e-2, atol=2e-2)
