"""Linear stages of 1 to 4 batch rows (GPU): operands at the ends of the number range,
fp32 results against fp64, and the wide matrices whose row groups own several
weight rows.  From two batch rows on the sums take two bf16 products per
instruction (v_dot2_f32_bf16); one row takes scalar FMAs."""

import pytest
import torch

from ezops import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _stage(X, W, epi, norm=0, W2=None, R=None, w=None):
    M, K = X.shape
    N = W.shape[0]
    Y = torch.full((M + 1, N), 7.0, dtype=torch.float32 if epi == 3 else BF, device=DEV)
    _hip.call("ezops_linear_stage_bf16", X.data_ptr(), K, W.data_ptr(), _hip.ptr(W2), Y.data_ptr(), N, _hip.ptr(R), N,
              _hip.ptr(w), norm, 1e-6, epi, M, N, K, None, 0, _hip.stream())
    torch.cuda.synchronize()
    assert (Y[M] == 7.0).all()
    return Y[:M]


INF, NAN, TINY = float("inf"), float("nan"), 2.0 ** -130  # TINY: a subnormal bf16
# (x, w) pairs, everything else zero; the exact sum
OPERANDS = [
    ([(TINY, 2.0 ** 100)], 2.0 ** -30), ([(2.0 ** 100, TINY)], 2.0 ** -30), ([(TINY, 1.0), (TINY, 1.0)], 2 * TINY),
    ([(2.0 ** -70, 2.0 ** -65), (2.0 ** -70, 2.0 ** -66)], 2.0 ** -135 + 2.0 ** -136),
    ([(2.0 ** -60, 2.0 ** -60), (2.0 ** -60, -2.0 ** -60), (2.0 ** -70, 2.0 ** -65)], 2.0 ** -135),
    ([(2.0 ** 12, 2.0 ** 12), (-2.0 ** 12, 2.0 ** 12), (1.0, 3.0)], 3.0), ([(2.0 ** 64, 2.0 ** 63)], 2.0 ** 127),
    ([(INF, 1.0)], INF), ([(-INF, 2.0), (1.0, 1.0)], -INF), ([(2.0 ** 120, 2.0 ** 10)], INF),
    ([(INF, 1.0), (INF, -1.0)], NAN), ([(INF, 0.0)], NAN), ([(NAN, 1.0)], NAN), ([(1.0, NAN)], NAN),
]


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("at", [0, 1, 9, 1022])  # the place in the row: pairs and pieces of a thread, split pairs
def test_extreme_operands(M, at):
    K = 2048
    X = torch.zeros(len(OPERANDS), K, device=DEV, dtype=BF)
    W = torch.zeros(len(OPERANDS), K, device=DEV, dtype=BF)
    for i, (pairs, _) in enumerate(OPERANDS):
        for j, (x, w) in enumerate(pairs):
            X[i, at + j], W[i, at + j] = x, w
    want = torch.tensor([s for _, s in OPERANDS], device=DEV)
    for i in range(len(OPERANDS)):
        got = _stage(X[i].expand(M, K).contiguous(), W[i:i + 1].expand(3, K).contiguous(), 3)
        torch.testing.assert_close(got, want[i].expand(M, 3), rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("K", [256, 4096, 16384])
def test_sums_against_fp64(M, K):
    """A thread chains at most K / 256 + 8 products (8 to a piece), then a tree over 64 lanes and 4 waves: each error is
    within that many roundings (2^-24 each) of the sum of magnitudes.  In the root mean square it is within 2.5
    roundings of the results' (scalar FMA chains: 0.9 at K = 256 to 1.6 at 16384); a sum that kept fewer than 24 bits
    between the terms would be outside."""
    gen = torch.Generator(device=DEV).manual_seed(K + M)
    X = torch.randn(M, K, generator=gen, device=DEV).to(BF)
    W = (torch.randn(512, K, generator=gen, device=DEV) * 0.02).to(BF)
    ref, mag = X.double() @ W.double().T, X.double().abs() @ W.double().abs().T
    err = (_stage(X, W, 3).double() - ref).abs()
    assert (err <= (K / 256 + 8 + 6 + 4) * 2.0 ** -24 * mag).all()
    assert err.pow(2).mean().sqrt() <= 2.5 * 2.0 ** -24 * ref.pow(2).mean().sqrt()


# N: enough blocks for 2, 4 and 8 weight rows per group and a partly empty last one, at 1 to 4 chunks per thread
@pytest.mark.parametrize("M", [2, 3, 4])
@pytest.mark.parametrize("N,K", [(4101, 2048), (4090, 2048), (4101, 3080), (4101, 4096), (2051, 8192), (16405, 1024),
                                 (16405, 520)])
@pytest.mark.parametrize("epi,norm", [(0, 0), (1, 1), (2, 0), (2, 1), (3, 1)])
def test_wide_matrices(M, N, K, epi, norm):
    """Against fp32 torch on the same GPU with the reference's bf16 staging; bar of the other linear stages."""
    gen = torch.Generator(device=DEV).manual_seed(N + K + M)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(BF)  # noqa: E731
    X, W, W2, R, w = r(M, K), r(N, K) * 2.0 ** -6, r(N, K) * 2.0 ** -6, r(M, N), r(K) * 0.125 + 1
    Xn = X.float()
    if norm:
        Xn = (Xn * torch.rsqrt(Xn.pow(2).mean(-1, keepdim=True) + 1e-6) * w.float()).to(BF).float()
    ref = Xn @ W.float().T
    if epi != 3:
        ref = ref.to(BF).float()
    if epi == 1:
        ref = (R.float() + ref).to(BF).float()
    elif epi == 2:
        ref = torch.nn.functional.silu(ref).to(BF).float() * (Xn @ W2.float().T).to(BF).float()
    got = _stage(X, W, epi, norm, W2, R, w).float()
    torch.testing.assert_close(got, ref, rtol=1e-2, atol=2e-2)


def test_bf16_rounding_of_every_exponent():
    """fp32 results rounded to bf16 (to nearest even) over all exponents, subnormal ones, ties, the largest values and
    NaN, bit for bit as torch rounds them.  A result is the exact sum of three bf16 parts, scaled by 2^60 in W and back
    in X below 2^-60 so that the parts are normal numbers."""
    gen = torch.Generator().manual_seed(0)
    bits = torch.randint(0, 1 << 32, (8192,), generator=gen)
    bits[:2048] = bits[:2048] & ~0xffff | 0x8000  # ties
    bits[2048:3072] = bits[2048:3072] & 0x80ffffff  # subnormal, and the smallest normal numbers
    bits[3072:3200] = bits[3072:3200] & 0x8000ffff | 0x7f7f0000  # about the largest bf16: to it or to infinity
    v = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).to(torch.int32).view(torch.float32)
    v = v[torch.isfinite(v)]
    small = v.abs() < 2.0 ** -60
    u = torch.where(small, v.double() * 2.0 ** 60, v.double())
    trunc = lambda x: (x.float().view(torch.int32) & -65536).view(torch.float32).double()  # noqa: E731
    hi = trunc(u)
    mid = trunc(u - hi)
    lo = u - hi - mid
    assert (trunc(lo) == lo).all()
    for sel, scale in ((~small, 1.0), (small, 2.0 ** -60)):
        W = torch.zeros(int(sel.sum()), 8, dtype=BF, device=DEV)
        for j, part in enumerate((hi, mid, lo)):
            W[:, j] = part[sel].to(BF).to(DEV)
        X = torch.zeros(1, 8, dtype=BF, device=DEV)
        X[0, :3] = scale
        got = _stage(X, W, 0)[0].cpu()
        assert torch.equal(got.view(torch.int16), v[sel].to(BF).view(torch.int16))
    nan = _stage(torch.ones(1, 8, dtype=BF, device=DEV), torch.full((1, 8), NAN, dtype=BF, device=DEV), 0)
    assert torch.isnan(nan).all()
