"""Row ops at row lengths that are not multiples of the access width, rows that
start at any element, and softmax rows cut into chunks (GPU) against torch in
fp64.  Bars: softmax atol 1e-6 / rtol 1e-5, fp32 RMSNorm 1e-5 (the ops' own),
bf16 RMSNorm one bf16 ulp (2^-7 relative) of the fp64 result."""

import pytest
import torch

import ezops
from ezops import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _softmax(X, Out):
    _hip.call("ezops_softmax_f32", X.data_ptr(), Out.data_ptr(), X.shape[0], X.shape[1], _hip.stream())
    torch.cuda.synchronize()


def _offset(rows, dim, dtype, off, seed=0):
    """A [rows, dim] tensor whose first element sits `off` elements into its buffer, and the buffer."""
    buf = torch.full((rows * dim + off + 16,), 5.0, dtype=dtype, device=DEV)
    t = buf[off: off + rows * dim].view(rows, dim)
    t.copy_(torch.randn(rows, dim, generator=torch.Generator().manual_seed(seed)) * 3)
    return t, buf


# remainders at each dispatch bound: 64-, 256- and 1024-thread rows, then the chunked rows (5 chunks and up)
@pytest.mark.parametrize("dim", [1, 3, 5, 1023, 2047, 2049, 8191, 8195, 32765, 32768, 32769, 40961, 151936, 524287,
                                 524288, 524289])
@pytest.mark.parametrize("off", [0, 1])
def test_softmax_any_row(dim, off):
    rows = 3
    X, _ = _offset(rows, dim, torch.float32, off)
    Out, buf = _offset(rows, dim, torch.float32, off)
    want = torch.softmax(X.double().cpu(), -1)
    _softmax(X, Out)
    torch.testing.assert_close(Out.double().cpu(), want, rtol=1e-5, atol=1e-6)
    assert (buf[off + rows * dim:] == 5.0).all() and (buf[:off] == 5.0).all()
    _softmax(X, X)  # in place
    torch.testing.assert_close(X.double().cpu(), want, rtol=1e-5, atol=1e-6)


def test_softmax_chunked_nonfinite():
    """A chunk of -inf alone weighs nothing; NaN, +inf and a row of -inf make the row NaN, as in the one-block rows."""
    dim = 40000
    X = torch.randn(6, dim, generator=torch.Generator().manual_seed(1)).to(DEV)
    X[0, :9000] = float("-inf")
    X[1, 20000] = float("nan")
    X[2, 39999] = float("inf")
    X[3] = float("-inf")
    X[4] = torch.finfo(torch.float32).min
    X[5, 1000:] = torch.finfo(torch.float32).min
    Out = torch.empty_like(X)
    _softmax(X, Out)
    want = torch.softmax(X.double().cpu(), -1)
    got = Out.double().cpu()
    torch.testing.assert_close(got[[0, 4, 5]], want[[0, 4, 5]], rtol=1e-5, atol=1e-6)
    assert torch.isnan(got[1:4]).all()


# one block per row of 64 / 256 / 1024 threads, rows in chunks, and in place (the three-pass kernel beyond 32768)
@pytest.mark.parametrize("dim", [1000, 5001, 20000, 40003])
@pytest.mark.parametrize("inplace", [False, True])
def test_softmax_large_maxima(dim, inplace):
    """Finite rows far from zero, where exp(x - max) must come from the difference: a full mask of the type's lowest
    value, of -1e10 or of the largest value, values near +-256 (where the formula changes) and near +-3e38, and a
    maximum on either side of 256 in one chunk alone.  Bar: the op's (rtol 1e-5, atol 1e-6) of torch's fp64 softmax."""
    big = torch.finfo(torch.float32).max
    base = torch.randn(10, dim, generator=torch.Generator().manual_seed(dim)) * 3
    X = base.clone()
    X[0], X[1], X[2] = -big, -1e10, big
    X[3] = base[3] - 1e6
    X[4] = base[4] + 250.0  # maxima about 260
    X[5] = base[5] - 262.0
    X[6, : dim // 2], X[6, dim // 2:] = 3e38, -3e38
    X[7, dim // 3:] = -big
    X[8, dim - 1], X[8, 0] = 300.0, 296.0
    X[9] = base[9] - 300.0
    X[9, 1] = 5.0
    want = torch.softmax(X.double(), -1)
    X = X.to(DEV)
    Out = X if inplace else torch.empty_like(X)
    _softmax(X, Out)
    torch.testing.assert_close(Out.double().cpu(), want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("dim", [1, 7, 513, 1025, 2050, 8197, 16391, 32767, 65535])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("off", [0, 1])
def test_rmsnorm_any_row(dim, dtype, off):
    rows = 5
    X, _ = _offset(rows, dim, dtype, off)
    Out, buf = _offset(rows, dim, dtype, off)
    op = ezops.RmsNormOp(rows, dim, "hip", dtype=dtype, weighted=dtype == torch.bfloat16)
    x = X.double().cpu()
    want = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)
    if dtype == torch.bfloat16:
        W, _ = _offset(1, dim, dtype, off, seed=2)
        op(X, W[0], Out)
        want = want * W[0].double().cpu()
        tol = dict(rtol=2.0 ** -7, atol=1e-6)
    else:
        op(X, Out)
        tol = dict(rtol=1e-5, atol=1e-5)
    torch.cuda.synchronize()
    torch.testing.assert_close(Out.double().cpu(), want, **tol)
    assert (buf[off + rows * dim:] == 5.0).all() and (buf[:off] == 5.0).all()


# batches of 256 threads x 8 float4, the block counts' bounds, partial batches, the streamed arrays
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 8191, 8193, 32771, 1000003, (1 << 20) + 1, 4194307, (1 << 25) - 3, (1 << 25) + 8197,
                               (3 << 24) - 1, (3 << 24) + 8197])
def test_sum_any_alignment(n):
    """Full sum of an array that starts at any element: the same bits as at 16 bytes, within 1e-6 of fp64 (fp32 partial
    sums of non-negative terms: chains of at most 64 values, then a tree), and nothing outside [0, n) in it."""
    A = torch.rand(n, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV)
    buf = torch.full((n + 32,), float("nan"), device=DEV)
    ws = torch.zeros(max(256, _hip.size("ezops_reduce_sum_workspace_size", n)), dtype=torch.uint8, device=DEV)
    got = []
    for off in (16, 17, 18, 19):
        buf.fill_(float("nan"))
        buf[off:off + n] = A
        Out = torch.zeros(1, device=DEV)
        _hip.call("ezops_reduce_sum_f32", buf.data_ptr() + 4 * off, Out.data_ptr(), n, ws.data_ptr(), ws.numel(),
                  _hip.stream())
        got.append(float(Out))
    want = float(A.double().sum())
    assert abs(got[0] - want) <= 1e-6 * want
    assert got[1:] == got[:1] * 3
