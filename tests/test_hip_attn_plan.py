"""Decode attention at the edges of the split plan for many units (GPU): one split,
splits of at least 512 rows, ragged batches whose sequences take different
split counts (empty and one-row ones among them), 64 sequences.  Bar: allclose
1e-2 / 1e-2 (the op's) against the fp32 formula."""

import pytest
import torch

from ezops import AttnDecodeOp, PagedAttnDecodeOp
from ezops.ops.attn_decode import gqa_decode_reference
from ezops.ops.paged_attn_decode import paged_to_contiguous

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,D,S", [(64, 32, 8, 128, 512), (64, 32, 8, 128, 1023), (64, 16, 8, 64, 1024),
                                         (33, 32, 8, 128, 1536), (40, 16, 1, 128, 2080), (2, 16, 8, 128, 700)])
@pytest.mark.parametrize("ragged", [False, True])
def test_attn_decode_plan_edges(B, H, Hkv, D, S, ragged):
    g = torch.Generator(device="cuda").manual_seed(B + S)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    Q, K, V = r(B, H, 1, D), r(B, Hkv, S, D), r(B, Hkv, S, D)
    lens = None
    if ragged:
        lens = torch.randint(1, S + 1, (B,), generator=g, device="cuda").to(torch.int32)
        lens[0], lens[1] = 1, S
        for b, n in enumerate(lens.tolist()):  # rows past the length do not reach the result
            K[b, :, n:], V[b, :, n:] = float("nan"), float("nan")
    out = AttnDecodeOp(B, H, S, D, "hip", Hkv)(Q, K, V, *([] if lens is None else [lens]))
    want = gqa_decode_reference(Q, K.nan_to_num(0.0), V.nan_to_num(0.0), lens)
    torch.testing.assert_close(out.float(), want.float(), rtol=1e-2, atol=1e-2)


def test_paged_attn_decode_plan_zero_length():
    B, H, Hkv, D, P, M = 64, 32, 8, 128, 64, 40
    g = torch.Generator(device="cuda").manual_seed(3)
    op = PagedAttnDecodeOp(B, H, Hkv, D, P, M, backend="hip")
    Q, Kp, Vp, bt, _ = op.gen_data("cuda")
    lens = torch.randint(1, M * P + 1, (B,), generator=g, device="cuda").to(torch.int32)
    lens[5], lens[63] = 0, 2049
    out = op(Q, Kp, Vp, bt, lens, 2560)
    live = lens.long() > 0
    want = gqa_decode_reference(Q, paged_to_contiguous(Kp, bt), paged_to_contiguous(Vp, bt), lens.clamp(min=1))
    torch.testing.assert_close(out[live].float(), want[live].float(), rtol=1e-2, atol=1e-2)
    assert (out[5] == 0).all()


# more sequences than a block's length scan holds (64): equal splits of the longest for every sequence
@pytest.mark.parametrize("B,H,Hkv,D,S", [(65, 32, 8, 128, 600), (65, 8, 8, 128, 1024), (80, 16, 8, 64, 2080),
                                         (100, 16, 1, 128, 1536), (130, 4, 2, 128, 1040)])
@pytest.mark.parametrize("long", [0, 64])
def test_attn_decode_many_sequences(B, H, Hkv, D, S, long):
    """One long sequence among short ones (an empty one too): every split but the long sequence's first is empty."""
    g = torch.Generator(device="cuda").manual_seed(B + S)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    Q, K, V = r(B, H, 1, D), r(B, Hkv, S, D), r(B, Hkv, S, D)
    lens = torch.randint(1, 40, (B,), generator=g, device="cuda").to(torch.int32)
    lens[long], lens[5] = S, 0
    for b, n in enumerate(lens.tolist()):
        K[b, :, n:], V[b, :, n:] = float("nan"), float("nan")
    out = AttnDecodeOp(B, H, S, D, "hip", Hkv)(Q, K, V, lens)
    want = gqa_decode_reference(Q, K.nan_to_num(0.0), V.nan_to_num(0.0), lens.clamp(min=1))
    live = lens.long() > 0
    torch.testing.assert_close(out[live].float(), want[live].float(), rtol=1e-2, atol=1e-2)
    assert (out[5] == 0).all()
