"""Prefill layer around the 64-token line between the linear stages and the GEMM
(GPU), fresh and over cached prefixes, against the op's own reference formulas
on the same GPU (the op's check: relative Frobenius < 1e-2), and the cache rows
it writes against theirs."""

import pytest
import torch

from ezops import Qwen3PrefillOp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,past", [([1], [0]), ([4], [7]), ([5], [0]), ([3, 0, 2], [0, 5, 31]), ([16], [100]),
                                         ([17], [0]), ([20, 13, 31], [0, 64, 1]), ([64], [0]), ([60, 5], [3, 0])])
@pytest.mark.parametrize("IS,page", [(3072, None), (1032, None), (3072, 64)])
def test_prefill_layer_few_tokens(q_lens, past, IS, page):
    torch.manual_seed(sum(q_lens))
    args = (len(q_lens), 256, 1024, IS, 16, 128, q_lens, past)
    kw = dict(num_kv_heads=8, norm_weights=True, rope_theta=1e6, page_size=page)
    op, ref = Qwen3PrefillOp(*args, backend="hip", **kw), Qwen3PrefillOp(*args, backend="ref", **kw)
    d = op.gen_data("cuda")
    K, V = d[1].clone(), d[2].clone()
    want = ref(d[0], K, V, *d[3:])
    out = op(*d)
    assert op.check(out, want)
    for got, w in ((d[1], K), (d[2], V)):
        torch.testing.assert_close(got.float(), w.float(), rtol=2e-2, atol=2e-2)
