"""GPU: each kernel form at the sizes where its dispatch or its tiling can go wrong (tile edges,
remainders, the smallest of its range), against the oracle or the form it must equal bit for bit."""
import pytest
import torch

import h3attn
from h3attn import ops, sla

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blk", [64, 96, 128])
def test_sparse_attention_sequence_major_output(gpu, blk):
    """seq_major writes [1,S,H,D] memory; the values are those of the head-major output."""
    torch.manual_seed(0)
    q, k, v = (torch.randn(1, 3, 777, 128, device=gpu).bfloat16() for _ in range(3))
    want = sla.sparse_attention(q, k, v, 0.4, blk)
    got = sla.sparse_attention(q, k, v, 0.4, blk, seq_major=True)
    assert want.is_contiguous() and got.transpose(1, 2).is_contiguous()
    assert torch.equal(got, want)
