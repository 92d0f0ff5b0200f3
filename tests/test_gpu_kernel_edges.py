"""GPU: each kernel form at the sizes where its dispatch or its tiling can go wrong (tile edges,
remainders, the smallest of its range), against the oracle or the form it must equal bit for bit."""
import pytest
import torch

import h3attn
from h3attn import sla

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


@pytest.mark.parametrize("rows,nk,fill", [(1, 1, 1.0), (3, 63, 0.5), (5, 64, 0.0), (7, 65, 0.7), (9, 256, 0.3),
                                          (6, 257, 0.9), (1030, 659, 0.2)])
def test_block_map_to_lut_chunk_edges(gpu, rows, nk, fill):
    """One wave per row, four 64-block chunks at a time: the LUT, its default width and its truncation."""
    torch.manual_seed(rows)
    m = (torch.rand(1, 1, rows, nk) < fill).to(torch.uint8)
    counts = m.sum(-1, dtype=torch.int32)
    width = max(1, int(counts.max()))
    for max_k in (None, max(1, width // 2)):
        lut, cnt = h3attn.block_map_to_lut(m.to(gpu), max_k)
        k = width if max_k is None else max_k
        want = torch.full((1, 1, rows, k), -1, dtype=torch.int32)
        for r in range(rows):
            nz = m[0, 0, r].nonzero().flatten()[:k].int()
            want[0, 0, r, :len(nz)] = nz
        assert torch.equal(lut.cpu(), want) and torch.equal(cnt.cpu(), counts.clamp(max=k))
