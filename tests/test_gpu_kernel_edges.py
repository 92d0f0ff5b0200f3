"""GPU: each kernel form at the sizes where its dispatch or its tiling can go wrong (tile edges,
remainders, the smallest of its range), against the oracle or the form it must equal bit for bit."""
import numpy as np
import pytest
import torch

import h3attn
import oracle
from conftest import assert_close_absmax, from_dev_bf16, randn_bf16, to_dev_bf16
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


@pytest.mark.parametrize("blk_q,blk_k,Sq,Skv", [(16, 16, 130, 4113), (48, 80, 1000, 2065), (96, 96, 65, 8200),
                                                (256, 240, 700, 2048), (112, 32, 500, 31), (1040, 1 << 21, 3000, 777)])
def test_tile_lut_chunk_and_slice_edges(gpu, blk_q, blk_k, Sq, Skv):
    """Tile LUTs against their element mask: shared map rows, split columns, ragged ends, several
    256-column chunks."""
    torch.manual_seed(Sq)
    nq, nk = -(-Sq // blk_q), -(-Skv // blk_k)
    m = (torch.rand(1, 2, nq, nk) < 0.4).to(torch.uint8)
    lut, cnt = ops.block_map_to_tile_lut(m.to(gpu), blk_q, blk_k, Sq, Skv)
    nsub, ncols = -(-Sq // 64), -(-Skv // 32)
    rows, keys = torch.arange(4 * nsub) * 16, torch.arange(2 * ncols) * 16
    sub = m[:, :, (rows // blk_q).clamp(max=nq - 1)][..., (keys // blk_k).clamp(max=nk - 1)].bool()
    sub &= (rows < Sq)[:, None] & (keys < Skv)
    bit = torch.tensor([[1 << (2 * i + j) for j in range(2)] for i in range(4)])
    mask = (sub.view(1, 2, nsub, 4, ncols, 2) * bit[:, None, :]).sum((3, 5))
    lut, cnt = lut.cpu(), cnt.cpu()
    assert torch.equal(cnt.long(), (mask != 0).sum(-1))
    for h in range(2):
        for qs in range(nsub):
            cols = mask[0, h, qs].nonzero().flatten()
            want = torch.full((ncols,), -1, dtype=torch.int32)
            want[:len(cols)] = ((cols << 8) | mask[0, h, qs, cols]).int()
            assert torch.equal(lut[0, h, qs], want)


@pytest.mark.parametrize("S,H,blk,rot", [(63, 3, 64, 128), (64, 4, 64, 64), (65, 8, 64, 128), (1, 1, 64, 128),
                                         (130, 14, 48, 96), (4104, 56, 64, 128), (2100, 60, 16, 32),
                                         (2100, 60, 16, 128)])
def test_pooled_prologue_tokens_heads_edges(gpu, S, H, blk, rot):
    """The pooling prologue in 4-head and 8-head workgroups, ragged heads and last blocks of fewer tokens
    than waves: its rows and means equal the plain prologue's and block_pool's bit for bit."""
    torch.manual_seed(S)
    qkv = torch.randn(S, 3 * H * 128, device=gpu).bfloat16()
    rope = torch.randn(1, S, 1, rot // 2, 2, 2, device=gpu)
    w = [torch.randn(128, device=gpu).bfloat16() for _ in range(2)]
    got, want = qkv.clone(), qkv.clone()

    def heads(x):
        f = x.view(1, S, 3, H, 128)
        return f[:, :, 0], f[:, :, 1]

    means = ops.qk_rmsnorm_rope_(*heads(got), rope, *w, pool_blk=blk)
    ops.qk_rmsnorm_rope_(*heads(want), rope, *w)
    assert torch.equal(got, want)
    for m, x in zip(means, heads(want)):
        assert torch.equal(m, ops.block_pool(x.transpose(1, 2), blk))


@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 1, 1), (1, 2, 63, 64), (1, 3, 65, 65), (2, 2, 64, 128), (1, 2, 300, 300),
                                        (2, 3, 129, 191), (1, 28, 700, 700), (1, 1, 40, 3000), (1, 2, 1000, 1090),
                                        (2, 14, 580, 1100)])
def test_short_tiles_match_oracle(gpu, B, H, Sq, Skv):
    """Launches of few tiles (128- and 64-row tiles, whole or in key ranges) at ragged rows and keys, down
    to ranges in which one group has no stage."""
    rng = np.random.default_rng(Sq + Skv)
    q, k, v = (randn_bf16(rng, (B, H, n, 128)) for n in (Sq, Skv, Skv))
    dev = [to_dev_bf16(x, gpu) for x in (q, k, v)]
    out = torch.full((B, Sq, H, 128), float("nan"), dtype=torch.bfloat16, device=gpu).transpose(1, 2)
    ops.attn_fwd(*dev, out=out)
    got = oracle.bf16_to_f32(from_dev_bf16(out)).reshape(out.shape)
    assert_close_absmax(got, oracle.attn_fwd(q, k, v), what=f"{B}x{H}x{Sq}x{Skv}")


@pytest.mark.parametrize("H,Sq,Skv", [(1, 5000, 5000), (4, 8000, 4100), (10, 1500, 1500), (28, 2500, 2600), (3, 100, 20000)])
def test_short_tiles_and_key_ranges_match_whole_tiles(gpu, H, Sq, Skv):
    torch.manual_seed(H)
    q, k, v = (torch.randn(1, H, n, 128, device=gpu).bfloat16() for n in (Sq, Skv, Skv))
    got = ops.attn_fwd(q, k, v).float()
    want = ops.attn_fwd(q, k, v, split_tail=False).float()
    d = (got - want).abs()
    # Both round O (2^-9 relative) and every p (2^-9 each, averaging out over the keys): on the mean
    # the two differ by less than the sum of the four bounds.
    assert d.max() <= 1e-2 * want.abs().max() and d.mean() <= 2.0 ** -7 * want.abs().mean()


@pytest.mark.parametrize("H,Sq,Skv,stride", [(1, 64, 200, (1 << 23) + 8), (3, 4000, 200, (1 << 23) + 8),
                                             (28, 700, 600, (1 << 22) + 8)])
def test_short_tiles_wide_kv_stride(gpu, H, Sq, Skv, stride):
    """K/V whose rows lie so far apart that a slice passes 2^32 bytes (per-stage descriptors), in 64- and
    (the last) 128-row tiles."""
    torch.manual_seed(1)
    buf = torch.empty(Skv * stride, dtype=torch.bfloat16, device=gpu)
    q = torch.randn(1, H, Sq, 128, device=gpu).bfloat16()
    k, v = (torch.randn(1, H, Skv, 128, device=gpu).bfloat16() for _ in range(2))
    kw, vw = (buf.as_strided((1, H, Skv, 128), (0, 128, stride, 1), off * 128 * H) for off in (0, 1))
    kw.copy_(k)
    vw.copy_(v)
    assert torch.equal(ops.attn_fwd(q, kw, vw), ops.attn_fwd(q, k, v))


@pytest.mark.parametrize("B,H,Sq,Skv,rows,split", [(32, 48, 26, 73, 64, False), (32, 35, 22, 449, 64, True),
                                                   (32, 34, 100, 198, 128, False), (32, 35, 74, 576, 128, True)])
def test_short_tiles_queued(gpu, B, H, Sq, Skv, rows, split):
    """Four rounds and more of 128- and 64-row tiles on the persistent grid, where an item's query rows land
    in the buffers of the last one's exchange, alone and followed by a split tail: equal to the unsplit
    256-row tiles within rounding, to the oracle on the last head, and to itself over garbage counters."""
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("the shapes are chosen for 256 CUs")
    tiles = B * H * -(-Sq // rows)
    need = ops.attn_workspace_bytes(B, H, Sq, Skv)
    one = tiles % 256 * rows * 130 * 4  # partials of one range of each tail tile
    assert tiles >= 1024 and (need - 1024 >= 2 * one and (need - 1024) % one == 0 if split else need == 1024)
    rng = np.random.default_rng(Sq + Skv)
    q, k, v = (randn_bf16(rng, (B, H, n, 128)) for n in (Sq, Skv, Skv))
    dev = [to_dev_bf16(x, gpu) for x in (q, k, v)]
    outs = []
    for fill in (0, 0x7F):
        torch.full((need,), fill, dtype=torch.uint8, device=gpu)  # freed: the next workspace's bytes
        outs.append(ops.attn_fwd(*dev))
    assert torch.equal(*outs)
    want = ops.attn_fwd(*dev, split_tail=False).float()
    d = (outs[0].float() - want).abs()
    assert d.max() <= 1e-2 * want.abs().max() and d.mean() <= 2.0 ** -7 * want.abs().mean()
    got = oracle.bf16_to_f32(from_dev_bf16(outs[0][-1:, -1:].contiguous())).reshape(1, 1, Sq, 128)
    assert_close_absmax(got, oracle.attn_fwd(*(x[-1:, -1:] for x in (q, k, v))), what=f"{rows}-row tiles, queued")


@pytest.mark.parametrize("H,nq,nk", [(1, 1, 1), (2, 5, 64), (3, 17, 128), (14, 65, 65), (4, 33, 129), (60, 65, 65),
                                     (140, 65, 40), (30, 157, 385), (5, 40, 768)])
def test_block_select_rows_per_workgroup(gpu, H, nq, nk):
    """Block selection in workgroups of 4, 8 and 16 rows (by how many there are), on integer vectors, where
    every order of summation gives the same scores and ties abound."""
    g = torch.Generator().manual_seed(nk)
    pq, pk = (torch.randint(-2, 3, (1, H, n, 128), generator=g).float() for n in (nq, nk))
    keep = max(1, nk // 3)
    bmap, lut, cnt = ops.block_select(pq.to(gpu), pk.to(gpu), keep, 64, 64, force_diag=True)
    score = pq @ pk.transpose(2, 3)
    want = torch.zeros(1, H, nq, nk, dtype=torch.uint8)
    want.scatter_(3, score.sort(dim=3, descending=True, stable=True).indices[..., :keep], 1)
    d = torch.arange(min(nq, nk))
    want[:, :, d, d] = 1
    assert torch.equal(bmap.cpu(), want)
    assert torch.equal(cnt.cpu(), want.sum(3, dtype=torch.int32))
    idx = torch.where(want.bool(), torch.arange(nk), nk).sort(3).values[..., :lut.shape[3]]
    assert torch.equal(lut.cpu(), torch.where(idx < nk, idx, -1).int())


@pytest.mark.parametrize("H,blk_q,blk_k,Sq,Skv", [(1, 64, 64, 64, 64), (2, 64, 64, 333, 1000), (3, 64, 128, 1000, 1090),
                                                  (2, 64, 256, 640, 2500), (2, 192, 64, 700, 1100),
                                                  (4, 192, 192, 4096, 777), (5, 64, 64, 4096, 333),
                                                  (4, 64, 64, 4096, 1300), (5, 64, 64, 4096, 1300)])
def test_one_sparse_block_per_workgroup(gpu, H, blk_q, blk_k, Sq, Skv):
    """64-row query blocks with lists of 8 stages and more, few enough for one per CU (up to the last but
    one, 256; the last is just too many), and with shorter lists: both groups on one block's list, with
    empty, one-entry and full lists, against the masked oracle."""
    rng = np.random.default_rng(Sq + Skv)
    q, k, v = (randn_bf16(rng, (1, H, n, 128)) for n in (Sq, Skv, Skv))
    bmap = (rng.random((1, H, -(-Sq // blk_q), -(-Skv // blk_k))) < 0.4).astype(np.uint8)
    bmap[0, 0, 0] = 0
    bmap[0, -1, -1] = 1
    bmap[0, :, -2:-1] = 0
    bmap[0, :, -2:-1, -1] = 1
    lut, cnt = h3attn.block_map_to_lut(torch.from_numpy(bmap).to(gpu))
    out = torch.full((1, Sq, H, 128), float("nan"), dtype=torch.bfloat16, device=gpu).transpose(1, 2)
    ops.attn_fwd_blocksparse(*(to_dev_bf16(x, gpu) for x in (q, k, v)), lut, cnt, blk_q, blk_k, out=out)
    got = oracle.bf16_to_f32(from_dev_bf16(out)).reshape(out.shape)
    assert_close_absmax(got, oracle.attn_fwd(q, k, v, block_map=bmap, blk_q=blk_q, blk_k=blk_k),
                        what=f"{H} heads {blk_q}x{blk_k}")


def test_one_sparse_block_per_workgroup_wide_kv_stride(gpu):
    """The same with K/V whose rows lie so far apart that a slice passes 2^32 bytes (per-stage descriptors)."""
    torch.manual_seed(2)
    Sq, Skv, stride = 200, 600, (1 << 22) + 8  # lists of up to 10 stages
    buf = torch.empty(Skv * stride, dtype=torch.bfloat16, device=gpu)
    q = torch.randn(1, 1, Sq, 128, device=gpu).bfloat16()
    k, v = (torch.randn(1, 1, Skv, 128, device=gpu).bfloat16() for _ in range(2))
    kw, vw = (buf.as_strided((1, 1, Skv, 128), (0, 128, stride, 1), off * 128) for off in (0, 1))
    kw.copy_(k)
    vw.copy_(v)
    lut, cnt = h3attn.block_map_to_lut((torch.rand(1, 1, 4, 10, device=gpu) < 0.8).to(torch.uint8), 10)
    assert torch.equal(ops.attn_fwd_blocksparse(q, kw, vw, lut, cnt, 64, 64),
                       ops.attn_fwd_blocksparse(q, k, v, lut, cnt, 64, 64))
