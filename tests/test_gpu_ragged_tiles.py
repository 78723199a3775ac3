"""Query tiles whose last rows are missing (waves without rows do not compute, ragged tiles run last) and launches whose
workgroups have fetch-only waves: every count of key tiles around the depth of the fill pipeline, against the oracle and
against the same heads in a launch that is large enough to take the other form."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _rand(B, H, Lq, Lk, d, seed):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(B, H, L, d, generator=g) * 0.5).to(torch.bfloat16) for L in (Lq, Lk, Lk)], g


def _close(o, ref):
    return torch.allclose(o.float().cpu(), ref, atol=2e-2, rtol=1e-2)     # the attention tolerance of bf16 outputs


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("Lq,Lk", [(1, 1), (32, 64), (33, 65), (128, 128), (129, 192), (160, 193), (250, 257), (300, 330)])
def test_few_query_tiles(Lq, Lk, d):
    from lvar_amd import sparse_attn_ops as ops
    H = 270                                                     # more query tiles than compute units: no fetch-only waves; `part`: pairs of waves
    (q, k, v), g = _rand(1, H, Lq, Lk, d, seed=Lq + d)
    qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
    h = slice(H - 3, H)
    part = [t[:, h].contiguous() for t in (qg, kg, vg)]
    o, (M, L) = ops.dense_attn(*part)
    ob, (Mb, Lb) = ops.dense_attn(qg, kg, vg)
    assert torch.equal(o, ob[:, h]) and torch.equal(M, Mb[:, h]) and torch.equal(L, Lb[:, h])
    o_ref, M_ref, L_ref = oracle.dense_attn(q[:, h], k[:, h], v[:, h])
    assert _close(o, o_ref)
    assert torch.allclose((M + L.log2()).cpu(), M_ref + L_ref.log2(), atol=1e-3)
    for bk in (64, 128):
        mask = torch.rand(1, H, -(-Lq // 128), -(-Lk // bk), generator=g) < 0.6      # some lists are empty
        num, idx = oracle.block_mask_to_lists(mask)
        o, (M, L) = ops.block_sparse_attn(*part, num[:, h].contiguous().cuda(), idx[:, h].contiguous().cuda(), 128, bk)
        ob, (Mb, Lb) = ops.block_sparse_attn(qg, kg, vg, num.cuda(), idx.cuda(), 128, bk)
        assert torch.equal(o, ob[:, h]) and torch.equal(M, Mb[:, h]) and torch.equal(L, Lb[:, h])
        o_ref, _, _ = oracle.block_sparse_attn(q[:, h], k[:, h], v[:, h], num[:, h], idx[:, h], 128, bk)
        assert _close(o, o_ref)


# 128-row workgroups of four computing and four fetch waves, where 64-row ones (dense: and 96-row ones) are more than the compute
# units: every count of key tiles around the depth of the pipeline, waves without rows and empty lists, against a larger launch
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("Lk", [1, 64, 65, 128, 190, 257, 320])
@pytest.mark.parametrize("tiles,Lq,dense", [(1, 97, True), (1, 128, True), (2, 193, True), (2, 250, True), (1, 65, False), (1, 96, False), (2, 129, False), (2, 225, False)])
def test_four_computing_and_four_fetch_waves(tiles, Lq, dense, Lk, d):
    from lvar_amd import sparse_attn_ops as ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    H = cus // tiles
    g = torch.Generator(device="cuda").manual_seed(Lq + Lk + d)
    q, k, v = ((torch.randn(1, 2 * cus // tiles + 3, L, d, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for L in (Lq, Lk, Lk))
    part = [t[:, 1:H + 1].contiguous() for t in (q, k, v)]
    if dense:
        o, (M, L) = ops.dense_attn(q, k, v)
        o1, (M1, L1) = ops.dense_attn(*part)
    else:
        num, idx = ops.mask_to_lists(torch.rand(1, q.shape[1], tiles, -(-Lk // 64), generator=g, device="cuda") < 0.6)
        o, (M, L) = ops.block_sparse_attn(q, k, v, num, idx, 128, 64)
        o1, (M1, L1) = ops.block_sparse_attn(*part, num[:, 1:H + 1].contiguous(), idx[:, 1:H + 1].contiguous(), 128, 64)
    assert torch.equal(o1, o[:, 1:H + 1]) and torch.equal(M1, M[:, 1:H + 1]) and torch.equal(L1, L[:, 1:H + 1])
    if dense:
        assert _close(o1[:, :2], oracle.dense_attn(*(t[:, :2].cpu() for t in part))[0])


# rows of the last query group / tile: one, a wave less one row, a wave, all but a wave; heads that do not divide by eight
@pytest.mark.parametrize("B,H,rows", [(1, 1, 1), (1, 3, 31), (1, 9, 32), (2, 5, 33), (3, 3, 96), (1, 17, 160)])
def test_ragged_last_tile(B, H, rows):
    from lvar_amd import sparse_attn_ops as ops
    for d in (64, 128):
        Lq, Lk = 2 * 192 + rows, 700
        (q, k, v), g = _rand(B, H, Lq, Lk, d, seed=rows)
        G = -(-Lq // 192)
        idx = torch.randint(0, Lk, (B, H, G, Lk), generator=g, dtype=torch.int32)
        cnt = torch.randint(0, 301, (B, H, G), generator=g, dtype=torch.int32)
        o0 = (torch.randn(B, H, Lq, d, generator=g) * 0.5).to(torch.bfloat16)
        qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
        out = ops.csp_attn(qg, kg, vg, None, idx.cuda(), cnt.cuda(), o0.cuda(), 1)
        assert _close(out, oracle.csp_attn(q, k, v, None, idx, cnt, o0, 1))
        # 128-row tiles with the same remainder (256-row ones: test_ragged_last_tile_of_256_rows)
        Lq = 128 + min(rows, 127)
        o, _ = ops.dense_attn(qg[:, :, :Lq].contiguous(), kg, vg)
        assert _close(o, oracle.dense_attn(q[:, :, :Lq], k, v)[0])


# 256-row workgroups: one per compute unit of the launch's single round, seven 128-row tiles per head (1.75 per compute unit,
# the same round shared by two) in the other form; the last of four tiles has 40 of its 256 rows, six of eight waves idle
@pytest.mark.parametrize("Lk", [1, 64, 65, 128, 190, 257, 320])
def test_ragged_last_tile_of_256_rows(Lk):
    from lvar_amd import sparse_attn_ops as ops
    H, Lq = torch.cuda.get_device_properties(0).multi_processor_count // 4, 3 * 256 + 40
    (q, k, v), g = _rand(1, H, Lq, Lk, 128, seed=7)
    qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
    o, (M, L) = ops.dense_attn(qg, kg, vg)
    h = slice(H - 2, H)
    part = [t[:, h].contiguous() for t in (qg, kg, vg)]
    o1, (M1, L1) = ops.dense_attn(*part)      # few tiles: 64-row workgroups of pairs of waves
    assert torch.equal(o1, o[:, h]) and torch.equal(M1, M[:, h]) and torch.equal(L1, L[:, h])
    assert _close(o1, oracle.dense_attn(q[:, h], k[:, h], v[:, h])[0])
    mask = torch.rand(1, H, 4, -(-Lk // 64), generator=g) < 0.7          # lists of 256-row query blocks, some of them empty
    num, idx = oracle.block_mask_to_lists(mask)
    o, (M, L) = ops.block_sparse_attn(qg, kg, vg, num.cuda(), idx.cuda(), 256, 64)
    o1, (M1, L1) = ops.block_sparse_attn(*part, num[:, h].contiguous().cuda(), idx[:, h].contiguous().cuda(), 256, 64)
    assert torch.equal(o1, o[:, h]) and torch.equal(M1, M[:, h]) and torch.equal(L1, L[:, h])
    assert _close(o1, oracle.block_sparse_attn(q[:, h], k[:, h], v[:, h], num[:, h], idx[:, h], 256, 64)[0])


# token lists whose ragged groups run behind the whole ones: more groups than compute units, fewer than one per head in the
# last round, 30 of 192 rows in a head's last group
@pytest.mark.parametrize("d", [64, 128])
def test_ragged_groups_behind_the_whole_ones(d):
    from lvar_amd import sparse_attn_ops as ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    H, Lq, Lk = cus // 2 + 19, 192 + 30, 300
    assert cus < 2 * H and 2 * H - cus < H
    (q, k, v), g = _rand(1, H, Lq, Lk, d, seed=d)
    idx = torch.randint(0, Lk, (1, H, 2, Lk), generator=g, dtype=torch.int32)
    cnt = torch.randint(0, 201, (1, H, 2), generator=g, dtype=torch.int32)
    o0 = (torch.randn(1, H, Lq, d, generator=g) * 0.5).to(torch.bfloat16)
    out = ops.csp_attn(q.cuda(), k.cuda(), v.cuda(), None, idx.cuda(), cnt.cuda(), o0.cuda(), 1)
    assert _close(out, oracle.csp_attn(q, k, v, None, idx, cnt, o0, 1))
