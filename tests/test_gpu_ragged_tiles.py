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
    H = 270                                                     # more query tiles than compute units: no fetch-only waves
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
        # 256-row workgroups (many tiles) are covered by the full-size checks; here 128-row tiles with the same remainder
        Lq = 128 + min(rows, 127)
        o, _ = ops.dense_attn(qg[:, :, :Lq].contiguous(), kg, vg)
        assert _close(o, oracle.dense_attn(q[:, :, :Lq], k, v)[0])


def test_ragged_last_tile_of_256_rows():
    from lvar_amd import sparse_attn_ops as ops
    H, Lq, Lk = 80, 3 * 256 + 40, 200
    (q, k, v), _ = _rand(1, H, Lq, Lk, 128, seed=7)
    o, (M, L) = ops.dense_attn(q.cuda(), k.cuda(), v.cuda())
    h = slice(H - 2, H)
    o1, (M1, L1) = ops.dense_attn(*[t[:, h].contiguous().cuda() for t in (q, k, v)])      # few tiles: 128-row workgroups
    assert torch.equal(o1, o[:, h]) and torch.equal(M1, M[:, h]) and torch.equal(L1, L[:, h])
    assert _close(o1, oracle.dense_attn(q[:, h], k[:, h], v[:, h])[0])
