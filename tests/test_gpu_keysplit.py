"""Workgroup shapes of dense and block-list attention: launches that leave compute units idle or fill them once with 128-row
workgroups, and launches of 256-row workgroups, at the edges of tiles and with odd, short and empty lists."""
import pytest
import torch

import oracle
from conftest import make_qkv

pytestmark = pytest.mark.gpu


def _close(o, ref):
    assert torch.allclose(o.float().cpu(), ref, atol=2e-2, rtol=1e-2)


# at most one 128-row workgroup per compute unit
@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,d", [
    (1, 2, 2, 1, 193, 128), (1, 2, 2, 64, 256, 128), (2, 2, 1, 65, 257, 64), (1, 3, 3, 129, 319, 128), (1, 2, 2, 200, 449, 64),
    (1, 140, 140, 128, 512, 128), (1, 140, 140, 100, 577, 128), (1, 130, 65, 127, 513, 64), (2, 64, 64, 200, 640, 64),
    (1, 140, 140, 128, 1024, 128), (1, 140, 140, 100, 1090, 128),
])
def test_dense_128_row_workgroups(B, H, Hkv, Lq, Lk, d):
    from lvar_amd import sparse_attn_ops as ops
    q, k, v = make_qkv(B, H, Lq, Lk, d, seed=Lq + Lk)
    k, v = k[:, :Hkv].contiguous(), v[:, :Hkv].contiguous()
    o, (M, L) = ops.dense_attn(q.cuda(), k.cuda(), v.cuda())
    hs = slice(0, min(H, 6))
    kx, vx = k.repeat_interleave(H // Hkv, 1)[:, hs], v.repeat_interleave(H // Hkv, 1)[:, hs]
    o_ref, M_ref, L_ref = oracle.dense_attn(q[:, hs], kx, vx)
    _close(o[:, hs], o_ref)
    lse = (M + torch.log2(L))[:, hs].cpu()
    assert torch.allclose(lse, M_ref + torch.log2(L_ref), atol=1e-3, rtol=0)
    if H > 6:   # every head of the launch, against the statement in float32 on the device
        s = torch.matmul(q.cuda().float(), k.cuda().float().repeat_interleave(H // Hkv, 1).transpose(-1, -2).contiguous()) * d ** -0.5
        ref = torch.matmul(s.softmax(-1), v.cuda().float().repeat_interleave(H // Hkv, 1))
        assert torch.allclose(o.float(), ref, atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("B,H,Lq,Lk,d", [(2, 64, 257, 65, 128), (1, 200, 250, 300, 64), (2, 70, 385, 130, 128), (1, 256, 512, 64, 128), (1, 250, 512, 1, 128)])
def test_dense_256_row_workgroups(B, H, Lq, Lk, d):
    """More than one 128-row tile per compute unit and at most one 256-row tile (or whole rounds of them)."""
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(Lq)
    q, k, v = (torch.randn(B, H, L, d, generator=g, device="cuda").to(torch.bfloat16) for L in (Lq, Lk, Lk))
    o, (M, L) = ops.dense_attn(q, k, v)
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) * d ** -0.5
    assert torch.allclose(o.float(), torch.matmul(s.softmax(-1), v.float()), atol=2e-2, rtol=1e-2)
    assert torch.allclose(M + torch.log2(L), torch.logsumexp(s, -1, keepdim=True) * 1.4426950408889634, atol=1e-3, rtol=0)


def test_dense_growing_logits():
    """Row maxima that grow along the keys: the reference moves again and again."""
    from lvar_amd import sparse_attn_ops as ops
    q, k, v = make_qkv(1, 2, 100, 700, 128, seed=9)
    k = (k.float() * torch.linspace(0.1, 6.0, 700).view(1, 1, -1, 1)).to(torch.bfloat16)
    o, _ = ops.dense_attn(q.cuda(), k.cuda(), v.cuda())
    _close(o, oracle.dense_attn(q, k, v)[0])


@pytest.mark.parametrize("H,Lq,Lk,d,bq,bk", [(2, 300, 1000, 128, 128, 64), (3, 130, 900, 64, 128, 128), (2, 200, 1100, 128, 64, 64),
                                             (140, 128, 1024, 128, 128, 64), (135, 120, 1300, 64, 128, 256), (140, 120, 1000, 128, 128, 64)])
def test_block_lists_128_row_workgroups(H, Lq, Lk, d, bq, bk):
    from lvar_amd import sparse_attn_ops as ops
    q, k, v = make_qkv(1, H, Lq, Lk, d, seed=Lq)
    nQ, nK = -(-Lq // bq), -(-Lk // bk)
    g = torch.Generator().manual_seed(Lk)
    mask = torch.rand(1, H, nQ, nK, generator=g) < 0.4
    mask[0, 0, 0] = False                      # an empty list
    mask[0, 1, 0] = False
    mask[0, 1, 0, nK - 1] = True               # one block, the ragged last one
    num, idx = ops.mask_to_lists(mask.cuda())
    o, (M, L) = ops.block_sparse_attn(q.cuda(), k.cuda(), v.cuda(), num, idx, bq, bk)
    hs = slice(0, min(H, 6))
    o_ref = oracle.block_sparse_attn(q[:, hs], k[:, hs], v[:, hs], num.cpu()[:, hs], idx.cpu()[:, hs], bq, bk)[0]
    _close(o[:, hs], o_ref)
    assert bool((o[0, 0, :min(bq, Lq)] == 0).all())


@pytest.mark.parametrize("B,H,Lq,Lk,d,bq,bk", [(1, 3, 300, 500, 128, 128, 64), (2, 20, 1000, 900, 64, 128, 128), (1, 7, 700, 1100, 128, 64, 64),
                                               (2, 70, 640, 300, 128, 256, 256), (1, 9, 700, 800, 128, 256, 64), (2, 40, 520, 600, 128, 384, 128)])
def test_block_lists_of_several_workgroups(B, H, Lq, Lk, d, bq, bk):
    """Query blocks of several workgroups and of 256-row workgroups, a ragged last block among them."""
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(Lq + bk)
    q, k, v = (torch.randn(B, H, L, d, generator=g, device="cuda").to(torch.bfloat16) for L in (Lq, Lk, Lk))
    nQ, nK = -(-Lq // bq), -(-Lk // bk)
    num, idx = ops.mask_to_lists(torch.rand(1, 1, nQ, nK, generator=g, device="cuda") < 0.5)
    ref, _ = ops.block_sparse_attn(q, k, v, num, idx, bq, bk)
    assert torch.equal(ops.block_sparse_attn_out(q, k, v, num, idx, bq, bk), ref)
    m = torch.zeros(nQ, nK, dtype=torch.bool, device="cuda")
    for i in range(nQ):
        m[i, idx[0, 0, i, :int(num[0, 0, i])].long()] = True
    m = m.repeat_interleave(bq, 0)[:Lq].repeat_interleave(bk, 1)[:, :Lk]
    s = (torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) * d ** -0.5).masked_fill(~m, float("-inf"))
    assert torch.allclose(ref.float(), torch.matmul(s.softmax(-1).nan_to_num(0.0), v.float()), atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("H,G", [(40, 2), (128, 1), (130, 1), (80, 2), (150, 2), (200, 2)])
def test_token_lists_head_dim_64_both_workgroup_shapes(H, G):
    """192-row groups run as 8-wave or as two 3-wave workgroups, by how full the last round of 8-wave ones is: the same
    bits as with the lists repeated for groups of 96 rows (which always take the 3-wave form)."""
    from test_gpu_random_shapes import _csp_abi
    g = torch.Generator(device="cuda").manual_seed(H + G)
    Lq, Lk, d = G * 192 - 37, 330, 64
    q, o0, k, v = (torch.randn(1, H, L, d, generator=g, device="cuda").to(torch.bfloat16) for L in (Lq, Lq, Lk, Lk))
    idx = torch.randint(0, Lk, (1, H, G, Lk), generator=g, device="cuda", dtype=torch.int32)
    cnt = torch.randint(0, Lk + 1, (1, H, G), generator=g, device="cuda", dtype=torch.int32)
    st, out = _csp_abi(q, k, v, idx, cnt, o0, 192, -1)
    st2, out2 = _csp_abi(q, k, v, idx.repeat_interleave(2, dim=2).contiguous(), cnt.repeat_interleave(2, dim=2).contiguous(), o0, 96, -1)
    assert st == 0 and st2 == 0 and torch.equal(out, out2)
