"""Tiles that run longest list first where a launch ends on a short round: every tile is computed once, with the bits that its head has
alone (a launch of one round, in natural order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 128-row tiles per head and heads: whole heads per XCD and heads across two, a ragged last tile in the order and behind it, as many
# tiles as a wave has lanes and one more, launches with and without a short last round
@pytest.mark.parametrize("H,Lq", [(32, 2304), (40, 1920), (39, 2200), (24, 3010), (9, 8192), (9, 8300), (32, 2048), (300, 240)])
@pytest.mark.parametrize("lists", ["random", "shared", "equal"])
def test_tiles_by_length_give_the_bits_of_a_head_alone(H, Lq, lists):
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(H + Lq)
    Lk, nQ = 640, -(-Lq // 128)
    q, k, v = ((torch.randn(1, H, L, 128, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for L in (Lq, Lk, Lk))
    mask = torch.rand(1, 1 if lists == "shared" else H, nQ, Lk // 64, generator=g, device="cuda") < 0.5
    if lists == "equal":
        mask = torch.zeros_like(mask).scatter_(-1, torch.rand(mask.shape, generator=g, device="cuda").topk(4, dim=-1).indices, True)
    num, idx = ops.mask_to_lists(mask)
    o, (M, L) = ops.block_sparse_attn(q, k, v, num, idx, 128, 64)
    num, idx = num.expand(1, H, nQ), idx.expand(1, H, nQ, idx.shape[-1])
    for h in range(H):
        part = [t[:, h:h + 1].contiguous() for t in (q, k, v, num, idx)]
        o1, (M1, L1) = ops.block_sparse_attn(*part, 128, 64)
        assert torch.equal(o[:, h], o1[:, 0]) and torch.equal(M[:, h], M1[:, 0]) and torch.equal(L[:, h], L1[:, 0]), h
