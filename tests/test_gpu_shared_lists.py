"""Lists that every (batch, head) shares run longest first where the launch ends on a partial round: every tile is computed once, with
the bits of the same lists handed over per head (which keep their order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 128-row tiles per head and heads: whole heads per XCD and heads across two, a ragged last tile in the order and behind it, as many
# tiles as a wave has lanes and one more, launches with and without a partial last round
@pytest.mark.parametrize("H,Lq", [(32, 2304), (40, 2304), (39, 2200), (24, 3010), (9, 8192), (9, 8300), (32, 2048), (300, 200)])
@pytest.mark.parametrize("lengths", ["random", "equal"])
def test_shared_lists_give_the_bits_of_lists_per_head(H, Lq, lengths):
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(H + Lq)
    Lk, nQ = 640, -(-Lq // 128)
    q, k, v = ((torch.randn(1, H, L, 128, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for L in (Lq, Lk, Lk))
    mask = torch.rand(1, 1, nQ, Lk // 64, generator=g, device="cuda") < 0.5
    if lengths == "equal":
        mask = torch.zeros_like(mask).scatter_(-1, torch.rand(mask.shape, generator=g, device="cuda").topk(4, dim=-1).indices, True)
    num, idx = ops.mask_to_lists(mask)
    o, (M, L) = ops.block_sparse_attn(q, k, v, num, idx, 128, 64)
    per_head = num.expand(1, H, nQ).contiguous(), idx.expand(1, H, nQ, idx.shape[-1]).contiguous()
    o1, (M1, L1) = ops.block_sparse_attn(q, k, v, *per_head, 128, 64)
    assert torch.equal(o, o1) and torch.equal(M, M1) and torch.equal(L, L1)
