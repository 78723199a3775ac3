"""Launches whose waves work in pairs (64-row workgroups that have a compute unit each), and token lists in half groups, against
larger launches of the same heads, which do neither: the same bits, whatever the number of key tiles, ragged rows or keys and
growth of the row maximum."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(H, Lq, Lk, d, seed, growth):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(1, H, L, d, generator=g, device="cuda") for L in (Lq, Lk, Lk))
    # growing keys: the reference maximum of most rows moves again and again, in some tiles for a few rows of a wave only
    k = k * (0.5 + growth * torch.arange(Lk, device="cuda").div(64, rounding_mode="floor").float().view(1, 1, Lk, 1))
    return [t.to(torch.bfloat16) for t in (q * 0.5, k, v)]


@pytest.mark.parametrize("growth", [0.0, 0.7])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("Lq,Lk", [(1, 1), (33, 64), (64, 65), (65, 128), (96, 129), (127, 200), (128, 257), (130, 640), (40, 1000)])
def test_pairs_give_the_bits_of_larger_launches(Lq, Lk, d, growth):
    from lvar_amd import sparse_attn_ops as ops
    H = 2 * torch.cuda.get_device_properties(0).multi_processor_count + 3          # no launch of pairs
    q, k, v = _inputs(H, Lq, Lk, d, seed=Lq * 7 + Lk, growth=growth)
    o, (M, L) = ops.dense_attn(q, k, v)
    g = torch.Generator(device="cuda").manual_seed(Lk)
    nQ, nK = -(-Lq // 128), -(-Lk // 64)
    num, idx = ops.mask_to_lists(torch.rand(1, H, nQ, nK, generator=g, device="cuda") < 0.6)      # empty lists among them
    ob, (Mb, Lb) = ops.block_sparse_attn(q, k, v, num, idx, 128, 64)
    for h in (slice(0, 1), slice(5, 12), slice(H - 40, H)):
        part = [t[:, h].contiguous() for t in (q, k, v)]
        o1, (M1, L1) = ops.dense_attn(*part)
        assert torch.equal(o1, o[:, h]) and torch.equal(M1, M[:, h]) and torch.equal(L1, L[:, h])
        o1, (M1, L1) = ops.block_sparse_attn(*part, num[:, h].contiguous(), idx[:, h].contiguous(), 128, 64)
        assert torch.equal(o1, ob[:, h]) and torch.equal(M1, Mb[:, h]) and torch.equal(L1, Lb[:, h])


# rows: one part-filled pair, whole groups of 192, 64, 96 and 160 rows in the last one
@pytest.mark.parametrize("growth", [0.0, 0.7])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("Lq,Lk,keys", [(20, 70, 33), (192, 400, 64), (256, 700, 129), (288, 500, 200), (400, 900, 450), (544, 300, 300)])
def test_token_lists_give_the_bits_of_larger_launches(Lq, Lk, keys, d, growth):
    from lvar_amd import sparse_attn_ops as ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    H, G = cus + 3, -(-Lq // 192)                                                             # more groups than compute units
    q, k, v = _inputs(H, Lq, Lk, d, seed=Lq + keys, growth=growth)
    g = torch.Generator(device="cuda").manual_seed(keys)
    idx = torch.rand(1, H, G, Lk, generator=g, device="cuda").argsort(-1).int()
    cnt = torch.randint(0, keys + 1, (1, H, G), generator=g, device="cuda", dtype=torch.int32)  # empty and part-filled lists
    cache = torch.randn(1, H, Lq, d, generator=g, device="cuda").to(torch.bfloat16)
    o = ops.csp_attn(q, k, v, None, idx, cnt, cache, -1.0)
    pair_heads, half_heads = cus // -(-Lq // 64), cus // -(-Lq // 96)                         # the most that either form takes
    for h in (slice(0, 1), slice(H - pair_heads, H), slice(H - half_heads, H)):
        q1, k1, v1, idx1, cnt1, cache1 = (t[:, h].contiguous() for t in (q, k, v, idx, cnt, cache))
        o1 = ops.csp_attn(q1, k1, v1, None, idx1, cnt1, cache1, -1.0)
        assert torch.equal(o1, o[:, h])


# dense launches in 96-row workgroups: more 64-row ones than compute units, but not more 96-row ones
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("Lq,Lk", [(65, 64), (96, 130), (97, 700), (190, 321)])
def test_96_row_workgroups_give_the_bits_of_larger_launches(Lq, Lk, d):
    from lvar_amd import sparse_attn_ops as ops
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    q, k, v = _inputs(2 * cus + 3, Lq, Lk, d, seed=Lq, growth=0.7)
    o, (M, L) = ops.dense_attn(q, k, v)
    h = slice(5, 5 + cus // -(-Lq // 96))
    o1, (M1, L1) = ops.dense_attn(*(t[:, h].contiguous() for t in (q, k, v)))
    assert torch.equal(o1, o[:, h]) and torch.equal(M1, M[:, h]) and torch.equal(L1, L[:, h])


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("growth", [0.0, 0.7])
def test_pairs_against_float64(growth, d):
    """bf16 inputs, P rounded to bf16: 2^-9 per probability and per output, so 1 % of the largest output is four times that."""
    from lvar_amd import sparse_attn_ops as ops
    q, k, v = _inputs(3, 150, 500, d, seed=1, growth=growth)
    o, (M, L) = ops.dense_attn(q, k, v)
    s = (q.double().cpu() @ k.double().cpu().transpose(-1, -2).contiguous()) / d ** 0.5
    ref = s.softmax(-1) @ v.double().cpu()
    assert (o.double().cpu() - ref).abs().max() < 1e-2 * ref.abs().max()
    lse = (M.double() + L.double().log2()).cpu().reshape(1, 3, 150)
    assert torch.allclose(lse, s.logsumexp(-1) / 0.6931471805599453, rtol=1e-5, atol=1e-4)
