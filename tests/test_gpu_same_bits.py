"""Bits that must not depend on the launch shape or on the host path of a call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(B, H, Lq, Lk, d, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [(torch.randn(B, H, L, d, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for L in (Lq, Lk, Lk)]


# an image alone and in a batch: launches that leave compute units idle, that fill them once, and larger ones
@pytest.mark.parametrize("B,H,Lq,Lk,d", [(2, 16, 16, 21, 128), (2, 16, 144, 265, 128), (2, 16, 576, 1497, 128), (8, 16, 256, 680, 64),
                                         (4, 16, 256, 521, 64), (3, 24, 400, 921, 128), (2, 140, 100, 1090, 128), (4, 32, 700, 600, 128)])
def test_attention_of_a_head_does_not_depend_on_the_others(B, H, Lq, Lk, d):
    from lvar_amd import sparse_attn_ops as ops
    q, k, v = _rand(B, H, Lq, Lk, d, seed=Lq)
    o, (M, L) = ops.dense_attn(q, k, v)
    g = torch.Generator(device="cuda").manual_seed(Lk)
    num, idx = ops.mask_to_lists(torch.rand(B, H, -(-Lq // 128), -(-Lk // 64), generator=g, device="cuda") < 0.7)
    ob, (Mb, Lb) = ops.block_sparse_attn(q, k, v, num, idx, 128, 64)
    for b, h in ((0, slice(0, 1)), (B - 1, slice(H // 2, H // 2 + 3))):
        part = [t[b:b + 1, h].contiguous() for t in (q, k, v)]
        o1, (M1, L1) = ops.dense_attn(*part)
        assert torch.equal(o1[0], o[b, h]) and torch.equal(M1[0], M[b, h]) and torch.equal(L1[0], L[b, h])
        o1, (M1, L1) = ops.block_sparse_attn(*part, num[b:b + 1, h].contiguous(), idx[b:b + 1, h].contiguous(), 128, 64)
        assert torch.equal(o1[0], ob[b, h]) and torch.equal(M1[0], Mb[b, h]) and torch.equal(L1[0], Lb[b, h])


# head_dim 64: as many 128-row workgroups as two per compute unit hold, and one row more per head; lists of 128 and of 64 rows
@pytest.mark.parametrize("extra,bq", [(0, 128), (1, 128), (0, 64), (1, 64)])
def test_head_dim_64_on_both_sides_of_two_workgroups_per_compute_unit(extra, bq):
    from lvar_amd import sparse_attn_ops as ops
    H, Lk = torch.cuda.get_device_properties(0).multi_processor_count // 4, 300
    q, k, v = _rand(1, H, 1024 + extra, Lk, 64, seed=extra)               # 8 or 9 tiles of 128 rows per head
    g = torch.Generator(device="cuda").manual_seed(bq)
    num, idx = ops.mask_to_lists(torch.rand(1, H, -(-(1024 + extra) // bq), -(-Lk // 64), generator=g, device="cuda") < 0.6)
    o, (M, L) = ops.block_sparse_attn(q, k, v, num, idx, bq, 64)
    od, (Md, Ld) = ops.dense_attn(q, k, v)
    h = slice(H - 2, H)
    part = [t[:, h].contiguous() for t in (q, k, v)]
    o1, (M1, L1) = ops.block_sparse_attn(*part, num[:, h].contiguous(), idx[:, h].contiguous(), bq, 64)
    assert torch.equal(o1, o[:, h]) and torch.equal(M1, M[:, h]) and torch.equal(L1, L[:, h])
    o1, (M1, L1) = ops.dense_attn(*part)
    assert torch.equal(o1, od[:, h]) and torch.equal(M1, Md[:, h]) and torch.equal(L1, Ld[:, h])


@pytest.mark.parametrize("B,H,n,S", [(1, 4, 7, 20), (2, 16, 5, 12), (1, 8, 8, 24), (2, 16, 10, 40)])
def test_full_step_lists_do_not_depend_on_the_host_path(B, H, n, S, monkeypatch):
    """Column sums of three repeats of the same keys in other orders: scores that are equal up to the order of their sums."""
    from lvar_amd import mask_build as mb, sparse_attn_ops as ops
    from lvar_amd.sparse_diff_attn import SparseDiffAttn
    if ops._native() is None:
        pytest.skip("torch binding not built")
    scales = mb.INFINITY_SCALES[:n] + (S,)
    Lk = sum(s * s for s in scales)
    q, k, v = _rand(B, H, S * S, Lk, 128, seed=S)
    third = Lk // 3
    k[:, :, third:2 * third] = k[:, :, :third].flip(2)
    k[:, :, 2 * third:3 * third] = k[:, :, :third].roll(7, dims=2)
    got = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_native", lambda: None)
        layer = SparseDiffAttn(scales=scales, spsd_scale=len(scales) - 1)
        o = layer(q, k, v, None, do_full_step=True, scale_ind=len(scales) - 1)
        got.append((o, layer.out_cache, layer.indices[..., :layer.count_host], layer.counts))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_full_step_calls_a_replaced_colsum_operator():
    """``dense_colsum_attn`` is an attribute of the layer that a caller may replace."""
    from lvar_amd import mask_build as mb
    from lvar_amd.sparse_diff_attn import SparseDiffAttn
    scales = mb.INFINITY_SCALES[:7] + (20,)
    q, k, v = _rand(1, 2, 400, sum(s * s for s in scales), 128, seed=3)
    layer = SparseDiffAttn(scales=scales, spsd_scale=len(scales) - 1)
    plain = layer(q, k, v, None, do_full_step=True, scale_ind=len(scales) - 1)
    inner, calls = layer.dense_colsum_attn, []

    def reversed_sums(*a):
        calls.append(len(a))
        o, cs = inner(*a)
        return o, (-cs).contiguous()
    first = layer.indices[..., :layer.count_host].clone()
    layer.dense_colsum_attn = reversed_sums
    o = layer(q, k, v, None, do_full_step=True, scale_ind=len(scales) - 1)
    assert calls == [4] and torch.equal(o, plain)
    assert not torch.equal(layer.indices[..., :layer.count_host], first)      # the least-attended keys now
