"""Block selection against a stable descending sort: rows at the edges of the keys-per-lane steps, ties across the cut."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nK", [1, 2, 63, 64, 65, 128, 129, 193, 256, 257, 385, 513, 1000, 1025, 1537, 2048])
@pytest.mark.parametrize("kind", ["distinct", "ties", "equal", "signed"])
def test_block_topk_lists_against_a_stable_sort(nK, kind):
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator().manual_seed(nK)
    B, H, nQ = 1, 3, 5                                    # 15 rows: the last workgroup has one idle wave
    s = torch.rand(B, H, nQ, nK, generator=g)
    if kind == "ties":
        s = (s * 4).floor()
    elif kind == "equal":
        s = torch.zeros_like(s)
        s[..., ::2] = -0.0                                # ties with +0.0
    elif kind == "signed":
        s = s - 0.5
        s[0, 0, 0, 0] = float("-inf")
        s[0, 1, 0, nK - 1] = float("inf")
    base = torch.rand(nQ, nK, generator=g) < 0.2
    base[0] = False
    base[1] = True
    for target in sorted({0, 1, nK // 3, max(0, nK - 1), nK, nK + 5}):
        for m in (None, base):
            num, idx = ops.block_topk_lists(s.cuda(), target, None if m is None else m.cuda())
            keep = torch.zeros(B, H, nQ, nK, dtype=torch.bool) if m is None else m.expand(B, H, nQ, nK).clone()
            for h in range(H):
                for i in range(nQ):
                    extra = max(0, min(target, nK) - int(keep[0, h, i].sum()))
                    free = (~keep[0, h, i]).nonzero()[:, 0]
                    order = torch.sort(s[0, h, i][free] + 0.0, descending=True, stable=True).indices
                    keep[0, h, i, free[order[:extra]]] = True
            assert torch.equal(num.cpu(), keep.sum(-1, dtype=torch.int32))
            ref = torch.zeros(B, H, nQ, nK, dtype=torch.int32)
            for h in range(H):
                for i in range(nQ):
                    on = keep[0, h, i].nonzero()[:, 0].int()
                    ref[0, h, i, :len(on)] = on
            assert torch.equal(idx.cpu(), ref)


@pytest.mark.parametrize("cnt,L,Gs,Gk,Ks", [(1, 0, 1, 3, 64), (255, 64, 3, 5, 300), (2048, 704, 9, 22, 2048), (2049, 2047, 2, 7, 2100), (130, 5, 4, 2, 60)])
def test_remap_lists_at_the_edges_of_a_batch_of_reads(cnt, L, Gs, Gk, Ks):
    """(130 entries of rows of 60: entries are repeated.)"""
    from lvar_amd import mask_build as mb, sparse_attn_ops as ops
    g = torch.Generator().manual_seed(cnt)
    q_len, k_len = Gk * 192 - 5, max(cnt + L, 400)
    src = torch.randint(0, k_len + 50, (2, 3, Gs, Ks), generator=g, dtype=torch.int32)
    local = torch.randint(0, k_len, (Gk, L), generator=g) if L else None
    idx, counts = ops.remap_concat_lists(src.cuda(), cnt, q_len, k_len, None if local is None else local.cuda(), indices_pad_to=1)
    ref, rc = mb.map_inds_counts_across_scales(src, cnt, q_len, k_len)
    assert torch.equal(idx[..., :cnt].cpu(), ref) and bool((counts.cpu() == rc + L).all())
    if L:
        assert torch.equal(idx[..., cnt:cnt + L].cpu(), local.int().expand(2, 3, Gk, L))
    assert bool((idx[..., cnt + L:] == 0).all())
