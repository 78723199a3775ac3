"""Row statistics kernel (base-2 log-sum-exp without the product with v) against a float64 statement of it."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

LOG2E = 1.4426950408889634


def _ref(q, k, scale):
    group = q.shape[1] // k.shape[1]
    k = k.repeat_interleave(group, dim=1)
    s = torch.matmul(q.double().cpu(), k.double().cpu().transpose(-1, -2)) * (scale * LOG2E)
    return torch.logsumexp(s * math.log(2.0), dim=-1) / math.log(2.0)


def _check(q, k, scale):
    from lvar_amd import sparse_attn_ops as ops
    got = ops._lse_only(q, k, scale).double().cpu()
    ref = _ref(q, k, scale)
    # 32-bit sums of d products: d * 2^-24 of the sum of their magnitudes, which is at most |q||k| ~ the largest logit
    # here times a small factor; 2^-17 of the largest statistic and 2^-15 absolute cover both that and the exp2 sum
    tol = 2.0 ** -15 + 2.0 ** -17 * ref.abs().max()
    err = (got - ref).abs().max()
    assert err <= tol, (float(err), float(tol))


@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,d", [
    (1, 1, 1, 1, 1, 128), (1, 2, 2, 31, 17, 64), (2, 2, 1, 64, 32, 128), (1, 3, 3, 65, 33, 128), (2, 4, 2, 255, 64, 64),
    (1, 2, 2, 257, 65, 128), (1, 2, 2, 300, 127, 256), (2, 3, 3, 511, 680, 64), (1, 2, 2, 128, 4121, 128), (1, 2, 1, 700, 1497, 256),
    (2, 16, 16, 576, 1497, 128),
])
def test_row_lse_sizes(B, H, Hkv, Lq, Lk, d):
    g = torch.Generator().manual_seed(Lq * 7 + Lk)
    q = torch.randn(B, H, Lq, d, generator=g).to(torch.bfloat16).cuda()
    k = torch.randn(B, Hkv, Lk, d, generator=g).to(torch.bfloat16).cuda()
    _check(q, k, 1.0 / math.sqrt(d))


@pytest.mark.parametrize("kind", ["ramp_up", "ramp_down", "late_spike", "first_tile_low"])
def test_row_lse_references_far_from_the_first_tile(kind):
    """The reference follows the running sum (ramps), and a jump of more than 2^127 takes the tracked sweep (spike)."""
    g = torch.Generator().manual_seed(3)
    Lq, Lk, d = 200, 700, 128
    q = torch.zeros(1, 2, Lq, d)
    q[..., 0] = 1.0
    q[..., 1:] = torch.randn(1, 2, Lq, d - 1, generator=g) * 0.05
    k = torch.randn(1, 2, Lk, d, generator=g) * 0.05
    n = torch.arange(Lk, dtype=torch.float32)
    k[..., 0] = {"ramp_up": n * 2.0, "ramp_down": -n * 2.0, "late_spike": torch.where(n == 500, 900.0, 0.0),
                 "first_tile_low": torch.where(n < 40, -800.0, 3.0)}[kind]
    q[:, :, ::3, 0] = 0.25                     # lanes of one wave that jump by different amounts
    _check(q.to(torch.bfloat16).cuda(), k.to(torch.bfloat16).cuda(), 1.0)


def test_block_scores_without_the_column_sums():
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator().manual_seed(5)
    q = (torch.randn(1, 2, 512, 64, generator=g) * 0.5).to(torch.bfloat16).cuda()
    k = (torch.randn(1, 2, 700, 64, generator=g) * 0.5).to(torch.bfloat16).cuda()
    rows = q[:, :, ::4]
    got = ops._colsum_block_scores(rows, k, None, 32, 128)
    cs = ops.colsum(rows, k, None, q_group_size=32)
    ref = torch.nn.functional.pad(cs, (0, 68)).unflatten(-1, (6, 128)).sum(-1)
    assert got.shape == ref.shape and torch.allclose(got, ref, rtol=1e-5, atol=0)   # 128 terms in another order: 128 * 2^-24
