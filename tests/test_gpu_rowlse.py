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


# (position, logit in nats) of the largest keys of a row; the last 64-key stage begins at 640, key ranges end at 256, 384 or 512
LATE = [[(690, 60.0)], [(690, 69.5)], [(690, 87.5)], [(690, 88.0)], [(690, 88.5)], [(699, 88.5)], [(300, 60.0), (692, 100.0)],
        [(300, 30.0), (692, 90.0)], [(300, 62.0), (692, 104.0)], [(300, 88.5), (691, 88.5)], [(303, 88.5), (692, 88.5)], [(691, 88.5), (692, 88.5)],
        [(255, 88.5), (300, 88.5)], [(383, 88.5), (600, 88.5)], [(500, 88.5), (600, 88.5)], [(200, 88.5), (500, 88.5), (690, 88.5)]]


def _late_qk(peaks, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.zeros(1, 2, 200, 128)
    q[..., 0] = 1.0
    k = torch.randn(1, 2, 700, 128, generator=g) * 0.05
    k[..., 0] = 0.0
    for n, x in peaks:
        k[:, :, n, 0] = x
    q[:, :, 1::5, 0] = 0.5                     # lanes of one wave that jump by different amounts
    return q.to(torch.bfloat16).cuda(), k.to(torch.bfloat16).cuda()


@pytest.mark.parametrize("cut_keys", [False, True])
@pytest.mark.parametrize("peaks", LATE)
def test_row_lse_largest_keys_in_the_last_stage(peaks, cut_keys):
    """Sums that jump in the last stage of a range, by up to 2^128 against the reference, alone and beside a half of the
    lanes, or a range, whose reference has moved that far before."""
    from lvar_amd import sparse_attn_ops as ops
    q, k = _late_qk(peaks, 11)
    got = ops._lse_only(q, k, 1.0, cut_keys=cut_keys).double().cpu()
    ref = _ref(q, k, 1.0)
    assert (got - ref).abs().max() <= 2.0 ** -15 + 2.0 ** -17 * ref.abs().max()    # the bound of _check


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


# ---- scores of key blocks from the statistics sweep ----

def _scores_ref(q, k, scale, group, block_k):
    k = k.repeat_interleave(q.shape[1] // k.shape[1], dim=1)
    p = (torch.matmul(q.double().cpu(), k.double().cpu().transpose(-1, -2)) * scale).softmax(-1)
    Lq, Lk = p.shape[-2:]
    p = torch.nn.functional.pad(p, (0, -Lk % block_k, 0, -Lq % group))
    return p.unflatten(-1, (-1, block_k)).sum(-1).unflatten(-2, (-1, group)).sum(-2)


def _check_scores(q, k, scale, group, block_k, target, base=None):
    from lvar_amd import sparse_attn_ops as ops
    got = ops._block_scores_for_topk(q, k, scale, group, block_k, base, target)
    ref = _scores_ref(q, k, scale, group, block_k)
    assert got.shape == ref.shape
    # exponents carry 2^-24 of the largest logit and statistic (log2 units, < 2^11 here): 2^-13 ln2 relative, far less
    # for plain inputs; what lies 2^-100 below the largest score is not looked at
    big = float(ref.abs().max())
    assert torch.allclose(got.double().cpu(), ref, rtol=2e-4, atol=big * 1e-6), float((got.double().cpu() - ref).abs().max())
    two_pass = ops._colsum_block_scores(q, k, scale, group, block_k)
    lists, lists2 = ops.block_topk_lists(got, target, base), ops.block_topk_lists(two_pass, target, base)
    assert torch.equal(lists[0], lists2[0]) and torch.equal(lists[1], lists2[1])


@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,d,group,block_k", [
    (1, 1, 1, 1, 1, 128, 32, 128), (1, 2, 2, 33, 64, 64, 32, 64), (2, 2, 1, 95, 129, 128, 32, 128), (1, 3, 3, 256, 257, 128, 64, 128),
    (1, 2, 2, 300, 1000, 256, 128, 128), (1, 2, 2, 513, 2049, 64, 32, 128), (2, 2, 2, 700, 1500, 128, 128, 64), (1, 4, 2, 1024, 4096, 128, 32, 128),
    (1, 3, 3, 200, 640, 128, 96, 128), (1, 24, 24, 2048, 1024, 64, 32, 128), (1, 40, 40, 2048, 704, 128, 64, 64),
])
def test_block_scores_sizes(B, H, Hkv, Lq, Lk, d, group, block_k):
    """Edges of stages, key blocks, key ranges, wave tiles and groups (96: the two-pass form)."""
    g = torch.Generator().manual_seed(Lq + 3 * Lk)
    q = (torch.randn(B, H, Lq, d, generator=g) * 0.5).to(torch.bfloat16).cuda()
    k = (torch.randn(B, Hkv, Lk, d, generator=g) * 0.5).to(torch.bfloat16).cuda()
    nQ, nK = -(-Lq // group), -(-Lk // block_k)
    base = (torch.rand(nQ, nK, generator=g) < 0.2).cuda()
    _check_scores(q, k, d ** -0.5, group, block_k, max(1, nK // 3), base)
    _check_scores(q, k, d ** -0.5, group, block_k, max(1, nK // 2))


@pytest.mark.parametrize("kind", ["ramp_up", "ramp_down", "late_spike", "first_tile_low"])
def test_block_scores_references_far_from_the_first_tile(kind):
    g = torch.Generator().manual_seed(4)
    Lq, Lk, d = 200, 700, 128
    q = torch.zeros(1, 2, Lq, d)
    q[..., 0] = 1.0
    q[..., 1:] = torch.randn(1, 2, Lq, d - 1, generator=g) * 0.05
    k = torch.randn(1, 2, Lk, d, generator=g) * 0.05
    n = torch.arange(Lk, dtype=torch.float32)
    k[..., 0] = {"ramp_up": n * 2.0, "ramp_down": -n * 2.0, "late_spike": torch.where(n == 500, 900.0, 0.0),
                 "first_tile_low": torch.where(n < 40, -800.0, 3.0)}[kind]
    q[:, :, ::3, 0] = 0.25
    _check_scores(q.to(torch.bfloat16).cuda(), k.to(torch.bfloat16).cuda(), 1.0, 32, 128, 2)


@pytest.mark.parametrize("peaks", LATE)
def test_block_scores_largest_keys_in_the_last_stage(peaks):
    """A block sum counts from the row's first reference: one that lies further from the statistic than the exponent range
    must not come out as 0 or NaN."""
    q, k = _late_qk(peaks, 12)
    _check_scores(q, k, 1.0, 32, 128, 2)
    _check_scores(q, k, 1.0, 64, 64, 3)


def test_block_scores_ties_at_the_cut():
    """Equal key blocks in other orders: the two-pass ranking decides (one key range: the statistics have equal bits)."""
    g = torch.Generator().manual_seed(6)
    q = (torch.randn(1, 8, 1024, 128, generator=g) * 0.5).to(torch.bfloat16).cuda()
    one = torch.randn(1, 8, 1, 128, 128, generator=g) * 0.5
    k = one.repeat(1, 1, 3, 1, 1).to(torch.bfloat16)
    for j in range(1, 3):
        k[:, :, j] = k[:, :, j, torch.randperm(128, generator=g)]
    _check_scores(q, k.flatten(2, 3).contiguous().cuda(), 128 ** -0.5, 32, 128, 2)


def test_column_sums_of_queries_with_far_rows():
    """Query rows 4 MiB apart span more than the kernel's 32-bit offsets reach: the operator works on a copy."""
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(8)
    rows, k = ((torch.randn(1, 1, L, 64, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for L in (520, 300))
    far = torch.empty(520 << 21, dtype=torch.bfloat16, device="cuda").as_strided((1, 1, 520, 64), (1 << 31, 1 << 31, 1 << 21, 1))
    far.copy_(rows)
    assert torch.equal(ops.colsum(far, k, None, 192), ops.colsum(rows, k, None, 192))
    assert torch.equal(ops._colsum_block_scores(far, k, None, 32, 128), ops._colsum_block_scores(rows, k, None, 32, 128))
    assert torch.equal(ops._block_scores_for_topk(far, k, None, 32, 128, None, 1), ops._block_scores_for_topk(rows, k, None, 32, 128, None, 1))


@pytest.mark.parametrize("kind", ["zero_queries", "zero_keys", "some_heads", "some_rows", "few_ties", "far_below"])
@pytest.mark.parametrize("group,block_k,d", [(32, 128, 128), (64, 64, 64), (32, 192, 128), (128, 128, 256)])
def test_block_scores_rows_with_many_ties(kind, group, block_k, d):
    """Up to eight scores about the cut are computed one by one; rows with more of them take their scores from the column
    sums of their (batch, head)."""
    g = torch.Generator().manual_seed(21)
    q, k = torch.randn(2, 3, 420, d, generator=g) * 0.5, torch.randn(2, 3, 2000, d, generator=g) * 0.5
    if kind == "zero_queries":
        q[:] = 0
    elif kind == "zero_keys":
        k[:] = 0
    elif kind == "some_heads":
        q[0, 1] = 0
        q[1, 2, :, 5:] = 0
    elif kind == "some_rows":
        q[:, :, 64:160] = 0
        q[1, 0, 400:] = 0
    elif kind == "few_ties":
        nb = 5                                            # five equal blocks among others
        k[:, :, block_k:(nb + 1) * block_k] = k[:, :, :block_k].repeat(1, 1, nb, 1)
    else:                                                 # all mass in one block: the others' scores are 0 or next to it
        k[..., 0] = -900.0
        k[:, :, 3] = 0
        q[..., 0] = 1.0
    q, k = q.to(torch.bfloat16).cuda(), k.to(torch.bfloat16).cuda()
    nQ, nK = -(-420 // group), -(-2000 // block_k)
    base = (torch.rand(nQ, nK, generator=g) < 0.1).cuda()
    for target in (1, nK // 3, nK - 1):
        _check_scores(q, k, d ** -0.5, group, block_k, target)
        _check_scores(q, k, d ** -0.5, group, block_k, target, base)


def test_block_scores_of_equal_blocks_cost_no_more_than_two_passes():
    """Every score of every row about the cut: the scores must not be computed one by one (six times the two-pass form)."""
    from lvar_amd import sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(22)
    k = (torch.randn(1, 8, 16384, 128, generator=g, device="cuda") * 0.5).to(torch.bfloat16)
    q = torch.zeros(1, 8, 4096, 128, device="cuda", dtype=torch.bfloat16)

    def time_of(f):
        f()
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            f()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return sorted(times)[2]
    one, two = time_of(lambda: ops._block_scores_for_topk(q, k, None, 32, 128, None, 12)), time_of(lambda: ops._colsum_block_scores(q, k, None, 32, 128))
    assert one < 2 * two, (one, two)


@pytest.mark.parametrize("amp", [1.0, 16.0, 64.0, 256.0])
@pytest.mark.parametrize("group,low", [(32, 0.0), (64, 0.0), (32, 40.0)])
def test_block_scores_ties_at_the_cut_of_large_logits(amp, group, low):
    """The rounding of the exponents grows with their size, and so does the distance within which the two-pass sums decide.
    Six orders of one block; ``low``: behind a first stage of logits that far below, so that references and statistics part."""
    g = torch.Generator().manual_seed(7)
    q = torch.randn(1, 8, 1024, 128, generator=g) * 0.5 * amp
    one = torch.randn(1, 8, 1, 128, 128, generator=g) * 0.5
    k = one.repeat(1, 1, 7, 1, 1)
    for j in range(1, 7):
        k[:, :, j] = k[:, :, j, torch.randperm(128, generator=g)]
    if low:
        q[..., 0] = 1.0
        k[..., 0] = 0.0
        k[:, :, 0, :, 0] = -low * 128 ** 0.5
    k = k.flatten(2, 3) if low else k[:, :, 1:].flatten(2, 3)
    _check_scores(q.to(torch.bfloat16).cuda(), k.to(torch.bfloat16).contiguous().cuda(), 128 ** -0.5, group, 128, 3)


@pytest.mark.parametrize("amp,low", [(1, 0), (1, 60), (4, 45), (16, 0), (16, 30), (16, 60), (64, 0), (64, 20), (64, 30)])
def test_block_scores_differ_from_two_passes_by_less_than_half_the_distance_looked_at(amp, low):
    """Scores from one sweep, none computed again, against the column sums: half of the distance from the cut within which
    both forms are compared, 2^-20 + 2^-23 (D + log2(terms) + |log2(score)|), D = statistic less the first stage's maximum.
    (The other half is the other score's.  Measured: 4 units of 2^-24 for plain inputs, 80 at the largest logits here.)"""
    from lvar_amd import _lib, sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(amp * 100 + low)
    q = torch.randn(1, 4, 1024, 128, generator=g, device="cuda") * 0.5 * amp
    k = torch.randn(1, 4, 2048, 128, generator=g, device="cuda") * 0.5
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    k[:, :, :64, 0] = -low * 128 ** 0.5
    q, k, scale = q.to(torch.bfloat16), k.to(torch.bfloat16), 128 ** -0.5
    lib = _lib.load()
    one = torch.empty(1, 4, 32, 16, device="cuda")
    nbytes = lib.lvar_block_scores_scratch_bytes(1, 4, 1024, 2048, 32, 128)
    scratch = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    assert lib.lvar_block_scores_fwd(ops._view(q), ops._view(k), one.data_ptr(), None, 0, scratch.data_ptr(), nbytes, 1, 4, 4, 1024, 2048, 128,
                                     32, 128, scale, ops._stream(q)) == 0
    two = ops._colsum_block_scores(q, k, scale, 32, 128).double()
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * (scale * LOG2E)
    far = (torch.logsumexp(s * math.log(2.0), -1) / math.log(2.0) - s[..., :64].amax(-1)).unflatten(-1, (32, 32)).amax(-1, keepdim=True)
    limit = 2.0 ** -20 + 2.0 ** -23 * (far + math.log2(32 * 128) + two.clamp_min(2.0 ** -120).log2().abs())
    assert bool(((one.double() - two).abs() <= 0.5 * limit * two + 2.0 ** -120).all())


def _dense_stats(q, k, want_ml):
    """lvar_dense_attn_fwd without an output: LSE2 alone, or M and L."""
    from lvar_amd import _lib, sparse_attn_ops as ops
    B, H, Lq, d = q.shape
    out = torch.empty(2, B, H, Lq, device="cuda")
    none = _lib.LvarTensor(None, 0, 0, 0)
    a, b, c = (out[0].data_ptr(), out[1].data_ptr(), None) if want_ml else (None, None, out[0].data_ptr())
    assert _lib.load().lvar_dense_attn_fwd(ops._view(q), ops._view(k), none, none, a, b, c, B, H, k.shape[1], Lq, k.shape[2], d, d ** -0.5, ops._stream(q)) == 0
    return out[0] + torch.log2(out[1]) if want_ml else out[0]


# at most one 128-row workgroup of the attention kernel per compute unit, and more
@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,d", [(1, 2, 1, 128, 4121, 128), (2, 16, 16, 1024, 700, 64), (2, 16, 16, 1025, 700, 64), (1, 260, 130, 77, 300, 128),
                                             (1, 2, 2, 300, 127, 256), (3, 100, 100, 100, 65, 256)])
def test_statistic_alone_from_either_kernel(B, H, Hkv, Lq, Lk, d):
    g = torch.Generator(device="cuda").manual_seed(Lq)
    q = torch.randn(B, H, Lq, d, generator=g, device="cuda").to(torch.bfloat16)
    k = torch.randn(B, Hkv, Lk, d, generator=g, device="cuda").to(torch.bfloat16)
    got = _dense_stats(q, k, False)
    assert (got.double().cpu() - _ref(q, k, d ** -0.5)).abs().max() <= 2.0 ** -13      # 2^-17 of the largest statistic (< 2^4), see _check
    assert torch.allclose(got, _dense_stats(q, k, True), rtol=0, atol=2.0 ** -18)       # the sum's logarithm and one addition, rounded


def test_statistic_alone_of_few_rows_costs_no_more_than_with_the_maximum():
    """256 rows per workgroup and uncut keys take a third longer where the rows leave compute units idle."""
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k = (torch.randn(1, 2, L, 256, generator=g, device="cuda").to(torch.bfloat16) for L in (128, 8192))

    def time_of(want_ml):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                _dense_stats(q, k, want_ml)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return sorted(times[1:])[2]
    with_max = time_of(True)
    assert time_of(False) < 1.15 * with_max


# ---- video lists: calls whose rows are too few for the sweep ----

# both sides of the rule: workgroups of 256 rows against an eighth of the compute units (a quarter at head_dim 256), 32 stages of 64 keys
@pytest.mark.parametrize("H,frames,height,width,d", [(1, 3, 40, 16, 128), (1, 2, 32, 32, 128), (3, 3, 48, 16, 64), (16, 2, 32, 32, 128), (17, 2, 32, 32, 64),
                                                     (32, 2, 32, 32, 256), (33, 2, 32, 32, 256)])
def test_video_lists_of_few_and_many_rows(H, frames, height, width, d):
    from lvar_amd import mask_build as mb, sparse_attn_ops as ops
    L = frames * height * width
    g = torch.Generator(device="cuda").manual_seed(H + L)
    q, k = ((torch.randn(1, H, L, d, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for _ in range(2))
    num, idx, score = mb.video_window_topk_block_lists(q, k, None, 0.4, frames, height, width)
    hs = slice(H - 1, H)
    ref = _scores_ref(q[:, hs, ::4], k[:, hs], d ** -0.5, 32, 128)
    assert score.shape[1] == H and torch.allclose(score[:, hs].double().cpu(), ref, rtol=2e-4, atol=float(ref.max()) * 1e-6)
    nK = -(-L // 128)
    base = mb.video_window_base_mask(frames, height, width, 128, device="cuda")
    lists = ops.block_topk_lists(ops._colsum_block_scores(q[:, :, ::4], k, None, 32, 128), int(round(0.4 * nK)), base)
    # (the statistic of the two forms may differ in the order of its sum: 2^-20 of a score, a tie now and then)
    same = (lists[0] == num) & (lists[1] == idx).all(-1)
    assert bool((lists[0] == num).all()) and float((~same).float().mean()) <= 0.01


def test_video_lists_of_few_rows_cost_no_more_than_two_passes():
    """Uncut keys and 256 rows per workgroup: 8 workgroups took a quarter longer than statistics of 128 rows and column sums."""
    from lvar_amd import mask_build as mb, sparse_attn_ops as ops
    g = torch.Generator(device="cuda").manual_seed(4)
    q, k = ((torch.randn(1, 1, 8192, 256, generator=g, device="cuda") * 0.5).to(torch.bfloat16) for _ in range(2))

    def two_passes():
        base = mb.video_window_base_mask(2, 64, 64, 128, device="cuda")
        rows = q[:, :, ::4]
        lse2 = ops._dense_launch(rows, k, k, None, want_o=False, want_ml=False, want_lse2=True)[3]
        sums = ops._colsum_given_lse(rows, k, lse2, None, 32, want_block_sums=True, want_columns=False)[1]
        return ops.block_topk_lists(sums.unflatten(-1, (-1, 2)).sum(-1), 6, base)
    times = [[], []]
    for _ in range(7):
        for t, call in zip(times, (two_passes, lambda: mb.video_window_topk_block_lists(q, k, None, 0.1, 2, 64, 64))):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                call()
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
    assert min(times[1]) < 1.12 * min(times[0])
