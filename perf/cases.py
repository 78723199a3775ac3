"""The work that users of this package have it do, as cases that can be timed.

Every case goes through the public entry points of ``lvar_amd`` the way the callers of a next-scale-prediction model do:
dense attention at the scales that stay dense, the two steps of the column-sparse layers (``SparseDiffAttn``), the
sink + window block-sparse layers (``SparseFlexAttn``), block-sparse attention over lists that come from a score, the
list build itself, the key selection of a ScaleKV-style cache, and long video sequences.  Sizes are those of the
Infinity-2B schedule (13 scales up to 64 x 64), of VAR-d16 (head_dim 64) and of the video grid of the benchmark; drawn
cases spread over the same ranges with odd grids, batch sizes, head counts and head dimensions among them.
Inputs are synthetic: q, k, v i.i.d. N(0, 1) * 0.5 in bf16, as in ``bench.py``.
"""
import math

import torch

from lvar_amd import mask_build as mb
from lvar_amd import sparse_attn_config as cfg
from lvar_amd import sparse_attn_ops as ops
from lvar_amd.sparse_diff_attn import SparseDiffAttn
from lvar_amd.sparse_flex_attn import SparseFlexAttn

SCALES = mb.INFINITY_SCALES
WIN_SIZE = cfg.BASE_CONFIG["attn"]["win_size"]


def schedule(n, last):
    """The first ``n`` scales of the Infinity schedule and then a grid of side ``last``."""
    return SCALES[:n] + (last,)


def listed():
    return [
        # the smallest calls of an image: scales 1 .. 6 take one or two 64-key tiles, so latency and launches count
        dict(name="dense_scale_4", kind="dense", B=2, H=16, Hkv=16, d=128, Lq=16, Lk=21, layout="bhld"),
        dict(name="dense_scale_12", kind="dense", B=2, H=16, Hkv=16, d=128, Lq=144, Lk=265, layout="bhld"),
        # the middle scales, which do not fill the chip with 128-row query tiles
        dict(name="dense_scale_24", kind="dense", B=2, H=16, Hkv=16, d=128, Lq=576, Lk=1497, layout="bhld"),
        # VAR-d16, last scale, a batch of eight; q, k, v as views of a fused projection ([B, L, H, d] storage)
        dict(name="dense_var_d16", kind="dense", B=8, H=16, Hkv=16, d=64, Lq=256, Lk=680, layout="blhd"),
        # the last scale of an all-dense image
        dict(name="dense_scale_64", kind="dense", B=2, H=16, Hkv=16, d=128, Lq=4096, Lk=10521, layout="bhld"),
        # column-sparse layer, decision scale: dense attention + column sums + top-k key lists + output cache
        dict(name="cs4a_full_40", kind="full_step", B=2, H=16, d=128, n=10, S=40, top_keys=0.2),
        # column-sparse layer, last scale: list remap + gathered attention with the upsampled output cache
        dict(name="cs4a_sparse_64", kind="sparse_step", B=2, H=16, d=128, n=12, S=64, steps=2, top_keys=0.2),
        # sink + local-window layer at the scale before the last
        dict(name="csla_48", kind="csla", B=2, H=16, d=128, n=11, S=48, sink=5, block=128),
        # block-sparse attention at the last scale: sink + window + best-scoring blocks, 25 % of all
        dict(name="block_sparse_25", kind="block_sparse", B=2, H=16, d=128, n=12, S=64, density=0.25, mask="scored", bq=128, bk=64),
        # column sums in the self-contained two-pass form and the block lists that follow from them
        dict(name="block_lists_48", kind="block_lists", B=2, H=16, d=128, n=11, S=48, density=0.25, lse=False),
        # cache selection of one layer after the last scale: scores of all keys against 256 window queries
        dict(name="scalekv_64", kind="scalekv", B=2, H=16, d=128, Lq=4096, Lk=10521, W=256, capacity=2048, pool="avgpool", ksize=5),
        # long video: 8 frames of 64 x 64 tokens, lists from a 3-D window and column sums, 10 % of the 128 x 128 blocks
        dict(name="video_8x64x64", kind="video", B=1, H=24, d=128, frames=8, height=64, width=64, density=0.10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense", "dense", "dense", "full_step", "sparse_step", "csla", "block_sparse", "block_lists", "scalekv", "video"])
    B, H = rng.randint(1, 3), rng.choice([4, 8, 12, 16, 20, 24])
    d = rng.choice([64, 128, 128, 128])
    if kind == "dense":
        side = _log(rng, 1, 64)
        Lq = max(1, side * side - rng.choice([0, 0, 1, side // 2]))      # whole grids and ragged lengths
        Lk = Lq + _log(rng, 1, 2 * Lq + 1)                                # the keys of the scales before
        return dict(kind=kind, B=B, H=H, Hkv=rng.choice([H, H, H, H // 4]), d=rng.choice([64, 128, 128, 128, 256]), Lq=Lq, Lk=Lk,
                    layout=rng.choice(["bhld", "bhld", "blhd"]))
    if kind == "full_step":
        S = rng.randint(20, 44)
        return dict(kind=kind, B=B, H=H, d=d, n=sum(s < S for s in SCALES), S=S, top_keys=rng.choice([0.05, 0.1, 0.2, 0.3]))
    if kind == "sparse_step":
        S = rng.randint(30, 64)
        return dict(kind=kind, B=B, H=H, d=d, n=sum(s < S for s in SCALES), S=S, steps=rng.choice([1, 2]), top_keys=rng.choice([0.05, 0.1, 0.2, 0.3]))
    if kind == "csla":
        S = rng.randint(24, 64)
        return dict(kind=kind, B=B, H=H, d=d, n=sum(s < S for s in SCALES), S=S, sink=rng.choice([3, 5, 7]), block=rng.choice([64, 128, 128, 256]))
    if kind == "block_sparse":
        S = rng.randint(20, 64)
        bq, bk = rng.choice([(128, 64), (128, 64), (128, 128), (64, 64)])
        return dict(kind=kind, B=B, H=H, d=d, n=sum(s < S for s in SCALES), S=S, density=round(math.exp(rng.uniform(math.log(0.05), math.log(0.5))), 3),
                    mask=rng.choice(["scored", "bernoulli"]), bq=bq, bk=bk)
    if kind == "block_lists":
        S = rng.randint(20, 64)
        return dict(kind=kind, B=B, H=H, d=d, n=sum(s < S for s in SCALES), S=S, density=rng.choice([0.1, 0.25, 0.5]), lse=rng.choice([False, True]))
    if kind == "scalekv":
        S = rng.randint(12, 64)
        Lq, Lk = S * S, S * S + sum(s * s for s in SCALES if s < S)
        return dict(kind=kind, B=B, H=H, d=d, Lq=Lq, Lk=Lk, W=rng.randint(16, min(256, Lq)), capacity=rng.randint(Lk // 8, Lk // 2),
                    pool=rng.choice(["avgpool", "maxpool"]), ksize=rng.choice([3, 5, 7]))
    height, width = rng.choice([(32, 32), (32, 48), (48, 48), (40, 64), (64, 64)])
    frames = rng.randint(2, 8)
    # (the 3-D window alone keeps nine blocks of a row, a larger share of a shorter sequence)
    return dict(kind="video", B=1, H=rng.choice([8, 12, 16, 24]), d=d, frames=frames, height=height, width=width,
                density=rng.choice([0.08, 0.1]) if frames * height * width >= 16384 else 0.25)


def _grid_lengths(case):
    scales = schedule(case["n"], case["S"])
    return scales, case["S"] ** 2, sum(s * s for s in scales)


def _normal(shape, gen, layout="bhld"):
    """N(0, 1) * 0.5 in bf16, logically [B, H, L, d]; "blhd": a view of [B, L, H, d] storage."""
    B, H, L, d = shape
    if layout == "blhd":
        return (torch.randn((B, L, H, d), generator=gen, device="cuda") * 0.5).to(torch.bfloat16).permute(0, 2, 1, 3)
    return (torch.randn(shape, generator=gen, device="cuda") * 0.5).to(torch.bfloat16)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    st = {"case": dict(case)}
    if kind == "video":
        L = case["frames"] * case["height"] * case["width"]
        st["q"], st["k"], st["v"] = (_normal((case["B"], case["H"], L, case["d"]), gen) for _ in range(3))
        return st
    if kind == "dense":
        B, H, d, lay = case["B"], case["H"], case["d"], case["layout"]
        st["q"] = _normal((B, H, case["Lq"], d), gen, lay)
        st["k"], st["v"] = (_normal((B, case["Hkv"], case["Lk"], d), gen, lay) for _ in range(2))
        return st
    B, H, d = case["B"], case["H"], case["d"]
    if kind == "scalekv":
        st["q"], st["k"] = _normal((B, H, case["Lq"], d), gen), _normal((B, H, case["Lk"], d), gen)
        # distinct keys of the newest scale
        place = torch.rand((B, H, case["Lq"]), generator=gen, device="cuda").topk(case["W"], dim=-1).indices
        st["window"] = (place + (case["Lk"] - case["Lq"])).sort(dim=-1).values
        return st
    scales, Lq, Lk = _grid_lengths(case)
    if kind == "full_step":
        cfg.GLOBAL_CONFIG["attn"]["top_keys"] = case["top_keys"]
        st["layer"] = SparseDiffAttn(scales=scales, spsd_scale=len(scales) - 1)
    elif kind == "sparse_step":
        cfg.GLOBAL_CONFIG["attn"]["top_keys"] = case["top_keys"]
        first = len(scales) - 1 - case["steps"]                 # the decision scale: `steps` sparse scales follow it
        layer = SparseDiffAttn(scales=scales, spsd_scale=first)
        for si in range(first, len(scales) - 1):                # what the layer holds when the last scale begins
            n_k = sum(s * s for s in scales[:si + 1])
            q, k, v = _normal((B, H, scales[si] ** 2, d), gen), _normal((B, H, n_k, d), gen), _normal((B, H, n_k, d), gen)
            layer(q, k, v, None, do_full_step=si == first, scale_ind=si)
        st["layer"] = layer
    elif kind == "csla":
        st["layer"] = SparseFlexAttn([(s, s) for s in scales], WIN_SIZE, len(scales) - 1, case["sink"], case["block"], H, device="cuda")
    st["q"], st["k"], st["v"] = (_normal((B, H, L, d), gen) for L in (Lq, Lk, Lk))
    if kind == "block_sparse":
        bq, bk = case["bq"], case["bk"]
        nQ, nK = -(-Lq // bq), -(-Lk // bk)
        if case["mask"] == "bernoulli":                         # lists of uneven length, at least one block in each
            mask = torch.rand((B, H, nQ, nK), generator=gen, device="cuda") < case["density"]
            mask.scatter_(-1, torch.randint(0, nK, (B, H, nQ, 1), generator=gen, device="cuda"), True)
            st["num"], st["idx"] = ops.mask_to_lists(mask)
        else:
            score = mb.key_block_sums(ops.colsum(st["q"], st["k"], q_group_size=bq), bk)
            base = mb.sink_window_base_mask(bq, bk, 5, 1, scales, device="cuda")
            st["num"], st["idx"] = ops.block_topk_lists(score, max(1, round(case["density"] * nK)), base)
    elif kind == "block_lists":
        st["base"] = mb.sink_window_base_mask(128, 64, 5, 1, scales, device="cuda")
        st["lse"] = ops.dense_attn(st["q"], st["k"], st["v"])[1] if case["lse"] else None
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dense":
        o, (M, L) = ops.dense_attn(state["q"], state["k"], state["v"])
        return o, M, L
    if kind == "full_step":
        layer = state["layer"]
        o = layer(state["q"], state["k"], state["v"], None, do_full_step=True, scale_ind=len(layer.scales) - 1)
        # behind the count the list rows are left as allocated
        return o, layer.out_cache, layer.indices[..., :layer.count_host], layer.counts
    if kind == "sparse_step":
        layer = state["layer"]
        return layer(state["q"], state["k"], state["v"], None, scale_ind=len(layer.scales) - 1)
    if kind == "csla":
        return state["layer"](state["q"], state["k"], state["v"], None)
    if kind == "block_sparse":
        o, (M, L) = ops.block_sparse_attn(state["q"], state["k"], state["v"], state["num"], state["idx"], case["bq"], case["bk"])
        return o, M, L
    if kind == "block_lists":
        cs, bs = ops.colsum(state["q"], state["k"], q_group_size=128, lse=state["lse"], return_block_sums=True)
        num, idx = ops.block_topk_lists(bs, max(1, round(case["density"] * bs.shape[-1])), state["base"])
        return cs, bs, num, idx
    if kind == "scalekv":
        return ops.scalekv_keep_indices(state["q"], state["k"], state["window"], case["capacity"], case["ksize"], case["pool"])
    num, idx, score = mb.video_window_topk_block_lists(state["q"], state["k"], None, case["density"], case["frames"], case["height"], case["width"])
    o, (M, L) = ops.block_sparse_attn(state["q"], state["k"], state["v"], num, idx, 128, 128)
    return o, M, L, num, idx, score


def work(case):
    """Bytes: every input read once, every output written once.  Operations: two per multiply-add of the products; the
    column sums need Q K^T for the row statistics and again for the sums where the statistics are not handed over."""
    kind, H, d, B = case["kind"], case["H"], case["d"], case["B"]
    if kind == "video":
        L = case["frames"] * case["height"] * case["width"]
        blocks = B * H * (L // 128) ** 2
        return {"bytes": 2.0 * B * H * d * 4 * L + 8.0 * B * H * L + 8.0 * blocks,
                "flops": 4.0 * B * H * d * L * L * (0.25 + case["density"])}
    if kind == "dense":
        Lq, Lk, Hkv = case["Lq"], case["Lk"], case["Hkv"]
        return {"bytes": 2.0 * B * d * (2 * H * Lq + 2 * Hkv * Lk) + 8.0 * B * H * Lq, "flops": 4.0 * B * H * Lq * Lk * d}
    if kind == "scalekv":
        Lk, W = case["Lk"], case["W"]
        return {"bytes": B * H * (2.0 * d * (Lk + W) + 8.0 * W + 8.0 * case["capacity"]), "flops": 2.0 * B * H * d * (Lk + W)}
    scales, Lq, Lk = _grid_lengths(case)
    qo, kv, pairs = 4.0 * B * H * Lq * d, 4.0 * B * H * Lk * d, float(B * H * d) * Lq * Lk
    groups = -(-Lq // 192)
    if kind == "full_step":
        cnt = mb.indices_count(case["top_keys"], Lk, 64)
        return {"bytes": qo * 1.5 + kv + 4.0 * B * H * groups * (cnt + 1), "flops": 6.0 * pairs + 4.0 * B * H * d * Lq * cnt}
    if kind == "sparse_step":
        first = len(scales) - 1 - case["steps"]
        cnt = mb.indices_count(case["top_keys"], sum(s * s for s in scales[:first + 1]), 64)
        ws = cfg.BASE_CONFIG["attn"]["cs4a_ws"][-case["steps"]:]
        for j in range(case["steps"]):                         # every sparse scale appends its local run
            cnt += mb.local_group_runs(first + 1 + j, ws[j], scales=scales)[1]
        cnt = min(cnt, Lk)
        return {"bytes": qo + kv + 2.0 * B * H * d * scales[first] ** 2 + 4.0 * B * H * groups * cnt, "flops": 4.0 * B * H * d * Lq * cnt}
    if kind == "csla":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        mask = mb.flex_block_mask(len(scales) - 1, WIN_SIZE, case["sink"], case["block"], scales=[(s, s) for s in scales], device=dev)
        touched = float(mask.any(0).float().mean())
        return {"bytes": qo + kv * touched + 4.0 * mask.numel(), "flops": 4.0 * pairs * float(mask.float().mean())}
    if kind == "block_sparse":
        blocks = B * H * (-(-Lq // case["bq"])) * (-(-Lk // case["bk"])) * case["density"]
        return {"bytes": qo + kv + 8.0 * B * H * Lq + 4.0 * blocks, "flops": 4.0 * pairs * case["density"]}
    g = -(-Lq // 128)
    blocks = B * H * g * (-(-Lk // 64))
    return {"bytes": qo / 2 + kv / 2 + 4.0 * B * H * g * Lk + 8.0 * blocks + (8.0 * B * H * Lq if case["lse"] else 0.0),
            "flops": (2.0 if case["lse"] else 4.0) * pairs}


def tolerance(case):
    """bf16 outputs of products in bf16 with 32-bit sums; column sums are 32-bit sums of exponentials.  Lists may differ
    where two scores tie within the rounding of those sums."""
    if case["kind"] == "scalekv":
        return {"rel": 0.0, "differ": 0.01}
    if case["kind"] == "block_lists":
        return {"rel": 1e-4, "max": 1e-3, "differ": 0.01}
    return {"rel": 1e-2, "differ": 0.01}
