"""Performance cases: the work that a user of this library has it do, through its public entry points.

The library serves sparse attention inside a diffusion transformer.  A layer's attention is called on
every denoising step: on a few steps it is computed densely while the mask cache is refreshed, on all
others it runs from the cached lists; some callers derive a mask on every step (threshold or top-k),
some keep it as bits, some call the operators with lists of their own, and dense attention is what
layers without a mask use.  Each of these is a kind of case:

  dense          ``full_attn_ex`` / ``baseline_attn``: layers without a mask, text and image towers
  tokens         ``sp_attn`` with the caller's own key lists (64- or 128-row q-blocks)
  blocks         ``sp_attn_block`` with the caller's own lists of 64-key blocks, log-sum-exp wanted
  refresh        ``cached_attn_cuda`` on a step that refreshes the key lists
  step           ``cached_attn_cuda`` on a step that uses them
  block_refresh  ``blockcached_attn_cuda`` on a refresh step
  masked         ``attn_computed_with_sparse_mask_cuda``: threshold mask and attention on every step
  topk           ``attn_topkmask_cuda``: top-k key lists and attention on every step
  bit_step       ``bitmaskcached_attn_cuda`` on a step that decodes its bit-packed mask

Shapes are those of the library's configurations, tests and benchmark: 32760 and 75600 tokens are
video latents (ragged against the 128-row q-block), 1024 to 16384 the other configurations.
"""
import math

import torch

from fgattn_tk_cuda_amd.spattn import mask_utils
from fgattn_tk_cuda_amd.spattn import sparseattn_functionals as fn

ops = torch.ops.cuda_attn

# Shares of what a threshold of x mean weights (x / S) keeps on the inputs of _qkv: keys per 128-row q-block.
# 1e-3, the helpers' default, is 32 mean weights at 32760 tokens and keeps about 8 % of the keys.
KEPT_KEYS = {16: 0.16, 32: 0.085, 64: 0.039}


def listed():
    return [
        # The smallest call: one short sequence, key lists for a quarter of the 64-key blocks (latency).
        dict(name="tokens_1k", kind="tokens", B=1, H=4, S=1024, D=64, qblk=64, keep=0.25),
        # A padded batch of short sequences, e.g. text or one image: log-sum-exp, keys behind the padding ignored.
        dict(name="dense_1000_padded", kind="dense", B=2, H=12, S=1000, D=128, pad=40, lse=True),
        # An ordinary dense layer.
        dict(name="dense_4k", kind="dense", B=4, H=16, S=4096, D=64, pad=0, lse=False),
        # Block lists with 10 % of the blocks, even lengths: the benchmark's headline workload.
        dict(name="blocks_16k", kind="blocks", B=2, H=32, S=16384, D=128, qblk=64, keep=0.10, zipf=False),
        # Block lists of very uneven length on a long sequence.
        dict(name="blocks_64k_zipf", kind="blocks", B=1, H=8, S=65536, D=128, qblk=128, keep=0.28, zipf=True),
        # Mask cache refresh of one layer, d = 64, ragged sequence.
        dict(name="refresh_32k_d64", kind="refresh", B=1, H=24, S=32760, D=64, x=32),
        # The step that runs most often: one layer from its cached key lists.
        dict(name="step_32k", kind="step", B=1, H=12, S=32760, D=128, x=32),
        # Block-list cache refresh on a shorter, ragged clip.
        dict(name="block_refresh_9000", kind="block_refresh", B=1, H=12, S=9000, D=128, qblk=64, x=32),
        # A threshold mask of its own on every step, short ragged clip.
        dict(name="masked_6000", kind="masked", B=1, H=16, S=6000, D=128, x=32),
        # A top-k mask of its own on every step.
        dict(name="topk_32k_d64", kind="topk", B=1, H=24, S=32760, D=64, keep=0.08),
        # Step of a layer whose mask is kept as bits to save memory (40 heads).
        dict(name="bit_step_32k", kind="bit_step", B=1, H=40, S=32760, D=128, x=32),
        # The largest: cache refresh of one layer at the longest sequence and the most heads.
        dict(name="refresh_75600", kind="refresh", B=1, H=40, S=75600, D=128, x=64),
    ]


def draw(rng):
    """A case of the same kinds; sizes spread over the logarithm of their range."""
    kind = rng.choice(["dense", "tokens", "blocks", "refresh", "step", "block_refresh", "masked", "topk", "bit_step"])
    largest = {"tokens": 16384, "dense": 32768, "blocks": 65536}.get(kind, 75600)
    S = int(round(math.exp(rng.uniform(math.log(256), math.log(largest)))))
    if rng.random() < 0.25:
        S = max(256, S // 128 * 128)
    case = dict(kind=kind, B=rng.choice([1, 2, 4]) if S <= 8192 else 1, H=rng.choice([4, 8, 12, 16, 24, 32, 40]), S=S,
                D=rng.choice([64, 128]))
    if kind == "dense":
        case.update(pad=rng.choice([0, rng.randrange(1, S // 8)]), lse=rng.random() < 0.5)
    elif kind in ("tokens", "blocks"):
        case.update(qblk=rng.choice([64, 128]), keep=round(math.exp(rng.uniform(math.log(0.04), math.log(0.4))), 3))
        if kind == "blocks":
            case.update(zipf=rng.random() < 0.5)
    elif kind == "topk":
        case.update(keep=round(rng.uniform(0.03, 0.2), 3))
    else:
        case.update(x=rng.choice([16, 32, 64]))
        if kind == "block_refresh":
            case.update(qblk=rng.choice([64, 128]))
    return case


def _qkv(case, seed):
    """bf16 q, k, v.  Neighbouring tokens resemble each other, as video latents do: every 64 tokens of q and
    k share most (0.8) of their variance, and the logits have a standard deviation of 2.5."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]

    def tokens():
        return torch.randn((B, H, S, D), generator=g, device="cuda", dtype=torch.bfloat16)

    def alike():
        shared = torch.randn((B, H, (S + 63) // 64, D), generator=g, device="cuda", dtype=torch.bfloat16)
        x = tokens().mul_(math.sqrt(0.2 * 2.5))
        return x.add_(shared.repeat_interleave(64, dim=2)[:, :, :S], alpha=math.sqrt(0.8 * 2.5))

    return alike(), alike(), tokens(), g


def _block_lists(case, g):
    """Ascending lists of 64-key blocks per q-block that hold the diagonal block; the others are uniform.
    Equal counts, or counts that follow Zipf's law (exponent 1.2, clipped) with the asked mean."""
    B, H, S, qblk = case["B"], case["H"], case["S"], case["qblk"]
    nq, nk = (S + qblk - 1) // qblk, (S + 63) // 64
    rank = torch.rand((B, H, nq, nk), generator=g, device="cuda")
    rank.scatter_(3, ((torch.arange(nq, device="cuda") * qblk) // 64).clamp(max=nk - 1).view(1, 1, nq, 1).expand(B, H, nq, 1), -1.0)
    mean = max(1, round(case["keep"] * nk))
    if case.get("zipf"):
        # inverse of the tail P(count >= c) = c ** -0.2, clipped at the number of blocks; the mean of the
        # clipped law is 0.28 of the blocks at 1024 of them, shorter lists are scaled to the asked mean
        u = torch.rand((B, H, nq), generator=g, device="cuda").clamp(min=1e-7)
        counts = (u ** -5.0).clamp(max=float(nk))
        counts = (counts * (mean / counts.mean().clamp(min=1.0)).clamp(max=1.0)).clamp(min=1.0).to(torch.int32)
    else:
        counts = torch.full((B, H, nq), mean, dtype=torch.int32, device="cuda")
    width = int(counts.max())
    place = rank.argsort(dim=3).argsort(dim=3)              # place of every block in its row's draw
    keep = place < counts.unsqueeze(3)
    ids = torch.arange(nk, device="cuda", dtype=torch.int32).expand(B, H, nq, nk)
    lists = torch.where(keep, ids, torch.full_like(ids, nk)).sort(dim=3).values[..., :width]
    return torch.where(lists == nk, torch.full_like(lists, -1), lists).contiguous(), counts.contiguous()


def prepare(case, seed):
    q, k, v, g = _qkv(case, seed)
    kind, S = case["kind"], case["S"]
    st = dict(kind=kind, q=q, k=k, v=v)
    if kind == "dense":
        st.update(o=torch.empty_like(q), kv_len=S - case["pad"], lse=None)
        if case["lse"]:
            st["lse"] = torch.empty(q.shape[:3], dtype=torch.float32, device="cuda")
    elif kind in ("tokens", "blocks"):
        idx, cnt = _block_lists(case, g)
        st.update(o=torch.empty_like(q), qblk=case["qblk"])
        if kind == "blocks":
            st.update(idx=idx, cnt=cnt, lse=torch.empty(q.shape[:3], dtype=torch.float32, device="cuda"),
                      order=mask_utils.qblock_order_cuda(cnt))
        else:
            # the same lists as key ids, in rows of a multiple of 128 entries
            B, H, nq, w = idx.shape
            keys = (idx.unsqueeze(4) * 64 + torch.arange(64, device="cuda", dtype=torch.int32)).view(B, H, nq, w * 64)
            live = (idx >= 0).repeat_interleave(64, dim=3) & (keys < S)
            stride = (w * 64 + 127) // 128 * 128
            lists = torch.full((B, H, nq, stride), stride, dtype=torch.int32, device="cuda")
            lists[..., : w * 64] = torch.where(live, keys, torch.full_like(keys, stride))
            st.update(idx=lists, cnt=live.sum(dim=3).to(torch.int32))
    elif kind == "topk":
        st.update(select_k=max(1, round(case["keep"] * S)))
    else:
        st.update(thresh=case["x"] / S)
        if kind == "block_refresh":
            st.update(cache=mask_utils.BlockListCache([0]), qblk=case["qblk"])
        elif kind == "bit_step":
            st.update(cache=mask_utils.CompressedBitMaskCache([0]))
            fn.bitmaskcached_attn_cuda(q, k, v, 0, 0, thresh=st["thresh"], blocksz=128, mask_cache=st["cache"])
        elif kind in ("refresh", "step"):
            st.update(cache=mask_utils.NaiveMaskCache([0]))
            if kind == "step":
                fn.cached_attn_cuda(q, k, v, 0, 0, thresh=st["thresh"], blocksz=128, mask_cache=st["cache"])
    return st


def run(st):
    kind, q, k, v = st["kind"], st["q"], st["k"], st["v"]
    if kind == "dense":
        if st["lse"] is None and st["kv_len"] == q.shape[2]:
            return fn.baseline_attn(q, k, v)
        ops.full_attn_ex(st["o"], st["lse"], q, k, v, 0.0, st["kv_len"])
        return st["o"], st["lse"]
    if kind == "tokens":
        ops.sp_attn(st["o"], q, k, v, st["idx"], st["cnt"])
        return st["o"]
    if kind == "blocks":
        ops.sp_attn_block(st["o"], st["lse"], q, k, v, st["idx"], st["cnt"], st["order"], st["qblk"], 0.0, 0)
        return st["o"], st["lse"]
    if kind == "refresh":
        out = fn.cached_attn_cuda(q, k, v, 0, 0, thresh=st["thresh"], blocksz=128, mask_cache=st["cache"])
        return (out,) + tuple(st["cache"].get_mask_from_cache(0))
    if kind == "step":
        return fn.cached_attn_cuda(q, k, v, 0, 1, thresh=st["thresh"], blocksz=128, mask_cache=st["cache"])
    if kind == "block_refresh":
        out = fn.blockcached_attn_cuda(q, k, v, 0, 0, thresh=st["thresh"], blocksz=128, qblk=st["qblk"], mask_cache=st["cache"])
        return (out,) + tuple(st["cache"].get_mask_from_cache(0))
    if kind == "masked":
        return fn.attn_computed_with_sparse_mask_cuda(q, k, v, thresh=st["thresh"], blocksz=128)
    if kind == "topk":
        return fn.attn_topkmask_cuda(q, k, v, select_k=st["select_k"], blocksz=128)
    return fn.bitmaskcached_attn_cuda(q, k, v, 0, 1, thresh=st["thresh"], blocksz=128, mask_cache=st["cache"])


def work(case):
    """Multiply-adds count two.  A kept (row, key) pair is 4 D operations (scores and output); a refresh is
    dense attention, whose scores also decide the mask."""
    kind, B, H, S, D = case["kind"], case["B"], case["H"], case["S"], case["D"]
    pairs = float(B) * H * S * S
    qkvo = 2.0 * 4 * B * H * S * D
    rows = B * H * ((S + 127) // 128)
    padded = (S + 127) // 128 * 128
    if kind == "dense":
        return {"flops": 4 * D * pairs * (S - case["pad"]) / S, "bytes": qkvo + (4 * B * H * S if case["lse"] else 0)}
    if kind in ("tokens", "blocks"):
        nq, nk = (S + case["qblk"] - 1) // case["qblk"], (S + 63) // 64
        kept = max(1, round(case["keep"] * nk)) / nk
        entries = kept * B * H * nq * (nk if kind == "blocks" else S)
        return {"flops": 4 * D * pairs * kept, "bytes": qkvo + 4 * entries + (4 * B * H * S if kind == "blocks" else 0)}
    if kind == "topk":
        # the score of every key against every q-block's mean comes on top of the attention
        return {"flops": 4 * D * pairs * case["keep"] + 2.0 * D * rows * S, "bytes": qkvo}
    kept = KEPT_KEYS[case["x"]]
    if kind == "refresh":
        return {"flops": 4 * D * pairs, "bytes": qkvo + 4 * rows * padded}
    if kind == "block_refresh":
        return {"flops": 4 * D * pairs, "bytes": qkvo + 4 * rows * (128 // case["qblk"]) * (padded // 64)}
    if kind == "masked":
        return {"flops": 2 * D * pairs + 4 * D * pairs * kept, "bytes": qkvo}
    if kind == "step":
        return {"flops": 4 * D * pairs * kept, "bytes": qkvo + 4 * kept * rows * S}
    return {"flops": 4 * D * pairs * kept, "bytes": qkvo + rows * padded / 8}


def tolerance(case):
    """Outputs are bf16, and P is rounded to bf16 ahead of its product with V.  A key whose weight lies at
    the threshold within the rounding of the fp32 statistics may fall on either side of it, and shifts the
    list entries behind it by one."""
    tol = {"rel": 1e-2}
    if case["kind"] in ("refresh", "block_refresh"):
        tol["differ"] = 5e-3
    return tol
