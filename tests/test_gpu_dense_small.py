"""GPU: dense attention and its statistics on both sides of the rule that gives small launches 64-row q-blocks, at the
edges of q-blocks and key tiles, against attention in fp32.  The scores of both forms are the same bits, so their row
maxima and block maxima are too."""
import pytest
import torch

from tests.helpers import assert_close_o, assert_close_stat, f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,S,kv_len", [
    (64, 1, 0), (128, 1, 0), (64, 63, 0), (128, 64, 33), (64, 65, 64), (128, 127, 1), (64, 129, 65), (128, 129, 0), (64, 191, 128),
    (128, 200, 129), (64, 400, 0), (128, 385, 321), (64, 832, 767), (64, 832, 768), (64, 1090, 0),
])
def test_small_launches_match_large_ones(dev, D, S, kv_len):
    import fgattn_tk_cuda_amd.spattn.cuda_attn  # noqa: F401

    print("case dense small", D, S, kv_len, flush=True)
    ops = torch.ops.cuda_attn
    per_head = (S + 63) // 64
    few = max(1, 256 // per_head)                        # heads of the largest launch with one 64-row q-block per CU
    many = 768 // per_head + 1                           # heads that take 128-row q-blocks in every form
    mid = max(few, 768 // per_head)                      # the largest launch of three per CU
    g = torch.Generator(device=dev).manual_seed(S + D)
    q, k, v = (torch.randn((1, many, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    kv = kv_len or S
    sp = (S + 127) // 128 * 128

    def call(h):
        a = [t[:, :h].contiguous() for t in (q, k, v)]
        nan = lambda *shape: torch.full(shape, float("nan"), device=dev)
        o, lse, o2 = torch.empty_like(a[0]), nan(1, h, S), torch.empty_like(a[0])
        ops.full_attn_ex(o, lse, *a, 0.0, kv_len)
        m, d, m3, d3 = (nan(1, h, 1, sp) for _ in range(4))
        bm, bm3 = (nan(1, h, sp // 64, sp).to(torch.bfloat16) for _ in range(2))
        ops.fullattn_maxq_denom_blockmax(o2, m, d, bm, *a, 0.0, kv_len)
        ops.maxq_denom_blockmax(m3, d3, bm3, a[0], a[1], 0.0, kv_len)
        n = (kv + 63) // 64
        return dict(o=o, lse=lse, o2=o2, m=m, d=d, m3=m3, d3=d3, bm=bm[:, :, :n], bm3=bm3[:, :, :n])

    large, small, medium = call(many), call(few), call(mid)
    h = min(few, 3)
    qf, kf, vf = (t[:, :h].float().cpu() for t in (q, k, v))
    s = (qf @ kf[:, :, :kv].transpose(2, 3)) * D ** -0.5
    want, want_lse = f32(torch.softmax(s, -1) @ vf[:, :, :kv]), f32(torch.logsumexp(s, -1))
    for r in (large, small, medium):
        assert_close_o(f32(r["o"][:, :h]), want, "o")
        assert_close_o(f32(r["o2"][:, :h]), want, "o with statistics")
        assert_close_stat(f32(r["lse"][:, :h]), want_lse, "lse", atol=1e-4)
        assert torch.equal(r["m"], r["m3"]) and torch.equal(r["bm"][..., :S], r["bm3"][..., :S])
        # max_q is the raw maximum, denom the sum of exp((s - max) / sqrt(D)); rows behind S hold 0 and -inf
        row_max = f32(r["m"][:, :h, 0, :S]) * D ** -0.5
        for d in (r["d"], r["d3"]):
            assert_close_stat(row_max + f32(torch.log(d[:, :h, 0, :S])), want_lse, "statistics", atol=1e-4)
            assert bool((d[..., S:] == float("-inf")).all())
        assert bool((r["m"][..., S:] == 0).all())
        n = r["m"].shape[1]
        assert torch.equal(r["m"], large["m"][:, :n]) and torch.equal(r["bm"][..., :S], large["bm"][:, :n][..., :S])
