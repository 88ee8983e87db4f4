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


@pytest.mark.parametrize("D,S,kv_len", [
    (64, 705, 0), (64, 769, 768), (64, 900, 833), (64, 1472, 1409), (64, 1537, 0), (128, 704, 0), (128, 705, 0), (128, 897, 769),
    (128, 961, 960), (128, 961, 897), (128, 1100, 1025),
])
def test_two_groups_match_one(dev, D, S, kv_len):
    """Launches on both sides of the rules that let two groups of waves share a q-block, by numbers of heads and of key
    tiles (odd numbers leave the second group a tile without keys): outputs and statistics against fp32, row and block
    maxima bit for bit those of the largest launch."""
    import fgattn_tk_cuda_amd.spattn.cuda_attn  # noqa: F401

    print("case dense two groups", D, S, kv_len, flush=True)
    ops = torch.ops.cuda_attn
    n64, n128 = (S + 63) // 64, (S + 127) // 128
    heads = sorted({max(1, 256 // n64), 256 // n64 + 1, 256 // n128, 256 // n128 + 1, 768 // n64, 768 // n64 + 1})
    g = torch.Generator(device=dev).manual_seed(S + D)
    q, k, v = (torch.randn((1, heads[-1], S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    kv, sp = kv_len or S, n128 * 128
    s = (q[:, :2].float() @ k[:, :2, :kv].float().transpose(2, 3).contiguous()) * D ** -0.5
    want, want_lse = f32(torch.softmax(s, -1) @ v[:, :2, :kv].float()), f32(torch.logsumexp(s, -1))
    largest = None
    for h in reversed(heads):
        a = [t[:, :h].contiguous() for t in (q, k, v)]
        nan = lambda *shape: torch.full(shape, float("nan"), device=dev)
        o, o2, lse = torch.full_like(a[0], float("nan")), torch.full_like(a[0], float("nan")), nan(1, h, S)
        m, d, m3, d3 = (nan(1, h, 1, sp) for _ in range(4))
        bm, bm3 = (torch.full((1, h, sp // 64 + 1, sp), 7.0, device=dev, dtype=torch.bfloat16)[:, :, :-1].contiguous() for _ in range(2))
        ops.full_attn_ex(o, lse, *a, 0.0, kv_len)
        ops.fullattn_maxq_denom_blockmax(o2, m, d, bm, *a, 0.0, kv_len)
        ops.maxq_denom_blockmax(m3, d3, bm3, a[0], a[1], 0.0, kv_len)
        for out in (o, o2):
            assert_close_o(f32(out[:, :2]), want[:, :h], "o, %d heads" % h)
        assert_close_stat(f32(lse[:, :2]), want_lse[:, :h], "lse", atol=1e-4)
        tiles = (kv + 63) // 64
        assert torch.equal(m, m3) and torch.equal(bm[..., :S], bm3[..., :S])
        assert bool((bm[:, :, tiles:] == 7).all()) and bool((bm3[:, :, tiles:] == 7).all())   # blocks without a key stay unwritten
        for den in (d, d3):
            got = f32(m[:, :2, 0, :S]) * D ** -0.5 + f32(torch.log(den[:, :2, 0, :S]))
            assert_close_stat(got, want_lse[:, :h], "statistics", atol=1e-4)
            assert bool((den[..., S:] == float("-inf")).all())
        if largest is None:
            largest = m, bm
        assert torch.equal(m, largest[0][:, :h]) and torch.equal(bm[..., :S], largest[1][:, :h, :, :S])


@pytest.mark.parametrize("S,kv_len,heads,dense,stats", [
    # 9 q-blocks of 256 rows per head, the last with one row, over rows behind Sp: 450 of them, 360
    (2049, 0, (50, 40), (256, 128), (256, 128)),
    (2176, 2060, (50, 40), (256, 128), (256, 128)),            # key tiles behind the kv length, rows up to a multiple of 128
    (2304, 2304, (57, 60), (128, 128), (128, 128)),            # 513, 540: last round of one, of 28
    (2304, 0, (72, 57), (256, 128), (128, 128)),               # 648: a third round, more than half full
    (2048, 0, (64, 66), (256, 128), (256, 128)),               # 512: rounds that are full, 32 tiles
    (2303, 1985, (57, 56, 57), (128, 256, 128), (128, 256, 128)),   # 32 tiles
    (2100, 1984, (57, 56), (128, 128), (128, 128)),            # 31 tiles
])
def test_256_row_qblocks_give_the_same_bits(dev, S, kv_len, heads, dense, stats):
    """d = 128, launches on both sides of the rule for 256-row q-blocks (dense, stats: rows per q-block of the calls without
    and with statistics): outputs, statistics and block maxima of the heads they share are the same bits, and right."""
    import fgattn_tk_cuda_amd.spattn.cuda_attn  # noqa: F401
    from fgattn_tk_cuda_amd import capi

    print("case dense 256 rows", S, kv_len, heads, flush=True)
    for st, rows in ((0, dense), (1, stats)):
        assert tuple(capi.load().spattn_dense_form(128, 1, st, h, S, kv_len, 0) for h in heads) == tuple(10 * r + 1 for r in rows)
    ops = torch.ops.cuda_attn
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn((1, max(heads), S, 128), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    kv, sp = kv_len or S, (S + 127) // 128 * 128
    s = (q[:, :1].float() @ k[:, :1, :kv].float().transpose(2, 3).contiguous()) * 128 ** -0.5
    want, want_lse = f32(torch.softmax(s, -1) @ v[:, :1, :kv].float()), f32(torch.logsumexp(s, -1))
    first = None
    for h in heads:
        a = [t[:, :h].contiguous() for t in (q, k, v)]
        o, o2, lse = torch.full_like(a[0], float("nan")), torch.full_like(a[0], float("nan")), torch.empty((1, h, S), device=dev)
        m, d = (torch.full((1, h, 1, sp), float("nan"), device=dev) for _ in range(2))
        bm = torch.full((1, h, sp // 64, sp), 7.0, device=dev, dtype=torch.bfloat16)
        ops.full_attn_ex(o, lse, *a, 0.0, kv_len)
        ops.fullattn_maxq_denom_blockmax(o2, m, d, bm, *a, 0.0, kv_len)
        assert_close_o(f32(o[:, :1]), want, "o")
        assert_close_o(f32(o2[:, :1]), want, "o with statistics")
        assert_close_stat(f32(lse[:, :1]), want_lse, "lse", atol=1e-4)
        assert bool((d[..., S:] == float("-inf")).all()) and bool((m[..., S:] == 0).all())
        got = (o, o2, lse, m, d, bm)
        if first is None:
            first = got
        n = min(h, first[0].shape[1])
        assert all(torch.equal(x[:, :n], y[:, :n]) for x, y in zip(got, first))


@pytest.mark.parametrize("S,kv_len,heads,rows", [
    (1400, 0, (45, 32), (128, 256)),                # 270 and 192 q-blocks of 256 rows, 22 tiles
    (1345, 0, (43, 42, 24), (128, 256, 256)),       # 258, 252 and 144
    (1345, 1344, (43, 24), (128, 128)),             # 21 tiles
])
def test_256_row_qblocks_in_one_round(dev, S, kv_len, heads, rows):
    test_256_row_qblocks_give_the_same_bits(dev, S, kv_len, heads, rows, rows)


@pytest.mark.parametrize("S,kv_len,heads", [(1100, 0, (57, 56, 71, 72)), (1473, 1408, (45, 44, 53)), (700, 0, (2, 24, 70))])
def test_statistics_alone_at_d64_match_those_of_attention(dev, S, kv_len, heads):
    """Row maxima, denominators and block maxima of the statistics alone: bit for bit those of the sweep with V."""
    import fgattn_tk_cuda_amd.spattn.cuda_attn  # noqa: F401

    print("case statistics alone against attention", S, kv_len, heads, flush=True)
    ops = torch.ops.cuda_attn
    g = torch.Generator(device=dev).manual_seed(S)
    sp = (S + 127) // 128 * 128
    for h in heads:
        q, k, v = (torch.randn((1, h, S, 64), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
        o = torch.empty_like(q)
        m, d, m2, d2 = (torch.full((1, h, 1, sp), float("nan"), device=dev) for _ in range(4))
        bm, bm2 = (torch.full((1, h, sp // 64, sp), 7.0, device=dev, dtype=torch.bfloat16) for _ in range(2))
        ops.fullattn_maxq_denom_blockmax(o, m, d, bm, q, k, v, 0.0, kv_len)
        ops.maxq_denom_blockmax(m2, d2, bm2, q, k, 0.0, kv_len)
        assert torch.equal(m, m2) and torch.equal(d, d2) and torch.equal(bm[..., :S], bm2[..., :S])
