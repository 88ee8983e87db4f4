"""GPU: blockmax_to_packedmask (the threshold sweep over what the block maxima leave) against the full sweep
(booleanmask_packed, pinned to the oracle elsewhere), bit for bit, at the edges of its tiles: 32-row groups,
128-row q-blocks, 64-key blocks, the 64 pieces of 32 keys that a wave's words go out in, and the key chunks of
20480 (d = 128) and 32768 (d = 64) keys; and the key lists decoded with their tails filled."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,S,kv_len,x", [
    (64, 1, 0, 0.5), (128, 33, 0, 2), (64, 64, 63, 2), (128, 129, 65, 2), (64, 200, 1, 0.5), (128, 300, 0, 1e-6), (64, 300, 0, 1e6),
    (64, 8193, 0, 16), (128, 8256, 8191, 32), (64, 8300, 0, 1e-6), (128, 20480, 0, 32), (128, 20545, 0, 16), (64, 32768, 32700, 64),
    (64, 32900, 0, 32), (128, 20490, 0, 1e-6), (64, 100, 20, 1e-6), (128, 8224, 8220, 1e-6),
])
def test_votes_from_block_maxima(dev, D, S, kv_len, x):
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    print("case blockmax_to_packedmask", D, S, kv_len, x, flush=True)
    ops = torch.ops.cuda_attn
    H = 2
    g = torch.Generator(device=dev).manual_seed(S + D)
    q, k = (torch.randn((1, H, S, D), generator=g, device=dev) +
            torch.randn((1, H, (S + 63) // 64, D), generator=g, device=dev).repeat_interleave(64, dim=2)[:, :, :S] for _ in range(2))
    q, k = q.to(torch.bfloat16).contiguous(), k.to(torch.bfloat16).contiguous()
    thresh = x / (kv_len or S)
    max_q, denom = mu._stats_buffers(q)
    blockmax = mu.blockmax_buffer(q).fill_(float("nan"))     # blocks without a key stay unwritten and unread
    ops.maxq_denom_blockmax(max_q, denom, blockmax, q, k, 0.0, kv_len)
    want = mu.qk_packedmask_from_maxq_denom_cuda(max_q, denom, q, k, thresh, 128, kv_len)
    got = torch.full_like(want, 0x5a)
    ops.blockmax_to_packedmask(got, blockmax, max_q, denom, q, k, thresh, 0.0, kv_len)
    assert torch.equal(got, want)
    idx, num = (torch.full((1, H, want.shape[2], n), -7, dtype=torch.int32, device=dev) for n in (want.shape[3] * 8, 1))
    ops.packedmask_to_indexmask(idx, num, got, kv_len or S)
    filled, num2 = mu.packedmask_to_indexmask_cuda(got, kv_len or S)
    assert torch.equal(num.view(-1), num2.view(-1))
    tail = torch.arange(idx.shape[3], device=dev) >= num
    assert torch.equal(filled.masked_fill(tail, -7), idx) and bool((filled[tail] == idx.shape[3]).all())
    if x < 1e-3:                                              # a threshold below every weight keeps every key there is
        assert int(num.sum()) == (kv_len or S) * num.numel()
    with pytest.raises(RuntimeError):
        ops.blockmax_to_packedmask(got, blockmax[:, :1].contiguous(), max_q, denom, q, k, thresh, 0.0, kv_len)


@pytest.mark.parametrize("S,D", [(700, 64), (1300, 128)])
def test_refresh_in_groups_of_heads(dev, S, D):
    """cached_attn_cuda and qk_indexmask_cuda with a budget that holds some heads' block maxima only: output,
    lists and counts equal those of all heads at once and of the two full sweeps."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu, sparseattn_functionals as fn

    print("case head groups", S, D, flush=True)
    B, H = 2, 3
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn((B, H, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    per_head = mu.blockmax_bytes(q) // (B * H)
    got = []
    for kw in (dict(onepass=True), dict(onepass=False), dict(blockmax_budget_bytes=4 * per_head), dict(blockmax_budget_bytes=2 * per_head),
               dict(blockmax_budget_bytes=per_head)):
        cache = mu.NaiveMaskCache([0])
        out = fn.cached_attn_cuda(q, k, v, 0, 0, thresh=4.0 / S, blocksz=128, mask_cache=cache, **kw)
        got.append((out,) + tuple(cache.get_mask_from_cache(0)))
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))
    one, two = mu.qk_indexmask_cuda(q, k, 4.0 / S), mu.qk_indexmask_cuda(q, k, 4.0 / S, onepass=False)
    assert torch.equal(one[0], two[0]) and torch.equal(one[1], two[1]) and 0 < float(two[1].float().mean()) < S


@pytest.mark.parametrize("S,D,qblk", [(700, 64, 64), (1300, 128, 64), (1300, 64, 128), (65, 128, 128)])
def test_block_refresh_in_groups_of_heads(dev, S, D, qblk):
    """blockcached_attn_cuda above its budget: output, lists and counts equal those of the two full sweeps."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu, sparseattn_functionals as fn

    print("case block lists by head groups", S, D, qblk, flush=True)
    B, H = 2, 3
    g = torch.Generator(device=dev).manual_seed(S + qblk)
    q, k, v = (torch.randn((B, H, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    per_head = mu.blockmax_bytes(q) // (B * H)
    got = []
    for kw in (dict(onepass=False), dict(blockmax_budget_bytes=4 * per_head), dict(blockmax_budget_bytes=2 * per_head),
               dict(blockmax_budget_bytes=per_head)):
        cache = mu.BlockListCache([0])
        out = fn.blockcached_attn_cuda(q, k, v, 0, 0, thresh=8.0 / S, qblk=qblk, mask_cache=cache, **kw)
        got.append((out,) + tuple(cache.get_mask_from_cache(0)))
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))
    assert int(got[0][2].sum()) > 0


@pytest.mark.parametrize("H,S,D", [(16, 2000, 128), (26, 2000, 64), (40, 1400, 64), (9, 1990, 128), (50, 2049, 128)])
def test_groups_take_the_form_of_the_whole(dev, H, S, D):
    """Heads whose launch as a whole takes 128-row q-blocks (the last: 256-row ones), in groups small enough for 64-row
    ones: output, statistics and lists are the bits of all heads at once."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu, sparseattn_functionals as fn

    print("case groups of the whole", H, S, D, flush=True)
    ops = torch.ops.cuda_attn
    g = torch.Generator(device=dev).manual_seed(S + H)
    q, k, v = (torch.randn((1, H, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    per_head = mu.blockmax_bytes(q) // H
    kw = [dict(onepass=True), dict(onepass=False), dict(blockmax_budget_bytes=4 * per_head)]
    got = []
    for route in kw:
        cache = mu.NaiveMaskCache([0])
        out = fn.cached_attn_cuda(q, k, v, 0, 0, thresh=8.0 / S, blocksz=128, mask_cache=cache, **route)
        got.append((out,) + tuple(cache.get_mask_from_cache(0)))
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))
    one = [mu.qk_indexmask_cuda(q, k, 8.0 / S, onepass=r.get("onepass"), budget_bytes=r.get("blockmax_budget_bytes")) for r in kw]
    assert all(torch.equal(a, b) for other in one[1:] for a, b in zip(one[0], other))
    m, d = mu._stats_buffers(q)
    ops.maxq_denom_blockmax(m, d, mu.blockmax_buffer(q), q, k, 0.0, 0)
    some = q[:, 2:4].contiguous(), k[:, 2:4].contiguous()
    ms, ds = mu._stats_buffers(some[0])
    ops.maxq_denom_blockmax(ms, ds, mu.blockmax_buffer(some[0]), *some, 0.0, 0, H)
    assert torch.equal(ms, m[:, 2:4]) and torch.equal(ds, d[:, 2:4])
    ops.maxq_denom_blockmax(ms, ds, mu.blockmax_buffer(some[0]), *some, 0.0, 0)
    assert torch.equal(ms, m[:, 2:4]) and not torch.equal(ds, d[:, 2:4])   # a launch of its own: another order of the sums
    with pytest.raises(RuntimeError):
        ops.maxq_denom_blockmax(ms, ds, mu.blockmax_buffer(some[0]), *some, 0.0, 0, 1)


@pytest.mark.parametrize("D,S,kv_len,stride,x", [
    (128, 2048, 0, 2048, 16), (128, 2049, 2040, 2304, 16), (64, 4096, 0, 4096, 32), (64, 4225, 4225, 4480, 1e-6), (128, 1535, 0, 1536, 1e-6),
    (64, 15, 0, 128, 0.5), (128, 17, 16, 256, 0.5), (64, 6000, 127, 6016, 1e-6), (128, 2200, 0, 2304, 1e9),
])
def test_votes_by_rows(dev, D, S, kv_len, stride, x):
    """The tiles of sixteen listed rows: chunks of 16 (d = 128) and 32 (d = 64) q-blocks and their remainders, lists that
    are full before the chunk has ended (every row active), q-blocks and chunks without an active row, rows filled up
    to four, rows of bits longer than the sequence - the bits of the full sweep, whose rows of bits are as long."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    print("case votes by rows", D, S, kv_len, stride, x, flush=True)
    ops = torch.ops.cuda_attn
    H = 3
    g = torch.Generator(device=dev).manual_seed(S + D)
    q, k = (torch.randn((1, H, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    q[:, 1, : S // 2] = 0                                     # equal weights: no row of these passes at x > 1
    max_q, denom = mu._stats_buffers(q)
    blockmax = mu.blockmax_buffer(q).fill_(float("nan"))
    ops.maxq_denom_blockmax(max_q, denom, blockmax, q, k, 0.0, kv_len)
    got = torch.full((1, H, (S + 127) // 128, stride // 8), 0x5a, dtype=torch.uint8, device=dev)
    want = torch.full_like(got, 0xa5)
    thresh = x / (kv_len or S)
    ops.booleanmask_packed(want, max_q, denom, q, k, thresh, 128, 0.0, kv_len)
    ops.blockmax_to_packedmask(got, blockmax, max_q, denom, q, k, thresh, 0.0, kv_len)
    assert torch.equal(got, want) and bool(got.any()) == (x < 1e6)


@pytest.mark.parametrize("D,S,H,kv_len", [
    (64, 640, 100, 0), (128, 1000, 60, 999), (128, 1000, 90, 0), (128, 2300, 20, 0), (64, 1500, 60, 1473), (128, 1500, 64, 0),
    (64, 900, 170, 897), (128, 2100, 180, 2049),
])
def test_votes_by_length_of_the_chunks(dev, D, S, H, kv_len):
    """Chunks of 2, 3, 4 (the instantiation for short ones), 5, 6, 6, 8 and 12 q-blocks, the last of a head shorter: every row
    active, and some - the bits of the full sweep."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    print("case votes by chunks", D, S, H, kv_len, flush=True)
    ops = torch.ops.cuda_attn
    g = torch.Generator(device=dev).manual_seed(S + H)
    q, k = (torch.randn((1, H, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    max_q, denom = mu._stats_buffers(q)
    blockmax = mu.blockmax_buffer(q)
    ops.maxq_denom_blockmax(max_q, denom, blockmax, q, k, 0.0, kv_len)
    for x in (1e-6, 16):
        want = mu.qk_packedmask_from_maxq_denom_cuda(max_q, denom, q, k, x / (kv_len or S), 128, kv_len)
        got = torch.full_like(want, 0x5a)
        ops.blockmax_to_packedmask(got, blockmax, max_q, denom, q, k, x / (kv_len or S), 0.0, kv_len)
        assert torch.equal(got, want) and bool(got.any())


@pytest.mark.parametrize("value", [0x7fc0, 0xffc0, 0x7f80, 0xff80])   # NaNs of both signs, infinities
@pytest.mark.parametrize("D,S,bad", [(128, 2500, (2499, 700)), (64, 5000, (4999, 4096)), (128, 2100, (2048, 5)), (64, 300, (299, 31))])
def test_votes_beside_rows_that_are_not_finite(dev, D, S, bad, value):
    """A query row without a finite score never votes, in this sweep as in the full one, and no row votes for another
    q-block than its own - whichever row it is: the last, the first of the next chunk."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    print("case votes beside", hex(value), D, S, bad, flush=True)
    ops = torch.ops.cuda_attn
    g = torch.Generator(device=dev).manual_seed(S + D)
    q, k = (torch.randn((1, 1, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    bits = []
    for v in (value, 0):                                      # zeros: equal weights, no votes at this threshold
        q.view(torch.int16)[:, :, list(bad)] = v if v < 0x8000 else v - 0x10000
        max_q, denom = mu._stats_buffers(q)
        blockmax = mu.blockmax_buffer(q)
        ops.maxq_denom_blockmax(max_q, denom, blockmax, q, k, 0.0, 0)
        want = mu.qk_packedmask_from_maxq_denom_cuda(max_q, denom, q, k, 20.0 / S, 128, 0)
        got = torch.full_like(want, 0x5a)
        ops.blockmax_to_packedmask(got, blockmax, max_q, denom, q, k, 20.0 / S, 0.0, 0)
        assert torch.equal(got, want) and bool(got.any())
        bits.append(got)
    assert torch.equal(*bits)


@pytest.mark.parametrize("S,D,dense", [(1, 64, True), (65, 128, False), (300, 64, True), (1300, 128, True), (2049, 64, False)])
def test_onepass_operators_are_the_operators_one_by_one(dev, S, D, dense):
    """onepass_packedmask and onepass_blocklists: output, bits, lists with their tails and counts are those of the
    statistics with block maxima and the threshold on them; what those refuse stays refused."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    print("case onepass", S, D, dense, flush=True)
    ops = torch.ops.cuda_attn
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v = (torch.randn((2, 3, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    thresh, o = 4.0 / S, torch.empty_like(q)
    m, d = mu._stats_buffers(q)
    blockmax = mu.blockmax_buffer(q)
    if dense:
        ops.fullattn_maxq_denom_blockmax(o, m, d, blockmax, q, k, v, 0.0, 0)
    else:
        ops.maxq_denom_blockmax(m, d, blockmax, q, k, 0.0, 0)
    packed = mu.qk_packedmask_from_blockmax_cuda(blockmax, m, d, q, k, thresh)
    extra = lambda: (torch.zeros_like(q), q, k, v) if dense else (None, q, k, None)
    got, a = torch.full_like(packed, 0x5a), extra()
    ops.onepass_packedmask(got, *a, thresh)
    assert torch.equal(got, packed) and (not dense or torch.equal(a[0], o))
    for qblk in (64, 128):
        idx, cnt = mu.blockmax_to_blocklists_cuda(blockmax, m, d, thresh, S, D, qblk)
        gi, gc, a = torch.full_like(idx, 7), torch.full_like(cnt, 7), extra()
        ops.onepass_blocklists(gi, gc, *a, thresh, qblk)
        assert torch.equal(gi, idx) and torch.equal(gc, cnt) and (not dense or torch.equal(a[0], o))
    for bad in ((got[..., :-1].contiguous(), *extra(), thresh), (got, None, q, k, v, thresh), (got, None, q, k[:, :, :-1].contiguous(), None, thresh),
                (got, None, q.float(), k, None, thresh)):
        with pytest.raises(RuntimeError):
            ops.onepass_packedmask(*bad)
    with pytest.raises(RuntimeError):
        ops.onepass_blocklists(gi, gc, *extra(), thresh, 96)
