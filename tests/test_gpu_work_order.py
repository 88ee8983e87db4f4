"""GPU: the work order that sp_attn keeps for a counts tensor is that tensor's own: not that of an earlier one whose
storage was freed and handed out again, not that of other q-blocks per head, and not one from before the counts were
written, by torch or by an operator of the library."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 640   # q-blocks: more than one per CU, fewer than that have no order


def _fresh(ops, counts, per_head):
    order = torch.empty((counts.numel(),), dtype=torch.int32, device=counts.device)
    ops.qblock_schedule(order, counts, per_head)
    return order


def _counts(dev, seed):
    return torch.randint(1, 4000, (1, 8, N // 8), generator=torch.Generator().manual_seed(seed), dtype=torch.int32).to(dev)


def test_order_follows_the_counts(dev):
    from fgattn_tk_cuda_amd.spattn import cuda_attn, mask_utils as mu

    print("case sp_attn order follows the counts", flush=True)
    ops = torch.ops.cuda_attn
    want, ptrs = [], []
    for seed in (1, 2):                                   # the second tensor takes the storage that the first one freed
        c = _counts(dev, seed)
        ptrs.append(c.data_ptr())
        want.append(_fresh(ops, c, N // 8))
        assert torch.equal(cuda_attn.work_order_of(c, N // 8), want[-1])
        if seed == 1:
            del c
    assert ptrs[0] == ptrs[1] and not torch.equal(*want)
    assert cuda_attn.work_order_of(c, N // 8).data_ptr() == cuda_attn.work_order_of(c, N // 8).data_ptr()   # kept
    one_head = cuda_attn.work_order_of(c, N)
    assert torch.equal(one_head, _fresh(ops, c, N)) and torch.equal(cuda_attn.work_order_of(c, N // 8), want[1])
    c.copy_(_counts(dev, 3))                              # written by torch
    assert torch.equal(cuda_attn.work_order_of(c, N // 8), _fresh(ops, c, N // 8))
    # written by an operator of the library
    S = 128 * (N // 8)
    packed = mu.pack(torch.rand((1, 8, N // 8, S), generator=torch.Generator().manual_seed(4)) <
                     torch.rand((1, 8, N // 8, 1), generator=torch.Generator().manual_seed(5))).to(dev)
    lists = torch.empty((1, 8, N // 8, S), dtype=torch.int32, device=dev)
    before = _fresh(ops, c, N // 8)
    ops.packedmask_to_indexmask(lists, c, packed, S)
    after = _fresh(ops, c, N // 8)
    assert not torch.equal(before, after) and torch.equal(cuda_attn.work_order_of(c, N // 8), after)


def test_no_order_up_to_one_qblock_per_cu(dev):
    from fgattn_tk_cuda_amd.spattn import cuda_attn

    print("case sp_attn without an order", flush=True)
    c = _counts(dev, 6).view(-1)
    assert cuda_attn.work_order_of(c[:256].contiguous(), 32) is None and cuda_attn.work_order_of(c[:257].contiguous(), 257) is not None


@pytest.mark.parametrize("H,ordered", [(31, False), (32, True)])
def test_lists_used_once_take_their_own_order(dev, monkeypatch, H, ordered):
    """Masks derived on every call: from 2048 q-blocks on each call orders its own counts, below none does, and the
    output is that of the lists in index order."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu, sparseattn_functionals as fn

    print("case lists used once", H, flush=True)
    S, D, seen = 8192, 64, []
    order_of = mu.qblock_order_cuda
    monkeypatch.setattr(mu, "qblock_order_cuda", lambda c: (seen.append(c.clone()), order_of(c))[1])
    cache = mu.CompressedBitMaskCache([0])
    for seed in (1, 2):
        g = torch.Generator(device=dev).manual_seed(seed)
        q, k, v = (torch.randn((1, H, S, D), generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
        lists, counts = mu.qk_indexmask_cuda(q, k, 8.0 / S)
        want = torch.empty_like(q)
        torch.ops.cuda_attn.sp_attn_ex(want, None, q, k, v, lists, counts, None, 0.0, 0)
        fn.bitmaskcached_attn_cuda(q, k, v, 0, 0, thresh=8.0 / S, blocksz=128, mask_cache=cache)
        for call in (lambda: fn.attn_computed_with_sparse_mask_cuda(q, k, v, thresh=8.0 / S, blocksz=128),
                     lambda: fn.bitmaskcached_attn_cuda(q, k, v, 0, 1, thresh=8.0 / S, blocksz=128, mask_cache=cache)):
            seen.clear()
            assert torch.equal(call(), want)
            assert len(seen) == int(ordered) and all(torch.equal(c, counts) for c in seen)
    seen.clear()
    fn.attn_topkmask_cuda(q, k, v, select_k=100, blocksz=128)
    assert not seen                                       # lists of equal length


def test_flat_counts(dev):
    """Counts without their heads: sorted as a whole, not as one head; a cache that stores them knows the heads from the
    lists."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    print("case flat counts", flush=True)
    H, SB = 16, 256
    c = torch.randint(1, 4000, (1, H, SB), generator=torch.Generator().manual_seed(7), dtype=torch.int32).to(dev)
    by_heads, as_one = _fresh(torch.ops.cuda_attn, c, SB), _fresh(torch.ops.cuda_attn, c, H * SB)
    whole = torch.empty_like(by_heads)
    torch.ops.cuda_attn.qblock_order(whole, c)
    assert not torch.equal(by_heads, as_one) and not torch.equal(whole, as_one)
    assert torch.equal(mu.qblock_order_cuda(c), by_heads) and torch.equal(mu.qblock_order_cuda(c.view(-1)), whole)
    cache = mu.NaiveMaskCache([0])
    cache.update_cache(0, torch.empty((1, H, SB, 128), dtype=torch.int32, device=dev), c.view(-1))
    assert torch.equal(cache.get_order(0), by_heads)
