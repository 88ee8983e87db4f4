"""GPU: lists of 128-row q-blocks in launches that leave the chip idle run by workgroups of 64 rows, two to a list: bit for bit
what the same lists, each given to both of its 64-row q-blocks, give, in index order and in a work order."""
import ctypes

import pytest
import torch

from fgattn_tk_cuda_amd import build as bld, capi, workloads as wl

pytestmark = pytest.mark.gpu


def _lists(dev, H, S):
    """Block lists and token lists of 128-row q-blocks, short, long and empty ones, and a work order."""
    nq, nkb = wl.ceil_div(S, 128), wl.ceil_div(S, 64)
    cnt = wl.zipf_counts(1, H, nq, s=1.1, lo=1, hi=nkb, seed=32)
    cnt[:, :, ::5] = cnt[:, :, ::5].clip(max=3)
    blk, bc = wl.ragged_block_lists(1, H, S, 128, 64, cnt, seed=33)
    blk = torch.nn.functional.pad(blk, (0, max(0, 5 - blk.shape[3])), value=-1)   # as wide as the rule asks for
    bc[:, :, ::7] = 0
    tok, num = wl.blocks_to_tokens(blk, bc, S)
    if tok.shape[3] < 256:
        tok = torch.nn.functional.pad(tok, (0, 256 - tok.shape[3]), value=256)
    order = torch.randperm(H * nq, generator=torch.Generator().manual_seed(34)).to(torch.int32).to(dev)
    return {"tokens": (tok.to(dev), num.to(dev)), "blocks": (blk.to(dev), bc.to(dev))}, order


def _call(lib, kind, qkv, idx, n, qblk, kv_len, order=None):
    q, k, v = qkv
    _, H, S, D = q.shape
    o, lse = torch.full_like(q, float("nan")), torch.full((1, H, S), float("nan"), device=q.device)
    name = {"tokens": "spattn_sp_attn", "blocks": "spattn_sp_attn_blocks"}[kind] + ("" if order is None else "_ordered")
    e = getattr(lib, name)(o.data_ptr(), lse.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), idx.data_ptr(), n.data_ptr(),
                           *([] if order is None else [order.data_ptr()]), int(idx.shape[3]), qblk, 1, H, S, D, kv_len, 0.0,
                           torch.cuda.current_stream().cuda_stream)
    assert e == 0
    torch.cuda.synchronize()
    return o.view(torch.int16), lse.view(torch.int32)


@pytest.mark.parametrize("D,H,S,kv_len,halved", [
    (64, 3, 100, 0, True), (64, 3, 129, 100, True),          # a q-block and a half; two, the second with one row
    (64, 5, 1050, 0, True), (64, 8, 2048, 2000, True),       # the last q-block ends in its first half; one per CU
    (64, 24, 2048, 0, True), (64, 24, 1100, 1023, False),    # three per CU; more than one per CU and too short
    (64, 25, 2048, 0, False),                                # behind three per CU
    (128, 5, 1650, 0, True), (128, 8, 2048, 0, True), (128, 1, 16384, 0, True),   # up to one per CU
    (128, 5, 900, 767, False), (128, 9, 2048, 0, False),     # too short; behind one per CU
])
def test_halves_give_the_bits_of_64_row_lists(dev, D, H, S, kv_len, halved):
    print("case halves", D, H, S, kv_len, flush=True)
    lib = capi.load()
    qkv = [t.to(dev) for t in wl.randn_qkv(1, H, S, D, seed=31)]
    lists, order = _lists(dev, H, S)
    for kind, (idx, n) in lists.items():
        twice = [t.repeat_interleave(2, dim=2)[:, :, :wl.ceil_div(S, 64)].contiguous() for t in (idx, n)]
        want = _call(lib, kind, qkv, *twice, 64, kv_len)
        o = want[0].view(torch.bfloat16).float()
        assert torch.isfinite(o).all()
        for by in (None, order):
            got = _call(lib, kind, qkv, idx, n, 128, kv_len, by)
            assert all(torch.equal(a, b) for a, b in zip(got, want)) == halved, (kind, by is not None)
            # both forms round P to bf16 ahead of its product with V, and O (2^-9)
            assert float((got[0].view(torch.bfloat16).float() - o).norm()) <= 1e-2 * float(o.norm())


@pytest.mark.parametrize("D,H,S,few", [(64, 25, 2048, 3), (64, 24, 2048, 5), (128, 9, 2048, 1), (128, 8, 1700, 3)])
def test_some_heads_give_the_bits_of_all(dev, D, H, S, few):
    """Some heads of a computation that runs by whole lists, and of one that runs by halves, through the operators and the
    functional, in index order and in a work order; without of_heads the former would run by halves."""
    from fgattn_tk_cuda_amd.spattn import cuda_attn, mask_utils, sparseattn_functionals as fn  # noqa: F401

    print("case some heads", D, H, S, few, flush=True)
    ops = torch.ops.cuda_attn
    q, k, v = (t.to(dev) for t in wl.randn_qkv(1, H, S, D, seed=36))
    lists, order = _lists(dev, H, S)

    def call(kind, heads, order=None, of_heads=0):
        qh, kh, vh, idx, n = (t[:, heads].contiguous() for t in (q, k, v, *lists[kind]))
        o, lse = torch.empty_like(qh), torch.empty(qh.shape[:3], device=dev)
        if kind == "tokens":
            ops.sp_attn_ex(o, lse, qh, kh, vh, idx, n, order, 0.0, 0, of_heads)
        else:
            ops.sp_attn_block(o, lse, qh, kh, vh, idx, n, order, 128, 0.0, 0, of_heads)
        return o, lse, (qh, kh, vh, idx, n)

    nq = wl.ceil_div(S, 128)
    for kind in lists:
        whole = call(kind, slice(0, H), order)
        for h0 in range(0, H, few):
            heads = slice(h0, min(H, h0 + few))
            some = torch.randperm((heads.stop - h0) * nq, generator=torch.Generator().manual_seed(h0)).to(torch.int32).to(dev)
            for by in (None, some):
                o, lse, _ = call(kind, heads, by, H)
                assert torch.equal(o, whole[0][:, heads]) and torch.equal(lse, whole[1][:, heads]), (kind, h0)
        o, _, part = call(kind, slice(0, few))
        assert kind != "tokens" or torch.equal(o, whole[0][:, :few]) == (H * wl.ceil_div(S, 64) <= (768 if D == 64 else 256))
        cache = (mask_utils.NaiveMaskCache if kind == "tokens" else mask_utils.BlockListCache)([0])
        cache.update_cache(0, *part[3:])
        step = fn.cached_attn_cuda if kind == "tokens" else fn.blockcached_attn_cuda
        assert torch.equal(step(*part[:3], 0, 1, blocksz=128, mask_cache=cache, of_heads=H), whole[0][:, :few])
    with pytest.raises(RuntimeError):
        call("tokens", slice(0, 2), None, 1)


@pytest.mark.parametrize("D,H,S", [(128, 16, 1100), (64, 56, 900)])
def test_large_list_launches_read_no_freed_slot(dev, D, H, S):
    """Lists of 128-row q-blocks behind the rule, one workgroup to a list, in the NaN-poisoning build."""
    print("case poison large lists", D, H, S, flush=True)
    poison = ctypes.CDLL(str(bld.POISON_LIB))
    for name, (res, args) in capi._SIGNATURES.items():
        getattr(poison, name).restype, getattr(poison, name).argtypes = res, args
    qkv = [t.to(dev) for t in wl.randn_qkv(1, H, S, D, seed=35)]
    for kind, (idx, n) in _lists(dev, H, S)[0].items():
        good, bad = (_call(lib, kind, qkv, idx, n, 128, 0) for lib in (capi.load(), poison))
        assert all(torch.equal(a, b) for a, b in zip(good, bad))
