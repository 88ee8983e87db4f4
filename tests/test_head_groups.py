"""Host logic of the one-sweep refresh in groups of heads."""
import pytest
import torch


def test_head_groups_cover_all_heads_within_half_the_budget():
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    q = torch.empty((2, 20, 75600, 128), dtype=torch.bfloat16, device="meta")
    per_head = mu.blockmax_bytes(q) // 40
    groups = mu.head_groups(q)
    assert groups[0][0] == 0 and groups[-1][1] == 40 and all(a[1] == b[0] for a, b in zip(groups, groups[1:]))
    sizes = [hi - lo for lo, hi in groups]
    assert max(sizes) * per_head <= mu.BLOCKMAX_BUDGET_BYTES // 2 and max(sizes) - min(sizes) <= 1
    assert mu.head_groups(q, True) == [(0, 40)] and mu.head_groups(q, False) is None
    assert mu.head_groups(q, None, 40 * per_head) == [(0, 40)] and mu.head_groups(q, None, per_head) is None


@pytest.mark.parametrize("bad", ["k", "v"])
@pytest.mark.parametrize("shape", [(3, 2, 300, 64), (2, 3, 64, 300), (1, 6, 300, 64), (2, 3, 600, 32)])
def test_other_shapes_of_as_many_numbers_are_refused(bad, shape):
    """The refreshes hand the operators views over all heads: k and v of another shape are refused all the same."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu, sparseattn_functionals as fn

    t = {n: torch.empty(shape if n == bad else (2, 3, 300, 64), dtype=torch.bfloat16, device="meta") for n in "qkv"}
    args = t["q"], t["k"], t["v"], 0, 0
    with pytest.raises(RuntimeError, match=bad + " must have the shape of q"):
        fn.cached_attn_cuda(*args, thresh=0.01, blocksz=128, mask_cache=mu.NaiveMaskCache([0]))
    with pytest.raises(RuntimeError, match=bad + " must have the shape of q"):
        fn.blockcached_attn_cuda(*args, thresh=0.01, mask_cache=mu.BlockListCache([0]), blockmax_budget_bytes=2 * mu.blockmax_bytes(t["q"]) // 6)
    if bad == "k":
        with pytest.raises(RuntimeError, match="k must have the shape of q"):
            mu.qk_indexmask_cuda(t["q"], t["k"], 0.01)


def test_masks_of_every_step_keep_to_the_callers_route_and_budget(monkeypatch):
    """attn_computed_with_sparse_mask_cuda takes the routes that its keywords name, as the refreshes do."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu, sparseattn_functionals as fn

    q = torch.empty((2, 3, 300, 64), dtype=torch.bfloat16, device="meta")
    per_head, seen = mu.blockmax_bytes(q) // 6, []
    by_groups = mu.packedmask_by_groups
    monkeypatch.setattr(mu, "packedmask_by_groups", lambda groups, *a: (seen.append(groups), by_groups(groups, *a))[1])

    def groups(**kw):
        seen.clear()
        fn.attn_computed_with_sparse_mask_cuda(q, q, q, thresh=0.01, blocksz=128, **kw)
        return list(seen)

    assert groups() == groups(onepass=True) == groups(blockmax_budget_bytes=6 * per_head) == [[(0, 6)]]
    assert groups(blockmax_budget_bytes=4 * per_head) == [[(0, 2), (2, 4), (4, 6)]]
    assert groups(onepass=False) == groups(blockmax_budget_bytes=per_head) == []


@pytest.mark.parametrize("groups", [[(0, 6)], [(0, 2), (2, 6)]])
@pytest.mark.parametrize("buffers", [True, False])
def test_a_callers_sweep_runs_over_every_group(groups, buffers):
    """Also where all heads go at once and the caller has no use for the statistics."""
    from fgattn_tk_cuda_amd.spattn import mask_utils as mu

    q = torch.empty((2, 3, 300, 64), dtype=torch.bfloat16, device="meta")
    seen = []
    max_q, denom = mu._stats_buffers(q) if buffers else (None, None)
    packed = mu.packedmask_by_groups(groups, lambda lo, hi, blockmax, *t: seen.append((lo, hi, blockmax.shape[1], t[0].shape[1])), q, q,
                                     max_q, denom, 0.01)
    assert seen == [(lo, hi, hi - lo, hi - lo) for lo, hi in groups] and packed.shape == (2, 3, 3, 48)
