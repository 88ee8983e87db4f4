"""Host logic of the one-sweep refresh in groups of heads."""
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
