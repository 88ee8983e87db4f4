"""GPU: the edge cases of list-driven attention through the kernels with one workgroup per 128-row list.

The cases of test_gpu_attention.py and test_gpu_random_shapes.py are small launches, and lists of 128-row q-blocks run by halves
there.  The same cases run here as part of a computation of so many heads that no launch takes the halves, against the oracle."""
import pytest

import test_gpu_attention as edges
import test_gpu_random_shapes as random_shapes
from fgattn_tk_cuda_amd import capi

pytestmark = pytest.mark.gpu
MANY = 1 << 20


@pytest.fixture
def whole_lists(monkeypatch):
    """capi.sp_attn and capi.sp_attn_blocks as a part of MANY heads; yields the calls that went to 128-row lists: (tokens, D)."""
    calls = []

    def patched(name, tokens):
        run = getattr(capi, name)

        def call(o, q, k, v, idx, num, *, qblk, kv_len=0, **kwargs):
            B, H, S, D = q.shape
            rows = capi.load().spattn_list_form(D, qblk, tokens, B * H, S, kv_len, idx.shape[3], MANY)
            assert rows == qblk
            if qblk == 128:
                calls.append((tokens, D))
            run(o, q, k, v, idx, num, qblk=qblk, kv_len=kv_len, of_heads=MANY, **kwargs)

        monkeypatch.setattr(capi, name, call)

    patched("sp_attn", 1)
    patched("sp_attn_blocks", 0)
    return calls


@pytest.mark.parametrize("D", [64, 128])
def test_edge_cases_of_token_lists(dev, whole_lists, D):
    print("case whole token lists", D, flush=True)
    edges.test_sp_attn_permuted_all_keys_equals_sdpa(dev, D, 128, 1000)
    edges.test_sp_attn_ragged_token_lists(dev, D, 128)
    edges.test_sp_attn_long_lists_with_entries_that_name_no_key(dev, D, 128)
    edges.test_sp_attn_first_tiles_without_a_key(dev, D, 128)
    assert len(whole_lists) == 7 and set(whole_lists) == {(1, D)}


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("growth", ["ramp", "jump"])
def test_growing_scores(dev, whole_lists, D, growth):
    print("case whole lists, growing scores", D, growth, flush=True)
    edges.test_sp_attn_scores_that_outgrow_the_running_maximum(dev, D, 128, growth)
    edges.test_sp_attn_blocks_matches_oracle_and_token_path(dev, D, 128, 1000)
    assert sorted(whole_lists) == [(0, D), (0, D), (1, D), (1, D)]


def test_empty_lists_and_bad_indices(dev, whole_lists):
    print("case whole lists, empty ones", flush=True)
    edges.test_sp_attn_empty_list_and_bad_indices(dev)
    edges.test_sp_attn_single_key_returns_v_row(dev)
    assert whole_lists == [(1, 64), (1, 128)]


def test_random_lists(dev, whole_lists):
    """Random sizes, kv lengths, work orders and entries."""
    for seed in range(24):
        random_shapes.test_token_lists_random(dev, seed)
        random_shapes.test_block_lists_random(dev, seed)
    assert all(whole_lists.count((tokens, D)) >= 5 for tokens in (0, 1) for D in (64, 128))
