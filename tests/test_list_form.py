"""How list-driven attention is split (spattn_list_form, host only): lists of 128-row q-blocks run by workgroups of 64 rows where a
launch leaves the chip idle.  The halves add a row's keys in another order, so a launch over some heads of a computation goes by
all of its heads."""
import pytest

from fgattn_tk_cuda_amd import capi


def form(D, tokens, heads, S, kv_len=0, stride=0, of_heads=0, qblk=128):
    return capi.load().spattn_list_form(D, qblk, tokens, heads, S, kv_len, stride or (1024 if tokens else 16), of_heads)


@pytest.mark.parametrize("tokens", [0, 1])
@pytest.mark.parametrize("D,S,whole", [(64, 2048, 8), (64, 2048, 24), (64, 2048, 25), (128, 2048, 8), (128, 2048, 9), (64, 500, 40), (128, 9000, 12)])
def test_some_heads_go_by_all_heads(D, S, whole, tokens):
    """Alone, some heads of a large computation take the halves that the whole does not."""
    want = form(D, tokens, whole, S)
    for some in range(1, whole + 1):
        assert form(D, tokens, some, S, of_heads=whole) == want
    assert form(D, tokens, 1, S) == 64


def test_workgroups_count_and_not_blocks_of_64_rows():
    """Thirteen and 25 blocks of 64 rows a head: a list's second half may be empty, its workgroup is started all the same."""
    assert form(128, 0, 18, 800) == 64 and form(128, 0, 19, 800) == 128    # 252 and 266 workgroups
    assert form(64, 0, 29, 1600) == 64 and form(64, 0, 30, 1600) == 128    # 754 and 780


@pytest.mark.parametrize("D,tokens,heads,S,stride,rows", [
    (128, 0, 4, 4096, 1, 128), (128, 0, 4, 4096, 2, 64),
    (128, 1, 4, 4096, 128, 128), (128, 1, 4, 4096, 256, 64),          # rows shorter than the sequence
    (128, 1, 9, 1600, 1664, 128), (128, 1, 9, 1601, 1664, 64),        # 4 % of the keys: one tile, two
    (64, 0, 4, 4096, 1, 128), (64, 1, 4, 4096, 128, 64), (64, 1, 18, 800, 896, 64),
    (64, 0, 8, 4096, 6, 128), (64, 0, 8, 4096, 7, 64), (64, 1, 8, 4096, 256, 128), (64, 1, 8, 4096, 384, 64),
    (64, 1, 10, 3200, 3200, 128), (64, 1, 9, 3201, 3328, 64),
    (64, 0, 12, 4096, 4, 128), (64, 0, 12, 4096, 5, 64), (64, 1, 12, 4096, 128, 128), (64, 1, 12, 4096, 256, 64),
    (64, 1, 29, 1600, 1664, 128), (64, 1, 29, 1601, 1664, 64),
])
def test_lists_that_lose_by_halves_keep_their_form(D, tokens, heads, S, stride, rows):
    assert form(D, tokens, heads, S, 0, stride) == rows


def test_what_the_rule_does_not_reach():
    assert form(64, 1, 1, 64, qblk=64) == form(128, 0, 400, 9000, qblk=64) == 64
    assert form(128, 1, 400, 9000) == form(64, 0, 400, 9000) == 128


def test_what_the_calls_refuse_has_no_form():
    assert form(96, 1, 1, 128) == -2 and form(64, 1, 1, 128, qblk=96) == -4 and form(64, 1, 1, 128, stride=100) == -3
    for bad in ((64, 1, 0, 128), (64, 0, 1, 0), (64, 0, 1, 1 << 24), (64, 0, 2, 128, 0, 0, 1), (64, 0, 1, 128, 0, -1)):
        assert form(*bad) == -6
