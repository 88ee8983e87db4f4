"""Host: how a dense launch is split (rows of a q-block, groups of waves that share one), by its size and by that of the
computation that its heads are a part of."""
import pytest

from fgattn_tk_cuda_amd import capi


def form(D, has_v, stats, heads, S, kv_len=0, of_heads=0):
    return capi.load().spattn_dense_form(D, has_v, stats, heads, S, kv_len, of_heads)


@pytest.mark.parametrize("heads,S,of_heads,whole", [(3, 9000, 12, 2561), (6, 9000, 12, 2561), (5, 2049, 50, 2561), (3, 5000, 24, 2561)])
def test_some_heads_take_256_row_qblocks_by_their_own_number(heads, S, of_heads, whole):
    """128- and 256-row q-blocks give the same bits: a part of a computation that 256-row ones would leave idle (216, 72
    and 108, 45, 60 of them for 256 CUs) takes 128-row ones, also where the whole does not."""
    assert form(128, 1, 1, of_heads, S) == whole
    last = heads * -(-S // 256) % 256
    assert form(128, 1, 1, heads, S, 0, of_heads) == (2561 if last == 0 or last > 128 else 1281)


def test_256_row_qblocks_with_statistics_by_rounds():
    """648 q-blocks of 256 rows of 36 key tiles and 660 of 219: behind two rounds from 64 tiles on; five rounds and six."""
    assert form(128, 1, 1, 72, 2304) == 1281 and form(128, 1, 1, 12, 14000) == 2561
    assert form(128, 1, 1, 44, 4033) == 2561 and form(128, 1, 1, 44, 4032) == 1281   # 64 and 63 tiles, 704 q-blocks
    assert form(128, 1, 1, 16, 20480) == 2561 and form(128, 1, 1, 24, 16384) == 1281


def test_forms_that_add_in_another_order_go_by_the_whole():
    assert form(128, 1, 1, 4, 2000, 0, 16) == form(128, 1, 1, 16, 2000) == 1282 and form(128, 1, 1, 4, 2000) == 641
    assert form(64, 1, 1, 4, 2000, 0, 26) == form(64, 1, 1, 26, 2000) != form(64, 1, 1, 4, 2000)
    assert form(128, 0, 1, 2, 9000, 0, 12) == form(128, 0, 1, 12, 9000) == 1281


def test_what_the_calls_refuse_has_no_form():
    assert form(96, 1, 0, 1, 128) == -2
    for bad in ((64, 0, 0, 1, 128), (64, 1, 0, 0, 128), (64, 1, 0, 1, 0), (64, 1, 0, 1, 1 << 24), (64, 1, 0, 2, 128, 0, 1)):
        assert form(*bad) == -6


def test_256_row_qblocks_in_one_round():
    """From 22 key tiles on where they fit one round that is more than half full, 32 otherwise."""
    assert form(128, 1, 0, 24, 1345) == form(128, 1, 1, 42, 1345) == 2561              # 144 and 252 q-blocks
    assert form(128, 1, 0, 43, 1345) == form(128, 1, 1, 24, 1345, 1344) == 1281        # 258; 21 tiles
    assert form(128, 1, 0, 80, 1506) == 1281                                            # 480 of 24 tiles


def test_statistics_at_d64_take_the_form_of_attention_with_statistics():
    """Other forms add a row's sum in another order: a key at its threshold would be in the mask of a call that takes the
    statistics alone and not in that of a refresh, or the other way round."""
    for heads in (1, 3, 8, 24, 44, 56, 57, 64, 71, 72, 90, 240):
        for S, kv_len in ((64, 0), (300, 0), (577, 0), (767, 0), (1100, 0), (1100, 767), (1473, 1408), (2050, 0), (8508, 0), (32760, 0)):
            assert form(64, 0, 1, heads, S, kv_len) == form(64, 1, 1, heads, S, kv_len), (heads, S, kv_len)


def test_two_groups_from_ten_tiles_at_d64():
    assert [form(64, v, s, 8, S) for v, s in ((1, 0), (1, 1), (0, 1)) for S in (576, 577)] == [641, 642] * 3
