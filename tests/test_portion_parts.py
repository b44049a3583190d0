"""Into how many parts the keys of a portion's row blocks are cut on a chip of 256 compute units: parts are for the turns that the
units take them in, and none for row blocks that fill the units or contexts too short to cut."""
import pytest
import torch

from arle_amd.kernels import ops

DEVICE = torch.device("cuda", 0)


@pytest.fixture(autouse=True)
def _units(monkeypatch):
    monkeypatch.setattr(ops, "_compute_units", lambda index: 256)


def _parts(rows, behind, head_dim, heads=32, kv_heads=8, portions=1):
    return ops.portion_key_splits(rows * portions, rows, portions, heads, kv_heads, head_dim, rows + behind, DEVICE)


@pytest.mark.parametrize("head_dim", [64, 96, 128, 160, 192, 256])
@pytest.mark.parametrize("rows,parts", [(520, 3), (640, 3)])      # 136 and 160 row blocks: three parts in two turns
def test_row_blocks_for_more_than_half_of_the_units_are_cut_by_turns(head_dim, rows, parts):
    assert _parts(rows, 3100, head_dim) == parts
    assert _parts(rows, 15000, head_dim) >= parts
    assert _parts(rows, 0, head_dim) == 1


@pytest.mark.parametrize("head_dim,behind,parts", [
    (64, 3100, 1), (64, 7000, 4), (96, 3100, 4), (96, 15000, 4), (128, 7000, 1), (128, 15000, 1), (256, 3100, 4), (256, 15000, 4)])
def test_three_quarters_of_the_units_in_three_turns_where_the_merge_is_worth_it(head_dim, behind, parts):
    assert _parts(768, behind, head_dim) == parts       # 192 row blocks


@pytest.mark.parametrize("head_dim", [64, 96, 128])
@pytest.mark.parametrize("rows,behind,parts", [(100, 15000, 8), (240, 15000, 4), (512, 15000, 2), (512, 600, 2), (512, 0, 1), (240, 1500, 2),
                                               (800, 15000, 1), (900, 15000, 1), (1024, 15000, 1), (2048, 15000, 1)])
def test_one_turn_or_none(head_dim, rows, behind, parts):
    assert _parts(rows, behind, head_dim) == (4 if head_dim == 128 and rows == 512 and behind == 15000 else parts)


@pytest.mark.parametrize("rows,parts", [(320, 3), (352, 5), (384, 5), (448, 4), (512, 4), (520, 3)])
def test_two_workgroups_a_unit_at_heads_of_128(rows, parts):
    assert _parts(rows, 4096, 128) == parts
    assert _parts(rows, 4095 - rows, 128) == (3 if parts == 3 else 2)


@pytest.mark.parametrize("rows,parts", [(100, 8), (360, 8), (400, 7), (512, 2), (800, 5), (832, 6), (900, 2), (1024, 1)])
def test_heads_beyond_128_take_the_fewest_turns(rows, parts):
    assert _parts(rows, 15000, 256) == parts
    items = -(-rows * 4 // 128) * 8
    if items < 256:
        cost = [-(-items * p // 256) / p for p in range(1, 9)]
        assert cost[parts - 1] == min(cost[1:])


def test_every_part_holds_512_keys_of_the_contexts_class():
    for head_dim in (64, 96, 128, 256):
        for rows in range(8, 1100, 12):
            for behind in (0, 100, 900, 2000, 5000, 40000):
                parts = _parts(rows, behind, head_dim)
                keys = 1 << ((rows + behind).bit_length() - 1)
                assert 1 <= parts <= 8 and (parts == 1 or parts * 512 <= keys)
                assert keys <= rows or parts == _parts(rows, keys - rows, head_dim)               # the class alone counts,
                assert keys < 4096 or parts == _parts(rows, 4096, head_dim)                       # up to 4,096


def test_several_portions_count_together():
    assert _parts(300, 15000, 64, portions=1) == 3 and _parts(300, 15000, 64, portions=2) == 4 and _parts(300, 15000, 64, portions=4) == 1


@pytest.mark.parametrize("head_dim", [64, 96, 128, 256])
@pytest.mark.parametrize("heads,kv_heads,rows,longest,parts", [
    (32, 8, (100, 20), 15020, 8), (16, 2, (512, 600, 20), 15020, 3), (32, 8, (20, 450), 7020, 3), (32, 8, (450, 450), 3450, 2),
    (32, 8, (200, 450), 3200, 2), (16, 2, (333, 512), 7512, 4), (32, 8, (20, 60), 1560, 2), (32, 8, (333, 500), 1833, 1)])
def test_unequal_portions_are_cut_for_the_few_row_blocks_with_the_most_keys(head_dim, heads, kv_heads, rows, longest, parts):
    assert ops.portion_key_splits(sum(rows), max(rows), len(rows), heads, kv_heads, head_dim, longest, DEVICE) == parts


def test_several_portions_have_two_parts_a_unit_of_1024_keys_each():
    for heads, kv_heads in ((32, 8), (16, 16), (16, 2)):
        for count in (2, 3, 6):
            for rows in range(17, 600, 13):
                for longest in (700, 1500, 3000, 9000):
                    items = -(-rows * (heads // kv_heads) // 128) * kv_heads * count
                    parts = ops.portion_key_splits(rows * count, rows, count, heads, kv_heads, 64, max(longest, rows), DEVICE)
                    keys = 1 << (max(longest, rows).bit_length() - 1)
                    assert 1 <= parts <= 8 and (parts == 1 or parts * 512 <= keys)
                    assert parts == 1 if items >= 256 else parts >= min(-(-512 // items), 8, keys // 1024)


def test_row_blocks_for_more_than_the_units_beside_decoded_tokens():
    def parts(rows, longest, heads=32, kv_heads=8, beside=True):
        return ops.portion_key_splits(sum(rows) + 4, max(rows), len(rows), heads, kv_heads, 128, longest, DEVICE, beside)

    assert parts((512, 512), 15512) == 2 and parts((512, 512), 15512, beside=False) == 1     # 256 row blocks
    assert parts((512, 512), 15512, 40) == 2 and parts((768, 768), 15768) == 2 and parts((769, 769), 15768) == 1
    assert parts((512, 512), 4095) == 1 and parts((1024,), 15512) == 1
    assert parts((333, 300), 7333) == parts((333, 300), 7333, beside=False) == 3


def test_more_parts_than_one_turn_are_for_the_keys_that_a_window_leaves():
    def parts(rows, head_dim, window, count=1):
        return ops.portion_key_splits(rows * count, rows, count, 32, 8, head_dim, 7000 + rows, DEVICE, False, window)

    for window in (512, 1024):
        assert parts(100, 64, window) == parts(100, 128, window) == 8 and parts(512, 128, window) == 2
        assert parts(520, 64, window) == parts(768, 64, window) == parts(768, 96, window) == 1
        assert parts(300, 64, window, 2) == window // 512
    assert parts(512, 128, 4096) == 4 and parts(520, 64, 4096) == 3 and parts(768, 64, 4096) == 4 and parts(300, 64, 4096, 2) == 4
