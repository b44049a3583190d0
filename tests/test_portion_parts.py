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
    assert _parts(rows, behind, head_dim) == parts


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
    assert _parts(300, 15000, 64, portions=1) == 3 and _parts(300, 15000, 64, portions=2) == 3 and _parts(300, 15000, 64, portions=4) == 1
