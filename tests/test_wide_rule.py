"""Where the product for prompt portions (`ops.gemm_wide`) is taken and in which workgroups, on the host."""
import pytest

from arle_amd.kernels import ops

# (rows, N, K), workgroups that were slower and faster ones (us): what an XCD gets of the column blocks decides, not their sum
PLANS = [
    (3072, 6144, 1024, (256, 320), (256, 160)),      # 67.5 / 47.2: 240 workgroups, but 36 on some XCDs of 32 places
    (1536, 6144, 1024, (128, 320), (256, 160)),      # 40.8 / 24.5
    (1152, 8192, 3072, (128, 320), (256, 192)),      # 98.9 / 63.2
    (2400, 19456, 2560, (256, 256), (256, 320)),     # 251.7 / 236.0
    (3072, 37888, 3584, (256, 256), (256, 320)),     # 708.5 / 661.9
    (3201, 24576, 4096, (256, 320), (256, 256)),     # 591.4 / 524.6
]


@pytest.mark.parametrize("rows,n,k,slower,faster", PLANS)
def test_turns_are_counted_by_the_fullest_xcd(rows, n, k, slower, faster):
    assert ops.wide_plan(rows, n, k, 1, 256)[0] == faster


def _order(row_blocks, col_blocks):
    """The (row block, column block) of every workgroup, in launch order, as gemm_wide's kernel works them out."""
    xcds, patch_rows, patch_cols = 8, 8, 4
    cols = -(-col_blocks // xcds)
    for place in range(row_blocks * cols * xcds):
        xcd, q = place % xcds, place // xcds
        group, q = divmod(q, row_blocks * patch_cols)
        cols_here = min(patch_cols, cols - group * patch_cols)
        row_group, q = divmod(q, patch_rows * cols_here)
        rows_here = min(patch_rows, row_blocks - row_group * patch_rows)
        yield row_group * patch_rows + q % rows_here, (group * patch_cols + q // rows_here) * xcds + xcd


@pytest.mark.parametrize("row_blocks", [1, 7, 8, 9, 10, 13, 16, 17, 20, 33])
@pytest.mark.parametrize("col_blocks", [1, 8, 9, 22, 33, 41, 76])
def test_every_block_has_one_workgroup_and_no_row_is_empty(row_blocks, col_blocks):
    taken = list(_order(row_blocks, col_blocks))
    assert all(0 <= r < row_blocks for r, _ in taken)
    inside = [p for p in taken if p[1] < col_blocks]
    assert len(inside) == len(set(inside)) == row_blocks * col_blocks
    assert len(taken) - len(inside) < 8 * row_blocks       # only the last column blocks' XCDs have places left
