"""Where the product for prompt portions (`ops.gemm_wide`) is taken and in which workgroups, on the host."""
import pytest

from arle_amd.kernels import ops

# (rows, N, K) of gate|up and which was faster by 3 % and more: gemm_wide, or what the other rules take (us on MI355X)
MEASURED = [
    ((65, 6144, 1024), True), ((256, 6144, 1024), True), ((3072, 6144, 1024), True), ((8192, 12288, 1024), True),     # 13.1 / 10.3, 17.5 / 10.8, 51.9 / 47.2, 221.9 / 200.1
    ((65, 4096, 2048), False), ((97, 8192, 3072), False), ((128, 8192, 3072), False), ((80, 16384, 3072), False),     # 13.4 / 16.3, 25.0 / 30.1, 26.6 / 32.1, 32.4 / 36.0
    ((160, 12288, 2048), True), ((512, 12288, 2048), True), ((2560, 12288, 2048), True), ((256, 16384, 3072), True),  # 29.3 / 24.2, 41.8 / 34.4, 130.3 / 115.2, 48.1 / 41.1
    ((65, 28672, 5120), False), ((160, 28672, 5120), False), ((192, 28672, 5120), False), ((384, 28672, 5120), False),  # 72.1 / 83.0, 82.5 / 97.0, 90.5 / 96.3, 122.1 / 135.2
    ((512, 28672, 5120), True), ((1792, 28672, 5120), True), ((256, 20480, 6144), True), ((128, 20480, 6144), False),  # 162.0 / 140.8, 549.4 / 446.4, 109.4 / 89.6, 76.5 / 83.3
    ((65, 22016, 4096), False), ((128, 28672, 4096), False), ((320, 28672, 4096), False), ((1280, 28672, 4096), True),  # 52.0 / 56.8, 63.6 / 71.7, 94.7 / 105.2, 302.4 / 260.3
    ((128, 57344, 8192), False), ((320, 57344, 8192), False), ((1536, 57344, 8192), False), ((320, 28672, 8192), False),  # 228 / 259, 336 / 415, 1,101 / 1,216, 171 / 209
]


@pytest.mark.parametrize("size,wide", MEASURED)
def test_the_faster_kernel_is_taken(size, wide):
    rows, n, k = size
    choice = ops.product_by_rules(rows, n, k, k, tiled=True, fused=True, partials_ok=False)
    assert (choice.kernel == "wide") == wide


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


@pytest.mark.parametrize("rows,n,k,fused,kernel", [
    (1000, 2560, 4096, False, "library_parts"),      # 29.5 us / gemm_wide's two parts 30.9
    (6272, 2560, 4096, False, "library"), (6400, 2560, 9728, False, "library"),     # 95.8 / 120.5, 208 / 261
    (6272, 5120, 8192, False, "library"), (6400, 5120, 25600, False, "library"),    # 341 / 449, 1,086 / 1,417
    (6410, 2560, 4096, False, "wide"), (6410, 2560, 9728, False, "wide"),           # 117.7 / 118.2, 267 / 262
    (6410, 5120, 8192, False, "wide"), (6410, 5120, 25600, False, "wide"),          # 578 / 423, 1,830 / 1,363
    (6400, 19456, 2560, True, "wide"), (6500, 19456, 2560, True, "library"), (6657, 19456, 2560, True, "wide"),   # 611 / 531, 540 / 558
    (6272, 24576, 4096, True, "library"), (6410, 24576, 4096, True, "wide"),        # 979 / 1,003, 1,135 / 1,026
])
def test_the_shipped_tables_have_their_lines_where_the_kernels_cross(rows, n, k, fused, kernel):
    """The library's 256 x 256 workgroups fill a last turn up to 6,400 rows (25 row blocks) of these widths."""
    import glob
    import os

    keep = dict(ops._PRODUCT_TABLE)
    try:
        for path in glob.glob(os.path.join(ops.PRODUCT_TABLE_DIR, "*.json")):
            ops.load_product_table(path)
        assert ops.choose_product(rows, n, k, k, tiled=True, fused=fused, partials_ok=True).kernel == kernel
    finally:
        ops._PRODUCT_TABLE.clear()
        ops._PRODUCT_TABLE.update(keep)


def test_operands_off_its_grid_do_not_go_to_it():
    """Weights that begin between two multiples of 16 bytes, or rows of x too far apart: the rules without gemm_wide."""
    widths = (6144, 1024)
    table = {"6144,1024,1,1": [[4096, "wide", [], 0]], "6144,1024,0,1": [[4096, "wide", [], 2]]}
    keep = dict(ops._PRODUCT_TABLE)
    try:
        for fused in (True, False):
            ops._PRODUCT_TABLE.clear()
            by_rules = ops.choose_product(300, *widths, 1024, tiled=True, fused=fused, partials_ok=True, w_aligned=False).kernel
            ops.load_product_table(table)
            on_grid = dict(tiled=True, fused=fused, partials_ok=True)
            assert ops.choose_product(300, *widths, 1024, **on_grid).kernel == "wide" != by_rules
            assert ops.choose_product(300, *widths, 1024, w_aligned=False, **on_grid).kernel == by_rules
            assert ops.choose_product(300, *widths, 1 << 20, **on_grid).kernel != "wide"
    finally:
        ops._PRODUCT_TABLE.clear()
        ops._PRODUCT_TABLE.update(keep)


def test_calls_look_where_their_weights_lie(monkeypatch):
    """gate_up_act and gemm_bf16 with a contiguous view that begins two bytes into its storage, and gate_up_act with rows of
    w further apart than K: none of them goes to gemm_wide (the last is then refused, as it was)."""
    import torch

    chosen = []
    monkeypatch.setattr(ops, "_gpu", lambda *tensors: None)
    monkeypatch.setattr(ops, "run_product", lambda choice, *args, **kw: chosen.append(choice.kernel))
    monkeypatch.setattr(ops, "_PRODUCT_TABLE", {(4096, 512, False, False): [(4096, ops.ProductChoice("wide", (), 1))]})
    x = torch.zeros(200, 512, dtype=torch.bfloat16)
    store = torch.zeros(4096 * 520 + 16, dtype=torch.bfloat16)
    first = next(i for i in range(8) if store[i:].data_ptr() % 16 == 0)
    straight, shifted = (store[first + i:first + i + 4096 * 512].view(4096, 512) for i in (0, 1))
    apart = store[first:first + 4096 * 520].view(4096, 520)[:, :512]
    for w in (straight, shifted, apart):
        ops.gate_up_act(x, w)
    for w in (straight, shifted):
        ops.gemm_bf16(x, w)
    assert chosen[0] == chosen[3] == "wide" and "wide" not in (chosen[1], chosen[2], chosen[4])
