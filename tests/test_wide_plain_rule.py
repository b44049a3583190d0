"""Which plain products without a table run whole in `ops.gemm_wide` (host only), and that the plan knows each shape's rows."""
import pytest

from arle_amd.kernels import ops

# (rows, N, K), and whether gemm_wide was faster (us on MI355X, the other rules / gemm_wide)
MEASURED = [
    ((9, 9728, 2560), True), ((64, 9728, 2560), True), ((256, 9728, 2560), True), ((1024, 9728, 2560), True),   # 15.2 / 14.8, 19.5 / 17.3, 38.4 / 26.3, 56.1 / 47.7
    ((2048, 10240, 2560), True), ((4096, 9728, 2560), True), ((1536, 12288, 3072), True),                       # 110 / 90, 191 / 170, 123 / 99
    ((1536, 9728, 2560), False), ((2048, 8192, 2048), False), ((3072, 9728, 2560), False),                      # 63 / 69, 55 / 62, 125 / 132
    ((9, 4096, 2560), False), ((112, 4096, 2560), False), ((2560, 4096, 1024), False), ((8, 9728, 2560), False),  # 10.2 / 12.1, 12.4 / 13.7, 27.8 / 28.7
]


@pytest.mark.parametrize("size,wide", MEASURED)
def test_the_faster_kernel_is_taken(size, wide):
    rows, n, k = size
    for tiled in (False, True):
        choice = ops.product_by_rules(rows, n, k, k, tiled=tiled, fused=False, partials_ok=False)
        assert (choice.kernel == "wide") == wide
    if wide:      # operands off the 16-byte grid keep the kernel they had
        for off in (dict(aligned=False), dict(w_aligned=False)):
            assert ops.product_by_rules(rows, n, k, k, tiled=True, fused=False, partials_ok=False, **off).kernel != "wide"


@pytest.mark.parametrize("rows", [9, 16, 40, 64])
def test_sums_that_may_stay_in_parts_stay_unrounded(rows):
    """A consumer that adds 32-bit parts itself goes on getting them where the kernels of few rows left them."""
    with_parts = ops.product_by_rules(rows, 8192, 2048, 2048, tiled=True, fused=False, partials_ok=True)
    assert with_parts.kernel in ("rows", "stream")


@pytest.mark.parametrize("k", [2048, 2560, 3072, 4096, 5120])
def test_sums_that_the_library_would_leave_in_parts_stay_unrounded(k):
    """o and down at 5,120 columns (no table names them): rounded to bfloat16 they would go into the 32-bit residual with fewer bits."""
    for rows in (65, 66, 97, 128, 192, 255, 256, 257, 384, 512, 513, 768, 1000, 1024):
        assert ops.library_k_splits(rows, 5120, k) > 1
        for tiled in (False, True):
            choice = ops.choose_product(rows, 5120, k, k, tiled=tiled, fused=False, partials_ok=True)
            assert choice.kernel in ("wide", "library_parts") and choice.splits > 1
            assert ops.product_by_rules(rows, 5120, k, k, tiled=tiled, fused=False, partials_ok=False) == ops.ProductChoice("wide", (), 1)
            off = ops.product_by_rules(rows, 5120, k, k, tiled=tiled, fused=False, partials_ok=True, w_aligned=False)
            assert off.kernel == "library_parts"


@pytest.mark.parametrize("rows,n,k", [(9, 6144, 2560), (64, 2560, 9728), (256, 4096, 2560), (257, 4096, 2560), (1024, 6144, 4096),
                                      (1025, 6144, 4096), (8192, 19456, 2560)])
def test_shapes_stay_within_their_rows(rows, n, k):
    for parts in (1, 4):
        shapes = [shape for shape, _ in ops.wide_shapes(rows, n, k, parts)]
        assert ops.wide_plan(rows, n, k, parts)[0] == shapes[0] and len(set(shapes)) == len(shapes)
        assert ((64, 64) in shapes) == (rows <= 256) and ((192, 192) in shapes) == (rows <= 1024) and (256, 320) in shapes
