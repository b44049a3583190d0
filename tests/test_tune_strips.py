"""A table that is measured or shipped does not undo what steps of up to eight rows gain where a projection, its add and its norm are one
kernel: that takes a reader in gemm_rows."""
import pytest

from arle_amd.kernels import ops, tune

ROWS, WIDE, LIBRARY = ops.ProductChoice("rows"), ops.ProductChoice("wide", (64, 64), 1), ops.ProductChoice("library")


def test_another_kernel_pays_for_the_norm_in_front():
    timed = {ROWS: 20e-6, WIDE: 17e-6, LIBRARY: 30e-6}
    assert tune.pick(timed, ROWS) == WIDE
    assert tune.pick(timed, ROWS, apart=3.5e-6) == ROWS
    assert tune.pick(timed, LIBRARY, apart=3.5e-6) == ROWS
    assert tune.pick({ROWS: 40e-6, WIDE: 20e-6}, ROWS, apart=3.5e-6) == WIDE       # far ahead all the same


def test_what_does_not_win_clearly_does_not_replace_the_rule():
    assert tune.pick({ROWS: 20e-6, WIDE: 19e-6}, ROWS) == ROWS and tune.pick({ROWS: 20e-6, WIDE: 19e-6}, WIDE) == WIDE


@pytest.mark.parametrize("hidden,q,kv,inter", [(2560, 4096, 1024, 9728), (4096, 4096, 1024, 12288)])
@pytest.mark.parametrize("rows", range(1, ops.STRIP_ROWS + 1))
def test_the_shipped_tables_read_scaled_rows(hidden, q, kv, inter, rows):
    assert len(tune.model_strips(hidden, q, kv, inter)) == 2
    for (n, k, fused), front in tune.model_strips(hidden, q, kv, inter).items():
        assert (n, k, fused, True) in ops._PRODUCT_TABLE and ops.strips_preferred(*front)
        assert ops.takes_scaled(rows, n, k, tiled=True, fused=fused)
