"""What comes with rows that a product still has to divide is looked at before anything is launched: the kernel reads whole rows of sums;
and which matrices leave such rows."""
import pytest
import torch

from arle_amd.kernels import ops

M, K = 3, 64


def _scaled(sums, count=4, rows=None, width=K):
    return ops.ScaledRows(torch.zeros(M, K, dtype=torch.bfloat16) if rows is None else rows, sums, count, width, 1e-6)


@pytest.mark.parametrize("sums,count", [
    (torch.zeros(M, 255), 4), (torch.zeros(M, 512), 4), (torch.zeros(M - 1, 256), 4), (torch.zeros(M * 256), 4),
    (torch.zeros(M, 256, dtype=torch.float64), 4), (torch.zeros(M, 256, dtype=torch.bfloat16), 4), (torch.zeros(256, M).T, 4),
    (torch.zeros(M, 512)[:, :256], 4), (torch.zeros(M * 256 + 1)[1:].view(M, 256), 4), (torch.zeros(M, 256), 0), (torch.zeros(M, 256), 257)])
def test_sums_that_the_kernel_could_not_read_are_refused(sums, count):
    scaled = _scaled(sums, count)
    with pytest.raises(ops.ShapeError, match="the sums of scaled rows"):
        ops.gemm_rows(scaled.rows, torch.zeros(16, K, dtype=torch.bfloat16), scaled=scaled)


def test_sums_of_other_rows_are_refused():
    w = torch.zeros(16, K, dtype=torch.bfloat16)
    scaled = _scaled(torch.zeros(M, 256))
    with pytest.raises(ops.ShapeError, match="those that the sums are of"):
        ops.gemm_rows(scaled.rows.clone(), w, scaled=scaled)
    for wrong in (_scaled(torch.zeros(M, 256), width=K - 1), _scaled(torch.zeros(9, 256), rows=torch.zeros(9, K, dtype=torch.bfloat16))):
        with pytest.raises(ops.ShapeError, match="those that the sums are of"):
            ops.gemm_rows(wrong.rows, w, scaled=wrong)
    with pytest.raises(ops.ShapeError, match="GPU only"):      # whole ones go on to what every call needs
        ops.gemm_rows(scaled.rows, w, scaled=scaled)


@pytest.mark.parametrize("n,k,columns,preferred", [
    (1024, 64, 4, True), (1024, 8192, 4, True), (1024, 8256, 4, False), (1024, 10240, 4, False), (1025, 8256, 5, True), (1280, 10240, 5, True),
    (1280, 10304, 5, False), (1792, 10240, 7, True), (1792, 12288, 7, False), (1793, 12288, 8, True), (2048, 24576, 8, True),
    (2560, 9728, 10, True), (2560, 32768, 10, True), (4096, 12288, 16, True), (4096, 32768, 16, True), (4097, 4096, 0, False),
    (768, 4096, 0, False), (769, 4096, 4, True), (2560, 96, 0, False), (2560, 32, 0, False)])
def test_which_matrices_are_cut_into_strips(n, k, columns, preferred):
    """Narrow strips only up to the K that was measured ahead of the product with the norm behind it."""
    assert (ops.strip_columns(n, k), ops.strips_preferred(n, k)) == (columns, preferred)
