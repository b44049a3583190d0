"""How many parts of a stack the norms fetch together, by width and rows: the rule, and the same bits on both sides of it."""
import pytest
import torch

from arle_amd.kernels import lib

F32, BF16 = 0, 1


def _ahead(width, rows, parts, taps=0, dtype=BF16):
    return lib.function("arle_layernorm_parts_ahead")(width, rows, parts, taps, dtype)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("width,most", [(512, 768), (1024, 768), (1028, 384), (2048, 384), (2052, 256), (2560, 256), (2564, 256), (4096, 256)])
def test_many_rows_take_one_term_after_the_other(width, most, dtype):
    for parts in (3, 8):
        assert _ahead(width, 1, parts, dtype=dtype) == _ahead(width, most, parts, dtype=dtype) == 8
        assert _ahead(width, most + 1, parts, dtype=dtype) == _ahead(width, 1 << 20, parts, dtype=dtype) == 0
    assert _ahead(width, 1, 9, dtype=dtype) == 0


@pytest.mark.parametrize("width", [256, 2560, 4096, 5120, 8192])
def test_terms_of_two_parts_are_fetched_together_whatever_the_rows(width):
    # (8,192 columns of 2,048 rows and more in bfloat16 have eight groups a lane)
    for rows in (1, 300, 2047, 1 << 20):
        assert _ahead(width, rows, 0, dtype=F32) == _ahead(width, rows, 2, dtype=F32) == 2
        assert _ahead(width, rows, 2) == (0 if width == 8192 and rows >= 2048 else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,most", [(1024, 768), (2048, 384), (2560, 256), (4096, 256)])
def test_rows_are_the_same_bits_on_both_sides_of_the_line(width, most, dtype):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    rows = most + 1
    residual, weight = rand(rows, width), rand(width).to(dtype)
    terms = [(rand(3, rows, width), rand(width).to(dtype)), (rand(8, rows, width), None)]
    part = [(t[:, 1:].contiguous(), b) for t, b in terms]
    sums, few = residual.clone(), residual[1:].clone()
    whole, less = ops.add_layernorm(sums, terms, weight, 1e-6, dtype), ops.add_layernorm(few, part, weight, 1e-6, dtype)
    assert torch.equal(whole[1:], less) and torch.equal(sums[1:], few)
    plain = torch.nn.functional.layer_norm(
        residual.double() + (terms[0][0].double().sum(0) + terms[0][1].double()) + terms[1][0].double().sum(0), (width,), weight.double(), eps=1e-6)
    # sums of twelve terms in 32 bits, a mean and a variance over them; a bfloat16 output is off by half a unit of its eight bits
    limit = 2e-6 if dtype == torch.float32 else 2.0 ** -8
    assert ((whole.double() - plain).abs() <= limit * (plain.abs() + 1)).all()


def test_wide_rows():
    assert _ahead(5120, 1 << 20, 8) == 8 and _ahead(5120, 1, 8, dtype=F32) == 0      # eight float32 parts would spill there
    assert _ahead(5120, 1, 8, taps=4) == 0 and _ahead(8192, 1, 8) == 0 and _ahead(8192, 1, 2, taps=4) == 0
    assert _ahead(16384, 1, 1) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("width", [1024, 2560, 4096])
@pytest.mark.parametrize("parts", [7, 8, 9, 17])
def test_rms_rows_are_the_same_bits_on_both_sides_of_the_line(width, parts):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width + parts)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    residual, stack, weight = rand(513, width), rand(parts, 513, width), rand(width)
    sums, few = residual.clone(), residual[1:].clone()
    whole = ops.add_rmsnorm(sums, stack, weight, 1e-6, torch.float32)
    less = ops.add_rmsnorm(few, stack[:, 1:].contiguous(), weight, 1e-6, torch.float32)
    assert torch.equal(whole[1:], less) and torch.equal(sums[1:], few)
    plain = residual.double() + stack.double().sum(0)
    plain = plain / (plain.square().mean(-1, keepdim=True) + 1e-6).sqrt() * weight.double()
    # a sum of up to eighteen terms in 32 bits, and a sum of squares over the row
    assert ((whole.double() - plain).abs() <= 2e-6 * (plain.abs() + 1)).all()
