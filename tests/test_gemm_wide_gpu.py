"""The product for prompt portions with both operands through LDS (`ops.gemm_wide`): every workgroup shape at one row and
column block and over their edges, strided rows, one to more stages of K than the LDS holds, parts of K, both output types,
the activation; against the float64 product.  bfloat16 operands are exact in float32, a sum of K terms in float32 is off
by at most K 2^-24 of the terms' absolute sum (1e-5 in relative norm here), a bfloat16 result by 2^-9 more."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SHAPES = [(128, 64), (128, 96), (128, 128), (128, 160), (128, 192), (128, 256), (128, 320), (256, 160), (256, 192), (256, 256),
          (192, 320), (256, 320)]


def _operands(M, N, K, seed, pad_x=0, pad_w=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    make = lambda r, c, pad: torch.randn(r, c + pad, generator=gen, device="cuda").bfloat16()[:, :c]
    return make(M, K, pad_x), make(N, K, pad_w)


def _rel(got, want):
    assert torch.isfinite(got.float()).all()
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("M,N,K,pad_x,pad_w", [(1, 32, 64, 0, 0), (33, 96, 128, 8, 0), (127, 352, 192, 0, 64), (256, 320, 256, 0, 0),
                                                (257, 672, 320, 24, 8), (300, 1952, 1088, 0, 0)])
def test_every_shape_over_its_edges(shape, M, N, K, pad_x, pad_w):
    from arle_amd.kernels import ops

    x, w = _operands(M, N, K, M + N, pad_x, pad_w)
    want = x.double() @ w.double().T
    assert _rel(ops.gemm_wide(x, w, torch.float32, shape=shape), want) < 1e-5
    assert _rel(ops.gemm_wide(x, w, shape=shape), want) < 2.0 ** -8
    gate_up = want.view(M, -1, 2, 16)
    act = (torch.nn.functional.silu(gate_up[:, :, 0]) * gate_up[:, :, 1]).reshape(M, -1)
    assert _rel(ops.gemm_wide(x, w, epilogue=ops.EPI_SILU_MUL, shape=shape), act) < 2.0 ** -8
    for parts in (2, 3, 5):
        if parts <= K // 64:
            stack = ops.gemm_wide(x, w, torch.float32, shape=shape, splits=parts)
            assert stack.dim() == 3 and _rel(stack.sum(0), want) < 1e-5


def test_the_activation_at_the_ends_of_its_range():
    """Gates far below and above zero: silu goes to -0 and to the gate itself, and no product with an infinity inside."""
    from arle_amd.kernels import ops

    gates = torch.tensor([-300.0, -100.0, -88.0, -20.0, -1.0, -0.0, 0.0, 1e-20, 1.0, 20.0, 90.0, 300.0, 3e4, -3e4, 5.0, -5.0])
    x = torch.zeros(1, 64, dtype=torch.bfloat16, device="cuda")
    x[0, 0] = 1.0
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device="cuda")
    w[:16, 0], w[16:, 0] = gates.bfloat16().cuda(), 2.0
    got = ops.gemm_wide(x, w, epilogue=ops.EPI_SILU_MUL)[0].double().cpu()
    want = (torch.nn.functional.silu(gates.bfloat16().double()) * 2).bfloat16().double()
    assert torch.isfinite(got).all() and torch.allclose(got, want, rtol=2.0 ** -8, atol=1e-30)


@pytest.mark.parametrize("rows", [65, 97, 300, 1153, 2048])
def test_gate_up_takes_it_by_the_rule_and_the_plan_fits(rows):
    from arle_amd.kernels import ops

    n, k = 6144, 512
    x, w = _operands(rows, n, k, rows)
    assert ops.choose_product(rows, n, k, k, tiled=False, fused=True, partials_ok=False).kernel == "wide"
    want = (x.double() @ w.double().T).view(rows, -1, 2, 16)
    want = (torch.nn.functional.silu(want[:, :, 0]) * want[:, :, 1]).reshape(rows, -1)
    assert _rel(ops.gate_up_act(x, w), want) < 2.0 ** -8


def test_what_it_does_not_take_goes_elsewhere():
    from arle_amd.kernels import ops

    for n, k, x_stride in ((6144, 544, 544), (6144 + 16, 512, 512), (6144, 512, 516)):
        assert not ops.gemm_wide_supported(n, k, x_stride)
    x, w = _operands(100, 6144, 544, 1)
    with pytest.raises(ops.ShapeError):
        ops.gemm_wide(x, w)
    want = (x.double() @ w.double().T).view(100, -1, 2, 16)
    want = (torch.nn.functional.silu(want[:, :, 0]) * want[:, :, 1]).reshape(100, -1)
    assert _rel(ops.gate_up_act(x, w), want) < 2e-2


@pytest.mark.parametrize("base,shape", [(-76, (128, 64)), (-50, (256, 320)), (-24, (128, 192)), (-9, (128, 320)), (2, (192, 320))])
def test_the_activation_keeps_the_error_of_a_whole_exponential_and_division(base, shape):
    """Gates that a float holds exactly, base + i / 1,024 up to base + 15.8, and ups of 1: the result is silu rounded to
    bfloat16, and it rounds the other way than the 64-bit silu where that lies within the 32-bit error of a middle between
    two bfloat16 numbers.  An error of e ulp in the mean does so for a share of e 2^-16 to 2 e 2^-16 of the values; expf and
    a division have 0.3 to 0.45 (1.4e-5 at most), the exponential and the reciprocal of the vector unit 3 to 15 below -5."""
    from arle_amd.kernels import ops

    rows, n = 128, 8192
    x = torch.zeros(rows, 64, device="cuda")
    x[:, 0], x[:, 1] = 1.0, torch.arange(rows, device="cuda") % 128
    w = torch.zeros(n // 32, 2, 16, 64, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(4)
    w[:, 0, :, 0] = base
    w[:, 0, :, 1] = torch.randint(0, 128, (n // 32, 16), device="cuda", generator=g) / 1024
    w[:, 1, :, 0] = 1.0
    x, w = x.bfloat16(), w.reshape(n, 64).bfloat16()
    gate = (x.double() @ w.view(n // 32, 2, 16, 64)[:, 0].reshape(-1, 64).double().T)
    want = (gate / (1 + torch.exp(-gate))).bfloat16()
    got = ops.gemm_wide(x, w, epilogue=ops.EPI_SILU_MUL, shape=shape)
    assert float((got != want).double().mean()) < 4e-5


def test_the_activation_below_where_the_reciprocal_leaves_the_floats():
    """exp(-x) from 2^126 on: the reciprocal of 1 + exp(-x) is no normal number, the result is one."""
    from arle_amd.kernels import ops

    gates = torch.tensor([-79.5, -80.0, -80.5, -87.0, -87.5, -88.0, -88.5, -100.0, 79.5, 80.0, 88.5, 3e38, float("inf"), float("nan"), 1.0, -1.0])
    x = torch.zeros(3, 64, dtype=torch.bfloat16, device="cuda")
    x[:, 0] = 1.0
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device="cuda")
    w[:16, 0], w[16:, 0] = gates.bfloat16().cuda(), 2.0
    got = ops.gemm_wide(x, w, epilogue=ops.EPI_SILU_MUL).float().cpu()
    exact = gates.bfloat16().double()
    want = (exact / (1 + torch.exp(-exact)) * 2).float()
    for row in got:
        assert torch.isnan(row[13]) and float(row[12]) == float("inf")
        keep = [i for i in range(16) if i not in (11, 12, 13)]
        assert torch.allclose(row[keep], want[keep], rtol=2.0 ** -8, atol=1e-38) and float(row[11]) == float("inf")


@pytest.mark.parametrize("shape,row_blocks,col_blocks", [((128, 64), 9, 8), ((128, 64), 10, 22), ((128, 96), 13, 33), ((128, 320), 17, 3),
                                                         ((256, 160), 10, 9), ((256, 256), 16, 41), ((192, 320), 11, 10), ((256, 320), 9, 40)])
def test_blocks_of_several_patches(shape, row_blocks, col_blocks):
    """More row blocks than a patch has, in numbers that eight does not divide, and column blocks to match: every block is
    somebody's, the last ones in part."""
    from arle_amd.kernels import ops

    M, N = shape[0] * row_blocks - 37, shape[1] * col_blocks - 32
    x, w = _operands(M, N, 128, row_blocks)
    want = x.double() @ w.double().T
    assert _rel(ops.gemm_wide(x, w, shape=shape), want) < 2.0 ** -8
    stack = ops.gemm_wide(x, w, torch.float32, shape=shape, splits=2)
    assert _rel(stack.sum(0), want) < 1e-5


@pytest.mark.parametrize("shape", [(128, 64), (192, 320), (256, 320)])
@pytest.mark.parametrize("scale", [79.875, 80.0, 300.0])
def test_one_wave_with_gates_beyond_the_short_form(shape, scale):
    """Gates of two rows reach `scale` with either sign, all others stay within 1: their waves take the whole exponential and
    division from 80 on, beside waves that do not.  Both forms are off by 3 ulp of a float at most, so every result is the
    64-bit one rounded to bfloat16, or its neighbour where that lies at a middle.  exp(-x) of a float is infinite from 2^128
    (x below -88.72) on, where the result is -0 instead of x / (1 + exp(-x)), 89 2^-128 at most."""
    from arle_amd.kernels import ops

    M, n = 300, 640
    x = torch.zeros(M, 64, dtype=torch.bfloat16, device="cuda")
    x[:, 0] = torch.linspace(-1, 1, M, device="cuda").bfloat16()
    x[37, 0], x[290, 0] = scale, -scale
    w = torch.zeros(n // 32, 2, 16, 64, dtype=torch.bfloat16, device="cuda")
    w[:, 0, :, 0] = torch.linspace(0.0625, 1, n // 2, device="cuda").bfloat16().view(n // 32, 16)
    x[:, 1], w[:, 1, :, 1] = 1.0, 1.0
    gate = x[:, :1].double() @ w[:, 0, :, 0].reshape(1, -1).double()
    want = gate / (1 + torch.exp(-gate))
    got = ops.gemm_wide(x, w.reshape(n, 64), epilogue=ops.EPI_SILU_MUL, shape=shape).double()
    assert torch.allclose(got, want, rtol=2.0 ** -8 * (1 + 2.0 ** -10), atol=89 * 2.0 ** -128)
