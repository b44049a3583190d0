"""The product for prompt portions (`ops.gemm_wide`) in its workgroups of three to five stages, and with W as operand tiles:
fewer stages of K than the LDS holds, as many, one more and many more; row and column edges; parts of K; both against the
float64 product (bounds as in test_gemm_wide_gpu), and tiles against rows bit for bit (the same products in the same order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEEP = [(64, 64), (64, 96), (64, 128), (128, 64), (128, 96), (128, 128), (128, 160), (128, 192), (128, 256), (192, 128), (192, 192),
        (192, 256), (256, 128), (256, 160)]


def _rel(got, want):
    assert torch.isfinite(got.float()).all()
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("M,N,K", [(1, 32, 64), (65, 96, 128), (193, 416, 192), (64, 224, 256), (129, 288, 320), (9, 64, 384), (257, 160, 1088)])
def test_every_depth_of_k(M, N, K):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=gen, device="cuda").bfloat16()[:, :K]
    w = torch.randn(N, K, generator=gen, device="cuda").bfloat16()
    tiles = ops.pack_weight_tiles(w)
    want = x.double() @ w.double().T
    gate_up = want.view(M, -1, 2, 16)
    act = (torch.nn.functional.silu(gate_up[:, :, 0]) * gate_up[:, :, 1]).reshape(M, -1)
    for shape in DEEP:
        whole = ops.gemm_wide(x, w, torch.float32, shape=shape)
        assert _rel(whole, want) < 1e-5, shape
        assert torch.equal(whole, ops.gemm_wide(x, w, torch.float32, shape=shape, tiles=tiles)), shape
        fused = ops.gemm_wide(x, w, epilogue=ops.EPI_SILU_MUL, shape=shape)
        assert _rel(fused, act) < 2.0 ** -8, shape
        assert torch.equal(fused, ops.gemm_wide(x, w, epilogue=ops.EPI_SILU_MUL, shape=shape, tiles=tiles)), shape
        for parts in (2, 3):
            if parts <= K // 64:
                stack = ops.gemm_wide(x, w, torch.float32, shape=shape, splits=parts, tiles=tiles)
                assert stack.dim() == 3 and _rel(stack.sum(0), want) < 1e-5, (shape, parts)


@pytest.mark.parametrize("shape", [(128, 320), (256, 192), (256, 256), (192, 320), (256, 320)])
def test_tiles_where_lines_are_touched_ahead(shape):
    """Two stages: the touched lines lie elsewhere in tiles than in rows."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(300, 640, generator=gen, device="cuda").bfloat16()
    w = torch.randn(736, 640, generator=gen, device="cuda").bfloat16()
    tiles = ops.pack_weight_tiles(w)
    assert torch.equal(ops.gemm_wide(x, w, torch.float32, shape=shape), ops.gemm_wide(x, w, torch.float32, shape=shape, tiles=tiles))
    # a matrix whose tiles are the first of a larger one's
    q_only = w[:320]
    assert torch.equal(ops.gemm_wide(x, q_only, shape=shape), ops.gemm_wide(x, q_only, shape=shape, tiles=tiles))
    with pytest.raises(ops.ShapeError):
        ops.gemm_wide(x, w, shape=shape, tiles=tiles[:20])
