"""The merge of a decoded token's sums inside a workgroup treats every column alike: where the keys' values are the same in all columns
so is the result, bit for bit.  The waves' sums nearly cancel here, so that a product rounded in another place would show in bfloat16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("splits", [2, 4])
def test_columns_of_equal_values_come_out_equal(D, splits):
    from arle_amd.kernels import lib, ops

    T, nq, nkv, P, cached = 64, 32, 8, 16, 511
    g = torch.Generator().manual_seed(D + splits)
    pages = (cached + 1) // P
    table = torch.randperm(T * pages, generator=g).to(torch.int32).view(T, pages).to(DEV)
    k_pages = torch.randn(T * pages, nkv, P, D, generator=g).bfloat16().to(DEV)
    v_pages = torch.zeros(T * pages, nkv, D, P, dtype=torch.bfloat16, device=DEV)
    per_wave = (cached + 1) // splits // P       # pages of a wave's keys: values of 1 and of -1 in turn
    for page in range(pages):
        v_pages[table[:, page].long()] = 1.0 if (page // per_wave) % 2 == 0 else -1.0
    rows = torch.randn(T, (nq + 2 * nkv) * D, generator=g)
    rows[:, :nq * D] *= 0.01                     # scores near each other
    rows[:, (nq + nkv) * D:] = -1.0
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    out = torch.empty(T, nq * D, dtype=torch.bfloat16, device=DEV)
    try:
        lib.function("arle_attn_decode_inwg")(1)
        ops.attn_decode_prep(rows.bfloat16().to(DEV), out, k_pages, v_pages, table, i32(list(range(T + 1))), i32(list(range(T))),
                             i32([cached] * T), max_kv_len=cached + 1, eps=1e-6, splits=splits, num_q_heads=nq, num_kv_heads=nkv,
                             head_dim=D, page_size=P, scale=D ** -0.5)
    finally:
        lib.function("arle_attn_decode_inwg")(-1)
    out = out.cpu().view(T, nq, D)
    assert torch.isfinite(out.float()).all() and 0 < out.float().abs().mean() < 0.05
    assert torch.equal(out, out[:, :, :1].expand_as(out))
