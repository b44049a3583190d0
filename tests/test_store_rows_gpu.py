"""`ops.qkv_norm_store` for steps of many rows (heads of 64, 128 and 256 elements in 16-byte accesses, values turned through
LDS) against the same in 64 bits: whole pages, requests that begin inside a page or a workgroup's rows, remainders, other
page sizes, q alone.  Outputs are bfloat16: half a unit in the last place, 2^-9 of the value."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,nq,nkv", [(64, 6, 2), (128, 5, 3), (256, 4, 1), (128, 4, 0)])
@pytest.mark.parametrize("spans,page", [([(0, 96)], 16), ([(0, 113)], 16), ([(3, 40), (16, 63), (31, 1)], 16), ([(0, 48), (32, 70)], 32), ([(5, 97)], 8)])
@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32, None])
def test_norms_and_pages(D, nq, nkv, spans, page, weights):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(D + nq + len(spans))
    T, per = sum(n for _, n in spans), 16
    y = torch.randn(T, (nq + 2 * nkv) * D, generator=gen, device="cuda").bfloat16()
    wq, wk = (None, None) if weights is None else (torch.randn(2, D, generator=gen, device="cuda").to(weights)).unbind(0)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    positions = [p for first, n in spans for p in range(first, first + n)]
    slots = [s for s, (_, n) in enumerate(spans) for _ in range(n)]
    table = torch.randperm(len(spans) * per, generator=torch.Generator().manual_seed(1)).view(len(spans), per).tolist()
    k_pages = torch.full((len(spans) * per, max(nkv, 1), page, D), 7.0, device="cuda").bfloat16()
    v_pages = torch.full((len(spans) * per, max(nkv, 1), D, page), 7.0, device="cuda").bfloat16()
    got = y.clone()
    q, k, v = got[:, :nq * D], got[:, nq * D:(nq + nkv) * D], got[:, (nq + nkv) * D:]
    extra = dict(slot_of_token=i32(slots), block_table=i32(table), k_pages=k_pages, v_pages=v_pages, page_size=page) if nkv else {}
    ops.qkv_norm_store(q, k if nkv else None, v if nkv else None, num_q_heads=nq, num_kv_heads=nkv, key_dim=D, value_dim=D, eps=1e-5,
                       q_weight=wq, k_weight=wk, temp_coef=0.3, temp_every=7, positions=i32(positions), **extra)

    def normed(t, heads, w):
        t = t.double().view(T, heads, D)
        t = t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5)
        return t if w is None else t * w.double()

    near = lambda a, b: torch.allclose(a.double(), b, rtol=2.0 ** -8, atol=1e-6)
    temp = 1 + 0.3 * torch.log(torch.floor((torch.tensor(positions, device="cuda").double() + 1) / 7) + 1)
    assert near(q.view(T, nq, D), normed(y[:, :nq * D], nq, wq) * temp[:, None, None])
    assert torch.equal(got[:, nq * D:], y[:, nq * D:])
    want_k, want_v = k_pages.double().clone().fill_(7.0), v_pages.double().clone().fill_(7.0)
    if nkv:
        kn, vn = normed(y[:, nq * D:(nq + nkv) * D], nkv, wk), y[:, (nq + nkv) * D:].double().view(T, nkv, D)
        for t, (p, s) in enumerate(zip(positions, slots)):
            want_k[table[s][p // page], :, p % page] = kn[t]
            want_v[table[s][p // page], :, :, p % page] = vn[t]
    assert near(k_pages, want_k) and torch.equal(v_pages.double(), want_v)


@pytest.mark.parametrize("D,Dv,nq,nkv", [(64, 36, 3, 1), (128, 128, 5, 3), (256, 8, 4, 1), (128, 128, 4, 0)])
@pytest.mark.parametrize("taps,parts", [(2, 0), (3, 1), (4, 4), (4, 9)])
def test_single_rows_with_the_convolution_in_front(D, Dv, nq, nkv, taps, parts):
    """`ops.conv_step_store` against `ops.conv_step` and the norm in 64 bits: the states and v bit for bit, q and k to half a unit in
    the last place of bfloat16, 2^-9 of the value, 2^-8 stated; other requests' states and pages stay as they are."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(D + taps)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    slots, positions, page = [4, 0, 2], [37, 0, 15], 16
    T, C = len(slots), (nq + nkv) * D + nkv * Dv
    u = rand(parts, T, C) if parts else rand(T, C).bfloat16()
    w, state, bias = rand(C, taps).bfloat16(), rand(5, taps - 1, C).bfloat16(), rand(C).bfloat16() if taps == 4 else None
    wq, wk = rand(2, D).bfloat16().unbind(0) if taps != 3 else (None, None)
    table = torch.randperm(20, generator=torch.Generator().manual_seed(1)).view(5, 4).tolist()
    k_pages, v_pages = rand(20, max(nkv, 1), page, D).bfloat16(), rand(20, max(nkv, 1), Dv, page).bfloat16()
    want_state, want_k, want_v = state.clone(), k_pages.double(), v_pages.clone()
    y = ops.conv_step(u, w, want_state, i32(slots), bias=bias)
    extra = dict(block_table=i32(table), k_pages=k_pages, v_pages=v_pages, page_size=page) if nkv else {}
    q = ops.conv_step_store(u, w, state, i32(slots), bias=bias, num_q_heads=nq, num_kv_heads=nkv, key_dim=D, value_dim=Dv, eps=1e-5,
                            q_weight=wq, k_weight=wk, temp_coef=0.3, temp_every=7, positions=i32(positions), **extra)

    def normed(t, heads, weight):
        t = t.double().view(T, heads, D)
        t = t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5)
        return t if weight is None else t * weight.double()

    near = lambda a, b: torch.allclose(a.double(), b, rtol=2.0 ** -8, atol=1e-6)
    temp = 1 + 0.3 * torch.log(torch.floor((torch.tensor(positions, device="cuda").double() + 1) / 7) + 1)
    assert torch.equal(state, want_state)
    assert near(q.view(T, nq, D), normed(y[:, :nq * D], nq, wq) * temp[:, None, None])
    if nkv:
        kn, vn = normed(y[:, nq * D:(nq + nkv) * D], nkv, wk), y[:, (nq + nkv) * D:].view(T, nkv, Dv)
        for t, (p, s) in enumerate(zip(positions, slots)):
            want_k[table[s][p // page], :, p % page] = kn[t]
            want_v[table[s][p // page], :, :, p % page] = vn[t]
    assert near(k_pages, want_k) and torch.equal(v_pages, want_v)
    assert not ops.conv_step_store_supported(w, state, 96, Dv) and not ops.conv_step_store_supported(w.float(), state.float(), D, Dv)
