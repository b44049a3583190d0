"""Kernels of steps in which every request brings one row: the convolution with its state (`ops.conv_step`) and PolyNorm of a
stack against the kernels that they stand for, bit for bit (the same sums in the same order, stacks rounded as the kernel that
adds them does), and alike for the layer norm with the convolution behind it; the mLSTM in one kernel (`ops.mlstm_decode`) against the 64-bit recurrence (bounds as in
test_mlstm_chunks_gpu); the layer norm at the edges of its workgroups' widths (two 32-bit passes: 1e-5), and it and PolyNorm in
steps of many rows, where a float32 row keeps its bits."""
import pytest
import torch

from test_mlstm_chunks_gpu import _case, _recurrence, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps,channels,rows", [(2, 4, 1), (3, 1020, 3), (4, 1028, 8), (4, 2560, 70)])
@pytest.mark.parametrize("biased,flags", [(False, {}), (True, dict(add_input=True)), (True, dict(silu=True))])
def test_the_convolution_and_its_state(dtype, taps, channels, rows, biased, flags):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(taps + channels)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    u, w, state = rand(rows, channels + 8)[:, :channels], rand(channels, taps), rand(rows + 2, taps - 1, channels)
    bias, out_bias = (rand(channels), rand(channels)) if biased else (None, None)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    slots = i32([rows + 1 - r for r in range(rows)])
    stack = torch.randn(3, rows, channels, generator=gen, device="cuda")
    for given, parts in ((u, None), (ops.sum_partials(stack, dtype), stack)):
        want_state, got_state = state.clone(), state.clone()
        want = ops.causal_conv(given, w, want_state, slots, bias=bias, out_bias=out_bias, **flags)
        ops.conv_state_update(given, want_state, i32(list(range(rows + 1))), slots, bias=bias)
        got = ops.conv_step(given if parts is None else parts, w, got_state, slots, bias=bias, out_bias=out_bias, **flags)
        assert torch.equal(got, want) and torch.equal(got_state, want_state)
    assert not ops.conv_step_supported(rand(channels, 5), state) and not ops.conv_step_supported(rand(6, 4), state)
    with pytest.raises(ops.ShapeError):
        ops.conv_step(u, w, state[:, :, :-4], slots)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [4, 2044, 2048, 2052, 4100, 9728, 10244, 14340, 24576])
def test_polynorm_of_a_stack(dtype, width):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width)
    stack = torch.randn(3, 5, width, generator=gen, device="cuda")
    coef, bias = torch.randn(4, generator=gen, device="cuda").to(dtype), torch.randn(width, generator=gen, device="cuda").to(dtype)
    whole = ops.sum_partials(stack, dtype)
    for b in (None, bias):
        got = ops.polynorm(stack, coef, 1e-6, bias=b, out_dtype=dtype)
        assert torch.equal(got, ops.polynorm(whole, coef, 1e-6, bias=b))
        z = whole.double() + (0 if b is None else b.double())
        n = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)
        c = coef.double()
        want = c[0] * n(z) + c[1] * n(z ** 2) + c[2] * n(z ** 3) + c[3]
        assert _rel(got, want) < (2.0 ** -8 if dtype == torch.bfloat16 else 1e-5)


@pytest.mark.parametrize("width", [2052, 4100, 6144, 8192, 8196])
def test_a_float32_row_of_polynorm_is_the_same_bits_in_any_step(width):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width)
    u, coef = torch.randn(1100, width, generator=gen, device="cuda"), torch.randn(4, generator=gen, device="cuda")
    whole = ops.polynorm(u, coef, 1e-6)
    pieces = [ops.polynorm(u[s].contiguous(), coef, 1e-6) for s in (slice(0, 1), slice(1, 9), slice(9, 1032), slice(1032, 1100))]
    assert torch.equal(torch.cat(pieces), whole)
    assert torch.equal(ops.polynorm(u[None, :64].contiguous(), coef, 1e-6, out_dtype=torch.float32), whole[:64])
    z, n = u.double(), lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)
    c = coef.double()
    assert _rel(whole, c[0] * n(z) + c[1] * n(z ** 2) + c[2] * n(z ** 3) + c[3]) < 1e-5


@pytest.mark.parametrize("rows", [256, 257, 1025])
@pytest.mark.parametrize("width", [4096, 4100, 8192, 8196])
def test_polynorm_of_many_bfloat16_rows(width, rows):
    """Both sides of the line between the workgroups; rounded once, half a unit in the last place: 2^-9 of a value, 2^-8 stated."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width + rows)
    u, coef = (torch.randn(*s, generator=gen, device="cuda").bfloat16() for s in ((rows, width), (4,)))
    z, c, n = u.double(), coef.double(), lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)
    assert _rel(ops.polynorm(u, coef, 1e-6), c[0] * n(z) + c[1] * n(z ** 2) + c[2] * n(z ** 3) + c[3]) < 2.0 ** -8


@pytest.mark.parametrize("rows,H,D,Dv,gate_std", [(1, 2, 128, 128, 1.0), (5, 3, 100, 64, 3.0), (9, 1, 32, 32, 20.0), (3, 2, 128, 32, 1.0), (2, 2, 7, 128, 1.0)])
def test_the_memory_in_one_kernel(rows, H, D, Dv, gate_std):
    from arle_amd.kernels import ops

    c = _case([1] * rows, H, D, Dv, gate_std, 7 + rows)
    want, states = _recurrence(c, H, D, Dv, 15.0)
    noise = torch.randn_like(c["qkvg"]) * 0.5
    wide = torch.cat([c["gates"], torch.zeros(rows, 16, device="cuda")], 1).contiguous()
    forms = [(c["qkvg"], c["gates"]), (torch.stack([c["qkvg"] - noise, noise]), torch.stack([wide * 0.25, wide * 0.5, wide * 0.25]))]
    whole = torch.stack([torch.cat([t, g], 1) for t, g in zip(forms[1][0], (wide * 0.25, wide * 0.75))])     # one product for both
    forms.append((whole, whole[..., c["qkvg"].shape[1]:]))
    for y, gates in forms:
        mine = [t.clone() for t in c["state"]]
        got = ops.mlstm_decode(y, gates, c["bi"], c["bf"], 15.0, *mine, c["row0"], c["slot"], c["weight"], 1e-6, torch.float32, heads=H,
                               key_dim=D, value_dim=Dv)
        assert _rel(got, want) < 2e-5
        for state, ref, before in zip(mine, states, c["state"]):
            assert _rel(state, ref) < 1e-6 and torch.equal(state[0], before[0])     # slot 0 belongs to nobody
    assert not ops.mlstm_decode_supported(160, 128, c["state"][0]) and not ops.mlstm_decode_supported(128, 96, c["state"][0])


@pytest.mark.parametrize("width", [1024, 1028, 2556, 2560, 2564, 4096, 4100, 5120, 5124, 8192, 8196, 16384])
@pytest.mark.parametrize("rows", [1, 300])
def test_layer_norm_at_the_edges_of_its_workgroups(width, rows):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    residual, stack, weight, bias = rand(rows, width) + 3, rand(3, rows, width), rand(width), rand(width)
    want = residual.double() + stack.double().sum(0) + bias.double()
    got = ops.add_layernorm(residual, [(stack, bias)], weight, 1e-6, torch.float32)
    assert _rel(residual, want) < 1e-6
    d = want - want.mean(-1, keepdim=True)
    assert _rel(got, d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-6) * weight.double()) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [1024, 2048, 2560, 4096, 5120, 8192, 8196])
def test_parts_of_both_terms_fetched_together(width, dtype):
    """As many parts as are fetched together, one less and one more, absent terms and biases.  A sum of n + 2 numbers in float32 is off
    by at most (n + 1) 2^-24 of the sum of their sizes: 1e-6 of the largest here; the outputs as in the tests beside this one."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    weight, other, bias, c = (rand(width).to(dtype) for _ in range(4))
    for parts in ((), (1,), (2,), (3,), (8,), (9,), (1, 1), (1, 2), (2, 1), (2, 2), (2, 3), (8, 1), (4, 6), (8, 8), (9, 1), (1, 9)):
        residual = rand(3, width) + 3
        terms = [(rand(n, 3, width), bias if n % 2 else None) for n in parts]
        want = residual.double() + sum((t.double().sum(0) + (0 if b is None else b.double()) for t, b in terms), torch.zeros_like(residual).double())
        a, b = ops.add_layernorm(residual, terms, weight, 1e-6, dtype, other, bias_b=c)
        d = want - want.mean(-1, keepdim=True)
        d = d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-6)
        assert _rel(residual, want) < 1e-6
        assert _rel(a, d * weight.double()) < (1e-5 if dtype == torch.float32 else 2.0 ** -8)
        assert _rel(b, d * other.double() + c.double()) < (1e-5 if dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("rows", [2047, 2048])
@pytest.mark.parametrize("width", [5124, 8192])
def test_layer_norm_of_many_bfloat16_rows(width, rows):
    """Both sides of the line between the workgroups; rounded once, half a unit in the last place: 2^-9 of a value, 2^-8 stated."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width + rows)
    residual, term = (torch.randn(rows, width, generator=gen, device="cuda") + 3 for _ in range(2))
    weight = torch.randn(width, generator=gen, device="cuda").bfloat16()
    want = residual.double() + term.double()
    got = ops.add_layernorm(residual, [(term, None)], weight, 1e-6, torch.bfloat16)
    d = want - want.mean(-1, keepdim=True)
    assert _rel(residual, want) < 1e-6
    assert _rel(got, d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-6) * weight.double()) < 2.0 ** -8


@pytest.mark.parametrize("width", [2052, 4100, 5120, 5124, 6144, 8192, 8196])
def test_a_float32_row_of_the_layer_norm_is_the_same_bits_in_any_step(width):
    from arle_amd.kernels import ops

    rows, taps = 1100, 3
    gen = torch.Generator(device="cuda").manual_seed(width)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    residual, term, weight = rand(rows, width) + 3, rand(rows, width), rand(width)
    at = [slice(0, 1), slice(1, 9), slice(9, 1032), slice(1032, 1100)]
    sums = residual.clone()
    whole = ops.add_layernorm(sums, [(term, None)], weight, 1e-6, torch.float32)
    pieces = [ops.add_layernorm(residual[s].clone(), [(term[s], None)], weight, 1e-6, torch.float32) for s in at]
    assert torch.equal(torch.cat(pieces), whole)
    d = residual.double() + term.double()
    d = d - d.mean(-1, keepdim=True)
    assert _rel(whole, d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-6) * weight.double()) < 1e-5
    w, state = rand(width, taps), rand(1100, taps - 1, width)
    slots = torch.arange(8, dtype=torch.int32, device="cuda")
    if ops.add_layernorm_conv_supported(residual, [(term, None)], weight, torch.float32, w, state):
        few = slice(0, 8)
        _, norm = ops.add_layernorm_conv(residual[few].clone(), [(term[few], None)], weight, 1e-6, torch.float32, w, state, slots)
        assert torch.equal(norm, whole[few])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width,rows,taps", [(4, 1, 2), (1024, 3, 4), (2044, 2, 3), (2560, 8, 4), (4100, 5, 4), (8192, 70, 2)])
@pytest.mark.parametrize("biased,both", [(False, False), (True, True), (True, False)])
def test_layer_norm_and_the_convolution_behind_it(dtype, width, rows, taps, biased, both):
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width + taps)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    typed = lambda *s: rand(*s).to(dtype)
    residual, weight, weight_b = rand(rows, width) + 3, typed(width), typed(width) if both else None
    terms = [(rand(3, rows, width), typed(width)), (rand(rows, width), None)] if biased else []
    bias, bias_b = typed(width) if biased else None, typed(width) if both else None
    w, state = typed(width, taps), typed(rows + 2, taps - 1, width)
    slots = torch.tensor([rows + 1 - r for r in range(rows)], dtype=torch.int32, device="cuda")
    res, got_state = residual.clone(), state.clone()
    out = ops.add_layernorm(residual, terms, weight, 1e-6, dtype, weight_b, bias=bias, bias_b=bias_b)
    norm, other = out if both else (out, out)
    want = ops.conv_step(norm, w, state, slots, add_input=True)
    got, got_other = ops.add_layernorm_conv(res, terms, weight, 1e-6, dtype, w, got_state, slots, weight_b, bias=bias, bias_b=bias_b)
    for a, b in ((got, want), (got_other, other), (got_state, state), (res, residual)):
        assert torch.equal(a, b)
    mixed = [(rand(rows, width).bfloat16(), None)]
    assert not ops.add_layernorm_conv_supported(res, mixed, weight, dtype, w, got_state)
    assert not ops.add_layernorm_conv_supported(rand(rows, 8196), [], weight, dtype, w, got_state)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [4096, 5120, 8192])
@pytest.mark.parametrize("parts", [1, 2, 3, 8])
def test_stacks_in_front_of_the_norm_with_a_convolution(dtype, width, parts):
    """Stacks of as many parts as are fetched at a time, fewer and more: bit for bit as without the convolution."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(width + parts)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    residual, terms = rand(2, width), [(rand(parts, 2, width), rand(width).to(dtype)), (rand(4 - min(parts, 3), 2, width), None)]
    weight, w, state = rand(width).to(dtype), rand(width, 4).to(dtype), rand(3, 3, width).to(dtype)
    slots = torch.tensor([2, 0], dtype=torch.int32, device="cuda")
    res, got_state = residual.clone(), state.clone()
    norm = ops.add_layernorm(residual, terms, weight, 1e-6, dtype)
    want = ops.conv_step(norm, w, state, slots, add_input=True)
    got, other = ops.add_layernorm_conv(res, terms, weight, 1e-6, dtype, w, got_state, slots)
    assert all(torch.equal(a, b) for a, b in ((got, want), (other, norm), (got_state, state), (res, residual)))
