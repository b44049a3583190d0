"""The short convolution that moves its requests' states on, against the convolution and the update one after the other, bit for bit:
segments of fewer rows than taps, of none, at the edges of the eight rows that a lane takes, steps on both sides of the row count
from which one kernel does both, and what only two kernels take."""
import pytest
import torch

from arle_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("lengths", [[128], [127], [1, 2, 3, 4, 5, 130], [8, 8, 120, 0, 1], [257, 7, 9], [1] * 140, [2, 1, 60]])
@pytest.mark.parametrize("channels,taps,kind", [(4, 2, torch.float32), (260, 3, torch.bfloat16), (2560, 4, torch.bfloat16), (1028, 4, torch.float32),
                                                (6, 4, torch.bfloat16), (64, 5, torch.bfloat16), (64, 1, torch.bfloat16)])
@pytest.mark.parametrize("flags", [dict(add_input=True), dict(silu=True, bias=True), dict(out_bias=True, bias=True)])
def test_one_call_makes_the_rows_and_moves_the_states_on(lengths, channels, taps, kind, flags):
    gen = torch.Generator().manual_seed(len(lengths) * 1000 + channels + taps)
    made = lambda *shape: torch.randn(*shape, generator=gen).to(kind).to(DEV)
    tokens, slots = sum(lengths), torch.randperm(len(lengths) + 3, generator=gen)[:len(lengths)].tolist()
    u = made(tokens, channels + 8)[:, :channels]
    w, state = made(channels, taps), made(len(lengths) + 3, taps - 1, channels) if taps > 1 else None
    given = dict(add_input=flags.get("add_input", False), silu=flags.get("silu", False))
    bias, out_bias = (made(channels) if flags.get(name) else None for name in ("bias", "out_bias"))
    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)
    row0 = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    slot_of = i32([s for s, n in zip(slots, lengths) for _ in range(n)])
    want_state = state.clone() if taps > 1 else None
    want = ops.causal_conv(u, w, want_state, slot_of, bias=bias, out_bias=out_bias, **given)
    if taps == 1:      # no state to move on
        with pytest.raises(ops.ShapeError):
            ops.causal_conv(u, w, None, slot_of, seg_row0=i32(row0), seg_slot=i32(slots))
        return
    ops.conv_state_update(u, want_state, i32(row0), i32(slots), bias=bias)
    got = ops.causal_conv(u, w, state, slot_of, bias=bias, out_bias=out_bias, seg_row0=i32(row0), seg_slot=i32(slots), **given)
    assert torch.equal(got, want) and torch.equal(state, want_state)


@pytest.mark.parametrize("lengths", [[128], [1, 2, 3, 4, 5, 130], [8, 8, 120, 0, 1], [1] * 140])
@pytest.mark.parametrize("channels,taps,kind", [(4, 2, torch.float32), (260, 3, torch.bfloat16), (1028, 4, torch.float32), (2560, 4, torch.bfloat16)])
@pytest.mark.parametrize("flags", [dict(add_input=True), dict(silu=True, bias=True), dict(out_bias=True, bias=True)])
@pytest.mark.parametrize("moves", [True, False])
def test_steps_of_many_rows_against_the_sums_in_64_bits(lengths, channels, taps, kind, flags, moves):
    """The kernel for 128 rows and more, with the segments and without them (then the states stay), against request by request on the CPU."""
    gen = torch.Generator().manual_seed(len(lengths) * 100 + channels + taps)
    made = lambda *shape: torch.randn(*shape, generator=gen).to(kind)
    tokens, slots = sum(lengths), torch.randperm(len(lengths) + 3, generator=gen)[:len(lengths)].tolist()
    u, w, state = made(tokens, channels), made(channels, taps), made(len(lengths) + 3, taps - 1, channels)
    bias, out_bias = (made(channels) if flags.get(name) else None for name in ("bias", "out_bias"))
    want, want_state, at = torch.empty(tokens, channels, dtype=torch.float64), state.double().clone(), 0
    rounded = lambda x: x.to(kind).double() if kind != torch.float32 else x.float().double()
    for slot, n in zip(slots, lengths):
        fresh = u[at:at + n].double() + (0.0 if bias is None else bias.double())
        rows = torch.cat([want_state[slot], fresh])
        y = sum(w[:, j].double() * rows[j:j + n] for j in range(taps)) + (0.0 if out_bias is None else out_bias.double())
        if flags.get("add_input"):
            y = y + fresh
        want[at:at + n] = y / (1.0 + torch.exp(-y)) if flags.get("silu") else y
        want_state[slot] = rounded(rows[n:]) if n else want_state[slot]
        at += n
    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)
    on = lambda t: None if t is None else t.to(DEV)
    held = state.to(DEV)
    segments = dict(seg_row0=i32([sum(lengths[:i]) for i in range(len(lengths) + 1)]), seg_slot=i32(slots)) if moves else {}
    got = ops.causal_conv(on(u), on(w), held, i32([s for s, n in zip(slots, lengths) for _ in range(n)]), bias=on(bias), out_bias=on(out_bias),
                          add_input=flags.get("add_input", False), silu=flags.get("silu", False), **segments)
    # sums of five terms of about 1 in 32 bits and one rounding to the type (2^-8 of a value in bfloat16)
    one = 2.0 ** -8 if kind == torch.bfloat16 else 1e-6
    assert float(((got.double().cpu() - want).abs() - one * want.abs()).max()) < 4e-6
    assert float((held.double().cpu() - (want_state if moves else state.double())).abs().max()) < 1e-6
