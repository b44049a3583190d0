"""The mLSTM matrix memory over chunks of 64 rows against the token-by-token kernels and a 64-bit recurrence: segments of one
row to several chunks with remainders, heads of unequal sizes, state slots out of order, gates far apart.  All 32-bit: both
kernels' outputs are within 2e-5 of the 64-bit ones (sums of up to 128 products and 64 rows, exponents to 1e-6; the
denominators of rows whose n . q nearly cancels amplify it), the states within 1e-6."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(lengths, H, D, Dv, gate_std, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    T, n = sum(lengths), len(lengths)
    row0 = [0]
    for length in lengths:
        row0.append(row0[-1] + length)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    return dict(qkvg=rand(T, 2 * H * (D + Dv)), gates=rand(T, 2 * H) * gate_std, bi=rand(H), bf=rand(H), weight=rand(H * Dv).bfloat16(),
                state=(rand(n + 1, H, D, Dv), rand(n + 1, H, D), rand(n + 1, H).abs()), row0=i32(row0), slot=i32(list(range(n, 0, -1))))


def _recurrence(c, H, D, Dv, cap):
    p, out = c["qkvg"].double(), []
    S, n, m = (t.double().clone() for t in c["state"])
    gate = cap * torch.tanh((c["gates"].double() + torch.cat([c["bi"], c["bf"]]).double()) / cap)
    i, f = gate[:, :H], torch.nn.functional.logsigmoid(gate[:, H:])
    for s, slot in enumerate(c["slot"].tolist()):
        for t in range(int(c["row0"][s]), int(c["row0"][s + 1])):
            q, k = p[t, :H * D].view(H, D) * D ** -0.5, p[t, H * D:2 * H * D].view(H, D)
            v, g = p[t, 2 * H * D:2 * H * D + H * Dv].view(H, Dv), p[t, 2 * H * D + H * Dv:]
            top = torch.maximum(f[t] + m[slot], i[t])
            keep, take = torch.exp(f[t] + m[slot] - top), torch.exp(i[t] - top)
            S[slot] = keep[:, None, None] * S[slot] + take[:, None, None] * k[:, :, None] * v[:, None, :]
            n[slot] = keep[:, None] * n[slot] + take[:, None] * k
            m[slot] = top
            o = torch.einsum("hdv,hd->hv", S[slot], q) / (torch.maximum((n[slot] * q).sum(-1).abs(), torch.exp(-top)) + 1e-6)[:, None]
            o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6)
            out.append(o.reshape(-1) * c["weight"].double() * torch.sigmoid(g))
    return torch.stack(out), (S, n, m)


def _rel(got, want):
    assert torch.isfinite(got.float()).all()
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("lengths,H,D,Dv,gate_std", [([1], 1, 32, 32, 1.0), ([64], 2, 128, 128, 1.0), ([65, 63], 2, 64, 96, 1.0),
                                                     ([130, 1, 200], 3, 96, 32, 3.0), ([1, 1, 129, 1], 2, 128, 64, 1.0), ([100], 1, 32, 128, 20.0)])
def test_chunks_give_the_recurrence(lengths, H, D, Dv, gate_std):
    from arle_amd.kernels import ops

    c = _case(lengths, H, D, Dv, gate_std, 5 + sum(lengths))
    want, states = _recurrence(c, H, D, Dv, 15.0)
    for dtype, bound in ((torch.float32, 2e-5), (torch.bfloat16, 2.0 ** -8)):
        mine = [t.clone() for t in c["state"]]
        got = ops.mlstm_chunks(c["qkvg"], c["gates"], c["bi"], c["bf"], 15.0, *mine, c["row0"], c["slot"], c["weight"], 1e-6, dtype,
                               heads=H, key_dim=D, value_dim=Dv)
        assert got.dtype == dtype and _rel(got, want) < bound
        for state, ref, before in zip(mine, states, c["state"]):
            assert _rel(state, ref) < 1e-6 and torch.equal(state[0], before[0])     # slot 0 belongs to nobody
    plain = [t.clone() for t in c["state"]]
    a, b = H * D, H * Dv
    num, nq, coefs = ops.mlstm_scan(c["qkvg"][:, :a], c["qkvg"][:, a:2 * a], c["qkvg"][:, 2 * a:2 * a + b], c["gates"], c["bi"], c["bf"],
                                    15.0, *plain, c["row0"], c["slot"], heads=H, key_dim=D, value_dim=Dv)
    by_row = ops.mlstm_output(num, nq, coefs, c["qkvg"][:, 2 * a + b:], c["weight"], 1e-6, torch.float32, heads=H, value_dim=Dv)
    assert _rel(by_row, want) < 2e-5


@pytest.mark.parametrize("lengths,D,Dv,bad", [([64], 128, 128, 63), ([130], 64, 96, 31), ([100, 70], 32, 64, 99), ([100, 70], 96, 32, 133),
                                              ([129], 128, 128, 128)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_a_value_that_is_no_number_reaches_its_row_and_later_ones_only(lengths, D, Dv, bad, value):
    """One entry of one head's v: the rows in front of it, the other requests and the other heads keep their bits, and the
    rows from it on hold no number where the token-by-token kernels hold none."""
    from arle_amd.kernels import ops

    H, T = 2, sum(lengths)
    c = _case(lengths, H, D, Dv, 1.0, 3 + bad)
    qk, vw = H * D, H * Dv
    spoilt = c["qkvg"].clone()
    spoilt[bad, 2 * qk + Dv + Dv // 2 + 1] = value       # head 1
    chunks = lambda p: ops.mlstm_chunks(p, c["gates"], c["bi"], c["bf"], 15.0, *[t.clone() for t in c["state"]], c["row0"], c["slot"],
                                        c["weight"], 1e-6, torch.float32, heads=H, key_dim=D, value_dim=Dv)
    clean, got = chunks(c["qkvg"]), chunks(spoilt)
    num, nq, coefs = ops.mlstm_scan(spoilt[:, :qk], spoilt[:, qk:2 * qk], spoilt[:, 2 * qk:2 * qk + vw], c["gates"], c["bi"], c["bf"], 15.0,
                                    *[t.clone() for t in c["state"]], c["row0"], c["slot"], heads=H, key_dim=D, value_dim=Dv)
    by_row = ops.mlstm_output(num, nq, coefs, spoilt[:, 2 * qk + vw:], c["weight"], 1e-6, torch.float32, heads=H, value_dim=Dv)
    end = next(int(e) for e in c["row0"].tolist()[1:] if e > bad)
    reached = torch.zeros(T, vw, dtype=torch.bool, device="cuda")
    reached[bad:end, Dv:] = True
    assert torch.equal(got[~reached], clean[~reached]) and torch.isfinite(clean).all()
    assert torch.equal(torch.isfinite(by_row), torch.isfinite(got))
