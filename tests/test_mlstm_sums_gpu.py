"""The mLSTM's chunks with their sums side by side and the states in front of them element by element (requests of 384 rows
and more) against the walk from chunk to chunk: more chunks than are fetched ahead, remainders, several requests of unequal
length, gates far apart; and which of the two a step takes.  Both are 32-bit sums of the same terms: within 1e-5 of each other, states within 2e-6."""
import pytest
import torch

from test_mlstm_chunks_gpu import _case, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,H,D,Dv,gate_std", [([384], 2, 128, 128, 1.0), ([577], 1, 32, 96, 3.0), ([1100, 1, 640], 2, 64, 32, 1.0),
                                                     ([70, 513], 3, 96, 128, 20.0), ([1], 1, 128, 64, 1.0)])
def test_sums_and_scan_give_what_the_walk_gives(lengths, H, D, Dv, gate_std):
    from arle_amd.kernels import ops

    c = _case(lengths, H, D, Dv, gate_std, 11 + sum(lengths))

    def run(longest):
        state = [t.clone() for t in c["state"]]
        out = ops.mlstm_chunks(c["qkvg"], c["gates"], c["bi"], c["bf"], 15.0, *state, c["row0"], c["slot"], c["weight"], 1e-6, torch.float32,
                               heads=H, key_dim=D, value_dim=Dv, longest=longest)
        return out, state

    (walked, s0), (summed, s1) = run(1), run(1 << 20)
    assert _rel(summed, walked.double()) < 1e-5
    for a, b, before in zip(s1, s0, c["state"]):
        assert _rel(a, b.double()) < 2e-6 and torch.equal(a[0], before[0])


@pytest.mark.parametrize("lengths,H,D,sums", [([384], 2, 128, True), ([384] * 8, 8, 128, False), ([640] * 2, 20, 128, True), ([639] * 2, 20, 128, False),
                                              ([700, 1, 1, 1, 1, 1, 1, 1, 1, 1], 8, 128, True), ([383], 1, 32, False)])
def test_which_of_them_a_step_takes(lengths, H, D, sums):
    """A walk that keeps the matrix cores busy stays (8 requests of 384 rows, 8 heads of 128: 56.6 against 65.7 us)."""
    from arle_amd.kernels import ops

    c = _case(lengths, H, D, D, 1.0, 5)

    def run(longest):
        state = [t.clone() for t in c["state"]]
        return ops.mlstm_chunks(c["qkvg"], c["gates"], c["bi"], c["bf"], 15.0, *state, c["row0"], c["slot"], c["weight"], 1e-6, torch.float32,
                                heads=H, key_dim=D, value_dim=D, longest=longest), state

    (got, state), (like, want) = run(max(lengths)), run(1 << 20 if sums else 1)
    assert torch.equal(got, like) and all(torch.equal(a, b) for a, b in zip(state, want))
