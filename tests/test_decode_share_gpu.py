"""Steps of single decoded tokens whose keys are shared out over all waves of a kv head: ragged and equal contexts,
more requests than a wave has lanes, windows, and the plan that later layers take from the first.  The unsplit form of
the same kernel (one wave a request and kv head) is the reference: it walks the keys in the same blocks, so the results
differ by the order of float32 sums and one rounding to bfloat16 (2^-9), stated as a relative norm of 4e-3."""
import random

import pytest
import torch

pytestmark = pytest.mark.gpu
D, P, NQ, NKV = 128, 16, 8, 2


def _case(contexts, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    pages = [-(-(c + 1) // P) for c in contexts]
    table = torch.zeros((len(contexts), max(pages)), dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(seed)).int(), 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    k, v = rand(at, NKV, P, D).bfloat16(), rand(at, NKV, D, P).bfloat16()
    parts = rand(2, len(contexts), (NQ + 2 * NKV) * D)
    i32 = lambda vals: torch.tensor(vals, dtype=torch.int32, device="cuda")
    n = len(contexts)
    return parts, k, v, table.cuda(), i32(list(range(n + 1))), i32(list(range(n))), i32(contexts)


def _run(case, contexts, **kw):
    from arle_amd.kernels import ops

    parts, k, v, table, row0, slot, start = case
    out = torch.full((len(contexts), NQ * D), float("nan"), dtype=torch.bfloat16, device="cuda")
    return ops.attn_decode_prep(parts, out, k.clone(), v.clone(), table, row0, slot, start, max_kv_len=max(contexts) + 1,
                                num_q_heads=NQ, num_kv_heads=NKV, head_dim=D, page_size=P, scale=D ** -0.5, eps=1e-6, **kw)


@pytest.mark.parametrize("contexts,window", [
    ([0], 0), ([31], 0), ([5000], 0),                                          # one request: one block, and more than 64 blocks
    ([0, 0, 0], 0), ([31, 32, 33, 4095, 0], 0), ([700] * 7, 0),
    ([random.Random(1).randrange(0, 900) for _ in range(63)] + [6000], 0),     # as many as lanes, one long
    ([random.Random(2).randrange(0, 300) for _ in range(65)], 0),              # one more than lanes
    ([3000] + [1] * 140 + [2500], 0),                                          # three lots of lanes
    ([17, 900, 64, 3], 50), ([random.Random(3).randrange(0, 400) for _ in range(70)], 33),
])
def test_shared_out_keys_give_what_one_wave_a_request_gives(contexts, window):
    from arle_amd.kernels import ops

    case = _case(contexts, 7 + len(contexts))
    want = _run(case, contexts, window=window, splits=1).float()
    splits, waves = ops.decode_share(len(contexts), NKV, max(contexts) + 1, sum(contexts) + len(contexts))
    for kw in (dict(total_kv_len=sum(contexts) + len(contexts)), dict(splits=5)):
        carry = {}
        got = _run(case, contexts, window=window, carry=carry, **kw)
        assert torch.isfinite(got.float()).all()
        assert float((got.float() - want).norm() / want.norm()) < 4e-3
        assert torch.equal(got, _run(case, contexts, window=window, carry=carry, **kw))    # a later layer: the plan is there
    assert waves == 0 or len(contexts) < waves <= max(512, 2 * len(contexts))


@pytest.mark.parametrize("segments,kv_heads,longest", [(1, 8, 1), (1, 8, 40), (3, 8, 4096), (64, 8, 2048), (100, 8, 2048), (700, 8, 900),
                                                       (2, 4096, 4096)])
def test_the_number_of_waves(segments, kv_heads, longest):
    from arle_amd.kernels import ops

    for total in (None, segments * longest, segments - 1 + longest):
        splits, waves = ops.decode_share(segments, kv_heads, longest, total)
        assert 1 <= splits <= 64 and (waves == 0 or (splits > 1 and segments < waves <= 65535))
