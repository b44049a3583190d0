"""Rows with a small top_k finished by one kernel (`sample_rows(..., small_k=True)`) against the passes of many workgroups: the
same tokens, for every draw.  Ties that fill more than the kernel's list (which then reads the row again), rows whose
kept tokens lie at the ends of groups and chunks, rows that do not reach the rank, greedy rows, NaN and infinities, new
buffers full of ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _logits(rows, vocab, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, vocab, generator=gen) * 2.5
    kinds = [lambda r: None, lambda r: r.fill_(0.25), lambda r: r.copy_(torch.where(torch.arange(vocab) % 61 == 0, 3.0, -30.0)),
             lambda r: r[[0, vocab - 1]].fill_(0).add_(0), lambda r: r.copy_((r * 2).round() / 2), lambda r: r.mul_(100.0),
             lambda r: r.masked_fill_(torch.arange(vocab) % 3 == 1, -float("inf")), lambda r: r.masked_fill_(torch.arange(vocab) % 7 == 2, float("nan")),
             lambda r: r.masked_fill_(torch.arange(vocab) % (vocab // 9) != 1, -float("inf"))]
    for i in range(rows):
        kinds[i % len(kinds)](x[i])
    x[0, 0] = x[0, vocab - 1] = 9.0
    return x.cuda()


@pytest.mark.parametrize("rows,vocab", [(1, 151936), (8, 151936), (64, 33000), (9, 8193), (5, 2048), (3, 333), (70, 50257), (2, 300000)])
def test_the_same_tokens(rows, vocab, monkeypatch):
    from arle_amd.kernels import ops

    logits = _logits(rows, vocab, rows + vocab)
    most = min(ops.sample_small_k(), vocab - 1)
    gen = torch.Generator().manual_seed(7)
    cycle = lambda values, dtype=torch.float32: torch.tensor([values[r % len(values)] for r in range(rows)], dtype=dtype, device="cuda")
    empty = torch.empty
    ones = lambda *a, **k: empty(*a, **k).view(torch.uint8).fill_(0xff).view(k["dtype"])
    for ks in ([50], [1], [most], [20, 3, 200 if most >= 200 else most, 1, 7]):
        for ps in ([1.0], [0.9], [0.95, 0.3, 1.0, 1e-6]):
            for ms in ([0.0], [0.0, 0.05, 0.5]):
                for temps in ([0.8], [1.2, 0.0, 0.3]):
                    args = [cycle(temps), cycle([min(k, vocab - 1) for k in ks], torch.int32), cycle(ps), cycle(ms)]
                    draws = [torch.rand(rows, generator=gen).cuda(), cycle([0.0, 0.99999994])]
                    for u in draws:
                        want = ops.sample_rows(logits, *args, u, use_top_p=min(ps) < 1)
                        monkeypatch.setattr(torch, "empty", ones)
                        got = ops.sample_rows(logits, *args, u, use_top_p=min(ps) < 1, small_k=True)
                        monkeypatch.setattr(torch, "empty", empty)
                        assert torch.equal(got, want), (ks, ps, ms, temps)


@pytest.mark.parametrize("rows,vocab", [(14, 151936), (14, 33003), (14, 5001), (14, 300001)])
@pytest.mark.parametrize("k", [1, 50, 256])
def test_flat_rows(rows, vocab, k):
    """Rows whose first digit leaves more than the list holds, about as many or somewhat fewer, and ties of any number at the
    threshold, below it and above it; odd lengths, so that rows begin anywhere on the 16-byte grid."""
    from arle_amd.kernels import ops

    gen = torch.Generator().manual_seed(vocab + k)
    x = torch.randn(rows, vocab, generator=gen)
    for i, spread in enumerate((0.005, 0.02, 0.05, 0.1, 0.2, 0.3, 0.5)):
        x[i] *= spread
    x[7] = torch.where(x[7] > 0.5, 1.0, 0.0)                                  # two values
    x[8] = torch.where(torch.arange(vocab) % 13 < k % 13, 0.1, 0.0)
    x[8, 5:5 + 100] = 0.11 + 0.001 * torch.arange(100)                          # some above the ties
    x[9] = 0.0
    x[9, vocab // 2:vocab // 2 + 300] = 1.0                                    # fewer than the list holds, more than top_k
    x[10] = (x[10] * 0.1 * 40).round() / 40
    x[11] = x[11] * 2 - 95                                                     # denormal e behind one large logit
    x[11, 17] = 0.0
    x[12] = torch.where(torch.arange(vocab) % 5 == 0, x[12] * 0.01, -float("inf"))
    x[13, :2500] = 3.0                                                         # ties that the list holds and the kept ones do not
    logits = x.cuda()
    full = lambda v, dtype=torch.float32: torch.full((rows,), v, dtype=dtype, device="cuda")
    for p in (1.0, 0.9, 0.02):
        for min_p in (0.0, 0.3, 1.0):
            for u in (torch.rand(rows, generator=gen).cuda(), full(0.0), full(0.99999994)):
                args = (logits, full(1.0), full(k, torch.int32), full(p), full(min_p), u)
                want = ops.sample_rows(*args, use_top_p=p < 1)
                assert torch.equal(ops.sample_rows(*args, use_top_p=p < 1, small_k=True), want), (p, min_p)


def test_the_sampler_promises_it_only_where_it_holds(monkeypatch):
    from arle_amd.kernels import ops
    from arle_amd.sampling import Sampler, SamplingParams

    logits, promised = _logits(4, 4000, 1), []
    whole = ops.sample_rows
    monkeypatch.setattr(ops, "sample_rows", lambda *a, **k: promised.append(k["small_k"]) or whole(*a, **k))
    most = ops.sample_small_k()
    for ks, small in (([5, 5, 5, 5], True), ([5, most, 1, 7], True), ([5, -1, 5, 5], False), ([5, 0, 5, 5], False), ([5, most + 1, 5, 5], False)):
        Sampler(logits.device).choose(logits, [(SamplingParams(temperature=0.8, top_k=k, top_p=0.9), i, i, []) for i, k in enumerate(ks)]).tokens()
        assert promised.pop() == small
    greedy = SamplingParams(temperature=0.0)
    Sampler(logits.device).choose(logits, [(greedy, 0, 0, []), (SamplingParams(temperature=0.8, top_k=5), 0, 0, [])] * 2).tokens()
    assert promised == [True]
