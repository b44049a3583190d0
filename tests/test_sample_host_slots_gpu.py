"""Tokens that the sampling kernel writes to pinned host memory by itself: what is read is what lies on the GPU, whether the results
are read at once, kept unread past the number of places, read out of order, or dropped."""
import gc

import pytest
import torch

from arle_amd.sampling import Sampler, SamplingParams
from arle_amd.sampling.sampler import _HostSlots

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(n, first, **more):
    p = SamplingParams(temperature=0.9, top_k=20, top_p=0.95, **more)
    return [(p, first + i, first, []) for i in range(n)]


@pytest.mark.parametrize("n", [1, 3, 64])
def test_tokens_written_by_the_kernel_are_those_on_the_gpu(n):
    logits = torch.randn(n, 5003, generator=torch.Generator().manual_seed(n)).to(DEV) * 3
    sampler = Sampler(logits.device)
    kept = [sampler.choose(logits, _rows(n, i)) for i in range(_HostSlots.SLOTS + 9)]      # more than there are places
    assert sum(c._slots is not None for c in kept) == _HostSlots.SLOTS
    for c in reversed(kept):
        assert c.tokens() == c.token_tensor.tolist() == c.tokens()
    assert len(sampler._slots.free) == _HostSlots.SLOTS
    for i in range(2 * _HostSlots.SLOTS):
        sampler.choose(logits, _rows(n, i))      # dropped unread
    gc.collect()
    torch.cuda.synchronize()
    assert len(sampler._slots.free) == _HostSlots.SLOTS
    after = sampler.choose(logits, _rows(n, 0))
    assert after.tokens() == kept[0].tokens()


def test_greedy_rows_and_log_probabilities_beside_it():
    logits = torch.randn(4, 999, generator=torch.Generator().manual_seed(5)).to(DEV)
    rows = _rows(3, 7, logprobs=True) + [(SamplingParams(), 0, 0, [])]
    chosen = Sampler(logits.device).choose(logits, rows)
    tokens, logprobs = chosen.tokens(), chosen.logprobs()
    assert tokens == chosen.token_tensor.tolist() and tokens[3] == int(logits[3].argmax())
    want = torch.log_softmax(logits.double().cpu(), -1)[range(4), tokens]
    assert float((torch.tensor(logprobs, dtype=torch.float64) - want).abs().max()) < 1e-5
