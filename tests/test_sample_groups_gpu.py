"""Rows with a small top_k by their groups' maxima (`sample_rows(..., small_k=True)`): parameters that travel with the launch, groups
of NaNs and infinities, more groups than a thread holds, few groups, and values that many groups end in.  The passes of many
workgroups give the expected tokens; every one has to be the same."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(vocab, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(10, vocab, generator=gen) * 2
    at = torch.arange(vocab)
    x[1] = float("nan")
    x[2] = -float("inf")
    x[3] = torch.where(at % 2 == 0, float("nan"), -float("inf"))
    x[4, vocab // 3] = float("inf")
    x[5, : vocab // 2] = float("nan")
    x[6] = (x[6] * 4).round() / 4                                     # ties at every value
    x[7] = torch.where(at % 64 == 63, 1.0, x[7] * 1e-3)               # every whole group ends in one value, few tokens do
    x[7, vocab - 1] = 1.5
    x[8] = torch.where(at % 7 == 0, 1.0, 1.0 - 1e-7)                  # neighbouring logits whose e are the same or next to it
    x[9, : vocab - 100] = -50.0                                       # all that counts in the last groups
    return x.cuda()


@pytest.mark.parametrize("vocab", [151936, 300000, 33001, 4099, 130])
def test_tokens_by_groups(vocab):
    from arle_amd.kernels import ops

    logits = _rows(vocab, vocab)
    rows = len(logits)
    gen = torch.Generator().manual_seed(3)
    for k in (1, 50, 256):
        k = min(k, vocab - 1)
        for p, min_p, temp in ((1.0, 0.0, 0.7), (0.9, 0.05, 1.3), (0.5, 1.0, 1.0), (1.0, 0.0, 0.0)):
            packed = np.empty((5, rows), dtype=np.float32)
            packed[:3] = [[temp], [p], [min_p]]
            packed[3] = torch.rand(rows, generator=gen).numpy()
            packed.view(np.int32)[4] = k
            dev = torch.from_numpy(packed).cuda()
            args = (dev[0], dev[4].view(torch.int32), dev[1], dev[2], dev[3])
            want = ops.sample_rows(logits, *args, use_top_p=p < 1)
            assert torch.equal(ops.sample_rows(logits, *args, use_top_p=p < 1, small_k=True), want), (k, p, min_p, temp)
            assert torch.equal(ops.sample_rows(logits, packed, use_top_p=p < 1, small_k=True), want), (k, p, min_p, temp)


def test_parameters_in_host_memory_are_refused_where_they_cannot_travel():
    from arle_amd.kernels import ops

    most = ops.sample_host_rows()
    logits = torch.zeros(most + 1, 300, device="cuda")
    packed = np.ones((5, most + 1), dtype=np.float32)
    with pytest.raises(ops.ShapeError):
        ops.sample_rows(logits, packed, small_k=True)                                # too many rows
    with pytest.raises(ops.ShapeError):
        ops.sample_rows(logits[:4], np.ones((5, 4), dtype=np.float32))                # the passes read them on the GPU
    with pytest.raises(ops.ShapeError):
        ops.sample_rows(logits[:4], np.ones((4, 4), dtype=np.float32), small_k=True)


def test_a_call_allocates_the_groups_maxima_alone():
    from arle_amd.kernels import ops

    rows, vocab = 64, 151936
    logits = torch.randn(rows, vocab, device="cuda")
    packed = np.full((5, rows), 0.5, dtype=np.float32)
    packed.view(np.int32)[4] = 50
    call = lambda: ops.sample_rows(logits, packed, small_k=True)
    first = call()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    assert torch.equal(call(), first)
    chunks = ops.lib.function("arle_argmax_chunks")(rows, vocab)
    groups = -(-(-(-vocab // chunks) + 3) // 64) + 1
    assert torch.cuda.max_memory_allocated() - before <= 4 * rows * chunks * groups + 4096
