"""Who owns the pinned memory that a sampling kernel writes its tokens to, with stubs in the place of the GPU: a call that fails behind
the launch gives its place back and never before the kernel is done with it, a result is read once by however many threads, and a
captured call takes no place."""
import threading

import pytest
import torch

from arle_amd.sampling import SamplingParams, sampler as module
from arle_amd.sampling.sampler import Chosen, Sampler

ROWS = [(SamplingParams(temperature=0.9, top_k=20, logprobs=True), 1, 0, [])] * 2


class Event:
    """Comes when `pending` is cleared."""

    def __init__(self):
        self.pending = self.launched = False
        self.records = 0

    def record(self):
        self.records += 1
        self.pending = self.launched
        self.launched = False

    def query(self):
        return not self.pending

    def synchronize(self):
        self.pending = False


class Place:
    written = True

    def __init__(self, rows):
        self.memory, self.event = torch.zeros(rows, dtype=torch.int32), Event()


@pytest.fixture
def stubbed(monkeypatch):
    """A sampler whose kernels run at once and are done only when their event is waited for."""
    made = []

    def sample_rows(logits, packed, host_out=None, **promises):
        if host_out is not None:
            place = next(p for p in made if p.memory.data_ptr() == host_out.data_ptr())
            assert not place.event.pending, "a kernel writes where an earlier one may still write"
            place.event.launched = True
            host_out.fill_(7 + len(made))
        return torch.full((len(logits),), 7 + len(made), dtype=torch.int32)

    def place(rows):
        made.append(Place(rows))
        return made[-1]

    monkeypatch.setattr(module, "_HostPlace", place)
    monkeypatch.setattr(module.ops, "sample_rows", sample_rows)
    monkeypatch.setattr(module.ops, "sample_small_k", lambda: 64)
    monkeypatch.setattr(module.ops, "sample_host_rows", lambda: 64)
    monkeypatch.setattr(module.ops, "token_logprobs", lambda logits, tokens: torch.zeros(len(tokens)))
    monkeypatch.setattr(module.torch.cuda, "is_current_stream_capturing", lambda: False)
    s = Sampler("cpu")
    s.made = made
    return s


LOGITS = torch.zeros(2, 100)


def test_log_probabilities_that_fail_lose_no_place(stubbed, monkeypatch):
    def fails(*a):
        raise RuntimeError("no memory")

    with monkeypatch.context() as m:
        m.setattr(module.ops, "token_logprobs", fails)
        for _ in range(3):
            with pytest.raises(RuntimeError):
                stubbed.choose(LOGITS, ROWS)
    # all are back, each with the event behind its kernel, which has not come: none is given out again before it has
    assert len(stubbed._slots.free) == len(stubbed.made) == 3
    assert [(p.event.records, p.event.pending, p.written) for p in stubbed.made] == [(1, True, False)] * 3
    stubbed.choose(LOGITS, ROWS)
    assert len(stubbed.made) == 4
    stubbed.made[0].event.pending = False
    stubbed.choose(LOGITS, ROWS)
    assert len(stubbed.made) == 4


def test_a_result_that_cannot_be_made_gives_its_place_back_behind_its_kernel(stubbed, monkeypatch):
    def fails(*a, **k):
        raise RuntimeError("no pinned memory")

    monkeypatch.setattr(module, "Chosen", fails)
    with pytest.raises(RuntimeError):
        stubbed.choose(LOGITS, ROWS)
    place, = stubbed._slots.free
    assert place.event.pending and not place.written


def test_a_failing_launch_gives_its_place_back(stubbed, monkeypatch):
    def fails(*a, **k):
        raise RuntimeError("refused")

    monkeypatch.setattr(module.ops, "sample_rows", fails)
    with pytest.raises(RuntimeError):
        stubbed.choose(LOGITS, ROWS)
    assert len(stubbed._slots.free) == 1


def test_a_second_reader_never_reads_what_a_later_call_wrote(stubbed):
    first = stubbed.choose(LOGITS, ROWS)
    want, got, event = first.token_tensor.tolist(), [], stubbed.made[0].event
    entered, go_on = threading.Event(), threading.Event()

    def waits():      # the slow reader stands in its wait while another may read and let go
        event.synchronize = lambda: None
        entered.set()
        go_on.wait(0.3)
        event.pending = False

    event.synchronize = waits
    slow = threading.Thread(target=lambda: got.append(first.tokens()))
    slow.start()
    assert entered.wait(10)
    fast = threading.Thread(target=lambda: got.append(first.tokens()))
    fast.start()
    fast.join(0.1)
    event.pending = False
    if stubbed._slots.free:      # the fast one came through: its place goes to another call
        other = stubbed.choose(LOGITS, ROWS)
        assert other._slots is not None
        stubbed.made[0].memory.fill_(99)
    go_on.set()
    slow.join(10)
    fast.join(10)
    assert got == [want, want]
    assert len(stubbed._slots.free) == len({id(p) for p in stubbed._slots.free}) == 1


def test_a_place_goes_back_once(stubbed):
    chosen = stubbed.choose(LOGITS, ROWS)
    held = chosen._slots
    barrier = threading.Barrier(4)

    def go():
        barrier.wait(10)
        held.let_go()

    readers = [threading.Thread(target=go) for _ in range(4)]
    for t in readers:
        t.start()
    for t in readers:
        t.join(10)
    chosen.tokens()
    del chosen
    held.__del__()
    assert len(stubbed._slots.free) == 1


def test_a_place_that_was_read_is_not_asked_for_its_event(stubbed):
    stubbed.choose(LOGITS, ROWS).tokens()
    place = stubbed.made[0]
    place.event.query = lambda: pytest.fail("the reader has waited for it")
    stubbed.choose(LOGITS, ROWS).tokens()
    assert stubbed.made == [place]


def test_a_captured_call_takes_no_place(stubbed, monkeypatch):
    """A graph would write to it at every replay, whoever has it by then."""
    monkeypatch.setattr(module.torch.cuda, "is_current_stream_capturing", lambda: True)
    chosen = stubbed.choose(LOGITS, ROWS)
    assert chosen._slots is None and not stubbed.made and chosen.tokens() == [7, 7]


def test_as_many_places_as_there_may_be_and_the_copy_beyond(stubbed, monkeypatch):
    monkeypatch.setattr(module._HostSlots, "SLOTS", 3)
    kept = [stubbed.choose(LOGITS, ROWS) for _ in range(5)]
    assert [c._slots is None for c in kept] == [False] * 3 + [True] * 2 and len(stubbed.made) == 3
    assert all(c.tokens() == c.token_tensor.tolist() for c in reversed(kept))
    assert isinstance(kept[0], Chosen) and len(stubbed._slots.free) == 3
