"""Choosing the next token of every row of a step's logits.

All rows greedy and without penalties: one argmax kernel.  Otherwise: penalties on the
logits (repetition, frequency, presence over the tokens generated so far), then per row
softmax(logits / T), min-p, top-k, top-p and an inverse-CDF draw in token order.

The uniform number of a draw is a pure function of (seed, request's own draw index), so a
request's tokens do not depend on which other requests share its steps.  The reference
draws one number per request per step from a shared generator in slot order
(infer/src/model/qwen3/forward.rs:458-508), which ties results to batch composition; that
is not kept.
"""
from __future__ import annotations

import threading
from array import array
from collections import deque

import numpy as np
import torch

from ..cache import native
from ..engine.batch import DeviceToken
from ..kernels import ops
from ..kernels.upload import upload
from .params import SamplingParams

_MASK = (1 << 64) - 1


def _splitmix64(x: int) -> int:
    x = (x + 0x9E3779B97F4A7C15) & _MASK
    z = x
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
    return z ^ (z >> 31)


def uniform(seed: int, index: int) -> float:
    """The index-th uniform number in [0, 1) of a request whose seed is `seed` (24 bits, exact in float32)."""
    return (_splitmix64(_splitmix64(seed & _MASK) ^ (index & _MASK)) >> 40) / float(1 << 24)


def _words(values) -> array:
    """The values modulo 2^64."""
    try:
        return array("Q", values)
    except OverflowError:
        return array("Q", [v & _MASK for v in values])


def uniforms(seeds, indices) -> np.ndarray:
    """uniform(seed, index) of every pair, float32, by the host runtime (64 pairs took 46 us in arithmetic on whole arrays,
    and 6 of these are left)."""
    s, i = _words(seeds), _words(indices)
    if len(s) != len(i):
        raise ValueError(f"{len(s)} seeds and {len(i)} indices do not make pairs")
    out = np.empty(len(s), dtype=np.float32)
    native.lib().arle_uniforms(len(out), s.buffer_info()[0], i.buffer_info()[0], out.ctypes.data)
    return out


class _HostPlace:
    """Pinned host memory that one sampling kernel at a time writes its tokens to, and the event behind that kernel; written: it is
    known to have come."""

    written = True

    def __init__(self, rows: int):
        self.memory = torch.empty((rows,), dtype=torch.int32, pin_memory=True)
        self.event = torch.cuda.Event()

    def __del__(self):
        event = getattr(self, "event", None)
        if event is not None:
            event.synchronize()      # the memory outlives the kernel that writes to it


class _HeldPlace:
    """A place of a `_HostSlots` and its owner: it goes back once, when the tokens have been read or nobody can read them any more."""

    def __init__(self, slots: "_HostSlots", place: _HostPlace, rows: int):
        place.written = False
        self.memory, self.event = place.memory[:rows], place.event
        self._free, self._places = slots.free, [place]

    def let_go(self, written: bool = False) -> None:
        """written: the event has been waited for."""
        try:
            place = self._places.pop()      # one thread gets it
        except IndexError:
            return
        place.written = written
        self._free.append(place)

    def __del__(self):
        self.let_go()


class _HostSlots:
    """Up to `SLOTS` places for tokens, made as they are needed.  A place is given out again once its holder has let go of it and
    its event has come; where there is none, `take` returns None and the tokens are copied as any others.  Nothing here waits.
    (One block for all places, made by a sampler's first call: 64.3 us that call, 64 rows of 151,936 logits; a place at a time 62.5, and
    61.7 with the copy, which costs every later call among others 40 instead of 34.)"""

    SLOTS = 256

    def __init__(self):
        self.free = deque()      # the longest unused first (append and popleft are atomic)
        self._made, self._lock = 0, threading.Lock()

    def take(self, rows: int):
        if torch.cuda.is_current_stream_capturing():
            return None      # a replay would write where another call's tokens are by then
        with self._lock:
            if self.free and (self.free[0].written or self.free[0].event.query()):
                return _HeldPlace(self, self.free.popleft(), rows)
            if self._made == self.SLOTS:
                return None
            place = _HostPlace(ops.sample_host_rows())
            self._made += 1
            return _HeldPlace(self, place, rows)


class Chosen:
    """The tokens that a step's sampling kernels chose, still on the GPU: handed to the next step as they are
    (`feed`), and on their way into pinned host memory, written there by the sampling kernel itself (a place of the sampler's, which
    goes back to it once they are read) or by a copy queued right behind the kernels, before anything
    else is launched, so that reading them (`tokens`, `logprobs`) waits for the step that chose them and not for
    the step launched after it.  Any thread may read them.  (The reference reads its argmax back asynchronously into a ring of pinned
    buffers: infer/src/model/qwen3/batch_decode.rs:728-774.  A copy stream of its own was tried here and taken
    out: while its wait for the step sits in a second hardware queue, every kernel of the step takes 0.7 us longer
    to start, 0.23 ms a step of the Qwen3-4B shape.)"""

    def __init__(self, token_tensor, logprob_tensor=None, read_back: bool = True, held: _HeldPlace | None = None):
        """held: the place that the kernel which made the tokens writes them to, its event recorded behind that kernel."""
        self._slots = held      # until they are read
        self._reading = threading.Lock()
        self.token_tensor = token_tensor       # int32 [rows]
        self.logprob_tensor = logprob_tensor   # float32 [rows] or None
        self._tokens = self._logprobs = self._arrived = None
        self._host = []
        copied = [logprob_tensor] if held is not None else [token_tensor, logprob_tensor]
        if held is not None:
            self._host.append(held.memory)
            self._arrived = held.event
        if read_back and token_tensor.is_cuda:
            for t in copied:
                if t is not None:
                    self._host.append(torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t, non_blocking=True))
            if held is None:
                self._arrived = torch.cuda.Event()
            if held is None or logprob_tensor is not None:
                self._arrived.record()

    def feed(self, row: int) -> DeviceToken:
        return DeviceToken(self.token_tensor, row)

    def _read(self) -> None:
        with self._reading:
            if self._tokens is not None:
                return
            if self._arrived is None:
                tokens = self.token_tensor.tolist()
                self._logprobs = None if self.logprob_tensor is None else self.logprob_tensor.tolist()
            else:
                self._arrived.synchronize()
                tokens = self._host[0].tolist()
                self._logprobs = self._host[1].tolist() if len(self._host) > 1 else None
            self._tokens = tokens
            held, self._slots, self._host = self._slots, None, []
            if held is not None:
                held.let_go(written=True)

    def tokens(self) -> list:
        self._read()
        return self._tokens

    def logprobs(self):
        self._read()
        return self._logprobs


class Sampler:
    def __init__(self, device):
        self.device = device
        self._slots = _HostSlots()

    def sample(self, logits: torch.Tensor, rows) -> list:
        """rows: one (SamplingParams, seed, draw_index, generated_tokens) per row of `logits`."""
        return self.sample_with_logprobs(logits, rows)[0]

    def sample_with_logprobs(self, logits: torch.Tensor, rows):
        """(token ids, log-probabilities): the second is None unless a row asks for `logprobs`; then it holds,
        for every row, log softmax(logits)[token] of the (penalised) logits, before temperature and truncation
        (for a greedy row: the reference's -log(sum exp(x - max)), crates/cuda-kernels/csrc/misc/sampling.cu:252-317)."""
        if not rows:
            if logits.shape[0] != 0:
                raise ValueError("one sampling row per row of logits is needed")
            return [], None
        chosen = self.choose(logits, rows)
        return chosen.tokens(), chosen.logprobs()

    def choose(self, logits: torch.Tensor, rows) -> Chosen:
        """As sample_with_logprobs, but nothing is read back: the kernels are queued and the result stays on the GPU."""
        if logits.shape[0] != len(rows):
            raise ValueError("one sampling row per row of logits is needed")
        # the parameters that differ, which every rule below asks alone: one where the requests share an object (64 rows with a
        # small top_k 40 us a call), else as many as there are objects, equal ones too (58 us)
        kinds = list({id(p): p for p, _, _, _ in rows}.values())
        if any(p.has_penalties() for p in kinds) and any(p.has_penalties() and gen for p, _, _, gen in rows):
            logits = logits.clone()
            self._penalise(logits, rows)
        chosen, held = self._choose(logits, rows, kinds)
        return Chosen(chosen, ops.token_logprobs(logits, chosen) if any(p.logprobs for p in kinds) else None, held=held)

    def _choose(self, logits: torch.Tensor, rows, kinds) -> tuple:
        """(the tokens, the _HeldPlace that they are written to as well or None)"""
        if all(p.is_greedy() for p in kinds):
            return ops.argmax_rows(logits), None
        n, vocab, small = len(rows), logits.shape[1], ops.sample_small_k()
        params, seeds, indices, _ = zip(*rows)
        packed = np.empty((5, n), dtype=np.float32)       # top_k as the bits of an int32
        if len(kinds) == 1:
            p = kinds[0]
            packed[:3] = [[p.temperature], [p.top_p], [p.min_p]]
            packed.view(np.int32)[4] = p.top_k
        else:
            packed[:3] = [[p.temperature for p in params], [p.top_p for p in params], [p.min_p for p in params]]
            packed.view(np.int32)[4] = [p.top_k for p in params]
        packed[3] = uniforms(seeds, indices)
        promises = dict(use_top_k=any(0 < p.top_k < vocab for p in kinds), use_top_p=any(p.top_p < 1.0 for p in kinds),
                        small_k=all(0 < p.top_k <= small and p.top_k < vocab or p.is_greedy() for p in kinds))
        if promises["small_k"] and n <= ops.sample_host_rows() and vocab <= ops.SAMPLE_FINISH_VOCAB:
            held = self._slots.take(n)      # the parameters travel with the launch
            if held is None:
                return ops.sample_rows(logits, packed, **promises), None
            try:
                return ops.sample_rows(logits, packed, host_out=held.memory, **promises), held
            finally:
                held.event.record()      # whatever fails from here on: the place is free when the kernel is done with it
        dev = upload(packed, self.device)      # one copy, queued: the host does not wait for the step that made the logits
        return ops.sample_rows(logits, dev[0], dev[4].view(torch.int32), dev[1], dev[2], dev[3], **promises), None

    def _penalise(self, logits, rows) -> None:
        indptr, toks, counts = [0], [], []
        for p, _, _, generated in rows:
            if p.has_penalties():
                seen: dict = {}
                for t in generated:
                    seen[t] = seen.get(t, 0) + 1
                toks.extend(seen.keys())
                counts.extend(seen.values())
            indptr.append(len(toks))
        i32 = lambda vals: torch.tensor(vals, dtype=torch.int32, device=self.device)
        f32 = lambda vals: torch.tensor(vals, dtype=torch.float32, device=self.device)
        ops.apply_penalties(logits, i32(indptr), i32(toks), i32(counts),
                            f32([p.repetition_penalty for p, _, _, _ in rows]),
                            f32([p.frequency_penalty for p, _, _, _ in rows]),
                            f32([p.presence_penalty for p, _, _, _ in rows]))
