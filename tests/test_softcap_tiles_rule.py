"""Which steps of the soft-capped attention at heads of 128 go to the kernel whose waves share their tiles, as far as sizes decide it;
the polynomial that this kernel caps scores with."""
import math
import os
import re

import pytest

from arle_amd.kernels import build, lib, ops


def _shares(lens, context, heads, kv_heads, known=True):
    longest = max(context + n for n in lens)
    return bool(lib.function("arle_attn_softcap_shares_tiles")(sum(lens), len(lens), max(lens), longest if known else 0, heads, kv_heads))


@pytest.mark.parametrize("heads,kv_heads", [(32, 4), (32, 8), (32, 16), (64, 8)])
def test_portions_that_fill_workgroups_share_them_from_144_on(heads, kv_heads):
    rows = 128 * kv_heads // heads                    # tokens of a workgroup
    blocks = -(-144 // kv_heads)
    for context in (0, 3000):
        assert _shares([rows * blocks], context, heads, kv_heads)
        assert not _shares([rows * (blocks - 1) - 1], context, heads, kv_heads)


@pytest.mark.parametrize("lens,heads,kv_heads,context,shares", [
    ([16] * 20, 32, 8, 0, False), ([16] * 20, 32, 8, 60, False), ([20] * 100, 32, 8, 0, False),     # short prompts, little to share
    ([20] * 100, 32, 8, 100, True), ([30] * 40, 32, 8, 0, True), ([64] * 12, 32, 8, 0, True),       # keys to share, or rows enough
    ([30] * 40, 32, 16, 100, False), ([8] * 100, 32, 16, 200, False), ([8] * 100, 32, 16, 400, True),   # two q heads a kv head
    ([64] * 20, 32, 16, 0, True), ([33] * 64, 32, 16, 40, True),
    ([16] * 20, 32, 4, 0, False), ([16] * 20, 32, 4, 400, False),           # a segment's rows fill one workgroup: 80 of them, not 160
    ([8] * 100, 32, 4, 100, True), ([33] * 64, 32, 4, 0, True),
])
def test_short_segments_share_tiles_where_they_are_many_or_long(lens, heads, kv_heads, context, shares):
    assert _shares(lens, context, heads, kv_heads) == shares


def test_decoded_rows_beside_a_portion_share_tiles_by_their_contexts():
    assert _shares([20] + [1] * 32, 1000, 32, 8) and not _shares([20] + [1] * 32, 10, 32, 8)
    assert _shares([20] + [1] * 32, 10, 32, 8, known=False)


def test_the_lines_lie_where_captured_steps_tell_contexts_apart():
    for line in (96, 224):
        assert ops.decode_split_cap(line) < ops.decode_split_cap(line + 1)


def test_the_caps_polynomial_is_as_far_off_as_it_says():
    with open(os.path.join(build.CSRC_DIR, "attention_softcap_portions.h")) as fh:
        text = fh.read()
    said, said_of_tanh = map(float, re.search(r"off by ([\d.e-]+), and t P from tanh by ([\d.e-]+);", text).groups())
    powers = [float(re.search(rf"c{n} = (-?[\d.]+)f \* sq", text).group(1)) for n in (1, 2, 3, 4)]
    off = off_of_tanh = 0.0
    for i in range(1, 20001):
        t = 0.5 * i / 20000
        p = 1.0 + sum(c * t ** (2 * n) for n, c in enumerate(powers, 1))
        off, off_of_tanh = max(off, abs(p - math.tanh(t) / t)), max(off_of_tanh, abs(t * p - math.tanh(t)))
    assert 0.9 * said < off < 1.1 * said and 0.9 * said_of_tanh < off_of_tanh < 1.1 * said_of_tanh
