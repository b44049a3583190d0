"""Which projections a pre_norm model leaves to the norm behind them (and lays out a further time for that): those with a norm behind
them that can run them, and a reader of its rows behind that."""
import types

import pytest
import torch

from arle_amd.parts.attention import PagedAttention
from arle_amd.parts.block import PreNormBlock


class Late:
    """A mixer or feed-forward whose last projection may be left."""

    def __init__(self, reads=True, laid=True):
        self.leaves_late, self.reads_scaled, self.laid, self.asked = False, reads, laid, 0

    def leave_late(self):
        self.asked += 1
        self.leaves_late = self.laid

    def forward(self, x, *step, late=False):
        return ("late" if late else "whole", x)


class Plain:
    def forward(self, x, *step):
        return ("whole", x)


class Norm:
    def add_norm(self, residual, delta):
        return delta

    def add_late(self, residual, late):
        raise AssertionError("nothing here is a LateProduct")


class NormOnly:
    def add_norm(self, residual, delta):
        return delta


def _block(mixer, ffn, norm=Norm):
    return PreNormBlock(mixer, ffn, {"mixer_in": norm(), "ffn_in": norm()})


def _left(block, rows=2):
    """What the mixer's and the feed-forward's projections were when a step of `rows` rows ran."""
    residual = torch.zeros(rows, 4)
    _, delta = block.forward(residual, None, None, None)
    return delta[1][0] if block.feed_forward is not None else None, delta[0]


def test_a_mixer_is_left_to_the_norm_of_its_own_feed_forward_and_that_one_to_the_next_layer():
    first, last = _block(Late(), Late()), _block(Late(), Late())
    first.followed_by(last)
    assert _left(first) == ("late", "late")
    assert _left(last) == ("late", "whole") and last.feed_forward.asked == 0      # the final norm reads it whole
    assert _left(first, rows=9) == ("whole", "whole")


@pytest.mark.parametrize("reader", [Plain(), Late(reads=False)])
def test_without_a_reader_nothing_is_left_and_nothing_laid_out(reader):
    block = _block(Late(), reader)
    assert _left(block)[0] == "whole" and block.mixer.asked == 0
    block, following = _block(Late(), Late()), _block(reader, Late())
    block.followed_by(following)
    assert _left(block) == ("late", "whole") and block.feed_forward.asked == 0


def test_without_a_norm_that_can_run_it_or_behind_another_arrangement():
    block = _block(Late(), Late(), NormOnly)
    block.followed_by(_block(Late(), Late(), NormOnly))
    assert _left(block) == ("whole", "whole") and block.mixer.asked == block.feed_forward.asked == 0
    block = _block(Late(), Late())
    block.followed_by(object())
    assert _left(block) == ("late", "whole")


def test_what_could_not_be_laid_out_is_not_left():
    block = _block(Late(laid=False), Late(laid=False))
    block.followed_by(_block(Late(), Late()))
    assert _left(block) == ("whole", "whole")


def test_without_a_feed_forward_the_mixer_is_left_to_the_next_layer():
    block = PreNormBlock(Late(), None, {"mixer_in": Norm()})
    block.followed_by(_block(Late(), Late()))
    assert _left(block) == (None, "late")
    alone = PreNormBlock(Late(), None, {"mixer_in": Norm()})
    assert _left(alone) == (None, "whole")


def test_a_layer_is_asked_about_the_product_that_it_runs():
    """A table entry of the q rows alone says nothing about a layer that writes its own cache."""
    part = PagedAttention.__new__(PagedAttention)
    part.qkv = types.SimpleNamespace(takes_scaled=lambda rows: True)
    part.q_only = types.SimpleNamespace(takes_scaled=lambda rows: False)
    assert part.takes_scaled(1) and part.takes_scaled(1, types.SimpleNamespace(writes=True))
    assert not part.takes_scaled(1, types.SimpleNamespace(writes=False))
