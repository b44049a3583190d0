"""What a decode step's captured graph is found by: the distinct answers of the model's parts, asked of one part of every kind
and sizes."""
import pytest

from arle_amd.models.decoder import DecoderModel, parts_that_answer
from arle_amd.parts.attention import PagedAttention
from arle_amd.parts.base import Part
from arle_amd.parts.mixer_pair import MixerPair
from arle_amd.parts.rotary_attention import RotaryAttention


class _Rt:
    is_f32 = False


def _made(kind, children=(), **attributes):
    part = object.__new__(kind)
    part.rt, part.child_parts = _Rt(), dict(children)
    for name, value in attributes.items():
        setattr(part, name, value)
    return part


def _paged(nkv=8, window=None, folds=True):
    return _made(PagedAttention, D=128, nkv=nkv, window=window, folds_preparation=folds)


def _rotary(nkv=4, window=0):
    return _made(RotaryAttention, Dk=128, Dv=128, nkv=nkv, softcap=0.0, window=window)


def _pair(left, right):
    return _made(MixerPair, {"left": left, "right": right}, left=left, right=right)


class _Silent(Part):
    def __init__(self, **children):
        super().__init__({}, {}, _Rt(), children)


class _Own(Part):
    """A part that answers and says nothing of its sizes."""

    def __init__(self, step):
        super().__init__({}, {}, _Rt())
        self.step = step

    def decode_launch_class(self, rows, max_context):
        return max_context // self.step


class _Stranger:
    """No `Part`, as a model's author may write one."""

    def decode_launch_class(self, rows, max_context):
        return rows + max_context


def _model(parts):
    model = object.__new__(DecoderModel)
    model.parts, model._answering = parts, parts_that_answer(parts)
    return model


def _asked_of_all(parts, rows, longest, total):
    found = set()
    for part in parts:
        for name, args in (("decode_launch_class", (rows, longest)), ("decode_spread_class", (rows, longest, total))):
            answer = getattr(part, name, lambda *a: None)(*args)
            if answer is not None:
                found.add((name, answer))
    return tuple(sorted(found, key=repr))


PARTS = {
    "layers alike": lambda: [_Silent() for _ in range(111)] + [_paged() for _ in range(36)],
    "windows and kv heads": lambda: [_paged(), _paged(window=64), _paged(nkv=2), _paged(folds=False), _paged()],
    "pairs": lambda: [_pair(_paged(), _rotary()), _pair(_paged(), _rotary()), _pair(_paged(), _rotary(window=32)), _pair(_Silent(), _Silent())],
    "own answers": lambda: [_Own(7), _Own(100), _Silent(inner=_paged(nkv=4)), _Stranger(), _Silent()],
}


@pytest.mark.parametrize("name", PARTS)
def test_the_answers_are_those_of_all_parts(name):
    parts = PARTS[name]()
    model = _model(parts)
    for rows in (1, 3, 19, 64, 200):
        for longest in (1, 40, 128, 700, 4096):
            for total in (rows * longest, rows - 1 + longest, None):
                assert model.decode_launch_class(rows, longest, total) == _asked_of_all(parts, rows, longest, total or rows * longest)


def test_one_part_of_a_kind_is_asked():
    """147 parts with 36 layers alike: one attention is asked, twice a step."""
    for name, most in (("layers alike", 1), ("windows and kv heads", 4), ("pairs", 2), ("own answers", 4)):
        assert len(parts_that_answer(PARTS[name]())) == most, name
