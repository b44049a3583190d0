"""Portions and decoded tokens in one launch of the portions kernel (head_dim 128): one, several and more workgroups of
decoded tokens than compute units, keys cut over workgroups, segments of a few tokens, windows, pages of 8 to 64 slots, and
what the merge of a portion's parts does at each head size and number of parts.  Against the plain attention in 64 bits:
queries, keys and values are bfloat16 on both sides, the probabilities and the result are rounded by 2^-9 each, so 4e-3 in relative norm
and twice that allowed, as for the kernels by themselves."""
import random

import pytest
import torch

from test_kernels_gpu import _mfma_case, _rel

pytestmark = pytest.mark.gpu


def _shorts(count, longest, seed, tokens=(1,)):
    rng = random.Random(seed)
    return [(rng.randint(0, longest), rng.choice(tokens)) for _ in range(count)]


@pytest.mark.parametrize("nq,nkv,P,segs,window,splits", [
    (32, 8, 16, [(1000, 1)] + [(64, 300)], 0, None),                                      # one decoded token
    (32, 8, 16, _shorts(3, 5000, 1) + [(0, 17)], 0, None),                                # cut over workgroups by the rule
    (32, 8, 16, _shorts(20, 200, 2) + [(130, 140)] + _shorts(20, 200, 3), 0, None),       # more pairs than compute units
    (8, 2, 8, _shorts(150, 60, 4, (1, 2, 3, 4)) + [(0, 90), (33, 5)], 0, None),           # segments of up to sixteen rows
    (6, 2, 64, [(700, 1), (31, 1), (32, 1), (0, 1), (511, 200)], 0, 16),                  # a group that is no power of two
    (16, 1, 32, [(900, 1), (5, 130), (64, 1)], 50, 12),                                   # windows, cut keys that none holds
    (5, 5, 16, [(40, 1), (3, 16), (0, 40)], 7, 4),                                        # one head a group
    (32, 8, 16, [(2000, 1), (600, 100), (2000, 128)], 0, None),                           # portions in parts beside decoded tokens
])
def test_decoded_tokens_beside_portions(nq, nkv, P, segs, window, splits):
    got, want = _mfma_case(nq, nkv, 128, P, segs, window, splits, 900 + len(segs), stale_nan=True)
    assert torch.isfinite(got).all()
    assert _rel(got, want) < 8e-3
    row = 0
    for _, n in segs:      # no segment hides behind the others
        assert _rel(got[row:row + n], want[row:row + n]) < 2.5e-2
        row += n


@pytest.mark.parametrize("D,P", [(64, 16), (128, 16), (96, 16), (256, 32)])
@pytest.mark.parametrize("parts", [2, 3, 4, 5, 8])
def test_parts_of_a_portion_put_together(D, P, parts):
    got, want = _mfma_case(4, 2, D, P, [(900, 70), (45, 9), (2, 131)], 0, 1, 950 + D, portion_splits=parts)
    assert torch.isfinite(got).all()
    assert _rel(got, want) < 8e-3
