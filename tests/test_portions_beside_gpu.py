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


@pytest.mark.parametrize("segs,splits,most", [
    (_shorts(32, 1000, 6) + [(64, 300)], None, 0),       # uncut keys leave no parts: nothing
    ([(3000, 1)] * 8 + [(64, 300)], None, 4),            # four workgroups a request
    ([(500, 1)] * 8 + [(64, 300)], 3, 0),                # three waves are less than a workgroup
])
def test_the_parts_of_decoded_tokens_take_what_they_hold(segs, splits, most):
    from arle_amd.kernels import ops

    nq, nkv, D, P = 32, 8, 128, 16
    rows, pages = sum(n for _, n in segs), [-(-(a + b) // P) for a, b in segs]
    table = torch.zeros(len(segs), max(pages), dtype=torch.int32)
    for i, n in enumerate(pages):
        table[i, :n] = torch.arange(n) + sum(pages[:i])
    row0 = [0]
    for _, n in segs:
        row0.append(row0[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    k_pages, v_pages = (torch.randn(sum(pages), nkv, *s, device="cuda", dtype=torch.bfloat16) for s in ((P, D), (D, P)))
    q = torch.randn(rows, nq * D, device="cuda", dtype=torch.bfloat16)
    out = torch.empty_like(q)
    fixed = (table.cuda(), i32(row0), i32(list(range(len(segs)))), i32([a for a, _ in segs]))
    call = lambda: ops.attn_paged_mfma(q, out, k_pages, v_pages, *fixed, max_qlen=max(n for _, n in segs), min_qlen=1, num_q_heads=nq,
                                       max_kv_len=max(a + b for a, b in segs), max_portion_kv_len=364, num_kv_heads=nkv, head_dim=D, page_size=P,
                                       scale=D ** -0.5, splits=splits, short_segments=len(segs) - 1)
    call()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    call()
    assert torch.cuda.max_memory_allocated() - before <= most * len(segs) * 4 * nq * (D + 2) * 4 + 4096
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("segs,splits", [
    (_shorts(5, 300, 8) + [(90, 200)], 1),                                   # whole keys: the workgroup writes the result
    ([(2500, 1), (40, 1), (0, 1), (700, 1), (2500, 130)], 16),               # parts over four workgroups, some of them empty
])
def test_a_sink_and_a_factor_beside_portions(segs, splits):
    from arle_amd.kernels import ops
    from test_kernels_gpu import DEV, _fill_cache, _g, _paged_setup

    nq, nkv, D, P, out_scale = 8, 2, 128, 16, 0.5
    lengths = [a + b for a, b in segs]
    table, k_pages, v_pages = _paged_setup(lengths, nkv, D, P, torch.bfloat16, 60)
    sink = torch.linspace(-3.0, 6.0, nq)
    qs, wants, row0 = [], [], [0]
    for s, (cached, n) in enumerate(segs):
        g = _g(61 + s)
        q, k, v = (torch.randn(rows, h, D, generator=g).bfloat16() for rows, h in ((n, nq), (cached + n, nkv), (cached + n, nkv)))
        _fill_cache(table, k_pages, v_pages, s, k, v, P)
        ahead = torch.arange(cached + n)[None, :] > cached + torch.arange(n)[:, None]
        want = torch.empty(n, nq, D, dtype=torch.float64)
        for h in range(nq):
            kv = h // (nq // nkv)
            scores = (q[:, h].double() @ k[:, kv].double().T / D ** 0.5).masked_fill(ahead, float("-inf"))
            probs = torch.softmax(torch.cat([scores, sink[h].double().expand(n, 1)], 1), -1)[:, :-1]     # the sink's share has no value
            want[:, h] = out_scale * (probs @ v[:, kv].double())
        wants.append(want.view(n, -1))
        qs.append(q.view(n, -1))
        row0.append(row0[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    q_all = torch.cat(qs).to(DEV)
    out = torch.full_like(q_all, float("nan"))
    ops.attn_paged_mfma(q_all, out, k_pages.to(DEV), v_pages.to(DEV), table.to(DEV), i32(row0), i32(list(range(len(segs)))),
                        i32([a for a, _ in segs]), max_qlen=max(n for _, n in segs), min_qlen=1, max_kv_len=max(lengths), num_q_heads=nq,
                        num_kv_heads=nkv, head_dim=D, page_size=P, scale=D ** -0.5, splits=splits, sink=sink.to(DEV), out_scale=out_scale)
    for want, first, last in zip(wants, row0, row0[1:]):
        assert _rel(out[first:last].cpu(), want) < (8e-3 if last - first > 1 else 2.5e-2)


def test_more_pairs_than_the_portions_list_holds():
    """1,100 decoded tokens beside a portion whose keys would be cut into parts: its row blocks times all segments are more
    than the list of pairs holds, without which there are no parts."""
    segs = [(i % 5, 1) for i in range(1100)] + [(700, 500)]
    got, want = _mfma_case(16, 4, 128, 16, segs, 0, None, 77, short=1100)
    assert torch.isfinite(got).all()
    assert _rel(got, want) < 8e-3 and _rel(got[-500:], want[-500:]) < 8e-3
