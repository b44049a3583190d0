"""Portions of the soft-capped attention at heads of 128 where the waves of a workgroup share their tiles: penalties from the table
and computed, scores within half the cap and beyond it, windows that begin inside a tile, pages of 16 to 64 slots, several requests
with decoded rows among them, and values that are no numbers."""

import pytest
import torch

from test_softcap_rows_gpu import _reference

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def _run(q, k_pages, v_pages, table, lens, contexts, nq, nkv, page, window, cap, r1, r2, out_scale=1.0):
    from arle_amd.kernels import ops

    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)
    row0 = [0]
    for n in lens:
        row0.append(row0[-1] + n)
    out = torch.empty(row0[-1], nq * D, dtype=torch.bfloat16, device=DEV)
    return ops.attn_softcap_mfma(q, out, k_pages, v_pages, table, i32(row0), i32(list(range(len(lens)))), i32(contexts), max_qlen=max(lens),
                                 num_q_heads=nq, num_kv_heads=nkv, key_dim=D, value_dim=D, page_size=page, scale=D ** -0.5, softcap=cap,
                                 r1=r1, r2=r2, window=window, out_scale=out_scale)


def _inputs(lens, contexts, nkv, page, seed, window=0):
    """Pages of keys and values; with a window, pages that no row sees any more have been given back (-1 in the table)."""
    g = torch.Generator().manual_seed(seed)
    need = [(c + n + page - 1) // page for c, n in zip(contexts, lens)]
    order = torch.randperm(sum(need), generator=g).to(torch.int32)
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    k_pages = torch.full((sum(need), nkv, page, D), float("nan"), dtype=torch.bfloat16)   # slots never written stay NaN
    v_pages = torch.full((sum(need), nkv, D, page), float("nan"), dtype=torch.bfloat16)
    keys, values, at = [], [], 0
    for i, (c, n) in enumerate(zip(contexts, lens)):
        k, v = (torch.randn(c + n, nkv, D, generator=g).bfloat16() for _ in range(2))
        table[i, :need[i]] = order[at:at + need[i]]
        at += need[i]
        where = torch.arange(c + n)
        pages = table[i, where // page].long()
        k_pages[pages, :, where % page] = k
        v_pages[pages, :, :, where % page] = v
        table[i, :max(0, c - window + 1) // page if window else 0] = -1
        keys.append(k)
        values.append(v)
    return g, table, k_pages, v_pages, keys, values


@pytest.mark.parametrize("lens,contexts,nq,nkv,page,window,cap,penalty,loud", [
    ([300, 70], [0, 100], 64, 16, 16, 100, 30.0, True, 1.0),        # the table
    ([200], [1500], 64, 16, 32, 1024, 30.0, True, 1.0),             # its longest window
    ([40, 33, 1] * 6, [0, 5, 70] * 6, 64, 16, 16, 1000, 30.0, True, 1.0),   # the little of it that short contexts take
    ([190], [2100], 64, 16, 64, 300, 30.0, True, 1.0),              # pages given back in front of the window
    ([200], [1500], 64, 16, 16, 1025, 30.0, True, 1.0),             # one more: computed
    ([400], [33], 64, 16, 16, 0, 30.0, True, 1.0),                  # no window: computed
    ([300, 31], [5, 64], 64, 32, 16, 40, 30.0, True, 1.0),          # a group of two
    ([250], [70], 128, 16, 64, 90, 30.0, False, 1.0),               # a group of eight, one page a tile
    ([300], [0], 64, 16, 16, 0, 2.0, True, 1.0),                    # scores beyond half the cap
    ([300], [10], 64, 16, 16, 77, 30.0, True, 12.0),                # ... of some tiles
    ([300], [10], 64, 16, 16, 64, 0.0, True, 1.0),                  # no cap
    ([300], [10], 64, 16, 16, 0, 0.0, False, 1.0),                  # neither
    ([150, 1, 1, 40, 128], [3, 500, 63, 64, 0], 64, 16, 16, 70, 30.0, True, 1.0),
])
def test_portions_whose_waves_share_tiles_match_64_bits(lens, contexts, nq, nkv, page, window, cap, penalty, loud):
    g, table, k_pages, v_pages, keys, values = _inputs(lens, contexts, nkv, page, 11 + len(lens), window)
    q = (torch.randn(sum(lens), nq * D, generator=g) * torch.linspace(0.1, loud, sum(lens))[:, None] if loud > 1.0
         else torch.randn(sum(lens), nq * D, generator=g)).bfloat16()
    r1, r2 = (torch.rand(nq, generator=g).bfloat16(), torch.rand(nq, generator=g).bfloat16()) if penalty else (None, None)
    up = lambda t: None if t is None else t.to(DEV)
    got = _run(up(q), up(k_pages), up(v_pages), up(table), lens, contexts, nq, nkv, page, window, cap, up(r1), up(r2), out_scale=0.5)
    got = got.cpu().double().view(sum(lens), nq, D)
    first = 0
    for i, (c, n) in enumerate(zip(contexts, lens)):
        rows = slice(first, first + n)
        first += n
        for h in range(0, nq, 9):
            kv = h // (nq // nkv)
            want, of_abs = _reference(q[rows, h * D:(h + 1) * D], keys[i][:, kv], values[i][:, kv], c + torch.arange(n), D ** -0.5, cap,
                                      None if r1 is None else float(r1[h]), None if r2 is None else float(r2[h]), window, 0, 0, None)
            # probabilities and the result are rounded to bfloat16, by up to 2^-8 each; 32-bit scores (errors of 1e-5) add less than a tenth
            bound = 0.5 * (2.0 ** -8 * 1.1 * (of_abs + want.abs()) + 1e-6)
            assert ((got[rows, h] - 0.5 * want).abs() <= bound).all(), (i, h)


@pytest.mark.parametrize("rows,context,nq,nkv,window,bad", [(230, 20, 64, 16, 0, 20 + 17), (230, 20, 64, 16, 40, 20 + 47), (230, 20, 64, 16, 40, 3),
                                                           (200, 70, 64, 32, 33, 71), (120, 0, 128, 16, 0, 31)])
def test_a_value_that_is_no_number_stays_in_the_blocks_of_sixteen_rows_that_see_it(rows, context, nq, nkv, window, bad):
    page = 16
    g, table, k_pages, v_pages, _, _ = _inputs([rows], [context], nkv, page, 5)
    q = torch.randn(rows, nq * D, generator=g).bfloat16().to(DEV)
    spoilt = v_pages.clone()
    spoilt[table[0, bad // page].long(), :, :, bad % page] = float("nan")
    clean, got = (_run(q, k_pages.to(DEV), v.to(DEV), table.to(DEV), [rows], [context], nq, nkv, page, window, 30.0, None, None) for v in (v_pages, spoilt))
    assert torch.isfinite(clean).all()
    for first in range(0, rows, 16):
        at = range(context + first, context + min(first + 16, rows))
        sees = [bad <= p and (not window or p - bad < window) for p in at]
        assert any(sees) or torch.equal(got[first:first + 16], clean[first:first + 16]), first
        for p, s in zip(at, sees):
            assert not s or torch.isnan(got[p - context]).all(), p
