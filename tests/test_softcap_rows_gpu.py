"""Portions in the matrix-core kernel of the soft-capped attention where a wave takes 32 rows, and just below."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

# q heads so many that the row blocks of 32 make waves enough for two blocks of sixteen a wave; the last one stays below
CASES = [
    # lens, contexts, nq, nkv, Dk, Dv, page, window, chunk, keep, cap, penalty, sink
    ([33, 1, 31, 32], [0, 5, 64, 7], 192, 48, 32, 32, 16, 0, 0, 0, 30.0, False, False),
    ([17, 65, 2], [40, 3, 0], 256, 128, 24, 16, 16, 9, 0, 0, 5.0, True, True),
    ([95, 16], [100, 1], 208, 208, 64, 48, 48, 40, 0, 21, 0.0, False, True),
    ([64, 63], [31, 32], 256, 64, 128, 128, 32, 33, 0, 0, 30.0, True, False),
    ([48, 49], [17, 0], 256, 64, 128, 112, 16, 0, 24, 0, 2.0, False, False),
    ([33, 15], [50, 9], 32, 8, 128, 128, 16, 20, 0, 0, 30.0, False, False),
]


def _reference(q, k, v, pos, scale, cap, r1, r2, window, chunk, keep, sink):
    """[n, Dk] queries of one head at positions pos over [S, D] keys and values, in 64 bits; and the same of |v|."""
    s = (q.double() @ k.double().T) * scale
    if cap > 0:
        s = cap * torch.tanh(s / cap)
    key = torch.arange(k.shape[0])
    gap = pos[:, None] - key[None]
    if r1 is not None:
        s = s - r1 * torch.log1p(r2 * gap.clamp(min=0))
    seen = gap >= 0
    if window:
        seen &= (gap < window) | (key[None] < keep)
    if chunk:
        seen &= key[None] // chunk == pos[:, None] // chunk
    s = s.masked_fill(~seen, -math.inf)
    top = s.amax(1, keepdim=True)
    if sink is not None:
        top = top.clamp(min=sink)
    p = torch.exp(s - top)
    total = p.sum(1, keepdim=True) + (0.0 if sink is None else torch.exp(sink - top))
    return p @ v.double() / total, p @ v.double().abs() / total


@pytest.mark.parametrize("case", CASES)
def test_rows_in_blocks_of_32_match_64_bit_attention(case):
    from arle_amd.kernels import ops

    lens, contexts, nq, nkv, Dk, Dv, page, window, chunk, keep, cap, penalty, with_sink = case
    g = torch.Generator().manual_seed(7)
    rnd = lambda *shape: torch.randn(*shape, generator=g)
    need = [(c + n + page - 1) // page for c, n in zip(contexts, lens)]
    order = torch.randperm(sum(need), generator=g).to(torch.int32)
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    k_pages = torch.full((sum(need), nkv, page, Dk), float("nan"), dtype=torch.bfloat16)   # slots never written stay NaN
    v_pages = torch.full((sum(need), nkv, Dv, page), float("nan"), dtype=torch.bfloat16)
    keys, values, at = [], [], 0
    for i, (c, n) in enumerate(zip(contexts, lens)):
        k, v = rnd(c + n, nkv, Dk).bfloat16(), rnd(c + n, nkv, Dv).bfloat16()
        table[i, :need[i]] = order[at:at + need[i]]
        at += need[i]
        for j in range(c + n):
            k_pages[table[i, j // page], :, j % page] = k[j]
            v_pages[table[i, j // page], :, :, j % page] = v[j]
        keys.append(k)
        values.append(v)
    T = sum(lens)
    q = rnd(T, nq * Dk).bfloat16()
    r1, r2 = (torch.rand(nq, generator=g), torch.rand(nq, generator=g)) if penalty else (None, None)
    sink = rnd(nq) if with_sink else None
    row0 = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    up = lambda t: None if t is None else t.to(DEV)
    i32 = lambda values_: torch.tensor(values_, dtype=torch.int32, device=DEV)
    out = torch.empty(T, nq * Dv, dtype=torch.bfloat16, device=DEV)
    ops.attn_softcap_mfma(up(q), out, up(k_pages), up(v_pages), up(table), up(row0), i32(list(range(len(lens)))), i32(contexts),
                          max_qlen=max(lens), num_q_heads=nq, num_kv_heads=nkv, key_dim=Dk, value_dim=Dv, page_size=page,
                          scale=Dk ** -0.5, softcap=cap, r1=up(r1), r2=up(r2), window=window, chunk=chunk, sink=up(sink),
                          keep_first=keep)
    got = out.cpu().double().view(T, nq, Dv)
    for i, (c, n) in enumerate(zip(contexts, lens)):
        rows = slice(int(row0[i]), int(row0[i]) + n)
        for h in range(0, nq, 11):
            kv = h // (nq // nkv)
            want, of_abs = _reference(q[rows, h * Dk:(h + 1) * Dk], keys[i][:, kv], values[i][:, kv], c + torch.arange(n),
                                      Dk ** -0.5, cap, None if r1 is None else float(r1[h]), None if r2 is None else float(r2[h]),
                                      window, chunk, keep, None if sink is None else float(sink[h]))
            # probabilities are rounded to bfloat16 in front of the second product and the result once more: eight significant
            # bits, so half a unit of the last is up to 2^-8 of the number; 32-bit scores (errors of 1e-5) add less than a tenth
            bound = 2.0 ** -8 * 1.1 * (of_abs + want.abs()) + 1e-6
            assert ((got[rows, h] - want).abs() <= bound).all(), (i, h)


@pytest.mark.parametrize("rows,context,window,keep,nq,bad", [(96, 20, 0, 0, 512, 20 + 17), (96, 20, 40, 0, 512, 20 + 47), (96, 20, 40, 0, 512, 3),
                                                             (70, 0, 33, 0, 512, 31), (96, 70, 40, 5, 512, 3), (96, 20, 40, 0, 8, 20 + 47)])
def test_a_value_that_is_no_number_stays_in_the_blocks_of_sixteen_rows_that_see_it(rows, context, window, keep, nq, bad):
    """The key's blocks of sixteen rows (counted from the portion's first) may all become NaN; every other block keeps its bits,
    with 32 rows a wave (the first five cases) as with sixteen."""
    from arle_amd.kernels import ops

    nkv, D, page = 8, 32, 16
    g = torch.Generator(device=DEV).manual_seed(3)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV).bfloat16()
    pages = -(-(rows + context) // page)
    q, k, v = rnd(rows, nq * D), rnd(pages, nkv, page, D), rnd(pages, nkv, D, page)
    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)

    def run(v_pages):
        out = torch.empty(rows, nq * D, dtype=torch.bfloat16, device=DEV)
        ops.attn_softcap_mfma(q, out, k, v_pages, i32([list(range(pages))]), i32([0, rows]), i32([0]), i32([context]), max_qlen=rows,
                              num_q_heads=nq, num_kv_heads=nkv, key_dim=D, value_dim=D, page_size=page, scale=D ** -0.5, softcap=30.0,
                              window=window, keep_first=keep)
        return out

    spoilt = v.clone()
    spoilt[bad // page, :, :, bad % page] = float("nan")
    clean, got = run(v), run(spoilt)
    assert torch.isfinite(clean).all()
    for first in range(0, rows, 16):
        at = range(context + first, context + min(first + 16, rows))
        sees = any(bad <= p and (not window or p - bad < window or bad < keep) for p in at)
        block = slice(first, first + 16)
        assert torch.equal(got[block], clean[block]) or sees, first
        for p in at:
            if bad <= p and (not window or p - bad < window or bad < keep):
                assert torch.isnan(got[p - context]).all(), p
