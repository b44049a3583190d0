"""Steps of single decoded tokens whose keys are shared out over all waves of a kv head: ragged and equal contexts,
more requests than a wave has lanes, windows, and the plan that later layers take from the first.  The unsplit form of
the same kernel (one wave a request and kv head) is the reference: it walks the keys in the same blocks, so the results
differ by the order of float32 sums and one rounding to bfloat16 (2^-9), stated as a relative norm of 4e-3."""
import random

import pytest
import torch

pytestmark = pytest.mark.gpu
D, P, NQ, NKV = 128, 16, 8, 2


def _case(contexts, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    pages = [-(-(c + 1) // P) for c in contexts]
    table = torch.zeros((len(contexts), max(pages)), dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(seed)).int(), 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    k, v = rand(at, NKV, P, D).bfloat16(), rand(at, NKV, D, P).bfloat16()
    parts = rand(2, len(contexts), (NQ + 2 * NKV) * D)
    i32 = lambda vals: torch.tensor(vals, dtype=torch.int32, device="cuda")
    n = len(contexts)
    return parts, k, v, table.cuda(), i32(list(range(n + 1))), i32(list(range(n))), i32(contexts)


def _run(case, contexts, **kw):
    from arle_amd.kernels import ops

    parts, k, v, table, row0, slot, start = case
    out = torch.full((len(contexts), NQ * D), float("nan"), dtype=torch.bfloat16, device="cuda")
    return ops.attn_decode_prep(parts, out, k.clone(), v.clone(), table, row0, slot, start, max_kv_len=max(contexts) + 1,
                                num_q_heads=NQ, num_kv_heads=NKV, head_dim=D, page_size=P, scale=D ** -0.5, eps=1e-6, **kw)


@pytest.mark.parametrize("contexts,window", [
    ([0], 0), ([31], 0), ([5000], 0),                                          # one request: one block, and more than 64 blocks
    ([0, 0, 0], 0), ([31, 32, 33, 4095, 0], 0), ([700] * 7, 0),
    ([random.Random(1).randrange(0, 900) for _ in range(63)] + [6000], 0),     # as many as lanes, one long
    ([random.Random(2).randrange(0, 300) for _ in range(65)], 0),              # one more than lanes
    ([3000] + [1] * 140 + [2500], 0),                                          # three lots of lanes
    ([17, 900, 64, 3], 50), ([random.Random(3).randrange(0, 400) for _ in range(70)], 33),
])
def test_shared_out_keys_give_what_one_wave_a_request_gives(contexts, window):
    from arle_amd.kernels import ops

    case = _case(contexts, 7 + len(contexts))
    want = _run(case, contexts, window=window, splits=1).float()
    splits, waves = ops.decode_share(len(contexts), NKV, max(contexts) + 1, sum(contexts) + len(contexts))
    for kw in (dict(total_kv_len=sum(contexts) + len(contexts)), dict(splits=5)):
        carry = {}
        got = _run(case, contexts, window=window, carry=carry, **kw)
        assert torch.isfinite(got.float()).all()
        assert float((got.float() - want).norm() / want.norm()) < 4e-3
        assert torch.equal(got, _run(case, contexts, window=window, carry=carry, **kw))    # a later layer: the plan is there
    assert waves == 0 or len(contexts) < waves <= max(512, 2 * len(contexts))


@pytest.mark.parametrize("segments,kv_heads,longest", [(1, 8, 1), (1, 8, 40), (3, 8, 4096), (64, 8, 2048), (100, 8, 2048), (700, 8, 900),
                                                       (2, 4096, 4096)])
def test_the_number_of_waves(segments, kv_heads, longest):
    from arle_amd.kernels import ops

    for total in (None, segments * longest, segments - 1 + longest):
        splits, waves = ops.decode_share(segments, kv_heads, longest, total)
        assert 1 <= splits <= 64 and (waves == 0 or (splits > 1 and segments < waves <= 65535))


def _exact(parts, k_pages, v_pages, table, contexts, D, nq, nkv, weights, angles, window):
    """The step in 64 bits: projections added, q and k normed and rotated, the new token's key and value rounded to bfloat16
    as the cache holds them."""
    y = parts.double() if parts.dim() == 2 else parts.double().sum(0)
    out = []
    for s, context in enumerate(contexts):
        q, k, v = (y[s, a * D:b * D].view(-1, D) for a, b in ((0, nq), (nq, nq + nkv), (nq + nkv, nq + 2 * nkv)))
        if weights is not None:
            q, k = (t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6) * w.double() for t, w in zip((q, k), weights))
        if angles is not None:
            rot = 2 * angles[0].shape[1]
            cos, sin = (t[context].double() for t in angles)
            turn = lambda t: torch.cat([t[:, :rot // 2] * cos - t[:, rot // 2:rot] * sin, t[:, rot // 2:rot] * cos + t[:, :rot // 2] * sin, t[:, rot:]], 1)
            q, k = turn(q), turn(k)
        pages = table[s, :context // P + 1].long()
        keys = k_pages[pages].transpose(1, 2).reshape(-1, nkv, D)[:context].double()
        values = v_pages[pages].permute(0, 3, 1, 2).reshape(-1, nkv, D)[:context].double()
        keys, values = torch.cat([keys, k.bfloat16().double()[None]]), torch.cat([values, v.bfloat16().double()[None]])
        first = max(0, context + 1 - window) if window else 0
        for h in range(nq):
            score = keys[first:, h * nkv // nq] @ q[h] * D ** -0.5
            out.append(torch.softmax(score, 0) @ values[first:, h * nkv // nq])
    return torch.stack(out).view(len(contexts), nq * D)


@pytest.mark.parametrize("D,nq,nkv,whole,normed,rot", [(128, 8, 2, False, True, 128), (128, 16, 1, True, True, 128), (64, 6, 2, True, True, 64),
                                                       (64, 8, 8, False, False, 0), (128, 4, 2, True, False, 64)])
@pytest.mark.parametrize("contexts,window", [([0, 31, 32, 33, 4095, 100], 0), ([700] * 5, 0), ([17, 900, 64, 3], 50), ([5000], 0),
                                             ([random.Random(2).randrange(0, 300) for _ in range(65)], 0)])
def test_shared_out_keys_against_64_bits(D, nq, nkv, whole, normed, rot, contexts, window):
    """Every form of the input at both head sizes.  Queries are rounded to bfloat16 in front of the first product, probabilities
    in front of the second and the result once more, each by at most 2^-9 of its size, with scores of a spread of one
    and averages over the keys behind the first two: 3e-3 in relative norm; half as much again is allowed."""
    from arle_amd.kernels import ops

    gen = torch.Generator(device="cuda").manual_seed(len(contexts) + D)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    pages = [c // P + 1 for c in contexts]
    table = torch.zeros((len(contexts), max(pages)), dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(1)).int(), 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    k_pages, v_pages = rand(at, nkv, P, D).bfloat16(), rand(at, nkv, D, P).bfloat16()
    width = (nq + 2 * nkv) * D
    parts = rand(len(contexts), width).bfloat16() if whole else rand(3, len(contexts), width) * 0.577
    weights = (1 + 0.1 * rand(D)).bfloat16(), (1 + 0.1 * rand(D)).bfloat16()
    weights = weights if normed else None
    angle = torch.arange(max(contexts) + 1, device="cuda")[:, None] * 10000.0 ** (-torch.arange(max(rot // 2, 1), device="cuda") / max(rot // 2, 1))
    angles = (torch.cos(angle).float().contiguous(), torch.sin(angle).float().contiguous()) if rot else None
    want = _exact(parts, k_pages, v_pages, table.cuda(), contexts, D, nq, nkv, weights, angles, window)
    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")
    n = len(contexts)
    for total in (sum(contexts) + n, None):
        out = torch.full((n, nq * D), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.attn_decode_prep(parts, out, k_pages.clone(), v_pages.clone(), table.cuda(), i32(list(range(n + 1))), i32(list(range(n))),
                             i32(contexts), max_kv_len=max(contexts) + 1, num_q_heads=nq, num_kv_heads=nkv, head_dim=D, page_size=P,
                             scale=D ** -0.5, eps=1e-6, q_weight=weights and weights[0], k_weight=weights and weights[1],
                             cos=angles and angles[0], sin=angles and angles[1], rotary_dim=rot, window=window, total_kv_len=total, carry={})
        err = float((out.double() - want).norm() / want.norm())
        assert err < 4.5e-3, (total, err)


def test_captured_steps_across_equal_and_ragged_contexts(tmp_path):
    """32 requests with 8 kv heads, a pair for every compute unit: contexts alike (splits inside a workgroup), then one graph
    for ragged ones, replayed with two other sets of ragged contexts, then the first graph again.  Every step's logits are
    those of an engine without graphs, bit for bit, and the plain implementation's within its bfloat16 tolerance."""
    import replay
    from arle_amd.config import Qwen3Config
    from arle_amd.engine import Engine
    from arle_amd.kernels import ops
    from arle_amd.weights import write_random_model
    from tiny import random_tokens, read_folder

    raw = dict(num_hidden_layers=2, hidden_size=96, num_attention_heads=8, num_key_value_heads=8, head_dim=64, intermediate_size=160,
               vocab_size=307, rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=True, max_position_embeddings=512)
    d = write_random_model(str(tmp_path / "m"), "Qwen3ForCausalLM", Qwen3Config.from_dict(raw), seed=5, std=0.08, norm_std=0.05)
    cfg, weights = read_folder(d)
    make = lambda graphs: Engine.from_folder(d, dtype="bfloat16", page_size=16, max_tokens=32 * 192, max_slots=32, max_request_tokens=192,
                                             cuda_graph=graphs)
    requests, steps = {}, []

    def phase(name, prompts, decoded, kept=()):
        """New requests of these lengths beside the kept ones, `decoded` steps of all 32; the new ones' names."""
        new = [f"{name}{i}" for i in range(len(prompts))]
        for rid, n in zip(new, prompts):
            requests[rid] = random_tokens(n, 307, len(requests))
        for first in range(0, len(new), 8):
            some = new[first:first + 8]
            steps.append({"entries": [(rid, list(requests[rid]), [len(requests[rid]) - 1]) for rid in some], "end": []})
        for _ in range(decoded):
            entries = []
            for rid in list(kept) + new:
                token = (7 * len(requests[rid]) + len(entries)) % 307
                entries.append((rid, [token], [0]))
                requests[rid].append(token)
            steps.append({"entries": entries, "end": []})
        return new

    alike = phase("a", [140] * 32, 3)
    assert ops.decode_share(32, 8, 143, 32 * 143)[1] == 0
    steps[-1]["end"] = alike[8:]
    short = phase("b", [10 + i for i in range(24)], 3, alike[:8])           # ragged: the first capture of that class
    assert ops.decode_share(32, 8, 146, 8 * 146 + sum(13 + i for i in range(24)))[1] > 0
    steps[-1]["end"] = short[:20] + alike[:4]
    long = phase("c", [1, 2, 150, 33, 64] * 4 + [5, 6, 120, 31], 3, alike[4:8] + short[20:])   # and replays of it
    steps[-1]["end"] = long + short[20:] + alike[4:8]
    phase("d", [141] * 32, 2)                                               # alike again
    eager = replay.run_steps(make(False), steps)
    engine = make(True)
    graphed = replay.run_steps(engine, steps)
    assert len([key for key in engine._graphs if key[0] == 32]) == 2 and engine.graph_replays >= 7
    assert eager.keys() == graphed.keys()
    for key in eager:
        assert torch.equal(eager[key], graphed[key]), key
    some = {rid: requests[rid] for rid in (alike[0], alike[9], short[3], short[22], long[2], long[0], "d31")}
    replay.check_rows(graphed, {rid: replay.plain_logits(cfg, weights, tokens) for rid, tokens in some.items()}, 2e-2,
                      "decode across classes", need_all=False)
