"""What `ops.attn_decode_prep` hands its launches as the plan of a pass, looked at on the host: a plan counts as made only
where an earlier launch of the pass has written it."""
import pytest
import torch

from arle_amd.kernels import ops

D, P, SEGMENTS = 128, 16, 64


@pytest.fixture
def launches(monkeypatch):
    """The plan and plan_made of every launch that would have gone out, in order."""
    seen = []
    monkeypatch.setattr(ops, "_gpu", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    names = ("splits", "ws_o", "ws_ml", "waves", "plan", "plan_made", "stream")
    monkeypatch.setattr(ops.lib, "call", lambda name, *args: seen.append(dict(zip(names, args[-len(names):]))))
    return seen


def _layer(kv_heads, keys, carry, **kw):
    heads = 8
    i32 = lambda values: torch.tensor(list(values), dtype=torch.int32)
    ops.attn_decode_prep(torch.zeros(1, SEGMENTS, (heads + 2 * kv_heads) * D), torch.zeros(SEGMENTS, heads * D, dtype=torch.bfloat16),
                         torch.zeros(1, kv_heads, P, D, dtype=torch.bfloat16), torch.zeros(1, kv_heads, D, P, dtype=torch.bfloat16),
                         torch.zeros(SEGMENTS, keys // P, dtype=torch.int32), i32(range(SEGMENTS + 1)), i32(range(SEGMENTS)),
                         i32([keys - 1] * SEGMENTS), max_kv_len=keys, num_q_heads=heads, num_kv_heads=kv_heads, head_dim=D, page_size=P,
                         scale=1.0, eps=1e-6, carry=carry, **kw)


def test_the_two_forms_meet_in_these_sizes():
    """64 requests of 128 keys: with 8 kv heads the splits stay inside a workgroup (which writes no plan), with 2 the keys are
    shared out over as many waves as the former has splits."""
    assert ops.decode_share(SEGMENTS, 8, 128) == (2, 0) and ops.decode_share(SEGMENTS, 2, 128) == (2, 128)


def _made(launches, layers):
    carry = {}
    for kv_heads, kw in layers:
        _layer(kv_heads, 128, carry, **kw)
    return [(call["waves"], call["plan_made"]) for call in launches]


@pytest.mark.parametrize("before", [[(8, {})], [(8, {"splits": 2})], [(2, {"splits": 2})], [(8, {}), (8, {})]])
def test_the_first_shared_out_layer_makes_the_plan_whatever_ran_before_it(launches, before):
    found = _made(launches, before + [(2, {}), (2, {})])
    assert found[-2:] == [(128, 0), (128, 1)] and all(made == 0 for _, made in found[:-1])
    assert launches[-1]["plan"] == launches[-2]["plan"]
