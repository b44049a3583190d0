"""A projection whose kernel adds into the residual and leaves the norm's division to the product that reads its rows, against the
float64 sums: strips of every kind of width (whole, 16 columns, a last one with columns missing), one to eight rows, K of one pair of
steps and of fewer pairs than waves, both types of norm weight; and the division in every variant of the reading product."""
import pytest
import torch

import plain_qwen3 as plain
from arle_amd.kernels import ops
from arle_amd.parts.linear import LateProduct, Linear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


def _made(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("N,K", [(1024, 64), (1500, 448), (2560, 4096), (2600, 640), (4096, 1088)])
@pytest.mark.parametrize("M,weight_type", [(1, torch.bfloat16), (2, torch.float32), (7, torch.bfloat16), (8, torch.float32)])
def test_strips_add_into_the_residual_and_leave_the_rows_and_their_squares(N, K, M, weight_type):
    x = _made(M, K + 8, seed=1).bfloat16().to(DEV)[:, :K]      # rows that do not lie side by side
    w = _made(N, K, seed=2, scale=0.05).bfloat16().to(DEV)
    residual = _made(M, N, seed=3, scale=3.0).to(DEV)
    weight = (1.0 + _made(N, seed=4, scale=0.3)).to(weight_type).to(DEV)
    want = residual.double() + x.double() @ w.double().T
    linear = Linear(w, tiles=True, strips=True)
    late = linear.late(x)
    assert isinstance(late, LateProduct)
    got = late.norm(residual, weight, EPS)
    # 32-bit sums of at most 4,096 exact products, and of N squares
    assert _rel(residual, want) < 1e-5
    squares = got.sums[:, :got.count].double().sum(1)
    assert _rel(squares, (want * want).sum(1)) < 1e-5
    # one rounding to bfloat16: half a unit of eight significant bits, 2^-8 of a value at most
    rows = want * weight.double()
    assert float(((got.rows.double() - rows).abs() - rows.abs() * 2.0 ** -8).max()) <= 1e-4
    assert (got.shape, got.dtype, got.count, got.width) == ((M, N), torch.bfloat16, -(-N // -(-N // 256)), N)


@pytest.mark.parametrize("N,K", [(2560, 9728), (2560, 4096), (1024, 3072), (2048, 6144), (4096, 4096)])
def test_the_residual_is_no_further_off_than_with_a_stack_of_partial_sums(N, K):
    """Its additions in 32 bits are ordered so that whole sums cost no accuracy against the product in parts that the norm adds."""
    whole, parts = 0.0, 0.0
    for seed in range(6):
        w = _made(N, K, seed=20 + seed, scale=0.02).bfloat16().to(DEV)
        linear = Linear(w, tiles=True, strips=True)
        for M in (1, 8):
            x = _made(M, K, seed=40 + seed).bfloat16().to(DEV)
            residual = _made(M, N, seed=60 + seed, scale=2.0).to(DEV)
            want = residual.double() + x.double() @ w.double().T
            by_parts, weight = residual.clone(), torch.ones(N, device=DEV)
            ops.add_rmsnorm(by_parts, linear(x, partials_ok=True), weight, EPS, torch.bfloat16)
            linear.late(x).norm(residual, weight, EPS)
            whole, parts = whole + _rel(residual, want), parts + _rel(by_parts, want)
    assert whole <= parts, (whole / 12, parts / 12)


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("variant,splits,fused", [(0, 1, False), (0, 3, False), (1, 2, False), (2, 1, False), (3, 1, False), (4, 2, False),
                                                  (0, 1, True), (1, 1, True), (3, 1, True), (4, 1, True)])
def test_the_reading_product_divides_its_sums(M, variant, splits, fused):
    N, K, count = 352, 1096, 250
    rows = _made(M, K, seed=5, scale=40.0).bfloat16().to(DEV)
    w = _made(N, K, seed=6, scale=0.05).bfloat16().to(DEV)
    sums = (_made(M, 256, seed=7).abs() * 800.0).to(DEV)
    sums[:, count:] = float("nan")      # behind the last strip's nothing was written
    scaled = ops.ScaledRows(rows, sums, count, K, EPS)
    divisor = torch.sqrt(sums[:, :count].double().sum(1, keepdim=True) / K + EPS)
    want = rows.double() @ w.double().T / divisor
    for tiles in (None, ops.pack_weight_tiles(w)):
        if fused:
            got = ops.gemm_rows(rows, w, torch.float32, ops.EPI_SILU_MUL, variant=variant, splits=1, tiles=tiles, scaled=scaled)
            pairs = want.view(M, -1, 2, 16)
            expected = (plain.silu(pairs[:, :, 0]) * pairs[:, :, 1]).reshape(M, -1)
        else:
            got = ops.gemm_rows(rows, w, torch.float32, variant=variant, splits=splits, tiles=tiles, scaled=scaled)
            got, expected = got.sum(0) if got.dim() == 3 else got, want
        assert _rel(got, expected) < 1e-5      # 32-bit sums of exact products, one division


def test_what_takes_no_strips_runs_as_before():
    w = _made(2560, 640, seed=8, scale=0.05).bfloat16().to(DEV)
    linear = Linear(w, tiles=True, strips=True)
    assert linear.strips is not None and not isinstance(linear.late(_made(9, 640, seed=9).bfloat16().to(DEV)), LateProduct)
    assert Linear(w, tiles=True).strips is None
    for n, k in ((512, 640), (5120, 640), (2560, 96)):      # too narrow, too wide, half a pair of steps left
        assert ops.strip_columns(n, k) == 0 and Linear(torch.zeros(n, k, dtype=torch.bfloat16, device=DEV), tiles=True, strips=True).strips is None
    wide = Linear(_made(4096, 640, seed=10).bfloat16().to(DEV), tiles=True, strips=True)
    assert wide.strips is wide.tiles      # sixteen columns: one layout
    rows = torch.zeros(9, 640, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ops.ShapeError):
        ops.gemm_strips(rows, linear.strips, torch.zeros(9, 2560, device=DEV), torch.ones(2560, device=DEV), EPS)
    with pytest.raises(ops.ShapeError):
        ops.gemm_rows(rows, w, scaled=ops.ScaledRows(rows, torch.zeros(9, 256, device=DEV), 4, 640, EPS))


def test_a_model_lays_strips_for_what_a_norm_runs_and_for_nothing_else():
    """o and down of every layer but the last down, which the final norm reads whole; steps of one to nine rows against the same model
    without copies of its weights."""
    from arle_amd.config import Qwen3Config
    from arle_amd.config.registry import detect_architecture
    from arle_amd.engine import Engine, StepEntry

    raw = dict(num_hidden_layers=3, hidden_size=1024, num_attention_heads=8, num_key_value_heads=2, head_dim=64, intermediate_size=1088,
               vocab_size=512, rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=True, max_position_embeddings=256)
    shapes = {"model.embed_tokens.weight": (512, 1024), "model.norm.weight": (1024,)}
    for i in range(3):
        p = f"model.layers.{i}."
        shapes |= {p + f"self_attn.{n}_proj.weight": s for n, s in (("q", (512, 1024)), ("k", (128, 1024)), ("v", (128, 1024)), ("o", (1024, 512)))}
        shapes |= {p + f"mlp.{n}_proj.weight": s for n, s in (("gate", (1088, 1024)), ("up", (1088, 1024)), ("down", (1024, 1088)))}
        shapes |= {p + f"self_attn.{n}_norm.weight": (64,) for n in "qk"}
        shapes |= {p + f"{n}_layernorm.weight": (1024,) for n in ("input", "post_attention")}
    weights = {n: (_made(*s, seed=100 + i, scale=0.04) if len(s) == 2 else 1.0 + _made(*s, seed=100 + i, scale=0.1)).bfloat16().to(DEV)
               for i, (n, s) in enumerate(sorted(shapes.items()))}
    recipe = detect_architecture({"architectures": ["Qwen3ForCausalLM"]}).recipe(Qwen3Config.from_dict(raw), ())
    engines = [Engine(recipe, dict(weights), dtype="bfloat16", max_slots=9, max_tokens=9 * 32, weight_tiles=tiles) for tiles in (True, False)]
    blocks = engines[0].model.blocks
    assert [b.mixer.o.strips is not None for b in blocks] == [True] * 3
    assert [b.feed_forward.down.strips is not None for b in blocks] == [True, True, False]
    assert all(b.mixer.o.strips is None and b.feed_forward.down.strips is None for b in engines[1].model.blocks)
    for rows in (1, 2, 7, 8, 9):
        logits = []
        for eng in engines:
            for r in range(rows):
                eng.add_request(r)
            eng.step([StepEntry(r, [5 + r, 6, 7], [2]) for r in range(rows)])
            logits.append(eng.step([StepEntry(r, [11 * r + 3], [0]) for r in range(rows)]).clone())
            for r in range(rows):
                eng.end_request(r)
        assert _rel(*logits) < 2e-2, rows      # three layers of bfloat16 rounding


def test_a_tuned_reader_is_charged_with_the_norm_in_front():
    """The tuner runs with a projection in front, and takes one in front of few rows into account only."""
    from arle_amd.kernels import tune

    n, k, front = 1536, 1024, (1024, 512)
    seen = []
    real = tune.pick
    try:
        tune.pick = lambda timed, ruled, apart=0.0: seen.append(apart) or real(timed, ruled, apart)
        table, report = tune.tune_products([("qkv", n, k, False, "norm")], device=DEV, rows=(1, 9), iters=4, behind={(n, k, False): front})
    finally:
        tune.pick = real
    assert list(table) == ["1536,1024,0,1"] and [r["rows"] for r in report] == [1, 9]
    assert seen[0] >= 0.0 and seen[1] == 0.0
    assert tune._apart(8, *front, DEV, 20) >= 0.0
