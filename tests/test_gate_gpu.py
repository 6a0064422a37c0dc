"""Gate products with SiLU in their epilogue, alone and grouped by expert, in every tile the row count picks: the four-wave tile, the smaller
ones, remainders of rows, columns and groups, empty and single-row groups.  Against the layers' equations in float64."""
import pytest
import torch

import lm_util as U
from oracle import layered_lm_oracle as O

pytestmark = pytest.mark.gpu


def run(cfg, rows, gain=1.5):
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    w = U.weights(cfg, 3, gain)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=torch.bfloat16, max_batch=64, max_context=512)
    n = -(-rows // 400)
    ts = [U.tokens(min(400, rows - 400 * i), cfg["vocab"], i) for i in range(n)]
    got = m.step([(m.open_sequence(), t, range(len(t))) for t in ts])
    return got, torch.cat([O.forward(cfg, w, t) for t in ts])


def mixer():
    return U.latent(1, 32, 32, 64)


@pytest.mark.parametrize("rows,ff", [(29, 100), (64, 330), (65, 330), (128, 70), (129, 330), (300, 2900), (700, 2900), (1100, 3000), (2300, 1300)])
def test_dense(rows, ff):
    got, want = run(U.stream_config([(mixer(), U.dense(ff))], width=320, vocab=120, streams=1, positions=400), rows)
    assert U.logit_error(got, want) < 3e-2


@pytest.mark.parametrize("rows,experts,top,ff", [(3, 5, 2, 40), (40, 6, 2, 300), (130, 7, 3, 300), (500, 9, 2, 200), (700, 4, 3, 200), (2100, 3, 2, 330), (1500, 40, 1, 70)])
def test_experts(rows, experts, top, ff):
    got, want = run(U.stream_config([(mixer(), U.moe(experts, top, ff))], width=320, vocab=120, streams=1, positions=400), rows)
    e = U.logit_errors(got, want).sort().values
    # a router between nearly equal logits may choose another expert at single rows
    assert float(e[int(0.9 * (len(e) - 1))]) < 3e-2 and float(e.median()) < 1e-2


def test_a_step_rounds_its_gates_alike_on_every_tile():
    """Up to 128 rows gates stay in fp32 until they are multiplied; 64 rows per expert and one K slice (128 rows, 8 experts, 4 of them, 2752
    columns) reach for another tile than 50 rows per expert do."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.stream_config([(mixer(), U.moe(8, 4, 1376))] * 2, width=320, vocab=120, streams=1, positions=64)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), U.weights(cfg, 3, 1.5), dtype=torch.bfloat16, max_batch=8, max_context=64)
    ts = [U.tokens(n, cfg["vocab"], n) for n in (50, 49, 29)]
    few, many = (m.step([(m.open_sequence(), t, range(len(t))) for t in part]) for part in (ts[:2], ts))
    assert torch.equal(few, many[:99])


@pytest.mark.parametrize("rows,experts,top,ff", [(1, 5, 2, 40), (3, 40, 7, 100), (8, 5, 3, 330), (9, 9, 1, 64), (16, 4, 2, 200), (17, 8, 4, 130), (40, 9, 2, 70),
                                                 (41, 16, 4, 70), (128, 110, 8, 30), (120, 110, 9, 30)], ids=str)
@pytest.mark.parametrize("alike", [False, True], ids=["spread", "one_choice"])
def test_experts_of_a_step(rows, experts, top, ff, alike):
    """Single tokens through the experts: a workgroup per choice and per expert, up to 8 and more than 16 choices of one expert, K of one unit, the most
    choices that go by themselves and the first that are sorted."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.stream_config([(mixer(), U.moe(experts, top, ff))], width=320, vocab=120, streams=2, positions=64)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=torch.bfloat16, max_batch=128, max_context=64)
    ts = [U.tokens(1, cfg["vocab"], 0 if alike else i) for i in range(rows)]
    got = m.step([(m.open_sequence(), t, [0]) for t in ts])
    want = torch.cat([O.forward(cfg, w, t) for t in ts[: 1 if alike else rows]]).expand(rows, -1)
    e = U.logit_errors(got, want)
    # (every row: no choice is so near with these weights that rounding turns it over)
    assert float(e.max()) < 3e-2 and float(e.median()) < 1e-2
    if alike:
        assert bool((got == got[:1]).all())


@pytest.mark.parametrize("streams,width", [(1, 320), (2, 2112), (4, 136), (5, 64)], ids=str)
def test_experts_between_products_of_a_step(streams, width):
    """Rows whose norm the router, the experts and the next projection finish: up to 48 rows, and the first that are normed whole; prompts beside tokens."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.stream_config([(U.ssm(2, 32, 32), U.moe(6, 1, 130)), (mixer(), U.dense(70)), (mixer(), U.moe(5, 1, 64))], width=width, vocab=120, streams=streams, positions=64)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=torch.bfloat16, max_batch=64, max_context=64)
    ts = [U.tokens(3, cfg["vocab"], i) for i in range(49)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, 8, 9, 33, 48, 49):
        slots = [m.open_sequence() for _ in range(n)]
        got = [m.step([(s, t[k : k + 1], [0]) for s, t in zip(slots, ts)]) for k in range(2)]
        for k in range(2):
            e = U.logit_errors(got[k], want[:n, k])
            assert float(e.max()) < 7e-2 and float(e.median()) < 3e-2, (n, k, e)
        if n == 8:  # the last token of each, beside a prompt
            got = m.step([(s, t[2:], [0]) for s, t in zip(slots, ts)] + [(m.open_sequence(), ts[40], [2, 0])])
            e = U.logit_errors(got, torch.cat([want[:8, 2], want[40, [2, 0]]]))
            assert float(e.max()) < 7e-2 and float(e.median()) < 3e-2
        for s in slots:
            m.close_sequence(s)
