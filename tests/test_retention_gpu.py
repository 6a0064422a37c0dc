"""Retention over prompts in bf16: the bits on record, whatever else is in the step."""
import os

import numpy as np
import pytest
import torch

import lm_util as U

pytestmark = pytest.mark.gpu

# heads, dim, vdim, coordinates that turn: every kind of width and of rotation; few heads, whose longer prompts are cut into segments of one chunk alone and beside others, and
# many, which are cut into fewer segments or none as more sequences are beside them
CASES = {"2x64": (2, 64, 64, 64), "3x96": (3, 96, 96, 64), "2x128": (2, 128, 128, 128), "5x64x32": (5, 64, 32, 6), "1x100x70": (1, 100, 70, 48),
         "40x64": (40, 64, 64, 64), "20x128": (20, 128, 128, 128)}
LENS = [2, 63, 64, 65, 129, 300, 700]


def rows_of(n):
    """First and last tokens, and those beside the edges of chunks."""
    return sorted({0, 1, n - 1} | {64 * c + d for c in range(1, n // 64 + 1) for d in (-1, 0) if 64 * c + d < n})


def results(case, groups, cut):
    """(logits of rows_of every prompt, one in 89 elements of the retention states behind them); the prompts read in groups, in two steps where ``cut`` is given."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    heads, dim, vdim, rot = CASES[case]
    cfg = U.config([U.retention(heads, dim, vdim, rot=rot)], width=64, vocab=60, ff=None)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), U.weights(cfg, 3, 1.5), dtype=torch.bfloat16, max_batch=8, max_context=704)
    ts, logits, states = [U.tokens(n, 60, n) for n in LENS], {}, {}
    for group in groups:
        slots = [m.open_sequence() for _ in group]
        done = [min(cut, LENS[i] - 1) for i in group]
        if cut:
            m.step([(s, ts[i][:k], []) for s, i, k in zip(slots, group, done)])
        wanted = [[r - k for r in rows_of(LENS[i]) if r >= k] for i, k in zip(group, done)]
        got = m.step([(s, ts[i][k:], w) for s, i, k, w in zip(slots, group, done, wanted)]).split([len(w) for w in wanted])
        for s, i, x in zip(slots, group, got):
            logits[i], states[i] = x.float().cpu(), m.state._slabs[0]["ret"][s].flatten()[::89].cpu()
            m.close_sequence(s)
    return torch.cat([logits[i] for i in range(len(LENS))]).numpy(), torch.cat([states[i] for i in range(len(LENS))]).numpy()


@pytest.mark.parametrize("groups,cut", [([[0, 1, 2, 3, 4, 5, 6]], 0), ([[0, 1, 2, 3, 4, 5, 6]], 37), ([[i] for i in range(7)], 0), ([[6, 0, 3], [1, 5], [4, 2]], 0)],
                         ids=["together", "together-37", "alone", "mixed"])
@pytest.mark.parametrize("case", CASES)
def test_prompts_keep_their_results(case, groups, cut):
    """The results on record were made by a workgroup per chunk, with the keys' weights in the keys' two parts, the values as the projection rounds them, every chunk's
    increment summed by itself and the states carried from chunk to chunk in order.  A prompt has those states alone and beside any others; logits also hang on the
    products, which round by the rows of a step."""
    want = np.load(os.path.join(os.path.dirname(__file__), "golden", "retention_bf16.npz"))
    logits, states = results(case, groups, cut)
    assert np.array_equal(states, want[f"{case}.{cut}.states"])
    if len(groups) == 1:
        assert np.array_equal(logits, want[f"{case}.{cut}.logits"])
