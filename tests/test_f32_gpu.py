"""fp32 products at the edges of their tiles: few rows, tiles with remainders, every count of K steps; one order of sums at every number of
rows; prompts through retention layers, whose first tokens show any other order; grouped rows; scans of every state size."""
import ctypes as C
import os

import numpy as np
import pytest
import torch

import lm_util as U
from moondream_amd import _lib
from oracle import layered_lm_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 130])
@pytest.mark.parametrize("n,k", [(64, 64), (192, 128), (320, 192), (64, 1472)])
@pytest.mark.parametrize("bias", [False, True])
def test_product(m, n, k, bias):
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, b = (torch.randn(*s, generator=g, device="cuda") for s in ((m, k + 8), (n, k), (n,)))
    for ldc in (n, n + 3):  # rows that 16-byte stores can and cannot take
        c = torch.full((m, ldc), 7.0, device="cuda")
        lin = _lib.MdLinear()
        lin.w, lin.b, lin.n, lin.k, lin.n_pad, lin.k_pad = w.data_ptr(), b.data_ptr() if bias else None, n, k, n, k
        _lib.check(lib.md_gemm_f32(a.data_ptr(), k + 8, C.byref(lin), c.data_ptr(), ldc, m, torch.cuda.current_stream().cuda_stream), "md_gemm_f32")
        want = a[:, :k].double() @ w.double().t() + (b.double() if bias else 0)
        # k products of rounding error 2^-24 each, added in fp32
        bound = (a[:, :k].abs().double() @ w.abs().double().t() + b.abs().double()) * (k + 1) * 2.0 ** -24
        assert bool(((c[:, :n].double() - want).abs() <= bound).all()) and bool((c[:, n:] == 7).all())


@pytest.mark.parametrize("n,k", [(64, 64), (192, 320), (2048, 1472)])
def test_a_row_has_the_same_sums_beside_any_others(n, k):
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(n + k)
    a, w = torch.randn(300, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")
    lin = _lib.MdLinear()
    lin.w, lin.b, lin.n, lin.k, lin.n_pad, lin.k_pad = w.data_ptr(), None, n, k, n, k
    got = []
    for m in (1, 16, 17, 32, 33, 64, 65, 300):
        c = torch.empty(m, n, device="cuda")
        _lib.check(lib.md_gemm_f32(a.data_ptr(), k, C.byref(lin), c.data_ptr(), n, m, torch.cuda.current_stream().cuda_stream), "md_gemm_f32")
        got.append(c)
    assert all(torch.equal(c, got[-1][: c.shape[0]]) for c in got)


RETENTION = U.config([U.retention(4, 32, 32), U.attention(4, 2, 32, 32, 50), U.retention(2, 96, 64), U.retention(1, 160, 32)], width=328, vocab=64, ff=600)
LENS = [1, 1, 7, 3, 60, 33]


def retention_logits(groups):
    """Logits of LENS's prompts and of a token behind each, the prompts read in groups."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    m = LayeredLM(LayeredLMConfig.from_dict(RETENTION), U.weights(RETENTION, 3), dtype=torch.float32, max_batch=8, max_context=128)
    ts, out = [U.tokens(n + 1, RETENTION["vocab"], i) for i, n in enumerate(LENS)], {}
    for group in groups:
        slots = {i: m.open_sequence() for i in group}
        a = m.step([(slots[i], ts[i][:-1], range(LENS[i])) for i in group])
        b = m.step([(slots[i], ts[i][-1:], [0]) for i in group])
        out.update(zip(group, zip(a.split([LENS[i] for i in group]), b.split(1))))
    return torch.cat([x for i in range(len(LENS)) for x in out[i]]).cpu()


@pytest.mark.parametrize("groups", [[[0, 1, 2, 3, 4, 5]], [[0, 1, 2], [3], [4], [5]], [[0, 3], [1, 2], [4, 5]], [[5, 0], [4, 1, 2, 3]]], ids=str)
def test_prompts_through_retention_layers_keep_their_results(groups):
    """A first token's retention is its value times q . k, normed: where q . k is small another order of any sum before it changes the result beyond
    fp32 rounding.  The results on record (made when every sum was one chain, token by token) stand, whatever else is in the step."""
    want = np.load(os.path.join(os.path.dirname(__file__), "golden", "retention_f32.npz"))["logits"]
    assert np.array_equal(retention_logits(groups).numpy(), want)


def forward(cfg, lens, context=192):
    """(logits of the prompts of one step and of a token behind each, the same in float64)"""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    w = U.weights(cfg, 3)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=torch.float32, max_batch=8, max_context=context)
    ts = [U.tokens(n + 1, cfg["vocab"], i) for i, n in enumerate(lens)]
    slots = [m.open_sequence() for _ in ts]
    got = [m.step([(s, t[:-1], range(len(t) - 1)) for s, t in zip(slots, ts)]), m.step([(s, t[-1:], [0]) for s, t in zip(slots, ts)])]
    want = [O.forward(cfg, w, t) for t in ts]
    return torch.cat(got), torch.cat([x[:-1] for x in want] + [x[-1:] for x in want])


@pytest.mark.parametrize("m,n,k", [(380, 2048, 192), (385, 2048, 64), (129, 4224, 128), (145, 2880, 448), (65, 8256, 64), (449, 2048, 320),
                                   (383, 2048, 384), (95, 8256, 192), (447, 2048, 256), (511, 2048, 1024)], ids=str)
def test_tiles_of_48_and_64_rows(m, n, k):
    """Tiles of 48 rows where they even out the CUs (380, 129, 145, 65, 383 and 95 rows: last tiles of 44, 33, 1, 17 and 47), of 64 elsewhere (385, 449, 447 and 511: of 1
    and 63); K of one step of 64, of odd and even numbers of them, and of several sums of 128: the bits of the kernel that takes up to 32 rows, row by row, and fp32
    rounding from 64 bits."""
    rows, cols = -(-m // 64), n // 64  # (the rule beside lm_gemm_f32)
    assert rows * cols > 128 and (-(-(-(-m // 48) * cols) // 256) * 48 * 22 < -(-rows * cols // 256) * 64 * 21) == (m in (380, 129, 145, 65, 383, 95))
    import ctypes as C

    from moondream_amd import _lib

    lib, g = _lib.load(), torch.Generator(device="cuda").manual_seed(m)
    a, w, b = (torch.randn(*s, device="cuda", generator=g) for s in ((m, k), (n, k), (n,)))
    lin = _lib.MdLinear(w.data_ptr(), b.data_ptr(), n, k, n, k)

    def product(rows):
        c = torch.full((rows.shape[0] + 1, n), float("nan"), device="cuda")
        _lib.check(lib.md_gemm_f32(rows.data_ptr(), k, C.byref(lin), c.data_ptr(), n, rows.shape[0], torch.cuda.current_stream().cuda_stream))
        assert bool(c[-1].isnan().all())
        return c[:-1]

    got = product(a)
    assert torch.equal(got, torch.cat([product(x) for x in a.split(32)]))
    want = a.double() @ w.double().t() + b.double()
    # a chain of at most 128 products and k / 128 sums of them: half an ulp each, added up as a walk
    assert float((got - want).pow(2).mean().sqrt()) < 2.0 ** -24 * k ** 0.5 * (min(k, 128) + k / 128) ** 0.5


@pytest.mark.parametrize("rows,experts,top", [(9, 40, 1), (64, 1, 1), (65, 1, 1), (130, 2, 1), (131, 3, 2), (150, 70, 4)])
def test_grouped_products(rows, experts, top):
    """Empty groups, groups of one row, of whole tiles and of a row more, gathered rows; groups that begin inside a tile's rows."""
    got, want = forward(U.stream_config([(U.ssm(1, 8, 8), U.moe(experts, top, 200))], width=320, vocab=64, streams=1, positions=160), [rows])
    # a sum of k products in fp32 is off by up to sqrt(k) 2^-24 of its size, through four products in a row: 1e-6 at k = 320; twenty times that
    assert U.logit_error(got, want) < 2e-5


@pytest.mark.parametrize("dim", [20, 64, 100, 160, 224, 256])
def test_retention_scans(dim):
    got, want = forward(U.config([U.retention(2, dim, 40, rot=dim // 4 * 2)], width=64, vocab=64, ff=None, eps=1e-2), [1, 16, 17, 40])
    assert U.logit_error(got, want) < 2e-5  # (the norm's eps keeps first tokens from enlarging it)


@pytest.mark.parametrize("state", [16, 64, 100, 140, 256, 300, 512])
def test_state_space_scans(state):
    got, want = forward(U.stream_config([(U.ssm(2, 24, state), None)], width=64, vocab=64, streams=1, positions=64), [1, 8, 9, 33])
    assert U.logit_error(got, want) < 2e-5
