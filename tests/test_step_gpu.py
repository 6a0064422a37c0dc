"""Decode steps of few rows: products that own whole columns and go on with the row-wise step (gemm_step.hip), at the edges of their row
tiles, for every count of streams that has a kernel of its own, beside the products that take more rows."""
import pytest
import torch

import lm_util as U
from oracle import layered_lm_oracle as O

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def build(name, weights=None, **kw):
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.CONFIGS[name] if isinstance(name, str) else name
    return LayeredLM(LayeredLMConfig.from_dict(cfg), weights or U.weights(cfg, 3, 1.5), dtype=BF16, max_batch=80, max_context=64, **kw)


ONE, TWO, FOUR = (U.stream_config([(U.ssm(4, 32, 32), U.dense(320)), (U.latent(4, 32, 32, 64), U.dense(96))], width=w, vocab=200, streams=n)
                  for n, w in ((1, 320), (2, 136), (4, 64)))


@pytest.mark.parametrize("name", ["odd", "shared", ONE, TWO, "streams", FOUR, "five_streams"],
                         ids=["odd", "shared", "one_stream", "two_streams", "streams", "four_streams", "five_streams"])
def test_rows_of_a_step(name):
    """Two tokens of 1 .. 64 sequences against the oracle (every row alone), and the logits of rows chosen among them in any order."""
    cfg = U.CONFIGS[name] if isinstance(name, str) else name
    m, w = build(name), U.weights(cfg, 3, 1.5)
    ts = [U.tokens(2, cfg["vocab"], i) for i in range(64)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])  # [64, 2, vocab]
    scale = (want - want.mean(-1, keepdim=True)).pow(2).mean().sqrt()
    # bf16 rounding through the layers, as in the other tests of whole models: 7e-2 at every row.  Routers, retention of first tokens and small
    # norm groups enlarge it at single rows, and at the same rows whatever product runs: there, twice what the products of 64 rows show
    limit = torch.full((2, 64), 7e-2, dtype=torch.float64)
    enlarges = isinstance(name, str)
    for n in (64, 1, 2, 8, 9, 16, 17, 28, 29, 32, 33, 48, 49):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(2):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)]).double().cpu()
            d = got - want[:n, k]
            e = (d - d.mean(-1, keepdim=True)).pow(2).mean(-1).sqrt() / scale
            if n == 64 and enlarges:
                top = e.sort().values
                assert float(top[57]) < 7e-2 and float(top[-1]) < 1.0
                limit[k] = torch.maximum(limit[k], 2 * e)
            assert bool((e < limit[k, :n]).all()), (n, k, e - limit[k, :n])
        for s in slots:
            m.close_sequence(s)
    # both tokens of 14 sequences at once (28 rows) and of 24 (48), logits of some of them
    for n in (14, 24):
        slots = [m.open_sequence() for _ in range(n)]
        places = [[1] if i % 3 == 0 else [1, 0] if i % 3 == 1 else [] for i in range(n)]
        got = m.step([(s, t, p) for s, t, p in zip(slots, ts, places)])
        ref = torch.cat([want[i][p] for i, p in enumerate(places) if p])
        at_most = torch.cat([limit[p, i] for i, p in enumerate(places) if p])
        assert bool((U.logit_errors(got, ref) < at_most).all())
        for s in slots:
            m.close_sequence(s)
    # more logits than rows, and more than the step products take
    t = U.tokens(9, cfg["vocab"], 5)
    for places in ([8, 0, 4] * 12, [8, 0, 4] * 17):
        got = m.step([(m.open_sequence(), t, places)])
        e = U.logit_errors(got, O.forward(cfg, w, t)[places]).sort().values
        assert float(e[len(e) // 2 if enlarges else -1]) < 7e-2 and float(e[-1]) < 1.0
    # no logits at all, then the state it left
    a, b = m.open_sequence(), m.open_sequence()
    assert m.step([(a, ts[0][:1], []), (b, ts[1][:1], [])]).shape[0] == 0
    got = m.step([(a, ts[0][1:], [0]), (b, ts[1][1:], [0])])
    assert bool((U.logit_errors(got, want[:2, 1]) < limit[1, :2]).all())


@pytest.mark.parametrize("heads,dim,vdim", [(40, 64, 64), (48, 96, 32), (64, 32, 32), (17, 128, 32), (40, 128, 32)], ids=str)
@pytest.mark.parametrize("own", [True, False])
def test_decode_attention_of_many_columns(heads, dim, vdim, own):
    """A step's queries, keys and values in two and four pieces per thread (more than 2048 and 4096 columns), more than 32 heads, and a layer that
    reads another one's keys; in two portions and then token by token."""
    layers = [U.attention(heads, heads // 2 if heads % 2 == 0 else 1, dim, vdim, 40)]
    if not own:
        layers.append(dict(U.attention(heads, heads // 2 if heads % 2 == 0 else 1, dim, vdim, 33, taps=1, kv_from=0)))
    cfg = U.config(layers, width=128, vocab=120, ff=None)
    m, w, ts = build(cfg), U.weights(cfg, 3, 1.5), [U.tokens(n, 120, n) for n in (50, 31)]
    want = [O.forward(cfg, w, t) for t in ts]
    slots = [m.open_sequence() for _ in ts]
    m.step([(s, t[:-12], []) for s, t in zip(slots, ts)])
    for k in range(12, 0, -1):
        got = m.step([(s, [t[-k]], [0]) for s, t in zip(slots, ts)])
        assert float(U.logit_errors(got, torch.stack([x[-k] for x in want])).max()) < 7e-2, k


@pytest.mark.parametrize("width", [2112, 4160])
def test_rows_of_wide_models(width):
    """More sums of squares per row than one pass of the step products takes (widths above 2048), and the rows from which such widths take tiles."""
    cfg = U.stream_config([(U.ssm(2, 32, 32), U.dense(128)), (U.latent(2, 32, 32, 64), None)], width=width, vocab=120, streams=2, positions=8)
    m, w = build(cfg), U.weights(cfg, 3, 1.5)
    ts = [U.tokens(2, 120, i) for i in range(49)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, 9, 17, 28, 29, 32, 33, 49):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(2):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)])
            assert float(U.logit_errors(got, want[:n, k]).max()) < 7e-2, (n, k)
        for s in slots:
            m.close_sequence(s)


@pytest.mark.parametrize("width,ff", [(64, 40), (600, 2040), (320, 2112), (1032, 4160), (1000, 4160), (2112, 4160)], ids=str)
def test_gates_of_up_to_eight_rows(width, ff):
    """Gates whose K two, four and eight waves share: one unit of K for eight waves, the most columns of one workgroup per CU and the first of
    more, and either side of the widths that two waves take."""
    cfg = U.stream_config([(U.latent(2, 32, 32, 64), U.dense(ff))], width=width, vocab=120, streams=2, positions=8)
    m, w = build(cfg), U.weights(cfg, 3, 1.5)
    ts = [U.tokens(2, 120, i) for i in range(9)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, 8, 9):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(2):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)])
            assert float(U.logit_errors(got, want[:n, k]).max()) < 7e-2, (n, k)
        for s in slots:
            m.close_sequence(s)


WIDE = [U.stream_config([(U.ssm(m, 32, 32), U.dense(ff)), (U.latent(4, 32, 32, 64), U.dense(96))], width=64, vocab=v, positions=8)
        for m, ff, v in ((8, 2112, 120), (64, 2120, 200), (130, 4168, 120), (128, 6208, 16500))]


@pytest.mark.parametrize("cfg", WIDE, ids=["gates", "pairs", "threes", "many"])
def test_columns_of_a_workgroup(cfg):
    """Products whose workgroups own one, two and three operands of columns, the last one fewer, at the edges of the row tiles."""
    m, w = build(cfg), U.weights(cfg, 3, 1.5)
    ts = [U.tokens(2, cfg["vocab"], i) for i in range(49)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (9, 16, 17, 32, 33, 48, 49):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(2):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)])
            assert float(U.logit_errors(got, want[:n, k]).max()) < 7e-2, (n, k)
        for s in slots:
            m.close_sequence(s)
    # a prompt and sequences that go on, logits of some rows in another order
    t = U.tokens(7, cfg["vocab"], 77)
    slots = [m.open_sequence() for _ in range(30)]
    for k in range(2):
        got = m.step([(s, [x[k]], [0]) for s, x in zip(slots, ts)] + ([(m.open_sequence(), t, [5, 0, 6])] if k else []))
    assert float(U.logit_errors(got[:30], want[:30, 1]).max()) < 7e-2
    assert float(U.logit_errors(got[30:], O.forward(cfg, w, t)[[5, 0, 6]]).max()) < 7e-2


@pytest.mark.parametrize("width,vdim,ff,vocab", [(64, 32, 64, 16500), (1000, 96, 330, 120), (1560, 32, 3080, 120), (2100, 130, 2080, 16500)], ids=str)
def test_weights_through_lds(width, vdim, ff, vocab):
    """Waves with no unit of K, with one, with as many as are under way and one more or less, in workgroups of one operand of columns to four, and gates, and residual
    products, at the edges of the row tiles: the ring of each wave comes round, ends early and is not used at all."""
    cfg = U.stream_config([(U.latent(4, 32, vdim, 64), U.dense(ff))], width=width, vocab=vocab, streams=2, positions=8)
    m, w = build(cfg), U.weights(cfg, 3, 1.5)
    ts = [U.tokens(2, vocab, i) for i in range(48)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, 8, 9, 16, 17, 32, 33, 48):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(2):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)])
            assert float(U.logit_errors(got, want[:n, k]).max()) < 7e-2, (n, k)
        for s in slots:
            m.close_sequence(s)


@pytest.mark.parametrize("width", [1088, 2624, 3648], ids=str)
def test_units_of_a_wave_past_two_rings(width):
    """Eight waves' parts of K of 2 and 3, 5 and 6, 7 and 8 units, two waves' of 8 and 9 (two or three units under way): the loop whose loads stand under no
    condition runs not at all, once, and more often, and leaves every number of units to the code behind it."""
    test_weights_through_lds(width, 32, width - 8, 120)


@pytest.mark.parametrize("rows", [3, 40, 200])
@pytest.mark.parametrize("which", ["in_proj", "out_proj", "gate_up", "down", "head"])
def test_misaligned_weights_are_refused(rows, which):
    """16-byte loads of the weights: at every number of rows."""
    from moondream_amd._lib import MoondreamHipError

    m = build(ONE)
    lin = m.w.model.head if which == "head" else getattr(m.w.model.layers[0], which)
    lin.w += 2
    with pytest.raises(MoondreamHipError):
        m.step([(m.open_sequence(), U.tokens(min(rows, 50), 200, i), [0]) for i in range(-(-rows // 50))])
    lin.w -= 2
    m.step([(m.open_sequence(), U.tokens(3, 200, 9), [0])])


@pytest.mark.parametrize("rows", [3, 40, 300])
@pytest.mark.parametrize("which", ["out_proj", "gate_up", "down"])
@pytest.mark.parametrize("cfg", [ONE, U.config([U.attention(4, 4, 32, 32, 64), U.attention(2, 2, 64, 64, 400)], width=328, vocab=200, ff=320)], ids=["streams", "plain"])
def test_biases_count_at_every_number_of_rows(cfg, which, rows):
    """The C structures allow a bias on every projection (the model folders have none there): bf16 beside fp32."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    out = {}
    for dtype in (BF16, torch.float32):
        m = LayeredLM(LayeredLMConfig.from_dict(cfg), U.weights(cfg, 3, 1.5), dtype=dtype, max_batch=2, max_context=320)
        lin, ids = getattr(m.w.model.layers[0], which), U.tokens(rows, 200, rows)
        for bias in (None, torch.linspace(-1.0, 1.0, lin.n_pad, device="cuda").to(BF16).to(dtype)):
            if bias is not None:
                bias[cfg["width"] if which != "gate_up" else lin.n_pad :] = 0  # (padded columns stay zero)
                lin.b = bias.data_ptr()
            s = m.open_sequence()
            out[dtype, bias is not None] = m.step([(s, ids, range(rows))])
            m.close_sequence(s)
    moved = U.logit_error(out[torch.float32, True], out[torch.float32, False].double().cpu())
    assert moved > 0.1 and U.logit_error(out[BF16, True], out[torch.float32, True].double().cpu()) < 0.25 * moved


@pytest.mark.parametrize("rows", [5, 28])
def test_residual_stream_behind_every_layer(rows):
    for cfg in (U.CONFIGS["shared"], TWO):
        m, t, ref, got = build(cfg), U.tokens(rows, cfg["vocab"], 0), [], []
        O.forward(cfg, U.weights(cfg, 3, 1.5), t, layers_out=ref)
        m.step([(m.open_sequence(), t, [])], layer_out=got)
        for a, b in zip(got[0].double().cpu(), ref):
            assert float((a - b).norm() / b.norm()) < 2e-2


@pytest.mark.parametrize("rows", [129, 256, 300, 700])
def test_prompts_whose_projections_leave_slices(rows):
    """Prompts of a few hundred tokens on layers wide enough for K slices and for segments of the state space, whole and in two portions."""
    cfg = U.stream_config([(U.ssm(8, 32, 32), U.dense(1100)), (U.latent(8, 32, 32, 64), U.dense(1030))], width=1032, vocab=200, streams=2, positions=900)
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    w = U.weights(cfg, 3, 1.5)
    t = U.tokens(rows, cfg["vocab"], rows)
    want = O.forward(cfg, w, t)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=2, max_context=1024)
    assert U.logit_error(m.step([(m.open_sequence(), t, range(rows))]), want) < 7e-2
    s, k = m.open_sequence(), rows - 130 if rows > 400 else 1
    got = torch.cat([m.step([(s, t[:k], range(k))]), m.step([(s, t[k:], range(rows - k))])])
    assert U.logit_error(got, want) < 7e-2


@pytest.mark.parametrize("lens", [[1], [1, 1, 1], [4, 1, 7], [28]], ids=str)
def test_prompts_through_retention_layers_round_alike(lens):
    """A first token's retention hangs on the sign of q . k: prompts of few rows get the bits that they get beside others."""
    cfg = U.config([U.retention(4, 32, 32), U.attention(4, 4, 32, 32, 64), U.retention(2, 64, 64)], width=328)
    m, prompts = build(cfg), [U.tokens(n, cfg["vocab"], i) for i, n in enumerate(lens)]

    def logits(texts):
        slots = [m.open_sequence() for _ in texts]
        got = m.step([(s, t, range(len(t))) for s, t in zip(slots, texts)])
        for s in slots:
            m.close_sequence(s)
        return got

    alone, beside = logits(prompts), logits(prompts + [U.tokens(30, cfg["vocab"], 9)])
    assert torch.equal(alone, beside[: sum(lens)])


@pytest.mark.parametrize("going", [1, 5])
@pytest.mark.parametrize("lens", [[1], [1, 1], [7], [3, 1, 9], [20]], ids=str)
def test_prompts_that_join_a_running_step_round_alike(lens, going):
    """The same beside sequences that go on, in a step of few rows (continuous batching)."""
    cfg = U.config([U.retention(4, 32, 32), U.attention(4, 4, 32, 32, 64), U.retention(2, 64, 64)], width=328)
    m, prompts = build(cfg), [U.tokens(n, cfg["vocab"], i) for i, n in enumerate(lens)]
    slots = [m.open_sequence() for _ in prompts]
    alone = m.step([(s, t, range(len(t))) for s, t in zip(slots, prompts)])
    for s in slots:
        m.close_sequence(s)
    running = [m.open_sequence() for _ in range(going)]
    m.step([(s, U.tokens(4 + i, cfg["vocab"], 20 + i), []) for i, s in enumerate(running)])
    entries = [(m.open_sequence(), t, range(len(t))) for t in prompts] + [(s, [i], [0]) for i, s in enumerate(running)]
    assert torch.equal(m.step(entries)[: sum(lens)], alone)


@pytest.mark.parametrize("heads,dim,vdim,most", [(6, 250, 200, 42), (33, 100, 130, 15), (16, 128, 128, 64), (40, 60, 40, 51)], ids=str)
def test_retention_of_many_sequences(heads, dim, vdim, most):
    """Decode steps whose workgroups hold all rows of a head's state (the most sequences that do, and one), and one sequence more, in which they take two
    after the other: rows and columns that are no multiple of what a pass takes."""
    cfg = U.config([U.retention(heads, dim, vdim)], width=64, vocab=60, ff=None)
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=most + 1, max_context=64)
    ts = [U.tokens(6, 60, i) for i in range(most + 1)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, most, most + 1):
        slots = [m.open_sequence() for _ in range(n)]
        m.step([(s, t[:3], []) for s, t in zip(slots, ts)])
        for k in range(3, 6):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)])
            assert float(U.logit_errors(got, want[:n, k]).max()) < 7e-2, (n, k)
        for s in slots:
            m.close_sequence(s)


@pytest.mark.parametrize("heads,dim,vdim,rot", [(2, 64, 64, 64), (3, 96, 96, 64), (2, 32, 128, 32), (5, 64, 32, 6), (1, 100, 70, 48), (2, 128, 128, 128), (2, 128, 32, 0),
                                                (40, 96, 64, 96)], ids=str)
def test_retention_prompts(heads, dim, vdim, rot):
    """Prompts at the edges of a chunk of 64 tokens, long ones in segments and without (heads enough), heads of every kind of width, coordinates that turn in pieces of
    eight, one by one and not at all; then the same cut in two, the second part on the state of the first."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.retention(heads, dim, vdim, rot=rot)], width=64, vocab=60, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=8, max_context=512)
    for lens in ([1, 63, 64, 65, 129], [450], [128, 2, 300]):
        ts = [U.tokens(n, 60, n) for n in lens]
        want = [O.forward(cfg, w, t) for t in ts]
        for cut in (0, 1, 64):
            slots = [m.open_sequence() for _ in ts]
            ks = [min(cut, n - 1) for n in lens]
            if cut:
                m.step([(s, t[:k], []) for s, t, k in zip(slots, ts, ks) if k])
            got = m.step([(s, t[k:], range(n - k)) for s, t, k, n in zip(slots, ts, ks, lens)])
            e = U.logit_errors(got, torch.cat([x[k:] for x, k in zip(want, ks)]))
            # bf16 through a layer: 7e-2 at every row, as in the tests of whole models (first tokens hang on q . k, which is nowhere small enough here to turn its sign)
            assert float(e.max()) < 7e-2, (lens, cut, e.sort().values[-8:])
            for s in slots:
                m.close_sequence(s)


@pytest.mark.parametrize("heads,dim,vdim", [(2, 64, 64), (3, 128, 128), (2, 96, 32), (1, 32, 128), (40, 64, 96)], ids=str)
def test_latent_prompts(heads, dim, vdim):
    """Prompts at the edges of a tile of 64 keys and of a block of 128 queries, short ones beside long ones (tiles that one group of waves has not got), few heads and more
    than a workgroup per compute unit; then cut, the second part on the context of the first."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.stream_config([(U.latent(heads, dim, vdim, 64), None)], width=64, vocab=60, positions=512)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=8, max_context=512)
    for lens in ([193], [2, 64, 65, 128, 256], [257, 1, 129], [450, 63], [320, 321, 450]):
        ts = [U.tokens(n, 60, n) for n in lens]
        want = [O.forward(cfg, w, t) for t in ts]
        for cut in (0, 1, 64, 190):
            slots = [m.open_sequence() for _ in ts]
            ks = [min(cut, n - 1) for n in lens]
            if cut:
                m.step([(s, t[:k], []) for s, t, k in zip(slots, ts, ks) if k])
            got = m.step([(s, t[k:], range(n - k)) for s, t, k, n in zip(slots, ts, ks, lens)])
            e = U.logit_errors(got, torch.cat([x[k:] for x, k in zip(want, ks)]))
            assert float(e.max()) < 7e-2, (lens, cut, e.sort().values[-4:])  # bf16 through a layer, as in the tests of whole models
            for s in slots:
                m.close_sequence(s)


@pytest.mark.parametrize("lens", [[1100], [517, 3, 580]], ids=str)
def test_state_space_prompts_that_fill_the_chip(lens):
    """Rows and columns enough for the convolution's 16 rows per thread (8224 columns), and a token behind each prompt, whose window is what
    the norm's launch left in the slots."""
    cfg = U.stream_config([(U.ssm(64, 128, 16), None)], width=72, vocab=200, streams=1, positions=1200)
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=4, max_context=1200)
    ts = [U.tokens(n + 1, cfg["vocab"], i) for i, n in enumerate(lens)]
    want = [O.forward(cfg, w, t) for t in ts]
    slots = [m.open_sequence() for _ in ts]
    got = m.step([(s, t[:-1], range(len(t) - 1)) for s, t in zip(slots, ts)])
    e = U.logit_errors(got, torch.cat([x[:-1] for x in want])).sort().values
    assert float(e[int(0.9 * len(e))]) < 7e-2 and float(e[-1]) < 1.0
    got = m.step([(s, t[-1:], [0]) for s, t in zip(slots, ts)])
    assert float(U.logit_errors(got, torch.cat([x[-1:] for x in want])).max()) < 7e-2


def test_rows_of_many_columns():
    """Step products of more than 16384 columns (the head), more than 8192 (an input projection) and of more than 4096 of K (the down product)."""
    cfg = U.stream_config([(U.ssm(64, 64, 16), U.dense(4200))], width=128, vocab=16600, streams=2, positions=8)
    m, w = build(cfg), U.weights(cfg, 3, 1.5)
    ts = [U.tokens(2, cfg["vocab"], i) for i in range(28)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, 8, 9, 16, 17, 28):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(2):
            got = m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)])
            assert float(U.logit_errors(got, want[:n, k]).max()) < 7e-2, (n, k)
        for s in slots:
            m.close_sequence(s)
        # rows in order, without an index: a decode step's logits
        slots = [m.open_sequence() for _ in range(n)]
        m.step([(s, t[:1], []) for s, t in zip(slots, ts)])
        logits = m._decode_logits(n)
        m._decode_lockstep(torch.tensor([t[1] for t in ts[:n]], dtype=torch.int32, device="cuda"), slots, 1)
        assert float(U.logit_errors(logits[:n, : cfg["vocab"]], want[:n, 1]).max()) < 7e-2, n
        for s in slots:
            m.close_sequence(s)


_REFS = {}


def errors_of_steps(m, cfg, w, tokens, n):
    """Single tokens of n sequences, ``tokens`` steps: errors of the logits [tokens, n], and the largest relative error of a row of the residual stream behind the
    first layer and behind the second."""
    key = (str(cfg), tokens)
    if key not in _REFS:
        _REFS.clear()
        taps, logits = [], []
        for i in range(49):
            taps.append([])
            logits.append(O.forward(cfg, w, U.tokens(tokens, cfg["vocab"], i), layers_out=taps[i]))
        _REFS[key] = torch.stack([torch.stack([x.double() for x in t]) for t in taps]), torch.stack(logits)
    taps, want = _REFS[key]
    slots, e, rows = [m.open_sequence() for _ in range(n)], [], []
    for k in range(tokens):
        out = []
        got = m.step([(s, [U.tokens(tokens, cfg["vocab"], i)[k]], [0]) for i, s in enumerate(slots)], layer_out=out)
        e.append(U.logit_errors(got, want[:n, k]))
        ref = taps[:n, :, k].transpose(0, 1)
        rows.append((out[0].double().cpu() - ref).norm(dim=-1) / ref.norm(dim=-1))
    for s in slots:
        m.close_sequence(s)
    return torch.stack(e), torch.stack(rows).amax((0, 2))


@pytest.mark.parametrize("groups", [1, 2, 4, 8])
@pytest.mark.parametrize("heads,vdim,state,width", [(16, 32, 32, 64), (40, 64, 16, 136), (88, 64, 16, 72)], ids=str)
def test_state_space_norm_groups_of_a_step(heads, vdim, state, width, groups):
    """The same with groups that are eighths, quarters and halves of the projection's K: more than eight heads to an eighth, and 49 rows, normed by a launch."""
    cfg = U.stream_config([(U.ssm(heads, vdim, state, norm_groups=groups), U.dense(64)), (U.ssm(heads, vdim, state, norm_groups=groups), U.dense(96))],
                          width=width, vocab=120, streams=2, positions=16)
    w = U.weights(cfg, 3, 1.5)
    for i in range(2):  # (groups of different size: another one's factor moves a row by about 0.5)
        w[f"l{i}.mix.D"] = torch.logspace(-1, 1, heads).to(BF16)
    m = build(cfg, w)
    # (a bound on the distribution of the logits' errors, as below; groups of few heads enlarge single rows there.  Behind a layer every row counts: rounding leaves
    # 0.01, up to 0.04 where a group of two heads nearly cancels, twice that behind the second layer)
    whole, rows = errors_of_steps(m, cfg, w, 3, 49)
    assert float(whole.median()) < 3e-2 and float(rows[0]) < 7e-2 and float(rows[1]) < 0.14
    for n in (1, 8, 9, 33, 48):
        e, rows = errors_of_steps(m, cfg, w, 3, n)
        assert float(rows[0]) < 7e-2 and float(rows[1]) < 0.14, (n, rows)
        e, ref = e.flatten().sort().values, whole[:, :n].flatten().sort().values
        assert float(e.median()) < (1.5 if n >= 8 else 4) * float(ref.median()) and float(e[int(0.8 * len(e))]) < (2 if n >= 8 else 8) * float(ref[int(0.8 * len(ref))]), (n, e, ref)


@pytest.mark.parametrize("heads,vdim,state,width", [(2, 32, 32, 64), (3, 20, 10, 72), (40, 32, 16, 136), (5, 100, 130, 320), (33, 72, 64, 64)], ids=str)
def test_state_space_norm_of_a_step(heads, vdim, state, width):
    """Rows whose norm the output projection finishes: heads padded, more heads than a lane holds sums of, at the edges of the row tiles."""
    # (more than one head in a norm: a first token's output is x times one factor per head, and a head's own norm leaves only the factor's sign)
    cfg = U.stream_config([(U.ssm(heads, vdim, state), U.dense(64)), (U.ssm(heads, vdim, state, conv=6), U.dense(96))],
                          width=width, vocab=120, streams=2, positions=16)
    m, w = build(cfg), U.weights(cfg, 3, 1.5)
    # a norm over few small values enlarges the rounding of single rows, other rows with every order of sums; so what is bounded is the distribution over
    # rows and steps, by that of rows that a launch of their own norms (49 rows).  Eight sequences and more: a median of 32 errors that spread
    # over a factor of ten is within a third, and the ninth in ten within a factor of two.  Behind a layer every row is bounded, as above
    whole, rows = errors_of_steps(m, cfg, w, 4, 49)
    assert float(whole.median()) < 3e-2 and float(rows[0]) < 7e-2 and float(rows[1]) < 0.14
    for n in (1, 8, 9, 33, 48):
        e, rows = errors_of_steps(m, cfg, w, 4, n)
        assert float(rows[0]) < 7e-2 and float(rows[1]) < 0.14, (n, rows)
        e, ref = e.flatten().sort().values, whole[:, :n].flatten().sort().values
        assert float(e.median()) < (1.5 if n >= 8 else 4) * float(ref.median()) and float(e[int(0.9 * len(e))]) < (2 if n >= 8 else 8) * float(ref[int(0.9 * len(ref))]), (n, e, ref)
