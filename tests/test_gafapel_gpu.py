"""What Gafapel's mechanisms promise, on the GPU: far keys and states, edges of the kernels' tiles, choices of experts, streams, positions."""

import pytest
import torch

import lm_util as U
from oracle import layered_lm_oracle as O

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16
TOL = {F32: 2e-5, BF16: 7e-2}
dtypes = pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])


def load(cfg, w, dtype, **kw):
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=dtype, **{"max_batch": 4, "max_context": 64, **kw})
    m.lib.md_lm_set_kernels(3)
    return m


def run(m, t, cuts):
    """Logits of every token of t, run as the portions ``cuts`` and then one by one."""
    s, at, got = m.open_sequence(), 0, []
    for n in list(cuts) + [1] * (len(t) - sum(cuts)):
        got.append(m.step([(s, t[at : at + n], range(n))]))
        at += n
    m.close_sequence(s)
    return torch.cat(got)


@dtypes
@pytest.mark.parametrize("rank", [40, 600], ids=["rank40", "rank600"])
def test_one_key_that_stands_out(dtype, rank):
    """The latent row of one token decides every later query, near and far, at the edges of the kernels' key tiles; nothing before it moves."""
    cfg = U.stream_config([(U.latent(3, 40, 24, rank, 1.0), None)], width=64, vocab=40, streams=1, positions=400)
    w = U.weights(cfg, 5)
    w["embed"][:, 0], w["embed"][:, 1], w["embed"][7] = 0.0, 4.0, 0.0
    w["embed"][7, 0], w["embed"][7, 1] = 8.0, 4.0
    w["pos"] = (w["pos"].float() * 0.1).to(BF16)
    for n in ("embed.norm", "l0.norm1"):
        w[n] = torch.ones_like(w[n])
    w["l0.mix.dkv"][0] = 0.0
    w["l0.mix.dkv"][0, 0] = 30.0  # latent coordinate 0: only the loud token has it
    w["l0.mix.uk"] = (w["l0.mix.uk"].float() * 0.3).to(BF16)
    w["l0.mix.uk"][:, 0] = 0.25
    w["l0.mix.q"] = (w["l0.mix.q"].float() * 0.3).to(BF16)
    w["l0.mix.q"][:, 1] = 0.5     # the same for every query
    m = load(cfg, w, dtype)
    base = [x if x != 7 else 8 for x in U.tokens(300, 40, 11)]
    plain = O.forward(cfg, w, base)
    for loud in (0, 1, 31, 32, 63, 64, 127, 128, 199, 255, 298):
        t = list(base)
        t[loud] = 7
        want = O.forward(cfg, w, t)
        shift = (want - plain).abs().amax(-1)
        assert shift[loud + 1 :].min() > 0.05 and (loud == 0 or shift[:loud].max() == 0)
        for cuts in ([300], [200], [64, 2, 63, 100], [257]):
            assert U.logit_error(run(m, t, cuts), want) < TOL[dtype], (loud, cuts)


@dtypes
@pytest.mark.parametrize("count", [17, 64, 133])
@pytest.mark.parametrize("heads, rank", [(40, 250), (5, 130), (33, 400)], ids=str)
def test_many_sequences_decode_together(dtype, count, heads, rank):
    """More sequences than share a weight or a split of the keys, of 1 to 330 positions; heads in one and in two groups."""
    cfg = U.stream_config([(U.latent(heads, 24, 20, rank), None), (U.ssm(9, 12, 20, groups=3, conv=3), None)], width=64, vocab=60, streams=2)
    w = U.weights(cfg, 7)
    m = load(cfg, w, dtype, max_batch=count, max_context=384)
    lens = [(1 + 37 * i) % 330 + 1 if i % 9 == 0 else 1 + (5 * i) % 23 for i in range(count)]
    ts = [U.tokens(n + 3, 60, i) for i, n in enumerate(lens)]
    slots = [m.open_sequence() for _ in ts]
    m.step([(s, t[:-3], []) for s, t in zip(slots, ts)])
    got = [m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)]) for k in (-3, -2, -1)]
    want = [O.forward(cfg, w, t)[-3:] for t in ts]
    for k in range(3):
        assert U.logit_error(got[k], torch.stack([x[k] for x in want])) < TOL[dtype]


@pytest.mark.parametrize("heads, vdim", [(40, 96), (72, 128), (9, 200)], ids=str)
def test_columns_of_a_head_between_workgroups(heads, vdim):
    """The last launch of a decode step's latent attention: a head's columns in one part, in as many as there are tiles, and in parts of which the
    last has fewer tiles; one sequence per workgroup and four."""
    cfg = U.stream_config([(U.latent(heads, 32, vdim, 100), None)], width=64, vocab=60, streams=2)
    w = U.weights(cfg, 7)
    m = load(cfg, w, BF16, max_batch=66, max_context=64)
    ts = [U.tokens(3, 60, i) for i in range(66)]
    want = torch.stack([O.forward(cfg, w, t) for t in ts])
    for n in (1, 8, 12, 15, 16, 30, 66):
        slots = [m.open_sequence() for _ in range(n)]
        for k in range(3):
            assert U.logit_error(m.step([(s, [t[k]], [0]) for s, t in zip(slots, ts)]), want[:n, k]) < TOL[BF16], (n, k)
        for s in slots:
            m.close_sequence(s)


def _slow_state(heads, vdim, state):
    cfg = U.stream_config([(U.ssm(heads, vdim, state, conv=2), None)], width=64, vocab=50, streams=2)
    w = U.weights(cfg, 2)
    w["l0.mix.A_log"] = torch.tensor([-9.0, -6.0, -30.0, 1.0])[:heads].to(BF16)
    return cfg, w


@dtypes
@pytest.mark.parametrize("sizes", [(2, 32, 64), (1, 96, 96), (3, 128, 128), (4, 30, 17)], ids=str)
def test_far_tokens_through_the_state(dtype, sizes):
    """Slow decays: what the first tokens wrote decides the last outputs, through chunks and segments of the prefill, portions and the cache.
    700 tokens of few heads run as several segments."""
    cfg, w = _slow_state(*sizes)
    ts = [U.tokens(700, 50, 4), U.tokens(700, 50, 4)]
    ts[1][:4] = [(x + 1) % 50 for x in ts[1][:4]]
    want = [O.forward(cfg, w, t) for t in ts]
    assert U.logit_error(want[1][690:], want[0][690:]) > 2e-3
    m = load(cfg, w, dtype)
    for t, ref in zip(ts, want):
        for cuts in ([700], [513, 2, 64, 100], [640]):
            assert U.logit_error(run(m, t, cuts), ref) < TOL[dtype]
    # several in one batch, of one and of many segments
    s = [m.open_sequence() for _ in range(3)]
    got = m.step([(s[0], ts[0], range(700)), (s[1], ts[1][:65], range(65)), (s[2], ts[1][:600], range(600))])
    tail = m.step([(s[2], ts[1][600:], range(100)), (s[1], ts[1][65:], range(635))])
    ref = torch.cat([want[0], want[1][:65], want[1][:600], want[1][600:], want[1][65:]])
    assert U.logit_error(torch.cat([got, tail]), ref) < TOL[dtype]


@dtypes
def test_fast_decays_and_large_steps(dtype):
    """Decays down to nothing within a token, steps far above 1: no overflow, no difference between the ways to compute them.  (Where a
    head's outputs nearly vanish, the norm enlarges the rounding: single positions may be ten times worse.)"""
    cfg = U.stream_config([(U.ssm(4, 32, 32, groups=2, conv=3, norm_groups=2), None)], width=64, vocab=50, streams=1)
    w = U.weights(cfg, 3)
    w["l0.mix.A_log"] = torch.tensor([3.0, 0.0, -3.0, 5.0]).to(BF16)
    w["l0.mix.dt_bias"] = torch.tensor([4.0, 30.0, -6.0, 0.0]).to(BF16)
    t = U.tokens(150, 50, 8)
    want, m = O.forward(cfg, w, t), load(cfg, w, dtype)
    for cuts in ([150], [2] * 40, [1]):
        e = U.logit_errors(run(m, t, cuts), want).sort().values
        assert float(e[-10]) < TOL[dtype] and float(e[-1]) < 10 * TOL[dtype]


@dtypes
def test_first_tokens(dtype):
    """Sequences shorter than the convolution, whole and token by token, in slots that held others."""
    cfg = U.CONFIGS["large_heads"]  # up to 6 taps
    w, m = U.weights(cfg, 3), None
    m = load(cfg, w, dtype, max_batch=1)
    for n in (1, 2, 3, 5, 6, 7):
        t = U.tokens(n, cfg["vocab"], n)
        want = O.forward(cfg, w, t)
        for cuts in ([n], [1], [max(1, n - 2)]):
            assert U.logit_error(run(m, t, cuts), want) < TOL[dtype]


def _expert_model(experts, top, ff, width=64):
    """The mixer adds nothing; embedding coordinates 0 .. 5 are +-3 and alone decide the router's logits, and no sublayer writes them: the
    choice is never close.  Every expert has a gain of its own."""
    cfg = U.stream_config([(U.ssm(1, 8, 8), U.moe(experts, top, ff))], width=width, vocab=64, streams=1)
    w = U.weights(cfg, 4)
    w["l0.mix.o"].zero_()
    bits = torch.tensor([[3.0 if (v >> b) & 1 else -3.0 for b in range(6)] for v in range(64)])
    w["embed"] = (w["embed"].float() * 0.5).to(BF16)
    w["embed"][:, :6] = bits.to(BF16)
    w["pos"] = (w["pos"].float() * 0.2).to(BF16)
    w["pos"][:, :6] = 0
    g = torch.Generator().manual_seed(9)
    r = torch.zeros(experts, width)
    r[:, :6] = torch.randn(experts, 6, generator=g)
    w["l0.mlp.router"] = r.to(BF16)
    for k in range(experts):
        w[f"l0.mlp.e{k}.down"][:6] = 0
        w[f"l0.mlp.e{k}.down"] = (w[f"l0.mlp.e{k}.down"].float() * (0.5 + k % 7)).to(BF16)
    return cfg, w


@dtypes
@pytest.mark.parametrize("shape", [(7, 1, 24), (7, 7, 24), (16, 2, 200), (40, 5, 64), (100, 4, 32), (150, 3, 32), (3, 2, 130)], ids=str)
def test_experts(dtype, shape):
    """Counts beyond one and beyond eight tiles, one expert, all experts; 1 to 400 rows a step (every tile height of the grouped product)."""
    cfg, w = _expert_model(*shape)
    t = U.tokens(400, 64, 6)
    want, m = O.forward(cfg, w, t), load(cfg, w, dtype)
    for cuts in ([400], [100, 300], [2] * 3 + [17, 130], [391]):
        e = U.logit_errors(run(m, t, cuts), want)
        # (a row whose k-th and next logits are close may choose otherwise in bf16)
        assert float(e.sort().values[-9 if dtype == BF16 else -1]) < TOL[dtype]


@pytest.mark.parametrize("width,ff", [(64, 64), (192, 320), (448, 384), (640, 512)], ids=str)
def test_weights_of_experts_through_lds(width, ff):
    """Waves with no unit of 64 of K, with as many as are under way and one more or less, for up to eight rows of an expert and for several passes of 16."""
    cfg, w = _expert_model(4, 2, ff, width=width)
    t = U.tokens(60, 64, 6)
    want, m = O.forward(cfg, w, t), load(cfg, w, BF16)
    for cuts in ([20] * 3, [1] * 10 + [5] * 10):
        assert float(U.logit_errors(run(m, t, cuts), want).sort().values[-2]) < TOL[BF16]  # (a row whose choice is close may choose otherwise in bf16)


@pytest.mark.parametrize("width,ff", [(832, 704), (896, 1024)], ids=str)
def test_units_of_an_experts_wave_past_two_rings(width, ff):
    """Two waves' parts of K of 6 and 7, 5 and 6, 7, and 8 units of 64, three under way: every number of units behind the loop whose loads stand under no condition."""
    test_weights_of_experts_through_lds(width, ff)


@dtypes
def test_one_expert_takes_every_row(dtype):
    """The other experts have no rows at all."""
    cfg, w = _expert_model(6, 1, 40)
    w["l0.mlp.router.b"] = torch.tensor([-90.0, -90.0, -90.0, 90.0, -90.0, -90.0]).to(BF16)
    t = U.tokens(200, 64, 6)
    want, m = O.forward(cfg, w, t), load(cfg, w, dtype)
    for cuts in ([200], [150]):
        assert U.logit_error(run(m, t, cuts), want) < TOL[dtype]


@dtypes
@pytest.mark.parametrize("streams", [1, 2, 3, 4, 7, 16])
def test_streams_alone(dtype, streams):
    """Mixers that add nothing, dense feed-forwards: what the streams' weights do."""
    cfg = U.stream_config([(U.ssm(1, 8, 8), U.dense(40)), (U.ssm(1, 8, 8), None), (U.ssm(1, 8, 8), U.dense(70))], width=100, vocab=60, streams=streams)
    w = U.weights(cfg, streams)
    for i in range(3):
        w[f"l{i}.mix.o"].zero_()
    t = U.tokens(140, 60, 1)
    want, m = O.forward(cfg, w, t), load(cfg, w, dtype)
    for cuts in ([140], [2, 130]):
        assert U.logit_error(run(m, t, cuts), want) < TOL[dtype]


def test_positions_end():
    """The last position works; one more token is an error before anything runs; generation stops there, sequence by sequence."""
    cfg = U.stream_config([(U.latent(2, 16, 16, 24), U.dense(32))], width=64, vocab=40, streams=1, positions=70)
    w = U.weights(cfg, 6)
    m = load(cfg, w, F32)
    t = U.tokens(71, 40, 2)
    s = m.open_sequence()
    assert U.logit_error(m.step([(s, t[:69], [68]), ]), O.forward(cfg, w, t[:69])[-1:]) < TOL[F32]
    assert U.logit_error(m.step([(s, t[69:70], [0])]), O.forward(cfg, w, t[:70])[-1:]) < TOL[F32]
    with pytest.raises(ValueError, match="positions"):
        m.step([(s, t[70:], [])])
    assert m.sequence_length(s) == 70
    m.close_sequence(s)
    with pytest.raises(ValueError, match="positions"):
        m.batch_generate_ids([t], max_tokens=2)
    got = m.batch_generate_ids([t[:66], t[:60]], max_tokens=30)
    assert [len(g) for g in got] == [5, 11]
    for p, g in zip((t[:66], t[:60]), got):
        full = list(p) + g
        assert g == O.forward(cfg, w, full[:-1])[len(p) - 1 :].argmax(-1).tolist()


def test_graph_replays_match_the_eager_steps():
    """Every replay of the captured decode against eager decoding, with other work between."""
    name = "streams"
    cfg = U.CONFIGS[name]
    w = U.weights(cfg, 3, 1.5)
    prompts = [U.tokens(n, cfg["vocab"], n) for n in (9, 31, 2)]
    eager, graph = load(cfg, w, BF16), load(cfg, w, BF16)
    graph.compile()
    want = eager.batch_generate_ids(prompts, max_tokens=50)
    for k in range(4):
        assert graph.batch_generate_ids(prompts, max_tokens=50) == want
        graph.batch_generate_ids([prompts[k % 3][:5]], max_tokens=3)
        torch.randn(1 << 16, device="cuda").sum().item()
        torch.cuda.synchronize()


@pytest.mark.parametrize("width,ff", [(256, 256), (192, 64)], ids=["four_wave_tile", "128_rows"])
def test_grouped_tiles_of_the_bf16_product_agree(width, ff):
    """One model, steps of different heights: the large tile of the grouped product (the four-wave one for 256 columns and more, 128 rows for
    fewer) and the 64-row one give the same rows within rounding."""
    cfg, w = _expert_model(2, 2, ff, width=width)
    t = U.tokens(1100, 64, 3)
    cfg["max_positions"] = 1200
    w["pos"] = torch.zeros(1200, width, dtype=BF16)
    m = load(cfg, w, BF16, max_batch=1)
    a, b, c = run(m, t, [1100]).double().cpu(), run(m, t, [200] * 5 + [100]).double().cpu(), run(m, t, [60] * 18 + [20]).double().cpu()
    assert U.logit_error(b, a) < 2e-2 and U.logit_error(c, a) < 2e-2
    assert U.logit_error(a[:120], O.forward(cfg, w, t[:120])) < TOL[BF16]


@pytest.mark.parametrize("width,ff,tokens", [(64, 64, 111), (64, 64, 112), (128, 320, 200), (192, 192, 257), (64, 1152, 419), (64, 1152, 560), (320, 1152, 280), (128, 1152, 897)], ids=str)
def test_grouped_tiles_of_a_few_dozen_rows(width, ff, tokens):
    """32 experts, eight a row: tiles of 128 x 128 from 28 rows a group on (and just below), of 256 x 128 where the four-wave tiles of 2304 columns leave most of a second
    round empty, experts of no row and of several tiles, columns and K at the edges of tiles and of the ring of slices; beside the products of a few rows."""
    cfg, w = _expert_model(32, 8, ff, width=width)
    cfg["max_positions"] = 900
    w["pos"] = torch.zeros(900, width, dtype=BF16)
    t = U.tokens(tokens, 64, 3)
    m = load(cfg, w, BF16, max_batch=1)
    got, few = run(m, t, [tokens]).double().cpu(), run(m, t, [8] * (tokens // 8)).double().cpu()
    assert float(U.logit_errors(got, O.forward(cfg, w, t)).max()) < TOL[BF16]
    # both are within the oracle's 7e-2, so within twice that of one another: a token whose eight experts nearly cancel is 0.037 apart (257 tokens)
    assert U.logit_error(got, few) < 2 * TOL[BF16]


@pytest.mark.parametrize("width,ff,tokens", [(64, 64, 112), (320, 320, 200), (192, 128, 257), (576, 576, 280), (1152, 1152, 560)], ids=str)
@pytest.mark.parametrize("copied", [True, False], ids=["gates_seen", "products_seen"])
def test_grouped_tiles_column_by_column(width, ff, tokens, copied):
    """Every number that the experts add to the residual stream against 64 bits, at the tiles of 128 x 128 and (560 tokens) 256 x 128: with ``copied`` the second product hands
    the gated columns on as they are, so that a wrong column of one expert shows whole, in either product."""
    cfg, w = _expert_model(32, 8, ff, width=width)
    cfg["max_positions"] = 600
    w["pos"] = torch.zeros(600, width, dtype=BF16)
    for k in range(32):
        if copied:
            w[f"l0.mlp.e{k}.down"] = torch.eye(width, ff).to(BF16)
    t, got, before = U.tokens(tokens, 64, 3), [], []
    m = load(cfg, w, BF16, max_batch=1, max_context=600)
    m.step([(m.open_sequence(), t, [])], layer_out=got)
    O.forward(dict(cfg, layers=[dict(layer, mlp=None) for layer in cfg["layers"]]), w, t, layers_out=before)
    d = {n: x.double().cuda() for n, x in w.items()}
    streams = before[0][None].cuda()
    h = (O.rms_norm(O.stream_input(streams, d["l0.hc2.in"]), cfg["norm"]["eps"]) * d["l0.norm2"]).to(BF16).double()  # (what the experts read is bf16)
    z = h @ d["l0.mlp.router"].T + d["l0.mlp.router.b"]
    top = z.topk(8, -1)
    share = torch.zeros_like(z).scatter(-1, top.indices, torch.softmax(top.values, -1))
    parts = torch.stack([share[:, k : k + 1] * O.gated_mlp(d, f"l0.mlp.e{k}.", h) for k in range(32)])
    want = O.stream_update(streams, d["l0.hc2.mix"], d["l0.hc2.out"], parts.sum(0)).sum(0)
    # Roundings to bf16 of up to 2^-9 each: what the experts read (seen by gate and input), gated values, results: 2^-7 of a value if all add up, and of a row's values for one
    # that its terms nearly cancel in; twice that for the largest of half a million, and twice again where a sum of such terms follows.  One expert's wrong column is a tenth of a
    # row's values and more.
    size = parts.abs().sum(0)
    far = float(((got[0][0].double() - want).abs() / (size + size.pow(2).mean(-1, keepdim=True).sqrt()) / d["l0.hc2.out"].abs()).max())
    assert far < (2.0 ** -6 if copied else 2.0 ** -5), far
