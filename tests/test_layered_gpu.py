"""Layered language models on the GPU, against the plain CPU oracle: every kernel family, both formats, every way to cut and batch."""
import json
import os
import subprocess
import sys

import pytest
import torch

import lm_util as U
from oracle import layered_lm_oracle as O

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32, BF16 = torch.float32, torch.bfloat16
TOL = {F32: 2e-5, BF16: 7e-2}
LENS = [67, 5, 1, 130]


def model(name, dtype, qk_gain=1.5, **kw):
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.CONFIGS[name]
    kw = {"max_batch": 2, "max_context": 64, **kw}
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), U.weights(cfg, 3, qk_gain), dtype=dtype, **kw)
    m.lib.md_lm_set_kernels(3)
    return m


def toks(name, lens=LENS):
    return [U.tokens(n, U.CONFIGS[name]["vocab"], i) for i, n in enumerate(lens)]


def error(got, want, name, dtype):
    return U.logit_error(got, want, name if dtype == BF16 else None)


def both(f):
    return pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])(pytest.mark.parametrize("name", sorted(U.CONFIGS))(f))


@both
def test_whole_prompts_in_one_ragged_batch(name, dtype):
    m, ts = model(name, dtype), toks(name)
    slots = [m.open_sequence() for _ in ts]
    got = m.step([(s, t, range(len(t))) for s, t in zip(slots, ts)])
    assert error(got, torch.cat(U.oracle_logits(name, LENS)), name, dtype) < TOL[dtype]


@both
def test_prompt_then_decode_together(name, dtype):
    """Sequences of different lengths decode as one batch, over chunk edges, beside sequences that stay idle."""
    m, ts = model(name, dtype), toks(name)
    slots = [m.open_sequence() for _ in ts]
    start = [25, 2, 0, 64]
    m.step([(slots[i], ts[i][: start[i]], []) for i in (0, 1, 3)])
    rows, want, ref = [], [], U.oracle_logits(name, LENS)
    for k in range(60):
        live = [i for i in (0, 1, 3) if start[i] + k < LENS[i]]
        rows.append(m.step([(slots[i], [ts[i][start[i] + k]], [0]) for i in live]))
        want += [ref[i][start[i] + k] for i in live]
    assert error(torch.cat(rows), torch.stack(want), name, dtype) < TOL[dtype]


@both
def test_token_by_token_from_the_first(name, dtype):
    m, t = model(name, dtype), toks(name)[0]
    s = m.open_sequence()
    got = torch.cat([m.step([(s, [x], [0])]) for x in t])
    assert error(got, U.oracle_logits(name, LENS)[0], name, dtype) < TOL[dtype]


@pytest.mark.parametrize("sizes", [[2] * 65, [3, 2, 16, 31, 33, 2, 43], [17, 64, 1, 48], [96, 34]], ids=str)
@both
def test_portions_of_a_prompt(name, dtype, sizes):
    m, t = model(name, dtype), toks(name)[3]
    s, got, at = m.open_sequence(), [], 0
    for n in sizes:
        got.append(m.step([(s, t[at : at + n], range(n))]))
        at += n
    assert at == 130 and error(torch.cat(got), U.oracle_logits(name, LENS)[3], name, dtype) < TOL[dtype]


@both
def test_mixed_step_of_prompts_portions_and_decodes(name, dtype):
    m, ts = model(name, dtype, max_step_rows=50), toks(name)
    slots = [m.open_sequence() for _ in ts]
    ref = U.oracle_logits(name, LENS)
    m.step([(slots[0], ts[0][:40], []), (slots[3], ts[3][:70], [])])
    got = m.step([(slots[0], ts[0][40:41], [0]), (slots[3], ts[3][70:], range(60)), (slots[1], ts[1], range(5)), (slots[2], ts[2], [0])])
    assert error(got, torch.cat([ref[0][40:41], ref[3][70:], ref[1], ref[2]]), name, dtype) < TOL[dtype]


@pytest.mark.parametrize("name", ["odd", "shared", "wide_heads", "streams", "wide_streams"])
def test_batch_changes_nothing_beyond_rounding(name):
    for dtype, tol in ((F32, 5e-6), (BF16, 6e-2)):
        m, ts = model(name, dtype), toks(name)
        alone = []
        for t in ts:
            s = m.open_sequence()
            alone.append(m.step([(s, t, range(len(t)))]))
            m.close_sequence(s)
        slots = [m.open_sequence() for _ in ts]
        got = m.step([(s, t, range(len(t))) for s, t in zip(slots, ts)])
        assert error(got, torch.cat(alone).double().cpu(), name, dtype) < tol


@both
def test_slots_are_used_again(name, dtype):
    """A shorter sequence in a slot that held a longer one, beside slots that go on."""
    m, ts = model(name, dtype, max_batch=1), toks(name)
    ref = U.oracle_logits(name, LENS)
    a = m.open_sequence()
    m.step([(a, ts[3], [])])
    b = m.open_sequence()  # grows the slabs: what slot a holds moves with them
    m.step([(b, ts[0][:30], [])])
    m.close_sequence(a)
    c = m.open_sequence()
    assert c == a and m.sequence_length(c) == 0
    got = m.step([(c, ts[1], range(5)), (b, ts[0][30:], range(37))])
    assert error(got, torch.cat([ref[1], ref[0][30:]]), name, dtype) < TOL[dtype]
    m.close_sequence(c)
    d = m.open_sequence()
    one = [m.step([(d, [x], [0])]) for x in ts[1]]
    assert error(torch.cat(one), ref[1], name, dtype) < TOL[dtype]


@pytest.mark.parametrize("name", sorted(U.CONFIGS))
def test_kernel_families_agree(name):
    """The plain kernels and the matrix-core / decode kernels on the same bf16 model, prompts' attention by size and as for long ones."""
    ts, out = toks(name), []
    for mask in (0, 1, 2, 3, 5, 7):
        m = model(name, BF16)
        m.lib.md_lm_set_kernels(mask)
        slots = [m.open_sequence() for _ in ts]
        rows = [m.step([(slots[0], ts[0][:50], range(50)), (slots[3], ts[3][:113], range(113))])]
        rows += [m.step([(slots[0], [ts[0][50 + k]], [0]), (slots[3], [ts[3][113 + k]], [0])]) for k in range(17)]
        out.append(torch.cat(rows).double().cpu())
        m.lib.md_lm_set_kernels(3)
    for o in out[1:]:
        assert error(o, out[0], name, BF16) < 6e-2


@pytest.mark.parametrize("fault", O.FAULTS + O.STREAM_FAULTS)
def test_product_is_not_the_faulty_design(fault):
    """The comparison above would have caught each planted mistake (planted in the oracle), in a prompt and decoded."""
    name = U.SHOWS[fault]
    m, t = model(name, F32), U.tokens(61, U.CONFIGS[name]["vocab"], 0)
    good, bad = U.oracle_logits(name, [61])[0], U.oracle_logits(name, [61], fault=fault)[0]
    a, b = m.open_sequence(), m.open_sequence()
    whole = m.step([(a, t, range(61))])
    dec = torch.cat([m.step([(b, [x], [0])]) for x in t])
    for got in (whole, dec):
        assert U.logit_error(got, good) < TOL[F32] and U.logit_error(got, bad) > 2e-3


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("decoded", [False, True], ids=["prompt", "decoded"])
def test_chunk_edges_with_one_key_that_stands_out(dtype, decoded):
    """Attention alone, the key of one token far above all others: it decides every query that sees it.  The chunk is 48 with the loud key
    at its first, second, last position, or just before it; queries at the edges and in between."""
    cfg = U.config([U.attention(4, 2, 32, 32, 48, taps=1, scale=1.0)], width=64, vocab=40, ff=None)
    w = U.weights(cfg, 5)
    # token 7's key points along every query's fixed part (the biases), all other tokens' keys along nothing
    w["embed"] = torch.randn(40, 64, generator=torch.Generator().manual_seed(9)).to(BF16)
    w["embed"][:, 0] = 0
    w["embed"][7] = 0
    w["embed"][7, 0] = 8.0
    for n in ("q", "k"):
        w[f"l0.mix.{n}"] = (w[f"l0.mix.{n}"].float() * 0.2).to(BF16)
        w[f"l0.mix.{n}.b"] = torch.zeros_like(w[f"l0.mix.{n}.b"])
        w[f"l0.mix.{n}.conv"] = torch.ones_like(w[f"l0.mix.{n}.conv"])
    w["l0.mix.q.b"] = torch.full_like(w["l0.mix.q.b"], 1.0)
    w["l0.mix.k"][:, 0] = 1.0
    w["l0.mix.talk"] = (torch.eye(4) + 0.05).to(BF16)
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=dtype, max_batch=4, max_context=256)
    base = [x if x != 7 else 8 for x in U.tokens(150, 40, 11)]
    for loud in (47, 48, 49, 80, 95, 96):
        t = list(base)
        t[loud] = 7
        want = O.forward(cfg, w, t)
        plain = O.forward(cfg, w, base)
        shift = (want - plain).abs().amax(-1)
        end = (loud // 48 + 1) * 48
        assert shift[loud + 1 : end].numel() == 0 or shift[loud + 1 : end].min() > 0.05, "the loud key must decide what sees it"
        assert shift[end:].max() == 0 and shift[:loud].max() == 0
        s = m.open_sequence()
        if decoded:
            head = m.step([(s, t[:40], range(40))])
            got = torch.cat([head] + [m.step([(s, [x], [0])]) for x in t[40:]])
        else:
            got = m.step([(s, t, range(150))])
        m.close_sequence(s)
        assert U.logit_error(got, want) < TOL[dtype]


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_far_tokens_through_retention(dtype):
    """Slow decays: what the first tokens wrote decides the last outputs, through several chunks of the prefill and through the cache."""
    cfg = U.config([U.retention(2, 32, 64, rot=0, decay=[0.9999, 1.0])], width=64, vocab=50, ff=None)
    w = U.weights(cfg, 2)
    ts = [U.tokens(300, 50, 4), U.tokens(300, 50, 4)]
    ts[1][:3] = [(x + 1) % 50 for x in ts[1][:3]]
    want = [O.forward(cfg, w, t) for t in ts]
    assert U.logit_error(want[1][290:], want[0][290:]) > 1e-3
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=dtype, max_batch=2, max_context=64)
    s = [m.open_sequence(), m.open_sequence()]
    got = [m.step([(s[0], ts[0][:257], range(257)), (s[1], ts[1][:200], range(200))])]
    a, b = got[0][:257], got[0][257:]
    tail = m.step([(s[0], ts[0][257:], range(43)), (s[1], ts[1][200:], range(100))])
    tol = TOL[F32] if dtype == F32 else 3e-2
    assert U.logit_error(torch.cat([a, tail[:43]]), want[0]) < tol and U.logit_error(torch.cat([b, tail[43:]]), want[1]) < tol


@pytest.mark.parametrize("name", ["odd", "shared", "streams", "five_streams"])
def test_residual_stream_layer_by_layer(name):
    cfg = U.CONFIGS[name]
    t, ref, got = toks(name)[0], [], []
    O.forward(cfg, U.weights(cfg, 3, 1.5), t, layers_out=ref)
    m = model(name, F32)
    m.step([(m.open_sequence(), t, [])], layer_out=got)
    for a, b in zip(got[0].double().cpu(), ref):
        assert float((a - b).abs().max() / b.abs().max()) < 1e-5


def _greedy_reference(name, prompts, n):
    """The oracle's greedy continuations and the smallest margin on the way."""
    cfg = U.CONFIGS[name]
    w = U.weights(cfg, 3, 1.5)
    out, margin = [], []
    for p in prompts:
        t, mg = list(p), float("inf")
        for _ in range(n):
            top = torch.topk(O.forward(cfg, w, t)[-1], 2)
            mg = min(mg, float(top.values[0] - top.values[1]))
            t.append(int(top.indices[0]))
        out.append(t[len(p):])
        margin.append(mg)
    return out, margin


@pytest.mark.parametrize("name", ["shared", "streams"])
@pytest.mark.parametrize("graphs", [False, True], ids=["eager", "graph"])
def test_greedy_generation(name, graphs):
    """batch_generate_ids: ragged prompts, lockstep decode, several runs (graph replays with other work between), groups, end token."""
    n = 20
    prompts = [t[:k] for t, k in zip(toks(name), (19, 5, 1, 33))]
    want, margin = _greedy_reference(name, prompts, n)
    m = model(name, F32)
    if graphs:
        m.compile()
    for _ in range(3):
        got = m.batch_generate_ids(prompts, max_tokens=n)
        for g, r, mg in zip(got, want, margin):
            assert g == r or mg < 1e-3
        m.batch_generate_ids([prompts[3]], max_tokens=3)
        torch.cuda.synchronize()
    assert m.batch_generate_ids(prompts, max_tokens=n, max_batch=3) == got
    eos = got[0][4]
    cut = m.batch_generate_ids(prompts, max_tokens=n, eos_id=eos)
    assert cut == [g[: g.index(eos)] if eos in g else g for g in got]
    assert m.state.pool.available() == m.state.slots


@pytest.mark.parametrize("name", ["wide_heads", "five_streams"])
@pytest.mark.parametrize("graphs", [False, True], ids=["eager", "graph"])
def test_long_bf16_decode_follows_its_own_logits(name, graphs):
    """150 greedy tokens over several chunks: feeding the ids back as a prompt gives the same choices within rounding."""
    m = model(name, BF16)
    if graphs:
        m.compile()
    p = toks(name)[0][:9]
    ids = m.batch_generate_ids([p, p[:4]], max_tokens=150)
    for prompt, gen in ((p, ids[0]), (p[:4], ids[1])):
        s = m.open_sequence()
        lg = m.step([(s, prompt + gen[:-1], range(len(prompt) - 1, len(prompt) + 149))]).float()
        m.close_sequence(s)
        chosen = lg.gather(1, torch.tensor(gen, device=lg.device)[:, None])[:, 0]
        assert float((lg.max(-1).values - chosen).max()) < 0.25
    ref = O.forward(U.CONFIGS[name], U.weights(U.CONFIGS[name], 3, 1.5), (p + ids[0][:-1]))
    s = m.open_sequence()
    assert error(m.step([(s, p + ids[0][:-1], range(158))]), ref, name, BF16) < TOL[BF16]


def test_sampled_generation_is_seeded_and_in_range():
    m = model("odd", BF16)
    prompts = [t[:k] for t, k in zip(toks("odd"), (9, 5))]
    run = lambda seed: m.batch_generate_ids(prompts, max_tokens=12, temperature=0.8, top_p=0.9,  # noqa: E731
                                            generator=torch.Generator(device="cuda").manual_seed(seed))
    a = run(1)
    assert a == run(1) and a != run(2) and all(0 <= t < U.CONFIGS["odd"]["vocab"] for g in a for t in g)


def test_text_interface():
    from moondream_amd.moondream import IdTokenizer

    m = model("odd", F32, tokenizer=IdTokenizer())
    ids = toks("odd")[1]
    text = m.generate(" ".join(map(str, ids)), {"temperature": 0, "max_tokens": 4})
    assert [int(x) for x in text.split()] == m.batch_generate_ids([ids], max_tokens=4)[0]


def test_bad_calls_are_refused():
    m = model("odd", BF16)
    s = m.open_sequence()
    for entries in ([(s, [], [])], [(s, [10 ** 6], [])], [(s, [1], [1])], [(s, [1], []), (s, [2], [])], [(99, [1], [])]):
        with pytest.raises(ValueError):
            m.step(entries)
    with pytest.raises(ValueError):
        m.batch_generate_ids([[]])


def test_fp32_gemm():
    from moondream_amd import _lib
    from moondream_amd.weights import PackedLinear
    import ctypes as C

    lib = _lib.load()
    g = torch.Generator().manual_seed(0)
    for m, n, k in ((1, 64, 64), (37, 130, 200), (130, 64, 320)):
        w, b, a = torch.randn(n, k, generator=g), torch.randn(n, generator=g), torch.randn(m, k, generator=g)
        p = PackedLinear(w, b, "cuda", F32)
        ap = torch.zeros(m, p.k_pad, device="cuda")
        ap[:, :k] = a.cuda()
        c = torch.empty(m, p.n_pad, device="cuda")
        _lib.check(lib.md_gemm_f32(ap.data_ptr(), p.k_pad, C.byref(p.struct()), c.data_ptr(), p.n_pad, m, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        want = a.double() @ w.double().T + b.double()
        assert float((c[:, :n].double().cpu() - want).abs().max()) < 1e-4


def test_argmax_of_fp32_rows_and_unaligned_vocabularies():
    m = model("odd", F32)
    lg = torch.randn(3, 136, device="cuda")
    lg[0, 130], lg[1, 5], lg[2, 0] = 9, 9, 9
    lg[:, 131:] = 99  # padding columns never win
    assert m._pick(lg, 0.0, 0.0, vocab=131).tolist() == [130, 5, 0]
    assert m._pick(lg.to(BF16), 0.0, 0.0, vocab=131).tolist() == [130, 5, 0]
    assert m._pick(lg, 0.0, 0.0, suppress_id=5, vocab=131).tolist()[1] != 5


@pytest.mark.parametrize("name", ["shared", "streams"])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_trace_runner(tmp_path, name, dtype):
    from safetensors.torch import save_file

    cfg = U.CONFIGS[name]
    (tmp_path / "m").mkdir()
    (tmp_path / "out").mkdir()
    (tmp_path / "m" / "config.json").write_text(json.dumps(cfg))
    save_file({k: v.contiguous() for k, v in U.weights(cfg, 3, 1.5).items()}, str(tmp_path / "m" / "model.safetensors"))
    ts, ref = toks(name), U.oracle_logits(name, LENS)
    steps = [{"step": 0, "entries": [{"id": "p", "tokens": ts[0][:60], "want": [59, 3]}, {"id": "q", "tokens": ts[1][:4], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "p", "tokens": ts[0][60:61], "want": []}, {"id": "q", "tokens": ts[1][4:], "want": []}], "end": ["q"]},
             {"step": 2, "entries": [{"id": "p", "tokens": ts[0][61:62], "want": [0]}], "end": ["p"]}]
    r = subprocess.run([sys.executable, os.path.join(REPO, "bin", "trace_run"), "--model", str(tmp_path / "m"), "--dtype", dtype, "--out",
                        str(tmp_path / "out"), "--max-tokens", "70"], input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert [x for x in r.stdout.splitlines() if x.startswith("done")] == ["done 0", "done 1", "done 2"]
    assert sorted(os.listdir(tmp_path / "out")) == ["0.f32", "2.f32"]
    read = lambda n: torch.frombuffer(bytearray((tmp_path / "out" / n).read_bytes()), dtype=F32).view(-1, cfg["vocab"])  # noqa: E731
    got = torch.cat([read("0.f32"), read("2.f32")])
    assert U.logit_error(got, ref[0][[59, 3, 61]]) < TOL[getattr(torch, dtype)]


@pytest.mark.parametrize("name", ["odd", "streams"])
def test_command_line(tmp_path, name):
    from safetensors.torch import save_file

    (tmp_path / "config.json").write_text(json.dumps(U.CONFIGS[name]))
    save_file({k: v.contiguous() for k, v in U.weights(U.CONFIGS[name], 3, 1.5).items()}, str(tmp_path / "model.safetensors"))
    p = toks(name)[1]
    r = subprocess.run([sys.executable, "-m", "moondream_amd", "generate", "--model", str(tmp_path), "--dtype", "float32", "--max-tokens", "5",
                        "--temperature", "0", "--prompt", " ".join(map(str, p)), "--prompt", "3 4"], capture_output=True, text=True, timeout=100, cwd=REPO)
    assert r.returncode == 0, r.stderr
    want = model(name, F32).batch_generate_ids([p, [3, 4]], max_tokens=5)
    assert [[int(x) for x in line.split()] for line in r.stdout.strip().splitlines()] == want


@pytest.fixture(params=[3, 7], ids=["by_size", "as_for_long_ones"])
def prompt_attention(request):
    """Attention over prompts by the kernels that their size chooses, and by those of long prompts."""
    from moondream_amd import _lib

    lib = _lib.load()
    lib.md_lm_set_kernels(request.param)
    yield
    lib.md_lm_set_kernels(3)


@pytest.mark.parametrize("heads,kv,dim,vdim", [(4, 4, 32, 32), (16, 4, 64, 64), (12, 12, 96, 128), (32, 32, 64, 64), (20, 5, 32, 64)], ids=str)
@pytest.mark.parametrize("lens,chunk", [([260], 2000), ([700], 2000), ([620, 3, 250, 431], 2000), ([900], 333)], ids=str)
def test_prompts_whose_tiles_are_cut_by_keys(heads, kv, dim, vdim, lens, chunk, prompt_attention):
    """Prefill attention of so few query tiles that their keys are divided between workgroups: first tiles whole and last ones in parts, ragged
    sequences, chunks that begin inside a part, and a second portion behind odd positions."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, kv, dim, vdim, chunk)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=4, max_context=1000)
    ts = [U.tokens(n, 120, n) for n in lens]
    want = [O.forward(cfg, w, t) for t in ts]
    slots = [m.open_sequence() for _ in ts]
    got = m.step([(s, t, range(len(t))) for s, t in zip(slots, ts)])
    assert float(U.logit_errors(got, torch.cat(want)).max()) < 7e-2
    s, cut = m.open_sequence(), lens[0] // 2 + 7
    got = torch.cat([m.step([(s, ts[0][:cut], range(cut))]), m.step([(s, ts[0][cut:], range(lens[0] - cut))])])
    assert float(U.logit_errors(got, want[0]).max()) < 7e-2


@pytest.mark.parametrize("heads,dim", [(4, 32), (16, 64), (17, 64), (32, 64), (33, 64), (32, 128)], ids=str)
def test_norms_of_prompts_sum_in_one_order(heads, dim):
    """Keys in the cache after a whole prompt (eight positions per workgroup, 256 to 1024 threads) are those of its tokens one at a time (a row per
    workgroup, 256 threads), bit for bit: fp32, where the products in front have one order of sums whatever their rows."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, heads, dim, dim, 2000)], width=64, vocab=60, ff=None)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), U.weights(cfg, 3, 1.5), dtype=F32, max_batch=2, max_context=64)
    text = U.tokens(43, 60, 1)
    whole, single = m.open_sequence(), m.open_sequence()
    m.step([(whole, text, [])])
    for t in text:
        m.step([(single, [t], [])])
    keys = m.state._slabs[0]["k"]
    assert bool(keys[whole].any()) and torch.equal(keys[whole], keys[single])


@pytest.mark.parametrize("copies", [1, 4])
@pytest.mark.parametrize("heads,kv,dim,vdim,chunk", [(3, 1, 20, 40, 2000), (4, 4, 32, 32, 33), (20, 5, 32, 24, 64), (24, 8, 64, 30, 33), (16, 16, 32, 32, 2000), (40, 40, 128, 128, 300), (64, 64, 128, 128, 300)], ids=str)
def test_fp32_rows_in_pairs(heads, kv, dim, vdim, chunk, copies):
    """561 rows in fp32, one at a time, and 2244: pairs of rows in one workgroup (16, 24 and 40 heads), pairs that two sequences or two chunks share, a last row without a second one, a
    second row with a tile of its own, heads whose pairs do not fit LDS; the same logits as those rows alone, up to the order in which a product's sums run."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, kv, dim, vdim, chunk)], width=64, vocab=60, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=F32, max_batch=24, max_context=600)
    ts = [U.tokens(n, 60, n) for n in (301, 64, 1, 130, 65)]
    slots = [m.open_sequence() for _ in range(copies * len(ts))]
    got = m.step([(s, t, range(len(t))) for s, t in zip(slots, copies * ts)])
    alone = torch.cat([m.step([(m.open_sequence(), t, range(len(t)))]) for t in ts[:3]])
    assert float(U.logit_errors(got, torch.cat(copies * [O.forward(cfg, w, t) for t in ts])).max()) < TOL[F32]
    assert float(U.logit_errors(got[: len(alone)], alone.double().cpu()).max()) < TOL[F32]


@pytest.mark.parametrize("heads,kv,dim,vdim,chunk", [(3, 1, 128, 96, 33), (17, 17, 64, 128, 2000), (32, 8, 30, 128, 45), (16, 16, 128, 128, 77), (1, 1, 32, 32, 2000), (30, 10, 64, 20, 300)], ids=str)
def test_prompts_whose_scores_go_through_memory(heads, kv, dim, vdim, chunk):
    """Heads that fill no wave's share, tiles whose queries lie in two chunks, blocks of 32 keys that begin before one, last keys at the edges of blocks and of a wave's
    share of them, one to eight waves; the second portion's convolution reads what the first one kept."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, kv, dim, vdim, chunk)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    text = U.tokens(900, 120, 9)
    ref = O.forward(cfg, w, text)  # (causal: a shorter text's logits are among them)
    for most, lens in ((900, [900]), (480, [2, 31, 32, 33, 64, 65, 255, 256, 257, 480]), (130, [5, 130])):
        m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=12, max_context=most)
        for cut in (0, 17):
            slots = [m.open_sequence() for _ in lens]
            if cut:
                m.step([(s, text[:cut], []) for s, n in zip(slots, lens) if n > cut])
            got = m.step([(s, text[cut * (n > cut) : n], range(n - cut * (n > cut))) for s, n in zip(slots, lens)])
            want = torch.cat([ref[cut * (n > cut) : n] for n in lens])
            assert float(U.logit_errors(got, want).max()) < 7e-2, (lens, cut)
            for s in slots:
                m.close_sequence(s)


@pytest.mark.parametrize("count", [1, 63, 64, 65, 130])
def test_scores_of_prompts_beside_many_running_sequences(count):
    """Tiles found by their slots among fewer sequences than a wave has lanes, as many, one more and twice as many: single tokens and prompts of several tiles in
    one step, at positions of every remainder; a second step reads the convolution's state that the first one kept."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(4, 2, 32, 32, 2000)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    text = U.tokens(210, 120, 9)
    ref = O.forward(cfg, w, text)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=count, max_context=256)
    at = [(29 * i) % 90 for i in range(count)]
    slots = [m.open_sequence() for _ in at]
    if any(at):
        m.step([(s, text[:n], []) for s, n in zip(slots, at) if n])
    for k in range(2):
        new = [(1 if i % 5 else 33 + i % 20) for i in range(count)]
        got = m.step([(s, text[a : a + n], range(n)) for s, a, n in zip(slots, at, new)])
        want = torch.cat([ref[a : a + n] for a, n in zip(at, new)])
        assert float(U.logit_errors(got, want).max()) < 7e-2, k
        at = [a + n for a, n in zip(at, new)]


@pytest.mark.parametrize("heads,kv,dim,vdim", [(4, 4, 32, 32), (12, 12, 96, 128), (32, 32, 64, 64)], ids=str)
@pytest.mark.parametrize("lens,chunk", [([260], 2000), ([700], 2000), ([620, 3, 250, 431], 2000), ([900], 333), ([300] * 13, 2000), ([530] * 8, 2000)], ids=str)
def test_prompts_whose_scores_stay_on_the_cu(heads, kv, dim, vdim, lens, chunk):
    """The kernels of longer prompts at the sizes that the others take: keys in parts, whole tiles in each of their orders."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, kv, dim, vdim, chunk)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=16, max_context=1000)
    text = U.tokens(max(lens), 120, 9)
    ref = O.forward(cfg, w, text)
    m.lib.md_lm_set_kernels(5)
    try:
        got = m.step([(m.open_sequence(), text[:n], range(n)) for n in lens])
    finally:
        m.lib.md_lm_set_kernels(3)
    assert float(U.logit_errors(got, torch.cat([ref[:n] for n in lens])).max()) < 7e-2


@pytest.mark.parametrize("lens", [[530] * 8, [300] * 16, [530] * 7 + [10], [530] * 7 + [500], [300] * 15, [300] * 13, [90] * 16],
                         ids=["eight", "sixteen", "ragged", "nearly", "fifteen", "thirteen", "short"])
def test_prompts_of_eight_sequences(lens, prompt_attention):
    """More query tiles than CUs: eight equal sequences (one to an XCD), sixteen, eight that differ, little and much, a last eight of seven, thirteen;
    short ones."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(4, 2, 32, 64, 2000)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=16, max_context=600)
    ts = [U.tokens(n, 120, i % 3) for i, n in enumerate(lens)]
    kept = {tuple(t): O.forward(cfg, w, t) for t in {tuple(t): t for t in ts}.values()}
    want = [kept[tuple(t)] for t in ts]
    got = m.step([(m.open_sequence(), t, range(len(t))) for t in ts])
    assert float(U.logit_errors(got, torch.cat(want)).max()) < 7e-2


@pytest.mark.parametrize("running,before,prompt", [(1, 300, 200), (3, 400, 290), (7, 20, 250), (15, 150, 40), (20, 300, 3), (31, 50, 330)], ids=str)
def test_prompts_beside_single_tokens(running, before, prompt, prompt_attention):
    """Sequences of one query tile beside one of many, keys in parts and whole: every tile of every sequence."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(4, 2, 32, 64, 2000)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=running + 1, max_context=640)
    ts = [U.tokens(before + 9 * (i % 4) + 1, 120, i % 5) for i in range(running)] + [U.tokens(prompt, 120, 77)]
    kept = {tuple(t): O.forward(cfg, w, t) for t in {tuple(t): t for t in ts}.values()}
    want = [kept[tuple(t)] for t in ts]
    for at in (running, 0, running // 2):  # the prompt's place
        slots = [m.open_sequence() for _ in ts]
        m.step([(s, t[:-1], []) for s, t in zip(slots[:running], ts)])
        entries = [(s, t[-1:], [0]) for s, t in zip(slots[:running], ts)]
        ref = [x[-1:] for x in want[:running]]
        entries.insert(at, (slots[running], ts[running], range(prompt)))
        ref.insert(at, want[running])
        assert float(U.logit_errors(m.step(entries), torch.cat(ref)).max()) < 7e-2
        for s in slots:
            m.close_sequence(s)


@pytest.mark.parametrize("heads,kv,dim,vdim", [(4, 4, 32, 32), (20, 5, 32, 64), (3, 1, 96, 128), (40, 40, 32, 32)], ids=str)
@pytest.mark.parametrize("count,ctx,chunk", [(128, 1100, 4000), (130, 2060, 4000), (128, 2060, 1700), (256, 1600, 4000)], ids=["a_tile", "two_tiles", "chunks", "five_blocks"])
def test_many_sequences_of_a_long_context(heads, kv, dim, vdim, count, ctx, chunk):
    """Decode attention whose splits are two, three and four blocks of 32 keys: a tile of 64 keys, two tiles of which the last is half of one, and splits that
    end within a tile, at a chunk's first key and before the split; every row."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, kv, dim, vdim, chunk)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=count, max_context=ctx)
    text = U.tokens(ctx, 120, 5)
    lens = [ctx, 1050, 700, 129, 97, 96, 65, 64, 33] + [1 + (7 * i) % 50 for i in range(count - 9)]  # (with the token of the step)
    ref = O.forward(cfg, w, text)  # (causal: a shorter text's logits are among them)
    slots = [m.open_sequence() for _ in lens]
    m.step([(s, text[: n - 1], []) for s, n in zip(slots, lens) if n > 1])
    got = m.step([(s, text[n - 1 : n], [0]) for s, n in zip(slots, lens)])
    e = U.logit_errors(got, ref[[n - 1 for n in lens]])
    assert float(e.max()) < 7e-2, e


@pytest.mark.parametrize("heads,dim,taps", [(8, 30, 1), (4, 64, 4), (2, 128, 2), (64, 32, 3), (12, 60, 3), (64, 100, 4), (48, 64, 3), (64, 64, 3)], ids=str)
@pytest.mark.parametrize("chunk", [4000, 300])
def test_decode_of_heads_with_keys_of_their_own(heads, dim, taps, chunk):
    """Scores and mixture in two launches: the first tokens (fewer than the convolution's taps), last keys at the edges of tiles of 16, of a
    workgroup's 128 and 256, sums of one, two and three workgroups; two steps, the second of which reads what the first one wrote."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(heads, heads, dim, dim, chunk, taps=taps)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=64, max_context=640)
    text = U.tokens(620, 120, 5)
    ref = O.forward(cfg, w, text)  # (causal: a shorter text's logits are among them)
    for lens in ([1, 2, 16, 17, 128, 129, 255, 256, 257, 299, 300, 301, 512, 513, 618], [4], [1 + (37 * i) % 600 for i in range(50)]):
        slots = [m.open_sequence() for _ in lens]
        m.step([(s, text[: n - 1], []) for s, n in zip(slots, lens) if n > 1])
        for k in range(2):
            got = m.step([(s, text[n - 1 + k : n + k], [0]) for s, n in zip(slots, lens)])
            e = U.logit_errors(got, ref[[n - 1 + k for n in lens]])
            assert float(e.max()) < 7e-2, (lens, k, e)
        for s in slots:
            m.close_sequence(s)


def test_captured_steps_of_many_sequences():
    """64 sequences in a graph with a context of 2048: splits of 64 keys; tokens and the last step's logits against the oracle."""
    from moondream_amd.config import LayeredLMConfig
    from moondream_amd.layered_lm import LayeredLM

    cfg = U.config([U.attention(6, 2, 32, 64, 4000)], width=96, vocab=120, ff=None)
    w = U.weights(cfg, 3, 1.5)
    m = LayeredLM(LayeredLMConfig.from_dict(cfg), w, dtype=BF16, max_batch=64, max_context=2048)
    m.compile()
    ts = [U.tokens(3 + (11 * i) % 60 if i else 200, 120, i) for i in range(64)]
    for _ in range(2):  # (the second time the graph is replayed at once)
        slots = [m.open_sequence() for _ in ts]
        m.step([(s, t[:-1], []) for s, t in zip(slots, ts)])
        logits = m._decode_logits(64)
        hist = m._decode_lockstep(torch.tensor([t[-1] for t in ts], dtype=torch.int32, device="cuda"), slots, 6).t().tolist()
        want = torch.stack([O.forward(cfg, w, t[:-1] + h[:-1])[-1] for t, h in zip(ts, hist)])
        assert float(U.logit_errors(logits[:64, :120], want).max()) < 7e-2
        for s in slots:
            m.close_sequence(s)
