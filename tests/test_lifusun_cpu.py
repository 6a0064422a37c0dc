"""Layered language models without a GPU: configuration, weight packing, slots, registry, and the oracle the GPU tests compare with."""
import ctypes
import json

import pytest
import torch

import lm_util as U
from moondream_amd import _lib
from moondream_amd.config import AttentionMixer, LayeredLMConfig, MoondreamConfig, RetentionMixer, load_config
from moondream_amd.state import SlotPool
from moondream_amd.weights import PackedLayeredLM, pad_heads, rope_table
from oracle import layered_lm_oracle as O


def test_configuration_is_read_in_full():
    cfg = LayeredLMConfig.from_dict(U.CONFIGS["shared"])
    assert (cfg.width, cfg.vocab, cfg.eps, len(cfg.layers)) == (128, 320, 1e-5, 4)
    a, b = cfg.layers[1].mixer, cfg.layers[2].mixer
    assert isinstance(a, AttentionMixer) and (a.heads, a.kv_heads, a.dim, a.vdim, a.chunk, a.taps, a.kv_from) == (4, 2, 32, 48, 24, 3, None)
    assert b.kv_from == 1 and b.taps == 1 and b.chunk == 40 and len(b.slopes) == 8 and b.slopes[7] == 2.0 ** -8
    r = cfg.layers[3].mixer
    assert isinstance(r, RetentionMixer) and r.rot_base == 500.0 and r.scale == 64 ** -0.5 and r.decay == (0.875,)
    assert LayeredLMConfig.from_dict(U.CONFIGS["odd"]).layers[1].ff == 0


@pytest.mark.parametrize("change", [
    lambda d: d.update(extra=1),
    lambda d: d["layers"][1]["mixer"].update(window=5),
    lambda d: d["layers"][1]["mixer"].update(heads=5),
    lambda d: d["layers"][1].update(type="delta"),
    lambda d: d["layers"][0]["mixer"].update(decay=[0.9]),
    lambda d: d["layers"][0]["mixer"]["rot"].update(dims=33),
    lambda d: d["layers"][2]["mixer"].update(kv_from=0),
    lambda d: d["layers"][2]["mixer"].update(dim=64),
    lambda d: d["layers"][2]["mlp"].update(kind="experts"),
])
def test_configuration_errors_are_named(change):
    d = json.loads(json.dumps(U.CONFIGS["shared"]))
    change(d)
    with pytest.raises(ValueError):
        LayeredLMConfig.from_dict(d)


def test_registry_chooses_by_configuration(tmp_path):
    from moondream_amd.layered_lm import LayeredLM
    from moondream_amd.moondream import MoondreamModel
    from moondream_amd.registry import model_class

    (tmp_path / "config.json").write_text(json.dumps(U.CONFIGS["odd"]))
    assert model_class(load_config(str(tmp_path))) is LayeredLM
    (tmp_path / "config.json").write_text(json.dumps({"text": {"n_layers": 2}}))
    cfg = load_config(str(tmp_path))
    assert isinstance(cfg, MoondreamConfig) and cfg.text.n_layers == 2 and model_class(cfg) is MoondreamModel
    (tmp_path / "config.json").write_text(json.dumps({"architecture": "Nothing"}))
    with pytest.raises(ValueError, match="Nothing"):
        load_config(str(tmp_path))


def _packed(name, dtype=torch.float32):
    cfg = U.CONFIGS[name]
    w = U.weights(cfg, seed=1)
    return cfg, w, PackedLayeredLM(LayeredLMConfig.from_dict(cfg), dict(w), "cpu", dtype)


def test_packing_pads_heads_and_keeps_every_weight():
    cfg, w, p = _packed("odd")
    m, o = cfg["layers"][2]["mixer"], p.layers[2]  # 6 query and 3 key / value heads of 20 and 12
    assert (o.dim_pad, o.vdim_pad, o.col_q, o.col_k, o.col_v, o.in_proj.n_pad, o.in_proj.k_pad) == (32, 32, 0, 192, 288, 384, 64)
    mats = {t.w.data_ptr(): t for t in p._keep if hasattr(t, "w")}
    lin = mats[o.in_proj.w]
    k = lin.w[192:288].view(3, 32, 64)
    assert torch.equal(k[:, :20, :52].reshape(60, 52), w["l2.mix.k"].float()) and k[:, 20:].abs().sum() == 0 and k[:, :, 52:].abs().sum() == 0
    assert torch.equal(lin.b[288:384].view(3, 32)[:, :12].reshape(-1), w["l2.mix.v.b"].float())
    out = mats[o.out_proj.w].w
    assert torch.equal(out[:52, :192].view(52, 6, 32)[:, :, :12].reshape(52, 72), w["l2.mix.o"].float()) and o.out_proj.k_pad == 192
    f32 = {t.data_ptr(): t for t in p._keep if torch.is_tensor(t)}
    assert torch.equal(f32[o.conv][:, 192:288].t().reshape(3, 32, 4)[:, :20].reshape(60, 4), w["l2.mix.k.conv"].float())
    assert o.norm1.stride == 0 and f32[o.norm1.w].item() == w["l2.norm1"].float().item()
    assert p.layers[1].ff == 0 and p.layers[0].ff_pad == 64 and p.layers[2].ff_pad == 128


def test_packing_names_missing_and_unknown_tensors():
    cfg = U.CONFIGS["retention"]
    c = LayeredLMConfig.from_dict(cfg)
    w = U.weights(cfg)
    with pytest.raises(ValueError, match="l0.mix.g is missing"):
        PackedLayeredLM(c, {k: v for k, v in w.items() if k != "l0.mix.g"}, "cpu")
    with pytest.raises(ValueError, match="l9.mix.q"):
        PackedLayeredLM(c, dict(w, **{"l9.mix.q": w["l0.mix.q"]}), "cpu")
    with pytest.raises(ValueError, match="shape"):
        PackedLayeredLM(c, dict(w, **{"l0.mix.q": w["l0.mix.q"][:-1]}), "cpu")
    with pytest.raises(ValueError, match="float16"):
        PackedLayeredLM(c, dict(w), "cpu", torch.float16)


def test_pad_heads_along_columns():
    t = torch.arange(12.0).view(2, 6)
    assert pad_heads(t, 2, 4, axis=1).tolist() == [[0, 1, 2, 0, 3, 4, 5, 0], [6, 7, 8, 0, 9, 10, 11, 0]]


def test_exact_rotation_table():
    t = rope_table(6, 5000, 1e4, exact=True)
    a = torch.tensor(4999.0, dtype=torch.float64) * 1e4 ** (-2.0 / 6)
    assert abs(t[4999, 1, 0] - a.cos()) < 1e-7 and abs(t[4999, 1, 1] - a.sin()) < 1e-7


def test_slots_are_reused_lowest_first():
    pool = SlotPool(2)
    a, b = pool.take(), pool.take()
    assert (a, b, pool.available()) == (0, 1, 0)
    pool.grow(4)
    assert pool.take() == 2
    pool.length[a] = 7
    pool.free(a)
    assert pool.length[a] == 0 and pool.take() == 0
    with pytest.raises(ValueError):
        pool.free(3)


def test_entry_points_validate_on_the_host():
    lib = _lib.load()
    assert lib.md_lm_workspace_bytes(None, None, 1) == 0
    assert lib.md_lm_forward(None, None, None, None, 0, None, 0, None, None, 0, None) == 1
    assert lib.md_gemm_f32(None, 0, None, None, 0, 1, None) == 1
    cfg, w, p = _packed("odd", torch.bfloat16)
    assert lib.md_lm_workspace_bytes(ctypes.byref(p.model), ctypes.byref(_lib.MdLmBatch(2, 7, 5, max_ctx=64)), 2) > 0


def test_steps_say_how_many_sequences_go_on():
    """The count lies where the structure had padding: everything else is where it was."""
    assert _lib.MdLmBatch.n_going.offset == 12 and _lib.MdLmBatch.tokens.offset == 16 and ctypes.sizeof(_lib.MdLmBatch) == 80
    lib, (cfg, w, p) = _lib.load(), _packed("retention", torch.bfloat16)
    size = lambda going: lib.md_lm_workspace_bytes(ctypes.byref(p.model), ctypes.byref(_lib.MdLmBatch(3, 9, 4, going, max_ctx=64, ctx_rows=40)), 3)  # noqa: E731
    assert size(0) == size(2) == size(3) > 0


@pytest.mark.parametrize("mixers", [[0, 1], [2, 3], [2]], ids=["attention_retention", "latent_state_space", "latent"])
@pytest.mark.parametrize("experts", [0, 32])
def test_a_workspace_of_the_largest_prompt_serves_all(mixers, experts):
    lib, linear = _lib.load(), lambda n, k: _lib.MdLinear(4096, None, n, k, n, k)  # (sizes only: nothing is read through the pointers)
    layers = (_lib.MdLmLayer * len(mixers))()
    for i, (l, mixer) in enumerate(zip(layers, mixers)):
        l.mixer, l.heads, l.kv_heads, l.kv_layer, l.taps, l.groups, l.norm_groups, l.rank, l.rank_pad = mixer, 32, 32, i, 4, 1, 1, 256, 256
        l.dim = l.dim_pad = l.vdim = l.vdim_pad = 64
        l.in_proj, l.out_proj, l.up_kv = linear(8192, 2048), linear(2048, 2048), linear(4096, 256)
        l.ff, l.ff_pad, l.gate_up, l.down, l.experts, l.top = 5440, 5440, linear(10880, 2048), linear(2048, 5440), experts, 4 if experts else 0
    m = _lib.MdLmModel(dtype=0, width=2048, width_pad=2048, vocab=51200, n_layers=len(mixers), layers=layers, head=linear(51200, 2048))
    for n_seq in (1, 8):
        batch = lambda n: _lib.MdLmBatch(n_seq, n * n_seq, n, 0, max_ctx=n, ctx_rows=n * n_seq)  # noqa: E731
        sizes = [lib.md_lm_workspace_bytes(ctypes.byref(m), ctypes.byref(batch(n)), 1) for n in range(2, 2100)]
        assert sizes == sorted(sizes) and sizes[0] > 0


def test_language_model_symbols_are_declared():
    assert set(_lib.LM_SYMBOLS) <= set(_lib.exported_symbols())


def test_oracle_retention_against_its_closed_form():
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(9, 2, n, generator=g, dtype=torch.float64) for n in (6, 6, 5))
    dec = torch.tensor([0.7, 1.0], dtype=torch.float64)
    t = torch.arange(9)
    d = (t[:, None] - t[None]).clamp(min=0)
    wt = torch.stack([torch.where(t[:, None] >= t[None], x ** d, torch.zeros(())) for x in dec])
    want = torch.einsum("hts,shv->thv", torch.einsum("thd,shd->hts", q, k) * wt, v)
    assert torch.allclose(O.retention(q, k, v, dec), want, atol=1e-12)


def test_oracle_attention_without_its_extras_is_plain_softmax():
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(7, 2, 8, generator=g, dtype=torch.float64) for _ in range(3))
    got = O.talking_chunk_attention(q, k, v, 0.3, torch.eye(2, dtype=torch.float64), 100, fault="no_slope")
    want = torch.nn.functional.scaled_dot_product_attention(q.transpose(0, 1), k.transpose(0, 1), v.transpose(0, 1), is_causal=True, scale=0.3)
    assert torch.allclose(got, want.transpose(0, 1), atol=1e-12)


def test_oracle_conv_and_rotation_by_hand():
    u = torch.tensor([[1.0], [2.0], [4.0]])
    assert O.causal_conv(u, torch.tensor([[10.0, 1.0]])).tolist() == [[1.0], [12.0], [24.0]]
    x = torch.tensor([[[1.0, 2.0, 3.0, 4.0, 9.0]]] * 2, dtype=torch.float64)
    y = O.rotate_half(x, 4, 100.0)
    c, s = torch.tensor(1.0).double().cos(), torch.tensor(1.0).double().sin()
    assert torch.equal(y[0], x[0]) and torch.allclose(y[1, 0, 0], 1 * c - 3 * s) and torch.allclose(y[1, 0, 2], 3 * c + 1 * s) and y[1, 0, 4] == 9


@pytest.mark.parametrize("fault", O.FAULTS + O.STREAM_FAULTS)
def test_every_planted_mistake_shows(fault):
    """The models the GPU tests run on would show each of these mistakes at 100 times the fp32 tolerance."""
    name = U.SHOWS[fault]
    good, bad = U.oracle_logits(name, [61]), U.oracle_logits(name, [61], fault=fault)
    assert U.logit_error(bad[0], good[0]) > 2e-3


@pytest.mark.parametrize("dim,vdim,resident", [(32, 32, 3), (32, 128, 2), (64, 64, 2), (64, 96, 2), (64, 128, 1), (96, 96, 1), (128, 32, 1), (128, 64, 1), (128, 128, 1), (160, 64, 0)])
def test_segments_of_retention_prompts(dim, vdim, resident):
    """As many as are resident by the kernel's LDS on 256 compute units, none of them empty, within the states that the largest step reserves."""
    lib = _lib.load()
    segments, most = lib._Z15lm_ret_segmentsiiiiiPi, lib._Z18lm_ret_most_statesiiiii  # (internal: lm_internal.hpp)
    for heads in (1, 3, 16, 40, 300):
        for n_seq in (1, 2, 7, 64):
            for n in (2, 64, 65, 130, 200, 500, 700, 2048, 100000):
                per = ctypes.c_int()
                segs, chunks = segments(n_seq, heads, dim, vdim, n, ctypes.byref(per)), -(-n // 64)
                assert (segs - 1) * per.value < chunks <= segs * per.value
                if segs > 1:
                    assert segs * n_seq * heads <= 256 * resident
                    assert all(n_seq * ((segs - 1) * per.value + 1) <= most(s, heads, dim, vdim, m) for s in (n_seq, 64) for m in (n, 100000))
                elif resident * 256 >= 4 * n_seq * heads:
                    assert chunks < 4
