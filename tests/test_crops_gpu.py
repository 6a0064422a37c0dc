"""Crops cut on the device (md_cut_crops) against the ones the host cuts with PIL: the same bytes (reference: image_crops.py:58-167)."""
import numpy as np
import pytest
import torch
from PIL import Image

from moondream_amd import image_crops
from moondream_amd.image_crops import overlap_crop_image

pytestmark = pytest.mark.gpu

# (height, width): a row more than a crop, tiny, both directions up, down and mixed, odd rows, long and flat, 3 megapixels
SIZES = [[(379, 378)], [(1, 1)], [(2, 1500)], [(120, 2)], [(300, 200)], [(768, 1024)], [(481, 643)], [(1400, 333)], [(1500, 2000)],
         [(378, 378), (768, 1024), (17, 31), (378, 379), (333, 1999), (1080, 1920)]]


@pytest.fixture(scope="module")
def model():
    from moondream_amd import synth
    from moondream_amd.config import get_config
    from moondream_amd.moondream import IdTokenizer, MoondreamModel

    cfg = get_config("tiny")
    return MoondreamModel(cfg, synth.synthetic_state_dict(cfg, seed=1, device="cuda"), device="cuda", tokenizer=IdTokenizer(), max_batch=4)


def pictures(sizes):
    rng = np.random.default_rng(sum(h + 3 * w for h, w in sizes))
    made = [rng.integers(0, 256, (h, w, 3), dtype=np.uint8) for h, w in sizes]
    return [Image.fromarray(np.where(a < 128, 0, 255).astype(np.uint8) if i % 2 else a) for i, a in enumerate(made)]  # (every other one: edges that overshoot)


@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "+".join("%dx%d" % x for x in s))
def test_the_same_bytes_as_pil(model, monkeypatch, sizes):
    monkeypatch.setattr(image_crops, "_pyvips", None)
    v = model.config.vision
    images = pictures(sizes)
    _, staged = model._stage_crops(images)
    got = []
    while staged:
        host, token, futs, plan = staged.pop(0)
        assert plan is not None
        part = [f.result() for f in futs]
        got.append(model._cut_crops(model._upload_pinned(host, token), plan, part))
    got = torch.cat(got).cpu().numpy()
    want = [overlap_crop_image(np.array(im), v.overlap_margin, v.max_crops, (v.crop_size, v.crop_size), v.enc_patch_size)["crops"] for im in images]
    assert np.array_equal(got, np.concatenate(want))


def test_what_stays_on_the_host(model, monkeypatch):
    plan = lambda *sizes: model._cut_plan([Image.new("RGB", (w, h)) for h, w in sizes], [(1, 1)] * len(sizes), 1 << 20)  # noqa: E731
    monkeypatch.setattr(image_crops, "_pyvips", None)
    assert plan((378, 378), (378, 300)) is not None
    assert plan((378, 378), (378, 378)) is None  # nothing to resize
    assert plan((378, 378), (650, 10)) is None   # PIL's other order
    assert plan((1024, 1024)) is None            # more bytes than asked for
    monkeypatch.setattr(image_crops, "_pyvips", object())
    assert plan((378, 300)) is None


def test_a_file_that_decodes_to_another_size(model, monkeypatch):
    """The named size decides how many crops there are, the decoded pixels what is in them, as on the host."""
    monkeypatch.setattr(image_crops, "_pyvips", None)
    v = model.config.vision
    other, plain = pictures([(310, 210), (500, 700)])
    grey = Image.new("L", (200, 300))
    monkeypatch.setattr(grey, "convert", lambda mode: other)
    _, staged = model._stage_crops([grey, plain])
    host, token, futs, plan = staged.pop(0)
    part = [f.result() for f in futs]
    got = model._cut_crops(model._upload_pinned(host, token), plan, part).cpu().numpy()
    want = [overlap_crop_image(np.array(im), v.overlap_margin, v.max_crops, (v.crop_size, v.crop_size), v.enc_patch_size)["crops"] for im in (other, plain)]
    assert np.array_equal(got, np.concatenate(want))
