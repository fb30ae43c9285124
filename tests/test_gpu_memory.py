"""Sizes of device memory: histograms past 2^32 words."""
import numpy as np
import pytest

import curfil_amd as cf

pytestmark = pytest.mark.gpu


def test_histograms_past_2_32_words(ctx, monkeypatch):
    """A histogram budget of 32 GiB lets a level's 307 nodes of 8192 features x 256 bins x 10 classes be cleared,
    counted and scored at once (6.4e9 words, 2.5 million workgroups of scores); the trees are those of the default
    budget, whose batches are a sixteenth of that."""
    rgb, depth, labels = cf.synth_dataset(4, 160, 120, sites=60, classes=9, zero_frac=0.05, seed0=4711)
    rng = np.random.default_rng(3)
    labels = np.where(rng.random(labels.shape) < 0.3, rng.integers(0, 10, labels.shape), labels).astype(np.uint8)
    im = cf.Images(ctx, 4, 160, 120)
    for i in range(4):
        im.set_rgbd_u8(i, rgb[i], depth[i])
        im.set_labels(i, labels[i])
    cfg = cf.TrainingConfiguration(4711, 15000, 8192, 2, 8, 30, 8, 255)
    want = cf.RandomForestImage.train(ctx, im, cfg, 5, 10, cf.MODE_BATCHED)
    monkeypatch.setenv("CURFIL_EVAL_BUDGET_MB", "32768")
    got = cf.RandomForestImage.train(ctx, im, cfg, 5, 10, cf.MODE_BATCHED)
    nodes = 0
    for t in range(5):
        (wn, wh), (gn, gh) = want.tree(t), got.tree(t)
        assert wn.tobytes() == gn.tobytes() and np.array_equal(wh, gh)
        nodes += int(((wn["level"] == 7) & (wn["num_samples"] >= 2) & ((wh > 0).sum(1) > 1)).sum())
    assert nodes * 8192 * 256 * 10 > 1 << 32
    assert want.profile()["slot_batches_max"] > 1 and got.profile()["slot_batches_max"] == 1
    im.close()
