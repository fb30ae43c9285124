"""Sizes of device memory: histograms past 2^32 words, what a context keeps between calls."""
import ctypes
import time

import numpy as np
import pytest

import curfil_amd as cf
from helpers import random_features, random_samples, random_u8_dataset

pytestmark = pytest.mark.gpu


def _free_bytes(ctx):
    """free device memory, from the HIP runtime that the library has loaded; the driver returns freed memory a
    millisecond or so after hipFree"""
    ctx.synchronize()
    time.sleep(0.25)
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


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


@pytest.mark.parametrize("call", ["counters", "best split", "refused"])
def test_tables_of_a_large_node_call_are_given_back(ctx, call):
    """The features of a single-node call are not limited in number: its tables (here 340 MiB) stay with the
    context up to 64 MiB only, also when the call is refused after its buffers were made."""
    rgb, depth, _ = random_u8_dataset(1, 64, 48, seed=5)
    im = cf.Images(ctx, 1, 64, 48)
    im.set_rgbd_u8(0, rgb[0], depth[0])
    rng = np.random.default_rng(2)
    s = random_samples(rng, 40, 1, 64, 48, depth.astype(np.int32))
    s["depth_mm"] = np.where(s["depth_mm"] > 0, s["depth_mm"], -1)
    s["label"] = rng.integers(0, 2, 40)
    hist = np.bincount(s["label"], minlength=2).astype(np.uint32)

    def run(F, T, bad=False):
        feats = random_features(rng, F, box_radius=10)
        thr = rng.normal(0, 200, (T, F)).astype(np.float32)
        if bad:
            thr[0, 0] = np.nan
        if call == "counters":
            cf.node_counters(ctx, im, s, feats, thr, 2)
        else:
            cf.node_best_split(ctx, im, s, feats, thr, 2, hist)

    run(10, 8)
    before = _free_bytes(ctx)
    if call == "refused":
        with pytest.raises(cf.CurfilError):
            run(4000000, 16, bad=True)
    else:
        run(400000, 64)
    assert before - _free_bytes(ctx) <= 80 << 20
    run(10, 8)
    im.close()


def test_workspace_of_a_large_training_is_trimmed_and_used_again(ctx):
    """A training whose workspace passes 1 GiB (a level of more than 50 nodes of 8192 features x 65 bins x 10 classes
    in its histograms alone) leaves at most that with the context; the next trainings on it, a small one and the
    same again, give the same trees as the first and as another context."""
    rgb, depth, labels = cf.synth_dataset(4, 160, 120, sites=60, classes=9, zero_frac=0.05, seed0=4711)
    rng = np.random.default_rng(3)
    labels = np.where(rng.random(labels.shape) < 0.3, rng.integers(0, 10, labels.shape), labels).astype(np.uint8)
    im = cf.Images(ctx, 4, 160, 120)
    for i in range(4):
        im.set_rgbd_u8(i, rgb[i], depth[i])
        im.set_labels(i, labels[i])

    def train(c, images, features, thresholds):
        cfg = cf.TrainingConfiguration(4711, 6000, features, 2, 6, 30, 8, thresholds)
        f = cf.RandomForestImage.train(c, images, cfg, 4, 10, cf.MODE_BATCHED)
        out = [f.tree(t) for t in range(4)]
        f.close()
        return out

    before = _free_bytes(ctx)
    own = cf.Context(0)
    im2 = cf.Images(own, 4, 160, 120)
    for i in range(4):
        im2.set_rgbd_u8(i, rgb[i], depth[i])
        im2.set_labels(i, labels[i])
    first = train(own, im2, 8192, 64)
    level = sum(int(((n["level"] == 5) & (n["num_samples"] >= 2) & ((h > 0).sum(1) > 1)).sum()) for n, h in first)
    assert level * 8192 * 65 * 10 * 4 > 1 << 30
    assert before - _free_bytes(own) <= (1 << 30) + (256 << 20)   # the images, the stream and the call's scratch beside it
    small = train(own, im2, 40, 10)
    again = train(own, im2, 8192, 64)
    want = train(ctx, im, 40, 10)
    for a, b in list(zip(first, again)) + list(zip(small, want)):
        assert a[0].tobytes() == b[0].tobytes() and np.array_equal(a[1], b[1])
    own.close()
    im.close()
