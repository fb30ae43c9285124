"""GPU counters, scores and best split of one node against the oracle at the edges of the launch shapes."""
import numpy as np
import pytest

import curfil_amd as cf
import oracle as orc
from helpers import random_features, random_samples, random_u8_dataset

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def frames(ctx):
    rgb, depth, labels = random_u8_dataset(3, 160, 120, seed=5)
    im = cf.Images(ctx, 3, 160, 120)
    for i in range(3):
        im.set_rgbd_u8(i, rgb[i], depth[i])
    return depth, labels, im, orc.Dataset.from_u8(rgb, depth, labels)


# one lane, a full and a broken workgroup of samples; feature tiles of 4 and 16 with remainders; enough chunks for
# the per-XCD order (64 of 256 samples) and one less; the widest threshold rows; classes from 1 to 32
@pytest.mark.parametrize("n,F,T,C", [(1, 1, 1, 1), (255, 4, 8, 6), (256, 5, 9, 6), (257, 17, 12, 6), (513, 3, 256, 2),
                                     (16128, 5, 13, 6), (16129, 5, 33, 6), (20000, 33, 20, 32), (700, 70, 65, 7)])
def test_node_counters_and_split_edges(ctx, frames, n, F, T, C):
    depth, labels, im, ds = frames
    rng = np.random.default_rng(n + F)
    s = random_samples(rng, n, 3, 160, 120, depth.astype(np.int32), labels=labels)
    s["depth_mm"] = np.where(s["depth_mm"] > 0, s["depth_mm"], -1)
    s["label"] = rng.integers(0, C, n)
    feats = random_features(rng, F, box_radius=40)
    thr = rng.normal(0, 200, (T, F)).astype(np.float32)
    if T > 8:
        thr[3], thr[5] = thr[4], 0.0          # equal thresholds share a rank
    got = cf.node_counters(ctx, im, s, feats, thr, C)
    want = ds.node_counters(s, feats, thr, C)
    assert np.array_equal(got, want.transpose(1, 2, 0, 3))   # the oracle has [C][F][T][2]
    hist = np.bincount(s["label"], minlength=C).astype(np.uint32)
    sc = orc.scores_from_counters(want, hist)
    f, t, score = cf.node_best_split(ctx, im, s, feats, thr, C, hist)
    bf, bt, bs = orc.argmax(sc)
    assert abs(score - bs) <= 4e-16
    assert (f, t) == (bf, bt)


# windows of 64 scores and segments of them, one score more and less; scans that take every score, none after the
# first, a few, and steps around the 1e-13 below which a larger score is not taken
@pytest.mark.parametrize("F,T", [(1, 1), (63, 1), (64, 1), (65, 1), (1024, 1), (1025, 1), (73, 15), (400, 50), (1200, 60)])
@pytest.mark.parametrize("order", ["random", "ascending", "descending", "equal", "ties", "steps"])
def test_argmax_scan_edges(ctx, F, T, order):
    rng = np.random.default_rng(F * T)
    n = F * T
    scores = rng.random(n)
    if order == "ascending":
        scores = np.sort(scores)
    elif order == "descending":
        scores = np.sort(scores)[::-1].copy()
    elif order == "equal":
        scores[:] = 0.25
    elif order == "ties":
        scores = 0.5 + rng.integers(0, 40, n) * 0.3e-13
    elif order == "steps":
        scores = 0.5 + np.arange(n) * rng.choice([0.2e-13, 0.6e-13, 1.1e-13], n)
    scores = scores.reshape(T, F)
    f, t, best = cf.argmax_scores(ctx, scores)
    bf, bt, bb = orc.argmax(scores)
    assert (f, t) == (bf, bt) and best == bb


# the number of scores past which sixteen waves take them, and segments of a few windows behind it
@pytest.mark.parametrize("F,T", [(3072, 1), (1024, 3), (3073, 1), (439, 7), (4097, 1), (512, 11)])
@pytest.mark.parametrize("order", ["random", "ascending", "ties", "steps", "infinite"])
def test_argmax_waves_edges(ctx, F, T, order):
    rng = np.random.default_rng(F * T)
    n = F * T
    scores = rng.random(n)
    if order == "ascending":
        scores = np.sort(scores)
    elif order == "ties":
        scores = 0.5 + rng.integers(0, 40, n) * 0.3e-13
    elif order == "steps":
        scores = 0.5 + np.arange(n) * rng.choice([0.2e-13, 0.6e-13, 1.1e-13], n)
    elif order == "infinite":
        scores[:n // 2] = -np.inf
        scores[rng.integers(0, n, 5)] = np.nan
    scores = scores.reshape(T, F)
    f, t, best = cf.argmax_scores(ctx, scores)
    bf, bt, bb = orc.argmax(scores)
    assert (f, t) == (bf, bt) and best == bb
