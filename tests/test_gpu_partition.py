"""GPU training against the oracle where a level's samples are cut into chunks and parts of chunks."""
import numpy as np
import pytest

import curfil_amd as cf
import oracle as orc
from helpers import random_samples, random_u8_dataset

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def frames(ctx):
    rgb, depth, labels = random_u8_dataset(3, 160, 120, seed=8)
    im = cf.Images(ctx, 3, 160, 120)
    for i in range(3):
        im.set_rgbd_u8(i, rgb[i], depth[i])
    return depth, labels, im, orc.Dataset.from_u8(rgb, depth, labels)


# a part of 512 samples, one less and one more; a whole chunk of 4096 and its neighbours; the numbers of chunks past which
# they are cut into 4, 2 and no parts instead of 8
@pytest.mark.parametrize("n", [511, 512, 513, 4095, 4096, 4097, 4096 * 128 + 1, 4096 * 256 + 1, 4096 * 512 + 1])
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("mode", [cf.MODE_BATCHED, cf.MODE_PLAIN])
def test_partition_edges_match_oracle(ctx, frames, n, flip, mode):
    depth, labels, im, ds = frames
    rng = np.random.default_rng(n)
    s = random_samples(rng, n, 3, 160, 120, depth.astype(np.int32), labels=labels)
    s["label"] = rng.integers(0, 5, n)
    s["flip"] = 2 if flip else 0
    s = s[s["depth_mm"] > 0]
    s = np.resize(s, n)
    params = dict(randomSeed=99, samplesPerImage=1, featureCount=3, minSampleCount=2, maxDepth=4, boxRadius=20,
                  regionSize=6, thresholds=2, horizontalFlipping=flip)
    forest = cf.RandomForestImage.train_tree_from_samples(ctx, im, cf.TrainingConfiguration(**params), 0, 5, 99, s,
                                                          mode=mode)
    nodes, hist = forest.tree(0)
    on, oh = ds.train_tree(orc.config(**params), 0, 5, 99, s)
    assert len(nodes) == len(on) > 1
    inner = on["is_leaf"] == 0
    for name in ("id", "level", "parent", "left", "right", "num_samples", "is_leaf"):
        assert np.array_equal(nodes[name], on[name]), name
    for name in ("feature", "threshold"):
        assert np.array_equal(nodes[name][inner], on[name][inner]), name
    assert np.array_equal(hist, oh)


# levels that hold both nodes of several chunks and nodes of one, which are scored where they are counted, with a
# broken last group of features; histograms too large for that (30 thresholds, 32 classes)
@pytest.mark.parametrize("T,C,flip", [(6, 5, False), (6, 5, True), (30, 32, False)])
def test_scored_where_counted_matches_oracle(ctx, frames, T, C, flip):
    depth, labels, im, ds = frames
    rng = np.random.default_rng(T)
    s = random_samples(rng, 24000, 3, 160, 120, depth.astype(np.int32), labels=labels)
    s["label"] = (s["x"] // 20 + 2 * (s["y"] // 30)) % C
    s["flip"] = 2 if flip else 0
    s = s[s["depth_mm"] > 0][:12000]
    params = dict(randomSeed=99, samplesPerImage=1, featureCount=2100, minSampleCount=20, maxDepth=7, boxRadius=20,
                  regionSize=6, thresholds=T, horizontalFlipping=flip)
    forest = cf.RandomForestImage.train_tree_from_samples(ctx, im, cf.TrainingConfiguration(**params), 0, C, 99, s,
                                                          mode=cf.MODE_BATCHED)
    nodes, hist = forest.tree(0)
    on, oh = ds.train_tree(orc.config(**params), 0, C, 99, s)
    assert len(nodes) == len(on) > 20
    inner = on["is_leaf"] == 0
    for name in ("id", "level", "parent", "left", "right", "num_samples", "is_leaf"):
        assert np.array_equal(nodes[name], on[name]), name
    for name in ("feature", "threshold"):
        assert np.array_equal(nodes[name][inner], on[name][inner]), name
    assert np.abs(nodes["score"][inner] - on["score"][inner]).max() <= 4e-16
    assert np.array_equal(hist, oh)


def test_coarsened_places_train_alike(ctx, monkeypatch):
    """190 trees over 700 frames of 1024x256 are 133000 (image, tree) segments a level: whole places (9 bits) would
    pass 2^26 buckets and one bit is dropped.  The order only decides which lanes evaluate what: the trees are those
    of levels that are not ordered by place."""
    n, trees = 700, 190
    rgb, depth, labels = random_u8_dataset(7, 1024, 256, seed=3)
    im = cf.Images(ctx, n, 1024, 256)
    for i in range(n):
        im.set_rgbd_u8(i, rgb[i % 7], depth[i % 7])
        im.set_labels(i, labels[i % 7])
    cfg = cf.TrainingConfiguration(4711, trees, 20, 5, 5, 30, 6, 4, subsamplingType="pixelUniform")
    forests = []
    for order in ("1", "0"):
        monkeypatch.setenv("CURFIL_ROW_ORDER", order)
        forests.append(cf.RandomForestImage.train(ctx, im, cfg, trees, 6, cf.MODE_BATCHED))
    im.close()
    for t in range(trees):
        (an, ah), (bn, bh) = forests[0].tree(t), forests[1].tree(t)
        assert len(an) > 7 and an.tobytes() == bn.tobytes() and np.array_equal(ah, bh)
