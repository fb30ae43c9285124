"""GPU prediction against the oracle where a response lies at or next to its split's threshold."""
import numpy as np
import pytest

import curfil_amd as cf
import oracle as orc
from helpers import config0_dataset, random_features

pytestmark = pytest.mark.gpu


# the float test of a depth split has to hand over to the exact one at the threshold, one float beside it, at the
# edge of its error bound, for boxes without valid pixels and for thresholds that are not finite
@pytest.mark.parametrize("edge", ["equal", "above", "below", "wide", "zero", "infinite"])
@pytest.mark.parametrize("use_depth", [True, False])
def test_threshold_edges_match_oracle(ctx, edge, use_depth):
    rgb, depth, _ = config0_dataset()
    depth = depth.copy()
    depth[1, 20:60, 30:90] = 0            # boxes without a valid pixel
    depth[2] = (depth[2] // 1000) * 1000 + 1000   # equal depths: differences of exactly zero
    im = cf.Images(ctx, 4, 160, 120)
    for i in range(4):
        im.set_rgbd_u8(i, rgb[i], depth[i])
    ds = orc.Dataset.from_u8(rgb, depth)
    rng = np.random.default_rng(len(edge) + 10 * use_depth)
    n = 48
    feats = random_features(rng, n, box_radius=20, region_size=6)
    feats[0] = 0 if use_depth else 1
    feats[9:] = 0 if use_depth else rng.integers(0, 3, (2, n))
    s = np.zeros(n, orc.SAMPLE_DTYPE)
    s["image"], s["x"], s["y"] = rng.integers(0, 4, n), rng.integers(40, 120, n), rng.integers(40, 80, n)
    s["depth_mm"] = depth[s["image"], s["y"], s["x"]]
    thr = np.nan_to_num(cf.feature_responses_paired(ctx, im, s, feats)).astype(np.float32)
    if edge == "above":
        thr = np.nextafter(thr, np.float32(np.inf))
    elif edge == "below":
        thr = np.nextafter(thr, np.float32(-np.inf))
    elif edge == "wide":
        thr = thr * np.where(np.arange(n) % 2, np.float32(1 + 2.0 ** -20), np.float32(1 - 2.0 ** -20))
    elif edge == "zero":
        thr[:] = np.where(np.arange(n) % 2, np.float32(0.0), np.float32(-0.0))
    elif edge == "infinite":
        thr[:] = np.where(np.arange(n) % 2, np.float32(np.inf), np.float32(-np.inf))
    for k in range(0, n, 8):
        trees = []
        for f in range(k, k + 8):
            nodes = np.zeros(3, cf.NODE_DTYPE)
            nodes["id"], nodes["level"], nodes["parent"] = [0, 1, 2], [1, 2, 2], [-1, 0, 0]
            nodes["left"], nodes["right"], nodes["is_leaf"] = [1, -1, -1], [2, -1, -1], [0, 1, 1]
            nodes["feature"][0], nodes["threshold"][0] = feats[:, f], thr[f]
            trees.append((nodes, np.array([[1, 1], [3 + f, 1], [1, 2 + f]], np.uint32)))
        forest = cf.RandomForestImage.from_trees(ctx, trees, 2)
        forest.normalizeHistograms(0.0, False)
        for img in range(4):
            labels, probs = forest.predict(im, img)
            want, wantp = ds.predict(img, [t[0] for t in trees], [forest.posteriors(t) for t in range(8)], 2)
            assert np.array_equal(labels, want)
            assert np.array_equal(probs.view(np.uint32), wantp.view(np.uint32))


# the waves that share a tile's trees: none, one tree each, two each, as many as there may be, and back to one thread
# per pixel; a frame of 0.02 Mpix and a batch of 0.15 Mpix on either side of the rule's line
@pytest.mark.parametrize("num_trees", [1, 2, 3, 4, 5, 7, 8, 9, 16, 17, 128, 129])
def test_tree_counts_match_oracle(ctx, num_trees):
    rgb, depth, _ = config0_dataset()
    im = cf.Images(ctx, 4, 160, 120)
    for i in range(4):
        im.set_rgbd_u8(i, rgb[i], depth[i])
    ds = orc.Dataset.from_u8(rgb, depth)
    rng = np.random.default_rng(num_trees)
    feats = random_features(rng, num_trees, box_radius=20, region_size=6)
    trees = []
    for t in range(num_trees):
        nodes = np.zeros(3, cf.NODE_DTYPE)
        nodes["id"], nodes["level"], nodes["parent"] = [0, 1, 2], [1, 2, 2], [-1, 0, 0]
        nodes["left"], nodes["right"], nodes["is_leaf"] = [1, -1, -1], [2, -1, -1], [0, 1, 1]
        nodes["feature"][0], nodes["threshold"][0] = feats[:, t], rng.normal(0, 300)
        trees.append((nodes, rng.integers(1, 50, (3, 7)).astype(np.uint32)))
    forest = cf.RandomForestImage.from_trees(ctx, trees, 7)
    forest.normalizeHistograms(0.0, False)
    posts = [forest.posteriors(t) for t in range(num_trees)]
    order = [0, 1, 2, 3, 3, 2, 1, 0]
    labels, probs = forest.predict_batch(im, order)
    for img in range(4):
        want, wantp = ds.predict(img, [t[0] for t in trees], posts, 7)
        one, onep = forest.predict(im, img)
        assert np.array_equal(one, want)
        assert np.array_equal(onep.view(np.uint32), wantp.view(np.uint32))
        for k in (img, 7 - img):
            assert np.array_equal(labels[k], want)
            assert np.array_equal(probs[k].view(np.uint32), wantp.view(np.uint32))
