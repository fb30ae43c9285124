"""GPU trainings whose levels are evaluated in one pass (k_eval_hist over several nodes at once) against the oracle,
and the sizes at which that kernel changes its tiles, its chunks and who scores."""
import numpy as np
import pytest

import curfil_amd as cf
import oracle as orc
from helpers import random_features, random_samples, random_u8_dataset

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def frames(ctx):
    rgb, depth, labels = random_u8_dataset(3, 160, 120, seed=8)
    im = cf.Images(ctx, 3, 160, 120)
    for i in range(3):
        im.set_rgbd_u8(i, rgb[i], depth[i])
    return depth, labels, im, orc.Dataset.from_u8(rgb, depth, labels)


def _compare_training(ctx, frames, s, C, mode, **params):
    _, _, im, ds = frames
    params = dict(dict(randomSeed=99, samplesPerImage=1, minSampleCount=5, boxRadius=20, regionSize=6), **params)
    forest = cf.RandomForestImage.train_tree_from_samples(ctx, im, cf.TrainingConfiguration(**params), 0, C, 99, s,
                                                          mode=mode)
    nodes, hist = forest.tree(0)
    on, oh = ds.train_tree(orc.config(**params), 0, C, 99, s)
    assert len(nodes) == len(on) > 1
    inner = on["is_leaf"] == 0
    for name in ("id", "level", "parent", "left", "right", "num_samples", "is_leaf"):
        assert np.array_equal(nodes[name], on[name]), name
    for name in ("feature_id", "feature", "threshold"):
        assert np.array_equal(nodes[name][inner], on[name][inner]), name
    assert np.abs(nodes["score"][inner] - on["score"][inner]).max(initial=0) <= 4e-16
    assert np.array_equal(hist, oh)
    return forest


# 256 thresholds do not fit the two passes' 8-bit bins; fewer take one pass with CURFIL_EVAL_DIRECT.  Nodes of
# several chunks and of less than one, all of a level together and (a budget of three nodes' histograms) in batches,
# and nodes small enough that near-ties of the argmax are replayed
@pytest.mark.parametrize("T,F,C", [(256, 24, 5), (20, 70, 5), (9, 33, 16)])
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("batches", [False, True])
def test_levels_in_one_pass_match_oracle(ctx, frames, monkeypatch, T, F, C, flip, batches):
    depth, labels, _, _ = frames
    rng = np.random.default_rng(T)
    s = random_samples(rng, 12000, 3, 160, 120, depth.astype(np.int32), labels=labels)
    s = s[s["depth_mm"] > 0][:6000]
    s["label"] = np.where(rng.random(6000) < 0.5, rng.integers(0, C, 6000), (s["x"] // 20 + 2 * (s["y"] // 30)) % C)
    s["flip"] = 2 if flip else 0
    if T < 256:
        monkeypatch.setenv("CURFIL_EVAL_DIRECT", "1")
    if batches:
        monkeypatch.setenv("CURFIL_EVAL_BUDGET_KB", str(3 * F * (T + 1) * C * 4 // 1024 + 1))
    forest = _compare_training(ctx, frames, s, C, cf.MODE_BATCHED, featureCount=F, maxDepth=12, thresholds=T,
                               minSampleCount=2, horizontalFlipping=flip)
    prof = forest.profile()
    print(f"nodes {prof['nodes']:.0f}, replays {prof['replays']:.0f}, launches {prof['eval_launches']:.0f}")
    if not flip:
        assert prof["replays"] > 0
    # a launch a level, or one for every three nodes
    if batches:
        assert prof["eval_launches"] > prof["nodes"] / 3 - 1
    else:
        assert prof["eval_launches"] == prof["levels"]


# a node of up to 512 samples is scored where it is counted: at the line, one sample less and more
@pytest.mark.parametrize("n", [511, 512, 513])
@pytest.mark.parametrize("F,T,C", [(17, 8, 5), (100, 33, 5), (16, 64, 32)])
def test_small_node_scoring_edges_match_oracle(ctx, frames, n, F, T, C):
    depth, labels, _, _ = frames
    rng = np.random.default_rng(n)
    s = random_samples(rng, 2 * n, 3, 160, 120, depth.astype(np.int32), labels=labels)
    s = s[s["depth_mm"] > 0][:n]
    s["label"] = rng.integers(0, C, n)
    _compare_training(ctx, frames, s, C, cf.MODE_PLAIN, featureCount=F, maxDepth=3, thresholds=T)


# tiles of 4 features below 512 full tiles of 16 (chunks x tiles of 16: 496, 512 and, with a broken last tile, 527);
# chunks of 512 samples instead of 256 past 2^20 (sample, tile) pairs
@pytest.mark.parametrize("n,F", [(31 * 256, 256), (31 * 256 + 1, 256), (31 * 256, 257), (65536, 256), (65537, 256)])
def test_tile_and_chunk_edges_match_oracle(ctx, frames, n, F):
    depth, labels, im, ds = frames
    T, C = 6, 6
    rng = np.random.default_rng(n + F)
    s = random_samples(rng, n, 3, 160, 120, depth.astype(np.int32), labels=labels)
    s["depth_mm"] = np.where(s["depth_mm"] > 0, s["depth_mm"], -1)
    s["label"] = rng.integers(0, C, n)
    feats = random_features(rng, F, box_radius=40)
    thr = rng.normal(0, 200, (T, F)).astype(np.float32)
    got = cf.node_counters(ctx, im, s, feats, thr, C)
    want = ds.node_counters(s, feats, thr, C)
    assert np.array_equal(got, want.transpose(1, 2, 0, 3))   # the oracle has [C][F][T][2]
