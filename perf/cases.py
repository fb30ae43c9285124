"""Performance cases of the framework: what programs that use it have it do, through its public Python API.

Kinds of pass:

  train    RandomForestImage.grow: a forest grown from sampled root pixels on resident integral images
           (the pixel sampling is data loading and belongs to prepare), the trees read back.  With
           "whole" the pass is RandomForestImage.train, sampling included.
  node     the plugin seams of one node: a feature table drawn from its samples, the counters, the
           scores and the argmax.
  frame    a frame as it arrives: upload, integral image, prediction with posteriors, one at a time.
  batch    predict_batch on resident frames: "device" leaves posteriors and labels in device memory,
           "host" returns both, "labels" returns the labels only.
  serve    the serving loop: frames of several sizes submitted together, all results waited for.
  lab      float-colour (CIELab) frames: set_rgbd_f32, and the integral images read back.

Frames are the seeded Voronoi frames of cf.synth_rgbd (smooth depth planes, noisy colour, missing
depth); the sizes are those of the benchmark and the tests, and odd ones between them.
"""
import math

import numpy as np
import torch

import curfil_amd as cf

_context = None


def _ctx():
    """One context for the process, as a program has."""
    global _context
    if _context is None:
        if torch.cuda.is_available():
            torch.cuda.init()
        _context = cf.Context(0)
    return _context


# ---------------------------------------------------------------- the cases


def listed():
    full = dict(kind="train", width=640, height=480, sites=30, classes=4, zero=0.08, box=120, region=20, min_samples=50,
                per_image=4000, flip=False, mode="batched", whole=False)
    return [
        # the smallest training a user runs: four small frames, one shallow tree, sampling included
        dict(name="train-small", kind="train", width=160, height=120, images=4, sites=12, classes=5, zero=0.05, trees=1,
             depth=8, features=100, thresholds=10, box=60, region=10, min_samples=32, per_image=1000, flip=False,
             mode="batched", whole=True),
        # an ordinary training: full-size frames, three trees (frames not a multiple of the device's XCDs)
        dict(full, name="train-full-frame", images=21, trees=3, depth=18, features=2000, thresholds=20),
        # the headline training configuration on a small data set: five trees to depth 20, 4000 x 32
        dict(full, name="train-batched", images=50, trees=5, depth=20, features=4000, thresholds=32),
        # a forest trained with mirrored samples (the reference's test configuration: 500 x 50)
        dict(full, name="train-flip", width=320, height=240, images=13, trees=2, depth=12, features=500, thresholds=50,
             per_image=1000, box=60, region=10, min_samples=32, flip=True),
        # the drop-in path: one node at a time
        dict(full, name="train-plain", images=8, trees=1, depth=9, features=1000, thresholds=20, mode="plain"),
        # the plugin seams on one node, as the reference's evaluator calls them
        dict(name="node-seams", kind="node", width=640, height=480, images=6, sites=30, classes=4, zero=0.08, samples=9000,
             features=500, thresholds=50, box=120, region=20),
        # one small frame at a time: latency and launches
        dict(name="frame-small", kind="frame", width=160, height=120, sites=12, classes=5, zero=0.05, trees=3, depth=10,
             box=60, region=10),
        # one full-size frame at a time through a ten-tree forest
        dict(name="frame-640x480", kind="frame", width=640, height=480, sites=30, classes=5, zero=0.05, trees=10, depth=16,
             box=120, region=20),
        # dense prediction of a large batch, results left on the device
        dict(name="batch-device", kind="batch", output="device", width=640, height=480, images=64, sites=30, classes=5,
             zero=0.05, trees=10, depth=18, box=120, region=20),
        # dense prediction of an odd batch into ordinary host arrays, the three-tree forest of a full training
        dict(name="batch-host", kind="batch", output="host", width=641, height=479, images=19, sites=30, classes=5, zero=0.05,
             trees=3, depth=16, box=120, region=20),
        # the serving loop with frames of three sizes (4 : 5 : 1)
        dict(name="serve-mix", kind="serve", small=12, middle=15, large=3, sites=30, classes=5, zero=0.05, trees=10, depth=16,
             box=120, region=20),
        # CIELab frames (the reference's default colour space) integrated for training
        dict(name="lab-integrals", kind="lab", width=640, height=480, images=3, sites=30, classes=5, zero=0.05),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "node", "frame", "frame", "batch", "batch", "serve", "lab"])
    zero = round(rng.uniform(0.02, 0.1), 3)
    if kind == "train":
        mode = rng.choice(["batched"] * 5 + ["plain"])
        # (features, thresholds) together as users set them, the number of responses per level bounded
        features, thresholds = _log(rng, 100, 4000), rng.choice([8, 10, 16, 20, 25, 32, 50])
        trees = rng.randint(1, 5)
        images = _log(rng, 3, 40)
        width, height = rng.choice([(160, 120), (320, 240), (321, 239), (640, 480), (600, 450)])
        per_image = _log(rng, 500, min(4000, width * height // 12))
        most = 8e6 if mode == "batched" else 1e6
        while images * per_image * trees * features / 250.0 > most:
            images = max(2, images * 3 // 4)
            features = max(100, features * 3 // 4)
        return dict(kind="train", width=width, height=height, images=images, sites=rng.randint(12, 30), classes=rng.randint(3, 7),
                    zero=zero, trees=trees, depth=rng.randint(6, 18) if mode == "batched" else rng.randint(5, 9), features=features,
                    thresholds=thresholds, box=rng.choice([60, 90, 120]), region=rng.choice([10, 15, 20]),
                    min_samples=rng.randint(32, 64), per_image=per_image, flip=mode == "batched" and rng.random() < 0.2, mode=mode,
                    whole=rng.random() < 0.2)
    if kind == "node":
        return dict(kind="node", width=rng.choice([320, 640]), height=rng.choice([240, 479, 480]), images=rng.randint(2, 8), sites=30,
                    classes=rng.randint(3, 9), zero=zero, samples=_log(rng, 50, 40000), features=_log(rng, 50, 1000),
                    thresholds=rng.choice([8, 10, 20, 32, 50]), box=rng.choice([60, 120]), region=rng.choice([10, 20]))
    if kind == "frame":
        width = _log(rng, 160, 1280)
        return dict(kind="frame", width=width, height=width * 3 // 4 + rng.randint(-3, 3), sites=rng.randint(12, 40),
                    classes=rng.randint(3, 9), zero=zero, trees=rng.randint(1, 12), depth=rng.randint(8, 17),
                    box=rng.choice([60, 90, 120]), region=rng.choice([10, 20]))
    if kind == "batch":
        width, height = rng.choice([(160, 120), (320, 240), (333, 251), (640, 480)])
        images = _log(rng, 2, 64)
        return dict(kind="batch", output=rng.choice(["device", "host", "labels"]), width=width, height=height, images=images,
                    sites=30, classes=rng.randint(3, 9), zero=zero, trees=rng.randint(1, 10), depth=rng.randint(8, 17),
                    box=rng.choice([60, 120]), region=rng.choice([10, 20]))
    if kind == "serve":
        return dict(kind="serve", small=rng.randint(1, 14), middle=rng.randint(1, 14), large=rng.randint(0, 3), sites=30, classes=5,
                    zero=zero, trees=rng.randint(3, 10), depth=rng.randint(10, 16), box=120, region=20)
    return dict(kind="lab", width=rng.choice([160, 321, 640]), height=rng.choice([120, 241, 480]), images=rng.randint(1, 4), sites=30,
                classes=5, zero=zero)


# ---------------------------------------------------------------- inputs

SERVE_SIZES = ((320, 240, "small"), (640, 480, "middle"), (1280, 960, "large"))


def _seed(seed, salt):
    return (seed * 1009 + salt * 7919) % 1000000007


def _frames(case, seed, n, width=None, height=None, salt=0):
    return cf.synth_dataset(n, width or case["width"], height or case["height"], sites=case["sites"], classes=case["classes"] - 1
                            if case["kind"] != "train" else case["classes"], zero_frac=case["zero"],
                            seed0=_seed(seed, 1 + salt) % 1000000)


def _images(rgb, depth, labels=None):
    n, height, width = depth.shape
    im = cf.Images(_ctx(), n, width, height)
    for i in range(n):
        im.set_rgbd_u8(i, rgb[i], depth[i])
        if labels is not None:
            im.set_labels(i, labels[i])
    return im


def _tree_tables(case, seed, frames, node_depth):
    """Complete trees of random splits over the training feature space; thresholds near the responses that the
    split's feature gives on the frames (a few sampled pixels), leaves Dirichlet(1).  Plain numpy."""
    rng = np.random.default_rng(_seed(seed, 77))
    n_nodes, n_split = (1 << node_depth) - 1, (1 << (node_depth - 1)) - 1
    idx = np.arange(n_nodes)
    level = np.zeros(n_nodes, np.int32)
    for d in range(node_depth):
        level[(1 << d) - 1:(2 << d) - 1] = d + 1
    col_int, dep_sum, dep_cnt = frames["integrals"]
    depth_mm = frames["depth"]
    h, w = depth_mm.shape
    ys, xs = np.nonzero(depth_mm)
    trees = []
    for _ in range(case["trees"]):
        nodes = np.zeros(n_nodes, cf.NODE_DTYPE)
        nodes["id"], nodes["level"] = idx, level
        nodes["parent"] = np.where(idx > 0, (idx - 1) // 2, -1)
        split = idx < n_split
        nodes["left"], nodes["right"] = np.where(split, 2 * idx + 1, -1), np.where(split, 2 * idx + 2, -1)
        nodes["is_leaf"] = ~split
        f = _random_features(rng, n_split, case["box"], case["region"])
        thr = np.full(n_split, np.nan)
        for _ in range(6):
            todo = np.flatnonzero(np.isnan(thr))
            if not len(todo):
                break
            pick = rng.integers(0, len(xs), len(todo))
            x, y = xs[pick], ys[pick]
            thr[todo] = _responses(col_int, dep_sum, dep_cnt, x, y, depth_mm[y, x], f[:, todo])
        nodes["feature"][:n_split] = f.T
        nodes["threshold"][:n_split] = np.where(np.isnan(thr), 0, thr).astype(np.float32)
        hist = np.ones((n_nodes, case["classes"]), np.uint32)
        e = rng.exponential(1.0, (n_nodes - n_split, case["classes"]))
        hist[n_split:] = np.rint(e / e.sum(1, keepdims=True) * (1 << 20)).astype(np.uint32)
        trees.append((nodes, hist))
    return trees


def _random_features(rng, n, box, region):
    f = np.zeros((11, n), np.int8)
    f[0] = rng.integers(0, 2, n)
    for r in (1, 2, 3, 4):
        f[r] = rng.integers(-box, box + 1, n)
    for r in (5, 6, 7, 8):
        f[r] = rng.integers(1, region + 1, n)
    color = f[0] == cf.COLOR
    f[9] = np.where(color, rng.integers(0, 3, n), 0)
    f[10] = np.where(color, rng.integers(0, 3, n), 0)
    return f


def _integrals(rgb, depth):
    """float32 colour sums and exact depth sums and counts of one frame, as the framework defines them"""
    col = np.cumsum(np.cumsum(rgb.astype(np.int64), axis=0), axis=1).transpose(2, 0, 1).astype(np.float32)
    dep = np.cumsum(np.cumsum(depth.astype(np.int64), axis=0), axis=1)
    cnt = np.cumsum(np.cumsum((depth > 0).astype(np.int64), axis=0), axis=1)
    return np.ascontiguousarray(col), dep, cnt


def _forest_parts(case, seed, width=None, height=None):
    """The tree tables of the case's forest, fitted to one frame of its own."""
    rgb, depth, _ = _frames(case, seed, 1, width, height, salt=5)
    return _tree_tables(case, seed, {"integrals": _integrals(rgb[0], depth[0]), "depth": depth[0]}, case["depth"])


def _forest(case, seed, width=None, height=None):
    forest = cf.RandomForestImage.from_trees(_ctx(), _forest_parts(case, seed, width, height), case["classes"])
    forest.normalizeHistograms(0.0, False)
    return forest


def _train_config(case, seed):
    return cf.TrainingConfiguration(_seed(seed, 3) % 60000, case["per_image"] * case["trees"], case["features"], case["min_samples"],
                                    case["depth"], case["box"], case["region"], case["thresholds"], ignored_labels=(0,),
                                    horizontalFlipping=case["flip"])


def _lab(rgb):
    """CIE L*a*b* (D65) of 8-bit RGB, [3][H][W] float32"""
    c = rgb.astype(np.float64) / 255.0
    c = np.where(c <= 0.04045, c / 12.92, ((c + 0.055) / 1.055) ** 2.4)
    xyz = c @ np.array([[0.4124564, 0.2126729, 0.0193339], [0.3575761, 0.7151522, 0.1191920], [0.1804375, 0.0721750, 0.9503041]])
    t = xyz / np.array([0.95047, 1.0, 1.08883])
    f = np.where(t > 216 / 24389, np.cbrt(t), (24389 / 27 * t + 16) / 116)
    lab = np.stack([116 * f[..., 1] - 16, 500 * (f[..., 0] - f[..., 1]), 200 * (f[..., 1] - f[..., 2])])
    return lab.astype(np.float32)


def _lab_frames(case, seed):
    rgb, depth, _ = _frames(case, seed, case["images"])
    return [(_lab(rgb[i]), depth[i].astype(np.int32)) for i in range(case["images"])]


def _node_inputs(case, seed):
    rng = np.random.default_rng(_seed(seed, 11))
    rgb, depth, labels = _frames(case, seed, case["images"])
    n = case["samples"]
    image, x, y = rng.integers(0, case["images"], n), rng.integers(0, case["width"], n), rng.integers(0, case["height"], n)
    samples = cf.make_samples(x, y, image, depth[image, y, x].astype(np.int32), labels[image, y, x])
    features = _random_features(rng, case["features"], case["box"], case["region"])
    # thresholds as a feature table has them: responses of the feature at sampled pixels
    thresholds = np.zeros((case["thresholds"], case["features"]), np.float32)
    ints = [_integrals(rgb[i], depth[i]) for i in range(case["images"])]
    for t in range(case["thresholds"]):
        k = rng.integers(0, n, case["features"])
        r = _responses_of(ints, samples[k], features)
        thresholds[t] = np.where(np.isnan(r), rng.normal(0, 100, case["features"]), r).astype(np.float32)
    histogram = np.bincount(samples["label"], minlength=case["classes"]).astype(np.uint32)
    return rgb, depth, samples, features, thresholds, histogram, ints


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        rgb, depth, labels = _frames(case, seed, case["images"])
        images = _images(rgb, depth, labels)
        config = _train_config(case, seed)
        state = {"images": images, "config": config, "mode": cf.MODE_PLAIN if case["mode"] == "plain" else cf.MODE_BATCHED,
                 "trees": case["trees"], "labels": case["classes"] + 1, "forest": None,
                 "rows": min((1 << case["depth"]) - 1, 4 * case["images"] * case["per_image"] // case["min_samples"] + 64)}
        if not case["whole"]:
            state["forest"] = cf.RandomForestImage.sample(_ctx(), images, config, case["trees"], case["classes"] + 1)
    elif kind == "node":
        rgb, depth, samples, features, thresholds, histogram, _ = _node_inputs(case, seed)
        state = {"images": _images(rgb, depth), "samples": samples, "features": features, "thresholds": thresholds,
                 "histogram": histogram, "classes": case["classes"], "box": case["box"], "region": case["region"],
                 "seed": _seed(seed, 13) % 100000}
    elif kind == "frame":
        rgb, depth, _ = _frames(case, seed, 1)
        state = {"rgb": rgb[0], "depth": depth[0], "images": cf.Images(_ctx(), 1, case["width"], case["height"]),
                 "forest": _forest(case, seed)}
    elif kind == "batch":
        rgb, depth, _ = _frames(case, seed, case["images"])
        state = {"images": _images(rgb, depth), "forest": _forest(case, seed), "indices": np.arange(case["images"], dtype=np.int32),
                 "output": case["output"]}
        if case["output"] == "device":
            shape = (case["images"], case["classes"], case["height"], case["width"])
            state["probs"] = torch.empty(shape, dtype=torch.float32, device="cuda:0")
            state["classes"] = torch.empty((shape[0],) + shape[2:], dtype=torch.uint8, device="cuda:0")
    elif kind == "serve":
        forest = _forest(case, seed, 640, 480)
        frames = []
        for k, (width, height, name) in enumerate(SERVE_SIZES):
            if case[name]:
                rgb, depth, _ = _frames(case, seed, case[name], width, height, salt=20 + k)
                frames += [(rgb[i], depth[i]) for i in range(case[name])]
        order = np.random.default_rng(17).permutation(len(frames))   # sizes arrive mixed
        state = {"server": cf.Server(_ctx(), forest), "frames": [frames[i] for i in order]}
    else:
        state = {"frames": _lab_frames(case, seed), "images": cf.Images(_ctx(), case["images"], case["width"], case["height"])}
    state["kind"] = kind
    return state


# ---------------------------------------------------------------- a pass


def _trees(forest, rows):
    """The forest's trees, each table padded with zeros to `rows` nodes (how many a tree has depends on the data)."""
    out = []
    for t in range(forest.num_trees):
        nodes, hist = forest.tree(t)
        n, split = len(nodes), nodes["is_leaf"] == 0
        rows = max(rows, n)
        whole = np.zeros((rows, 19), np.int32)
        for k, name in enumerate(("id", "level", "parent", "left", "right", "num_samples", "feature_id", "is_leaf")):
            whole[:n, k] = nodes[name]
        whole[:n, 8:] = np.where(split[:, None], nodes["feature"], 0)
        thresholds, scores, counts = np.zeros(rows, np.float32), np.zeros(rows), np.zeros((rows, hist.shape[1]), np.int32)
        thresholds[:n], scores[:n], counts[:n] = np.where(split, nodes["threshold"], 0), np.where(split, nodes["score"], 0), hist
        out.append({"nodes": whole, "thresholds": thresholds, "scores": scores, "histograms": counts})
    return out


def run(s):
    kind = s["kind"]
    if kind == "train":
        if s["forest"] is None:
            forest = cf.RandomForestImage.train(_ctx(), s["images"], s["config"], s["trees"], s["labels"], s["mode"])
        else:
            forest = s["forest"]
            forest.grow(s["config"], s["mode"])
        return _trees(forest, s["rows"])
    if kind == "node":
        ctx, thresholds = _ctx(), s["thresholds"]
        drawn = cf.generate_features(ctx, s["images"], s["samples"], s["seed"], thresholds.shape[1], thresholds.shape[0], s["box"],
                                     s["region"])
        counters = cf.node_counters(ctx, s["images"], s["samples"], s["features"], thresholds, s["classes"])
        scores = cf.scores(ctx, counters, s["histogram"])
        feature, threshold, score = cf.argmax_scores(ctx, scores)
        return {"drawn_features": drawn[0], "drawn_thresholds": drawn[1], "counters": counters.view(np.int32), "scores": scores,
                "feature": feature, "threshold": threshold, "score": score}
    if kind == "frame":
        s["images"].set_rgbd_u8(0, s["rgb"], s["depth"])
        labels, probs = s["forest"].predict(s["images"], 0)
        return {"labels": labels, "posteriors": probs}
    if kind == "batch":
        if s["output"] == "device":
            s["forest"].predict_batch_device(s["images"], s["indices"], s["probs"].data_ptr(), s["classes"].data_ptr())
            return {"labels": s["classes"], "posteriors": s["probs"]}
        labels, probs = s["forest"].predict_batch(s["images"], s["indices"], probabilities=s["output"] == "host")
        return {"labels": labels} if probs is None else {"labels": labels, "posteriors": probs}
    if kind == "serve":
        ids = [s["server"].submit(rgb, depth) for rgb, depth in s["frames"]]
        return [s["server"].wait(i)[:2] for i in ids]
    for i, (color, depth) in enumerate(s["frames"]):
        s["images"].set_rgbd_f32(i, color, depth)
    return [s["images"].integrals(i) for i in range(len(s["frames"]))]


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind == "train":
        # the integral images and root samples read, the trees written; a response (two box sums, their
        # difference and the thresholds it passes) of every sample and feature at every level that is evaluated
        px = case["images"] * case["width"] * case["height"]
        samples = case["images"] * case["per_image"] * case["trees"] * (2 if case["flip"] else 1)
        levels = min(case["depth"] - 1, math.log2(max(2, samples / case["trees"] / case["min_samples"])) + 1)
        return {"bytes": 20 * px + 16 * samples, "flops": samples * case["features"] * levels * (20 + case["thresholds"])}
    if kind == "node":
        px = case["images"] * case["width"] * case["height"]
        cells = case["features"] * case["thresholds"]
        return {"bytes": 20 * px + 16 * case["samples"] + cells * (8 * case["classes"] + 12),
                "flops": case["samples"] * case["features"] * (20 + case["thresholds"]) + cells * case["classes"] * 12}
    if kind == "lab":
        px = case["images"] * case["width"] * case["height"]
        return {"bytes": px * (12 + 4 + 20), "flops": px * 8}
    if kind == "serve":
        px = sum(w * h * case[name] for w, h, name in SERVE_SIZES)
    else:
        px = case.get("images", 1) * case["width"] * case["height"]
    # 5 bytes of a frame (20 where its integrals are resident), posteriors and label out; per tree and split level a
    # response of 20 operations
    inp = 20 if kind == "batch" else 5
    out = 1 + (0 if case.get("output") == "labels" else 4 * case["classes"])
    leaves = case["trees"] * ((1 << (case["depth"] - 1)) * (16 + 8 * case["classes"]))
    return {"bytes": px * (inp + out) + min(leaves, px * case["trees"] * (16 * case["depth"] + 8 * case["classes"])),
            "flops": px * case["trees"] * (case["depth"] - 1) * 20}


# ---------------------------------------------------------------- the same in 64 bits, plain numpy


def _responses(col_int, dep_sum, dep_cnt, x, y, mm, f):
    """Response of pixel i to feature column i; NaN where a box leaves the frame or has no valid depth."""
    h, w = dep_sum.shape
    d = mm.astype(np.float32) / np.float32(1000.0)
    with np.errstate(divide="ignore", invalid="ignore"):
        scaled = np.where(mm > 0, f[1:9].astype(np.float32) / d, 0).astype(np.int64)

    def box(k, plane):
        ox, oy, rx, ry = scaled[2 * k], scaled[2 * k + 1], np.maximum(scaled[4 + 2 * k], 1), np.maximum(scaled[5 + 2 * k], 1)
        lx, hx, uy, ly = x + ox - rx, x + ox + rx, y + oy - ry, y + oy + ry
        inside = (lx >= 0) & (hx < w) & (uy >= 0) & (ly < h)
        lx, hx, uy, ly = (np.where(inside, v, 0) for v in (lx, hx, uy, ly))

        def total(p):
            return (p(ly, hx) - p(uy, hx)) + (p(uy, lx) - p(ly, lx))

        c = total(lambda yy, xx: col_int[plane, yy, xx].astype(np.float64))
        s, n = total(lambda yy, xx: dep_sum[yy, xx]), total(lambda yy, xx: dep_cnt[yy, xx])
        with np.errstate(divide="ignore", invalid="ignore"):
            mean = np.where(n > 0, s / 1000.0 / n, np.nan)
        return np.where(inside, np.where(f[0] == cf.COLOR, c, mean), np.nan)

    r = box(0, f[9].astype(np.int64)) - box(1, f[10].astype(np.int64))
    return np.where(mm > 0, r, np.nan)


def _responses_of(ints, samples, features):
    r = np.full(len(samples), np.nan)
    for i, t in enumerate(ints):
        k = np.flatnonzero(samples["image"] == i)
        r[k] = _responses(*t, samples["x"][k].astype(np.int64), samples["y"][k].astype(np.int64), samples["depth_mm"][k], features[:, k])
    return r


def _classify(rgb, depth, trees, classes):
    h, w = depth.shape
    t3 = _integrals(rgb, depth)
    y, x = (v.reshape(-1) for v in np.mgrid[0:h, 0:w])
    mm = depth.reshape(-1).astype(np.int64)
    acc = np.zeros((h * w, classes))
    for nodes, hist in trees:
        at = np.zeros(h * w, np.int64)
        for _ in range(int(nodes["level"].max()) - 1):
            live = nodes["is_leaf"][at] == 0
            p, n = np.flatnonzero(live), at[live]
            r = _responses(*t3, x[p], y[p], mm[p], nodes["feature"][n].T)
            at[p] = np.where(r <= nodes["threshold"][n], nodes["left"][n], nodes["right"][n])
        leaf = hist[at].astype(np.float64)
        acc += leaf / leaf.sum(1, keepdims=True)
    return (acc / acc.sum(1, keepdims=True)).T.reshape(classes, h, w)


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        if case["width"] * case["height"] * case["trees"] * case["depth"] > 1.5e7:
            return None
        rgb, depth, _ = _frames(case, seed, 1)
        return {"labels": None, "posteriors": _classify(rgb[0], depth[0], _forest_parts(case, seed), case["classes"])}
    if kind == "batch":
        work_px = case["images"] * case["width"] * case["height"] * case["trees"] * case["depth"]
        if work_px > 1.5e7 or case["output"] == "labels":
            return None
        rgb, depth, _ = _frames(case, seed, case["images"])
        trees = _forest_parts(case, seed)
        return {"labels": None, "posteriors": np.stack([_classify(rgb[i], depth[i], trees, case["classes"]) for i in range(len(depth))])}
    if kind == "lab":
        out = []
        for color, _ in _lab_frames(case, seed):
            out.append((np.cumsum(np.cumsum(color.astype(np.float64), axis=1), axis=2), None, None))
        return out
    if kind == "node":
        n, features, thresholds, classes = case["samples"], case["features"], case["thresholds"], case["classes"]
        if n * features > 8e6:
            return None
        _, _, samples, feats, thr, histogram, ints = _node_inputs(case, seed)
        total = float(histogram.sum())
        scores = np.zeros((thresholds, features))

        def plogq(p, q):
            return np.where(p > 0, p * np.log2(np.where(p > 0, p, 1) / np.where(p > 0, q, 1)), 0)

        def xlogx(p):
            return -np.where(p > 0, p * np.log2(np.where(p > 0, p, 1)), 0)

        share = histogram / total
        for f in range(features):
            r = _responses_of(ints, samples, np.repeat(feats[:, f:f + 1], n, axis=1))
            with np.errstate(invalid="ignore"):
                goes_left = r[None, :] <= thr[:, f].astype(np.float64)[:, None]
            left = np.stack([(goes_left & (samples["label"] == c)).sum(1) for c in range(classes)], axis=1).astype(np.float64)
            right = histogram - left
            pl, pr = left.sum(1, keepdims=True) / total, right.sum(1, keepdims=True) / total
            gain = (plogq(left / total, pl * share) + plogq(right / total, pr * share)).sum(1)
            split, spread = (xlogx(pl) + xlogx(pr))[:, 0], xlogx(share).sum()
            gain = np.clip(gain, 0, 1)
            with np.errstate(divide="ignore", invalid="ignore"):
                scores[:, f] = np.where(gain == 0, 0, np.clip(2 * gain / (split + spread), 0, 1))
        return {"drawn_features": None, "drawn_thresholds": None, "counters": None, "scores": scores, "feature": None,
                "threshold": None, "score": float(scores.max())}
    return None
