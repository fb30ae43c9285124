"""CPU-side checks of the product library: it loads, exports every symbol the
C ABI header declares, validates configuration like the reference, and its
synthetic workload generator is deterministic.  No GPU compute here."""
import os
import re

import numpy as np
import pytest

import curfil_amd as cf

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "curfil_hip.h")).read()
    return sorted(set(re.findall(r"^(?:int|const char\*)\s+(cf_\w+)\(", text, re.M)))


def test_header_symbols_exported():
    names = _declared_functions()
    assert len(names) >= 30
    for n in names:
        assert hasattr(cf.lib, n), n


def test_struct_layouts_match_header():
    assert cf.SAMPLE_DTYPE.itemsize == 16
    assert cf.NODE_DTYPE.itemsize == 56
    assert cf.NODE_DTYPE.fields["score"][1] == 32
    assert cf.NODE_DTYPE.fields["feature"][1] == 40
    assert cf.NODE_DTYPE.fields["is_leaf"][1] == 51


def test_configuration_validation_like_reference():
    # random_tree.h:263-272 and random_tree.cpp:114-124
    with pytest.raises(ValueError, match="maxImages"):
        cf.TrainingConfiguration(4711, 500, 100, 32, 8, 60, 10, 10, maxImages=2, imageCacheSize=5)
    with pytest.raises(ValueError, match="acceleration mode"):
        cf.TrainingConfiguration(4711, 500, 100, 32, 8, 60, 10, 10, accelerationMode="tpu")
    c = cf.TrainingConfiguration(4711, 500, 100, 32, 8, 60, 10, 10, ignored_labels=[0]).to_c()
    assert (c.random_seed, c.feature_count, c.box_radius, c.num_ignored, c.ignored_labels[0]) == (4711, 100, 60, 1, 0)


def test_synthetic_frames_deterministic_and_shaped():
    a = cf.synth_rgbd(4711, 160, 120, 12, 5, 0.05)
    b = cf.synth_rgbd(4711, 160, 120, 12, 5, 0.05)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    rgb, depth, labels = a
    assert rgb.shape == (120, 160, 3) and depth.shape == (120, 160) and labels.shape == (120, 160)
    assert labels.max() <= 5
    zero = np.mean(depth == 0)
    assert 0.03 < zero < 0.07
    valid = depth[depth > 0]
    assert valid.min() >= 500 and valid.max() <= 5000
    c = cf.synth_rgbd(4712, 160, 120, 12, 5, 0.05)
    assert not np.array_equal(c[0], rgb)


def test_context_without_device_fails_cleanly():
    import ctypes
    n = 0
    try:
        import torch
        n = torch.cuda.device_count()
    except Exception:
        pass
    if n > 0:
        pytest.skip("a device is present")
    h = ctypes.c_void_p()
    assert cf.lib.cf_ctx_create(0, ctypes.byref(h)) != cf.CF_OK


class _RecordingLibrary:
    """Stands in for the native library: hands out handles and records the calls that release them."""

    def __init__(self):
        self.released, self.handles = [], 0

    def __getattr__(self, name):
        def call(*args):
            if name.endswith(("_destroy", "_free")):
                self.released.append((name, getattr(args[-1], "value", args[-1])))
            for a in args:
                if hasattr(a, "_obj"):
                    self.handles += 1
                    a._obj.value = self.handles
            return cf.CF_OK
        return call


@pytest.mark.parametrize("how", ["collected", "closed", "children first"])
def test_handles_are_released_before_their_context(monkeypatch, how):
    """A context and what lives on it that become garbage together (a cycle, or a script's globals at exit)
    are finalized in any order, their weak references already cleared: the native handles still go before
    the context's, the serving loop first, each once."""
    import ctypes
    import gc
    lib = _RecordingLibrary()
    monkeypatch.setattr(cf, "lib", lib)
    ctx = cf.Context(0)
    images = cf.Images(ctx, 1, 8, 8)
    forest = cf.RandomForestImage(None, ctypes.c_void_p(77))
    buffer = cf.DeviceBuffer(ctx, 64)
    server = cf.Server(ctx, forest)
    if how == "collected":
        cycle = [ctx, images, forest, buffer, server]
        cycle.append(cycle)
        del cycle
    elif how == "closed":
        ctx.close()
        assert images.h is None and forest.h is None and server.h is None
    else:
        server.close()
        forest.close()
        images.close()
    del ctx, images, forest, buffer, server
    gc.collect()
    names = [n for n, _ in lib.released]
    assert sorted(names) == ["cf_ctx_destroy", "cf_device_free", "cf_forest_destroy", "cf_images_destroy",
                             "cf_server_destroy"]
    assert names[0] == "cf_server_destroy" and names[-1] == "cf_ctx_destroy"
    assert ("cf_forest_destroy", 77) in lib.released


_TUNER_SCRIPT = """
import ctypes, os, sys
import curfil_amd as cf
choose = cf.lib._ZN2cf15evalTunerChooseEimPb
choose.argtypes = [ctypes.c_int, ctypes.c_size_t, ctypes.POINTER(ctypes.c_bool)]
record = cf.lib._ZN2cf15evalTunerRecordEimidd
record.argtypes = [ctypes.c_int, ctypes.c_size_t, ctypes.c_int, ctypes.c_double, ctypes.c_double]
record.restype = None
measure = ctypes.c_bool()
shape = choose(32, 1 << 24, ctypes.byref(measure))
print(shape, int(measure.value))
fastest = int(sys.argv[1])
while fastest >= 0 and measure.value:
    record(32, 1 << 24, shape, 1.0 if shape == fastest else 2.0, 1e9)
    shape = choose(32, 1 << 24, ctypes.byref(measure))
print(shape)
"""


def _tuner(path, fastest=-1):
    """First choice (shape, whether it is to be timed) and last for a large level of 32 thresholds in a process of
    its own, which times launches until its key is settled if `fastest` names a shape."""
    import subprocess
    import sys
    env = dict(os.environ, CURFIL_TUNE_FILE=str(path), CURFIL_TUNE_ROUNDS="1", PYTHONPATH=ROOT)
    for name in ("CURFIL_EVAL_SHAPE", "CURFIL_TUNE"):
        env.pop(name, None)
    out = subprocess.run([sys.executable, "-c", _TUNER_SCRIPT, str(fastest)], env=env, cwd=ROOT, check=True,
                         capture_output=True, text=True).stdout.split()
    return int(out[0]), int(out[1]), int(out[2])


def test_tune_file_of_another_build_is_tuned_again(tmp_path):
    """A tune file names a launch shape by what it is and the kernel it was measured on; lines that do not (an
    earlier build's shape numbers) or that name another kernel are not taken as choices."""
    path = tmp_path / "tuning.txt"
    path.write_text("32 2 4\n20 2 1\n")
    assert _tuner(path)[:2] == (0, 1)
    # what this build settles is read back as settled
    assert _tuner(path, fastest=2)[2] == 2
    assert _tuner(path)[:2] == (2, 0)
    line = [v.split() for v in path.read_text().splitlines() if v.startswith("32 2 ")][-1]
    assert tuple(int(v) for v in line[2:6]) == cf.eval_shape_info(2)
    path.write_text(" ".join(line[:-1] + [str(int(line[-1]) - 1)]) + "\n")
    assert _tuner(path)[:2] == (0, 1)


@pytest.mark.parametrize("width,height", [(1, 1), (160, 120), (640, 480), (1280, 960), (2048, 64), (32767, 32767)])
def test_level_order_keeps_as_many_place_bits_as_fit(width, height):
    """The keys of a level's order hold the (image, tree) segment and a sample's place in the image.  Where whole
    places would pass 2^26 buckets they are coarsened bit by bit, not left out (65534 segments of 640x480 and one
    more)."""
    import ctypes
    places_of = cf.lib._ZN2cf11levelPlacesEii
    bits_of = cf.lib._ZN2cf14levelPlaceBitsEmiPi
    bits_of.argtypes = [ctypes.c_uint64, ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    places = places_of(width, height)
    assert places == -(-width // 128) * -(-height // 4)
    full = (places - 1).bit_length()
    for segments in (1, 100, 65534, 65535, 131070, 131071, 1 << 20, (1 << 25) - 2, (1 << 25) - 1, (1 << 26) - 2, (1 << 27) - 1):
        shift = ctypes.c_int(-1)
        bits = bits_of(segments, places, ctypes.byref(shift))
        assert bits + shift.value == full and bits >= 0 and shift.value >= 0
        assert ((places - 1) >> shift.value).bit_length() <= bits
        assert bits == 0 or (segments + 2) << bits <= 1 << 26
        assert bits == full or (segments + 2) << (bits + 1) > 1 << 26
