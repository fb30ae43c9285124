"""GPU integration of float-colour frames against the oracle at the edges of the row chunks."""
import numpy as np
import pytest

import curfil_amd as cf
import oracle as orc

pytestmark = pytest.mark.gpu


# chunks of half a row up to 256 pixels: one-pixel chunks, blocks of 8 with and without a remainder, a short last
# chunk; one column and 6400 columns are past the LDS kernel's range
@pytest.mark.parametrize("W,H", [(1, 9), (2, 5), (3, 4), (15, 3), (16, 3), (33, 2), (511, 4), (512, 3), (513, 4), (769, 3),
                                 (6400, 2)])
def test_float_integral_chunk_edges(ctx, W, H):
    rng = np.random.default_rng(W)
    # values of very different size and both signs, so that every operation rounds
    color = (rng.normal(0, 1, (1, 3, H, W)) * 10.0 ** rng.integers(-6, 6, (1, 3, H, W))).astype(np.float32)
    depth = rng.integers(-1, 5000, (1, H, W)).astype(np.int32)
    im = cf.Images(ctx, 1, W, H)
    im.set_rgbd_f32(0, color[0], depth[0])
    got, want = im.integrals(0), orc.Dataset(color, depth).integrals(0)
    assert np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32))
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2])
