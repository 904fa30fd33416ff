"""References that take a whole wave in the raster kernels (tile-level ones and
those of 40 quads or more), which a work item's waves share: items of more
references than are listed at a time (1,024; 512 with multisampling) against
items of 256 references, bit for bit, and against the oracle.  And raster
matrices whose pictures are far larger than the frame, so that triangles leave
the compact form (16,384 sixteenths of a pixel) and differences of their
coordinates leave 24 bits, against the oracle."""
import numpy as np
import pytest

from edxraster_amd import configs, Renderer
from edxraster_amd import _lib as L
from test_direct_frame import frame, oracle_frame, same, triangles

pytestmark = pytest.mark.gpu


def long_items():
    """256x256, 180,000 triangles of about 14 pixels each way and 40 of the whole picture."""
    rng = np.random.default_rng(7)
    n = 180000
    c = np.stack([rng.uniform(-1.2, 1.2, n), rng.uniform(-1.2, 1.2, n), rng.uniform(-0.3, 0.3, n)], 1)
    corner = np.array([[-0.08, -0.08, 0.0], [0.08, -0.08, 0.0], [0.0, 0.08, 0.0]])
    small = c[:, None, :] + corner[None] + rng.uniform(-0.01, 0.01, (n, 3, 3))
    big = 20.0 * corner[None] + rng.uniform(-0.2, 0.2, (40, 3, 3))
    return triangles(np.concatenate([small, big]), 256, 256)


@pytest.mark.parametrize("msaa", [0, 1, 2, 3])
def test_long_items(built, msaa):
    w = long_items()
    r = Renderer(w.width, w.height)
    w.apply(r)
    r.set_msaa_mode(msaa)
    frames = []
    for per_cu in (0, 1):
        assert L.lib().edxr_set_state(r.ctx, L.STATE_RASTER_BLOCKS_PER_CU, per_cu) == 0
        r.render_mesh(w.mesh)
        frames.append(frame(r))
    assert same(frames[0], frames[1])
    r.close()
    if not msaa:
        assert same(frames[0][:2], oracle_frame(w))


@pytest.mark.parametrize("chunks", [0, 3])
@pytest.mark.parametrize("scale", [1, 8, 20, 300, 3000])
def test_large_raster_matrix(built, scale, chunks):
    w = configs.small_sphere(200, 136, 24, 12)
    raster = np.array(w.raster, np.float32).reshape(4, 4).copy()
    raster[:2, :3] *= scale
    w.raster = raster
    r = Renderer(w.width, w.height)
    w.apply(r)
    r.set_bin_chunks(chunks)
    r.render_mesh(w.mesh)
    assert same(frame(r)[:2], oracle_frame(w))
    r.close()
