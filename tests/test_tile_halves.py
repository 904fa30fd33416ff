"""Direct frames whose tiles two workgroups share, 16 rows each (up to 512 tiles),
and one beyond: pictures that end in a tile's upper or lower half, with triangles
of every walk (a lane, quads, a whole wave, trivially accepted), three frames of
one context so that count words left by a frame would show, against the general
path and the oracle."""
import numpy as np
import pytest

from edxraster_amd import configs, Renderer
from test_direct_frame import frame, oracle_frame, same, triangles

pytestmark = pytest.mark.gpu

SIZES = [(512, 1024), (27 * 32 - 5, 19 * 32 - 20), (33, 17), (40, 16), (70, 15), (64, 33), (100, 49), (320, 1)]


def mixed(width, height):
    """Triangles of 2, 12, 40 and 400 pixels or so."""
    rng = np.random.default_rng(width)
    v = []
    for size, n in ((2, 40), (12, 30), (40, 12), (400, 3)):
        c = rng.uniform(-1.5, 1.5, (n, 1, 3)) * [1.0, 1.0, 0.2]
        corner = np.array([[-1.0, -1.0, 0.0], [1.0, -1.0, 0.0], [0.0, 1.0, 0.0]]) * 1.7 * size / max(height, 60)
        v.append(c + corner + rng.uniform(-0.01, 0.01, (n, 3, 3)))
    return triangles(np.concatenate(v), width, height)


@pytest.mark.parametrize("hierarchical", [True, False])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "%dx%d" % s)
def test_frames(built, size, hierarchical):
    scenes = [mixed(*size), configs.small_sphere(*size, 20, 10)]
    scenes.append(scenes[0])
    r = Renderer(*size)
    r.set_hierarchical_rasterize(hierarchical)
    for w in scenes:
        w.apply(r)
        r.render_mesh(w.mesh)
        got = frame(r)
        r.set_bin_chunks(1)  # the general path
        r.render_mesh(w.mesh)
        assert same(got, frame(r))
        r.set_bin_chunks(0)
        if hierarchical:
            assert same(got[:2], oracle_frame(w))
    r.close()
