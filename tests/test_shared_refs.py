"""Multisampled tiles of few references that take a whole wave, which two or four
of a work item's eight waves share (one or two references: four, three or four:
two): tile-level triangles by quadrants, others by rows of quads, against the
oracle, in whole and partial tiles."""
import numpy as np
import pytest

from test_direct_frame import triangles
from test_msaa import assert_ms_parity, render_ms

pytestmark = pytest.mark.gpu


def tile_level(n, width, height):
    """Triangles that cover the frame or most of it."""
    rng = np.random.default_rng(n)
    corner = np.array([[-1.6, -1.4, 0.0], [1.6, -1.4, 0.0], [0.0, 1.5, 0.0]])
    return triangles(corner[None] + rng.uniform(-0.4, 0.4, (n, 3, 3)), width, height)


def quad_walked(n, width, height):
    """Triangles of about 30 pixels each way, within 2x2 tiles."""
    rng = np.random.default_rng(10 + n)
    s = 15.0 / max(width, height) * 3.4
    corner = s * np.array([[-1.0, -1.0, 0.0], [1.0, -1.0, 0.0], [0.0, 1.0, 0.0]])
    c = np.concatenate([rng.uniform(-0.2, 0.2, (n, 2)), rng.uniform(-0.3, 0.3, (n, 1))], 1)
    return triangles(c[:, None, :] + corner[None] + rng.uniform(-0.2 * s, 0.2 * s, (n, 3, 3)), width, height)


@pytest.mark.parametrize("hierarchical", [True, False])
@pytest.mark.parametrize("level", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("make", [tile_level, quad_walked])
def test_against_the_oracle(built, make, n, level, hierarchical):
    for width, height in ((96, 96), (49, 40)):
        w = make(n, width, height)
        r, o = render_ms(w, level, hierarchical)
        assert (o.ids() != 0xFFFFFFFF).any()
        assert_ms_parity(r, o, "%s %d, %dx%d" % (make.__name__, n, width, height))
        r.close()
