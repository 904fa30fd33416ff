"""Textured frames of more than 8,192 tiles, which are shaded a tile at a time
(one job, anisotropic) or along the work list (other filters, batches): one job
against the same job in a batch, bit for bit, both on the general path."""
import numpy as np
import pytest

from edxraster_amd import configs, Renderer
from edxraster_amd import _lib as L
from test_direct_frame import frame, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tex_filter", [L.FILTER_TRILINEAR, L.FILTER_ANISO_4X, L.FILTER_ANISO_16X])
@pytest.mark.parametrize("size", [(8192, 1024), (8192, 1025)], ids=["8192_tiles", "8448_tiles"])
def test_one_job_equals_batch(built, size, tex_filter):
    w = configs.textured_scene(*size, n=40, tex_filter=tex_filter)
    r = Renderer(*size)
    w.apply(r)
    r.set_bin_chunks(4)
    r.render_mesh(w.mesh)
    one = frame(r)
    assert (one[0] != 0xFFFFFFFF).sum() > 100000
    assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 8) == 0
    r.render_batch([configs.small_sphere(40, 40, 8, 4).job(), w.job()])
    rgba, depth, ids = r.batch_read(1)
    assert same((ids, depth.view(np.uint32), rgba), one)
    r.close()
