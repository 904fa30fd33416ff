"""The tile scan at the edges of its variants (one workgroup with 1, 2 or 4
tiles per thread, then workgroups of 1,024 tiles in two launches): frames of
1,024 to 4,097 tiles against the oracle (IDs and depth bit-exact), with tiles
of mostly tile-level triangles (finer segments) and of many small ones, also
with the capacities that force a re-run on the three-kernel column scan, and
the allocation-free frame against the plain one."""
import ctypes as C

import numpy as np
import pytest

from edxraster_amd import configs, Renderer
from edxraster_amd import _lib as L
from test_zz_no_alloc import device_mesh, noalloc_frame, plain_frame, assert_equal_frames

pytestmark = pytest.mark.gpu

SIZES = [(1024, 1024), (41 * 32, 25 * 32 - 5), (64 * 32 - 1, 1024), (50 * 32, 41 * 32), (2048, 2048 - 7),
         (241 * 32 - 3, 17 * 32)]  # 1024, 1025, 2048, 2050, 4096, 4097 tiles
IDS = ["%dx%d" % s for s in SIZES]


def scene(size, kind):
    if kind == "large":  # a few triangles over many tiles each, some clipped
        return configs.sphere_grid_1080p(size[0], size[1], grid=2, segments=8)
    return configs.heightfield_small(150, size[0], size[1], seed=5)


def check(r, o):
    assert np.array_equal(r.read_triangle_ids(), o.ids())
    assert np.array_equal(r.read_depth().view(np.uint32), o.depth().view(np.uint32))


@pytest.mark.parametrize("kind", ["large", "small"])
@pytest.mark.parametrize("size", SIZES, ids=IDS)
def test_frame_matches_oracle(built, size, kind):
    from oracle.oracle import Oracle
    w = scene(size, kind)
    o = Oracle()
    o.render_workload(w)
    r = Renderer(w.width, w.height)
    w.apply(r)
    r.render_mesh(w.mesh)
    check(r, o)
    assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 64) == 0
    r.render_mesh(w.mesh)
    assert r.stats()["retries"] > 0
    check(r, o)
    r.close()


@pytest.mark.parametrize("size", [SIZES[0], SIZES[5]], ids=[IDS[0], IDS[5]])
def test_noalloc_equals_plain_frame(built, size):
    w = scene(size, "large")
    r = Renderer(w.width, w.height)
    w.apply(r)
    dm, keep = device_mesh(w.mesh)
    got = noalloc_frame(r, w, dm)
    assert r.stats()["clipped"] > 0
    assert_equal_frames(got, plain_frame(r, w), "%dx%d" % size)
    r.close()


@pytest.mark.parametrize("size", [(2048, 2048), (65 * 32, 2048)], ids=["4096", "4160"])
def test_default_chunks_of_many_triangles(built, size):
    """2.2M triangles: the default number of binning chunks on either side of
    4,096 tiles, the frame as with every other number."""
    w = configs.heightfield_small(1050, size[0], size[1], seed=5)
    r = Renderer(w.width, w.height)
    w.apply(r)
    frames = []
    for chunks in (0, 4096, 700):
        r.set_bin_chunks(chunks)
        r.render_mesh(w.mesh)
        if chunks == 0:
            assert r.stats()["bin_chunks"] == (2048 if size[0] > 2048 else 2150)
        frames.append((r.get_back_buffer(), r.read_depth().view(np.uint32), r.read_triangle_ids()))
    for f in frames[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(f, frames[0]))
    r.close()
