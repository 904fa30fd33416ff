"""Triangles far longer than the frame: a raster matrix that shows a crop of a
large picture, unclipped triangles of up to 600,000 pixels whose tiles in the
frame are at most 2x2 (no corner tests) or more, with edges through pixel and
sample centres, against the oracle on the direct and the general path, in a
batch, in the allocation-free frame and with 4 samples; and their bin lists."""
import numpy as np
import pytest

from edxraster_amd import configs, Mesh, Renderer
from edxraster_amd import _lib as L
from test_direct_frame import frame, oracle_frame, same

pytestmark = pytest.mark.gpu

SCALE = 2.0 ** 20  # pixels per unit of clip space: sixteenths of a pixel up to 2^24 are exact


def crop(tris, width, height):
    """The triangles (N, 3, 2), corners in pixels of the picture, in both windings (one is culled)."""
    v = np.asarray(tris, np.float64)
    v = np.concatenate([v, v[:, ::-1]], 1).reshape(-1, 3, 2)
    z = np.repeat(np.random.default_rng(3).uniform(0.2, 0.8, len(v) // 2), 6).astype(np.float32)
    v = v.reshape(-1, 2)
    x, y = (v / SCALE).astype(np.float32).T
    assert np.array_equal(np.stack([x, y], 1).astype(np.float64) * SCALE, v) and np.abs(v).max() < SCALE
    c = np.random.default_rng(4).uniform(0, 1, (3, len(v))).astype(np.float32)
    one, zero = np.ones(len(v), np.float32), np.zeros(len(v), np.float32)
    mesh = Mesh(x, y, z, zero, zero, -one, *c, np.arange(len(v), dtype=np.uint32))
    eye = np.eye(4, dtype=np.float32)
    raster = np.diag([SCALE, SCALE, 1.0, 1.0]).astype(np.float32)
    return configs.Workload("crop", width, height, mesh, eye, eye, raster)


def strips(length, width, height, kind):
    """Adjoining quadrilaterals of two triangles each across the frame, their long sides through
    pixel centres and the centres of 4 samples."""
    span = width + height
    at = np.cumsum([0.5, 3.0, 2.875, 4.375, 3.25] * (span // 6))
    at = at[at < span]
    if kind == "diagonal":  # (every other one: their boxes all cover the same tiles, at most 48 for the direct path)
        at = at[::2] - height
    tris = []
    for a, b in zip(at[:-1], at[1:]):
        p, q, r, s = (a, -length), (b, -length + 0.5), (a, length), (b, length + 1.0)
        tris += [(p, q, r), (q, s, r)]
    v = np.array(tris)
    if kind == "horizontal":
        v = v[..., ::-1]
    elif kind == "diagonal":
        v[..., 0] = v[..., 0] + v[..., 1]
    return v


def fan(length, width, height, kind):
    """Triangles around a pixel centre of the frame, some of their sides one sixteenth off an axis."""
    c = np.array([width // 2 + 0.5, height // 2 + 0.5])
    e, m = 1.0 / 16.0, length
    far = [(m, 0), (m, e), (m, m / 2), (m / 2, m), (e, m), (0, m), (-e, m), (-m, m / 2), (-m, e), (-m, 0), (-m, -e),
           (-m, -m / 2), (-e, -m), (0, -m), (e, -m), (m, -m / 2), (m, -e)]
    return np.array([(c, c + a, c + b) for a, b in zip(far, far[1:] + far[:1])])


SHAPES = {"vertical": strips, "horizontal": strips, "diagonal": strips, "fan": fan}
LENGTHS = [500, 1040, 2100, 3000, 5000, 100000, 600000]


def check_bins(r, o):
    for a, b in zip(r.debug_bins(), o.bins()):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("size", [(64, 64), (20, 40), (150, 100)])
@pytest.mark.parametrize("length", LENGTHS)
@pytest.mark.parametrize("kind", list(SHAPES))
def test_against_the_oracle(built, kind, length, size):
    from oracle.oracle import Oracle
    from test_zz_no_alloc import device_mesh, noalloc_frame
    # (sheared corners stay within the picture)
    w = crop(SHAPES[kind](min(length, 400000) if kind == "diagonal" else length, *size, kind), *size)
    o = Oracle()
    o.render_workload(w, threads=1)
    want = o.ids(), o.depth().view(np.uint32)
    assert (want[0] != 0xFFFFFFFF).any()
    r = Renderer(*size)
    w.apply(r)
    got = []
    for chunks in (0, 2):  # direct, general
        r.set_bin_chunks(chunks)
        r.render_mesh(w.mesh)
        got.append(frame(r))
        assert same(got[-1][:2], want), "chunks %d" % chunks
        check_bins(r, o)
    assert same(*got)
    for capacity in (0, 8):  # direct, general
        assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, capacity) == 0
        r.render_batch([configs.small_sphere(40, 40, 8, 4).job(), w.job()])
        rgba, depth, ids = r.batch_read(1)
        assert same((ids, depth.view(np.uint32), rgba), got[0]), "batch, capacity %d" % capacity
    assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 0) == 0
    dm, keep = device_mesh(w.mesh)
    for chunks in (0, 2):
        r.set_bin_chunks(chunks)
        ids, depth, rgba = noalloc_frame(r, w, dm)
        assert same((ids, depth.view(np.uint32), rgba), got[0]), "allocation-free, chunks %d" % chunks
    r.close()


@pytest.mark.parametrize("length", LENGTHS)
@pytest.mark.parametrize("kind", list(SHAPES))
def test_samples_against_the_oracle(built, kind, length):
    from test_msaa import assert_ms_parity, render_ms
    w = crop(SHAPES[kind](min(length, 400000) if kind == "diagonal" else length, 64, 64, kind), 64, 64)
    r, o = render_ms(w, 2)
    assert_ms_parity(r, o, "%s %d" % (kind, length))
    r.close()
