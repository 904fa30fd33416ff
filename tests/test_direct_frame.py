"""Direct frames (small frames and batches in three launches, a fixed list per
tile) against the general path over the forms they accept, bit for bit, and
against the oracle at the limits that send a frame to the general path: a
tile's references (4,096; 2,048 in the allocation-free frame and beyond 8,192
tiles) and tile-level triangles (48), 416 triangle slots per tile, 32,768
tiles.  The general path is taken with a chunk count set by the caller (single
frames) or with the capacity testing aid (batches)."""
import numpy as np
import pytest

from edxraster_amd import configs, EdxrError, Mesh, Renderer
from edxraster_amd import _lib as L

pytestmark = pytest.mark.gpu

STATS = ("triangles_in", "trivially_rejected", "clipped", "near_clipped", "setup_records", "refs", "clip_vertices")


def frame(r):
    return r.read_triangle_ids(), r.read_depth().view(np.uint32), r.get_back_buffer()


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def stats(r):
    st = r.stats()
    assert st["retries"] == 0
    return [st[k] for k in STATS]


def oracle_frame(w):
    from oracle.oracle import Oracle
    o = Oracle()
    o.render_workload(w)
    return o.ids(), o.depth().view(np.uint32)


def triangles(v, width=96, height=96):
    """A workload of the given triangles (N, 3, 3) in front of an eye at (0, 0, -3), vertex colours seeded."""
    mv, p, r = configs.camera(width, height, (0.0, 0.0, -3.0), (0.0, 0.0, 0.0))
    v = configs._front_facing(np.array(v, np.float64), np.asarray(p, np.float64) @ np.asarray(mv, np.float64))
    v = v.reshape(-1, 3).astype(np.float32)
    c = np.random.default_rng(1).uniform(0, 1, v.shape).astype(np.float32)
    one, zero = np.ones(len(v), np.float32), np.zeros(len(v), np.float32)
    mesh = Mesh(v[:, 0], v[:, 1], v[:, 2], zero, zero, -one, c[:, 0], c[:, 1], c[:, 2], np.arange(len(v), dtype=np.uint32))
    return configs.Workload("triangles", width, height, mesh, mv, p, r)


def small_in_one_tile(n):
    rng = np.random.default_rng(n)
    c = np.stack([rng.uniform(-0.1, 0.1, n), rng.uniform(-0.1, 0.1, n), rng.uniform(-0.5, 0.5, n)], 1)
    return triangles(c[:, None, :] + rng.normal(0.0, 0.02, (n, 3, 3)) * [1, 1, 0])


def large(n):
    rng = np.random.default_rng(n)
    corner = np.array([[-1.4, -1.4, 0.0], [1.4, -1.4, 0.0], [0.0, 1.4, 0.0]])
    return triangles(corner[None] + rng.uniform(-0.1, 0.1, (n, 3, 3)))


SCENES = {
    "sphere": lambda: configs.small_sphere(333, 217, 40, 20),
    "clipped": lambda: configs.sphere_grid_1080p(640, 360, grid=3, segments=20),
    "clip_all": lambda: configs.clip_scene("all"),
    "one_pixel": lambda: configs.heightfield_small(9, 1, 1),
    "textured": lambda: configs.textured_scene(320, 200, 40),
    "reference_shader": lambda: _shader(configs.heightfield_small(60, 200, 150), 1, 200.0),
    "lambert": lambda: _shader(configs.heightfield_small(60, 2047, 2048), 0, 0.0),
    "below_slots": lambda: configs.small_sphere(96, 32, 39, 16),     # 1,248 triangles on 3 tiles: 416 a tile
    "above_slots": lambda: configs.small_sphere(96, 32, 40, 16),
    "tile_4095": lambda: small_in_one_tile(4095), "tile_4096": lambda: small_in_one_tile(4096),
    "tile_4097": lambda: small_in_one_tile(4097),
    "large_47": lambda: large(47), "large_48": lambda: large(48), "large_49": lambda: large(49),
}


def _shader(w, kind, shininess):
    w.shader, w.shininess = kind, shininess
    return w


@pytest.mark.parametrize("hierarchical", [1, 0])
@pytest.mark.parametrize("name", list(SCENES))
def test_equals_general_path_and_oracle(built, name, hierarchical):
    w = SCENES[name]()
    r = Renderer(w.width, w.height)
    w.apply(r)
    r.set_hierarchical_rasterize(hierarchical)
    got = []
    for chunks in (0, 3, 0, 0):
        r.set_bin_chunks(chunks)
        r.render_mesh(w.mesh)
        offs, refs = r.debug_bins()
        got.append((frame(r), stats(r), (offs, refs)))
    for f, st, bins in got[1:]:
        assert same(f, got[0][0]) and st == got[0][1] and same(bins, got[0][2])
    r.close()
    if hierarchical:
        assert same(got[0][0][:2], oracle_frame(w))


def test_sequence_of_frames_and_states(built):
    """The lists' counts are clear for every frame, whatever came before it: a
    frame sent to the general path, a bad index, forced capacities, graph mode,
    an allocation-free frame, a batch."""
    from test_zz_no_alloc import device_mesh, noalloc_frame
    r = Renderer(96, 96)
    a, b = large(20), small_in_one_tile(4500)
    want = {}
    for key, w in (("a", a), ("b", b)):
        w.apply(r)
        r.set_bin_chunks(2)
        r.render_mesh(w.mesh)
        want[key] = frame(r)
    r.set_bin_chunks(0)
    bad = Mesh(*a.mesh.planes(), np.array([0, 1, 999999], np.uint32))
    for step in ("a", "b", "a", "bad", "a", "graph", "a", "b", "a", "capacity", "a", "noalloc", "a", "batch", "a"):
        if step == "bad":
            with pytest.raises(EdxrError):
                r.render_mesh(bad)
        elif step == "graph":
            r.set_graph(True)
        elif step == "capacity":
            assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 4) == 0
            r.render_mesh(a.mesh)
            assert r.stats()["retries"] > 0 and same(frame(r), want["a"])
            assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 0) == 0
        elif step == "noalloc":
            dm, keep = device_mesh(a.mesh)
            ids, depth, rgba = noalloc_frame(r, a, dm)
            assert same((ids, depth.view(np.uint32), rgba), want["a"])
        elif step == "batch":
            r.render_batch([b.job(), a.job()])
            rgba, depth, ids = r.batch_read(1)
            assert same((ids, depth.view(np.uint32), rgba), want["a"])
        else:
            w = a if step == "a" else b
            for _ in range(3):
                r.render_mesh(w.mesh)
                assert same(frame(r), want[step]), step
    r.close()


@pytest.mark.parametrize("n", [2047, 2048, 2049])
def test_noalloc_list_limit(built, n):
    from test_zz_no_alloc import device_mesh, noalloc_frame
    w = small_in_one_tile(n)
    r = Renderer(w.width, w.height)
    w.apply(r)
    dm, keep = device_mesh(w.mesh)
    r.set_bin_chunks(2)
    r.render_mesh(w.mesh)
    want = frame(r)
    r.set_bin_chunks(0)
    for _ in range(2):
        ids, depth, rgba = noalloc_frame(r, w, dm)
        assert same((ids, depth.view(np.uint32), rgba), want)
    r.close()


@pytest.mark.parametrize("size", [(8192, 1024), (8192, 1025), (8192, 2048)],
                         ids=["8192_tiles", "8448_tiles", "16384_tiles"])
def test_tile_limits(built, size):
    w = configs.heightfield_small(64, size[0], size[1])
    r = Renderer(w.width, w.height)
    w.apply(r)
    got = []
    for chunks in (0, 4):
        r.set_bin_chunks(chunks)
        r.render_mesh(w.mesh)
        got.append(frame(r) + tuple(r.debug_bins()))
    assert same(*got)
    r.close()


@pytest.mark.parametrize("extra", [0, 1], ids=["32768_tiles", "32769_tiles"])
def test_batch_tile_limit(built, extra):
    jobs = [configs.heightfield_small(40, 4096, 2048, seed=k) for k in range(4)]
    jobs += [configs.small_sphere(32, 32, 8, 4)] * extra
    r = Renderer(64, 64)
    r.render_batch([w.job() for w in jobs])
    got = [r.batch_read(k) for k in range(len(jobs))]
    for w, (rgba, depth, ids) in zip(jobs, got):
        s = Renderer(w.width, w.height)
        w.apply(s)
        s.set_bin_chunks(4)
        s.render_mesh(w.mesh)
        assert same((ids, depth.view(np.uint32), rgba), frame(s))
        s.close()
    r.close()


@pytest.mark.parametrize("n,tmax", [(2, 300), (9, 3000), (70, 400)])
def test_batch_equals_general_path(built, n, tmax):
    jobs = configs.batch_jobs(n, seed_base=50, tmin=100, tmax=tmax, resolutions=(33, 96, 200))
    jobs.insert(1, configs.clip_scene("lateral"))
    empty = configs.small_sphere(64, 48)
    empty.mesh.indices = empty.mesh.indices[:0]
    jobs.insert(0, empty)
    out = []
    for capacity in (0, 8):
        r = Renderer(64, 64)
        assert L.lib().edxr_set_state(r.ctx, L.STATE_FLOAT_COLOR, 1) == 0
        assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, capacity) == 0
        arr = [w.job() for w in jobs]
        for _ in range(2):
            r.render_batch(arr)
            rgb = np.empty(3 * sum(w.width * w.height for w in jobs), np.float32)
            assert L.lib().edxr_copy_float_color(r.ctx, rgb.ctypes.data, rgb.nbytes) == 0
            out.append([rgb] + [x for k in range(len(jobs)) for x in r.batch_read(k)])
        r.close()
    for o in out[1:]:
        assert all(np.array_equal(x.view(np.uint8), y.view(np.uint8)) for x, y in zip(o, out[0]))
