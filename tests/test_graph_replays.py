"""Graph replays where frames take the general path (more than 416 triangles per
tile, or a chunk count set): each replay against the eager frame, with other
cameras, lights and meshes between."""
import numpy as np
import pytest

from edxraster_amd import configs, Mesh, Renderer
from test_direct_frame import frame, same

pytestmark = pytest.mark.gpu


def deep(slices=80, width=96, height=64):
    """A sphere of 80 x 40 x 2 triangles on 6 tiles."""
    w = configs.small_sphere(width, height, slices, 40)
    assert w.mesh.num_triangles > 416 * ((width + 31) // 32) * ((height + 31) // 32)
    return w


def turn(w, step, k=0):
    ang = 0.3 * step + 0.1 * k
    w.light = (float(np.cos(ang)), 1.0, float(np.sin(ang)))
    eye = 3.0 * np.array([np.cos(ang), 0.6, np.sin(ang)]) / np.sqrt(1.36)
    w.mv, w.proj, w.raster = configs.camera(w.width, w.height, eye, (0.0, 0.0, 0.0))


def pair(w, chunks):
    out = []
    for graph in (False, True):
        r = Renderer(w.width, w.height)
        r.set_graph(graph)
        r.set_bin_chunks(chunks)
        w.apply(r)
        out.append(r)
    return out


@pytest.mark.parametrize("chunks", [0, 3])
def test_replays_follow_the_camera(built, chunks):
    w = deep() if not chunks else configs.small_sphere(200, 136, 40, 20)
    eager, graph = pair(w, chunks)
    seen = []
    for step in range(5):
        turn(w, step)
        for r in (eager, graph):
            w.apply(r)
            r.render_mesh(w.mesh)
        seen.append(frame(graph))
        assert same(frame(eager), seen[-1]), "step %d" % step
    assert all(not same(a, b) for a, b in zip(seen, seen[1:]))
    eager.close()
    graph.close()


@pytest.mark.parametrize("chunks", [0, 3])
def test_replays_follow_the_mesh(built, chunks):
    import torch
    from test_zz_no_alloc import device_mesh
    w = deep() if not chunks else configs.small_sphere(200, 136, 40, 20)
    a = w.mesh
    b = Mesh(a.px + 0.35, a.py - 0.2, a.pz, a.nx, a.ny, a.nz, a.cb, a.cr, a.cg, a.indices)
    meshes = [device_mesh(m) for m in (a, b)]
    eager, graph = pair(w, chunks)
    seen = []
    for step in range(5):
        for r in (eager, graph):
            r.render_mesh(meshes[step % 2][0])
        seen.append(frame(graph))
        assert same(frame(eager), seen[-1]), "step %d" % step
    assert not same(seen[0], seen[1]) and same(seen[0], seen[2])
    eager.close()
    graph.close()
    torch.cuda.synchronize()


def test_batch_replays_follow_cameras_and_meshes(built):
    jobs = [deep(80), deep(100, 70, 50), deep(60, 64, 33), deep(90, 33, 96)]
    other = [Mesh(m.px + 0.2, m.py, m.pz - 0.1, m.nx, m.ny, m.nz, m.cg, m.cb, m.cr, m.indices)
             for m in (w.mesh for w in jobs)]
    first = [w.mesh for w in jobs]
    eager, graph = pair(jobs[0], 0)
    seen = []
    for step in range(5):
        for k, w in enumerate(jobs):
            turn(w, step // 2, k)
            w.mesh = (other if step % 2 else first)[k]
        arr = [w.job() for w in jobs]
        for r in (eager, graph):
            r.render_batch(arr)
        seen.append([graph.batch_read(k) for k in range(len(jobs))])
        for k in range(len(jobs)):
            assert same(eager.batch_read(k), seen[-1][k]), "job %d step %d" % (k, step)
    for k in range(len(jobs)):
        assert all(not same(x[k], y[k]) for x, y in zip(seen, seen[1:]))
    eager.close()
    graph.close()
