"""Which settings autotuning leaves behind: those it found for jobs of the general
path (more than 416 triangles per tile), the context's own for direct ones."""
import pytest

from edxraster_amd import configs, Renderer
from edxraster_amd import _lib as L
from test_direct_frame import same
from test_graph_replays import deep

pytestmark = pytest.mark.gpu


def chunks_of(r, jobs):
    """Chunks of a batch that takes the general path (the capacity testing aid)."""
    assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 8) == 0
    r.render_batch(jobs)
    assert L.lib().edxr_set_state(r.ctx, L.STATE_DEBUG_CAPACITY, 0) == 0
    return r.stats()["bin_chunks"]


def test_autotune_of_direct_jobs_keeps_the_settings(built):
    scenes = [configs.small_sphere(100, 70, 20, 10), configs.heightfield_small(20, 64, 64)]  # (keep the meshes)
    small = [s.job() for s in scenes]
    w = configs.heightfield_small(80, 128, 128)  # 12,482 triangles
    big = [w.job(), w.job()]
    T = w.mesh.num_triangles
    for tris, blocks in ((0, 0), (300, 5)):
        r = Renderer(64, 64)
        r.set_tuning(tris, blocks)
        t = r.autotune(small)
        assert (t["tris_per_chunk"], t["raster_blocks_per_cu"]) == (tris or 1024, blocks or 8) and t["frame_ms"] > 0
        assert chunks_of(r, big) == 2 * -(-T // (tris or 1024))
        r.close()


def test_autotune_of_general_jobs(built):
    scenes = [deep(80), deep(100, 70, 50)]
    jobs = [w.job() for w in scenes]
    r = Renderer(64, 64)
    r.render_batch(jobs)
    before = [r.batch_read(k) for k in range(2)]
    r.set_graph(True)
    t = r.autotune(jobs)
    assert t["tris_per_chunk"] in (512, 1024, 2048, 4096) and t["raster_blocks_per_cu"] in (4, 8, 16)
    for _ in range(3):
        r.render_batch(jobs)
        assert r.stats()["bin_chunks"] == sum(-(-j.mesh.num_triangles // t["tris_per_chunk"]) for j in jobs)
        assert all(same(before[k], r.batch_read(k)) for k in range(2))
    r.close()
