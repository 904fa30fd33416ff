"""Empty tiles, cleared four pixels at a time where every row of the picture
starts on 16 bytes and pixel by pixel elsewhere: batches of jobs of other sizes
(rows and first pixels on and off 16 bytes) after a batch that covered every
pixel, and frames into the caller's buffers at each offset to 16 bytes, on the
general and the direct path, with no triangle in sight too."""
import ctypes as C

import numpy as np
import pytest

from edxraster_amd import configs, Renderer
from edxraster_amd import _lib as L
from test_direct_frame import oracle_frame, same, triangles
from test_zz_no_alloc import device_mesh

pytestmark = pytest.mark.gpu

SIZES = [(64, 64), (61, 47), (100, 36), (33, 130), (34, 33), (256, 160), (96, 31), (1, 70), (200, 200)]


def read_batch(r, n):
    return [[a.view(np.uint32) if a.dtype == np.float32 else a for a in r.batch_read(k)] for k in range(n)]


@pytest.mark.parametrize("floats", [0, 1])
@pytest.mark.parametrize("dense", [0, 120])
def test_batch(built, dense, floats):
    """dense: stacks of the first job's sphere; with 120 of them the batch takes the general path."""
    full = np.array([[[-40.0, -40.0, 0.0], [40.0, -40.0, 0.0], [0.0, 60.0, 0.0]]])
    jobs = [configs.small_sphere(w, h, 12, 8) for w, h in SIZES]
    if dense:
        jobs[0] = configs.small_sphere(*SIZES[0], 2 * dense, dense)
    r = Renderer(64, 64)
    assert L.lib().edxr_set_state(r.ctx, L.STATE_FLOAT_COLOR, floats) == 0
    covered = [triangles(full, w, h) for w, h in SIZES]
    r.render_batch([w.job() for w in covered])
    assert all((ids == 0).all() for _, _, ids in read_batch(r, len(SIZES)))
    r.render_batch([w.job() for w in jobs])
    got = read_batch(r, len(jobs))
    for w, (rgba, depth, ids) in zip(jobs, got):
        assert same((ids, depth), oracle_frame(w)), (w.width, w.height)
        empty = ids == 0xFFFFFFFF
        assert (rgba[empty] == 0).all() and (rgba[~empty][:, 3] == 255).all()
    if floats:
        import torch
        out = torch.full((sum(w * h for w, h in SIZES), 3), -1.0).cuda()
        torch.cuda.synchronize()
        assert L.lib().edxr_copy_float_color(r.ctx, C.c_void_p(out.data_ptr()), out.numel() * 4) == 0
        want = np.concatenate([g[0].reshape(-1, 4)[:, :3] for g in got])
        assert np.array_equal((out.cpu().numpy() * np.float32(255.0) + np.float32(0.5)).astype(np.uint8), want)
    r.close()


@pytest.mark.parametrize("chunks", [0, 1])
@pytest.mark.parametrize("size", [(128, 96), (130, 96), (131, 70), (132, 33)], ids=lambda s: "%dx%d" % s)
def test_frame_into_any_buffers(built, size, chunks):
    import torch
    for seen in (True, False):
        w = configs.small_sphere(*size, 16, 8)
        if not seen:
            w.mv = configs.camera(*size, (0.0, 0.0, -3.0), (0.0, 0.0, -6.0))[0]
        want = oracle_frame(w)
        assert (want[0] != 0xFFFFFFFF).any() == seen
        r = Renderer(*size)
        w.apply(r)
        r.set_bin_chunks(chunks)
        dm, keep = device_mesh(w.mesh)
        n = size[0] * size[1]
        for off in ((0, 0, 0), (1, 0, 0), (0, 2, 0), (0, 0, 3)):
            bufs = [torch.full((n + 8,), 0x5A5A5A5A, dtype=torch.int32).cuda() for _ in off]
            torch.cuda.synchronize()
            ptr = [C.c_void_p(b.data_ptr() + 4 * (4 + k)) for b, k in zip(bufs, off)]
            assert L.lib().edxr_render_mesh_noalloc(r.ctx, C.byref(dm), *ptr) == 0
            host = [b.cpu().numpy().view(np.uint32) for b in bufs]
            color, depth, ids = (h[4 + k:4 + k + n].reshape(size[1], size[0]) for h, k in zip(host, off))
            for h, k in zip(host, off):  # and nothing beside the picture
                assert (h[:4 + k] == 0x5A5A5A5A).all() and (h[4 + k + n:] == 0x5A5A5A5A).all()
            assert same((ids, depth), want), (seen, off)
            assert (color[ids == 0xFFFFFFFF] == 0).all() and (color[ids != 0xFFFFFFFF] >> 24 == 255).all()
        r.close()
