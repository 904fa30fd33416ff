"""The adjoint kernel's per-tile tables at their limits, against the FP64
reference gradient (tests/adjoint_ref.py): tiles with more vertices than the
table of sums holds, with one large triangle, partial tiles at the image's
edges, few tiles (shared by several workgroups) and many, more jobs than a
wave, and a shininess that is no whole exponent.

Tolerance 1e-5 relative L2 per gradient: everything after the float32 inputs
is computed in double and rounded once, and what differs from the reference
by float32 rounding (the eye position, 6e-8) reaches a position's gradient
through sums that cancel by one to two decimal digits.
"""
import numpy as np
import pytest
import torch

from edxraster_amd import Mesh, configs
from tests import adjoint_ref as R

pytestmark = pytest.mark.gpu


def sphere_views(n_views, res, slices, stacks, light):
    """A unit sphere, the light from the camera's side (no negative N.H)."""
    mesh = Mesh.sphere(slices, stacks, 1.0, (0.0, 0.0, 0.0), color_seed=4)
    views = []
    for k in range(n_views):
        a = 0.02 * k
        mv, p, r = configs.camera(res[0], res[1], (-3.0 * np.sin(a), 0.1, -3.0 * np.cos(a)), (0.0, 0.0, 0.0))
        views.append(configs.Workload("v%d" % k, res[0], res[1], mesh, mv, p, r, light=light))
    return mesh, views


@pytest.mark.parametrize("n_views,res,seg,shininess", [
    (1, (33, 31), (160, 80), 32.0),     # most triangles under a pixel: the table of sums overflows
    (1, (97, 65), (4, 2), 32.0),        # a few triangles over many tiles
    (1, (1000, 900), (24, 12), 32.0),   # beyond 768 tiles: one workgroup per tile, partial last ones
    (1, (1000, 900), (300, 150), 20.5),
    (2, (70, 50), (40, 20), 20.5),      # pow
    (70, (32, 32), (16, 8), 7.0),       # more jobs than lanes
], ids=["dense", "large_triangles", "many_tiles", "many_tiles_pow", "pow", "70_jobs"])
def test_gradients_match_fp64(built, n_views, res, seg, shininess):
    from edxraster_amd import Renderer, diff
    light, material = (0.1, 0.2, -1.0), (0.2, 0.6, 0.3, shininess)
    mesh, views = sphere_views(n_views, res, seg[0], seg[1], light)
    g = np.random.default_rng(11).normal(size=(n_views, res[1], res[0], 3)).astype(np.float32)
    idx, planes = diff.mesh_tensors(mesh)
    for t in planes:
        t.requires_grad_(True)
    lt = torch.tensor(light, dtype=torch.float32, requires_grad=True)
    mt = torch.tensor(material, dtype=torch.float32, requires_grad=True)
    r = Renderer(64, 64)
    img = diff.render_views(r, views, idx, *planes, lt, mt)
    (img * torch.from_numpy(g).cuda()).sum().backward()
    ids = [r.batch_read(k)[2] for k in range(n_views)]
    r.close()
    th = R.theta_from(mesh, np.float32(light).astype(np.float64), np.float32(material).astype(np.float64))
    total = torch.zeros((), dtype=torch.float64)
    for v, i, gk in zip(views, ids, g):
        k = int(shininess) if shininess == int(shininess) else shininess
        col, (rows, xs) = R.image_fp64(th, mesh.indices, v, i, shininess_int=k)
        total = total + (col * torch.from_numpy(gk[rows, xs].astype(np.float64))).sum()
    total.backward()
    got = dict(zip(diff.PLANE_NAMES, planes), light=lt, material=mt)
    for name, t in got.items():
        a, b = t.grad.detach().cpu().double().numpy(), th[name].grad.numpy()
        err = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        assert err <= 1e-5, (name, err)
