"""What the adjoint decides by an exact value: a triangle whose vertices coincide
has no area and contributes nothing (clipped, it can cover pixels), and light in
the plane of the surface is not above it."""
import numpy as np
import pytest
import torch

from edxraster_amd import configs, diff, Mesh, Renderer
from edxraster_amd import _lib as L

pytestmark = pytest.mark.gpu


def gradients(mesh, view, light, shader):
    """(gradients of planes, light and material, covered pixels) of the summed image."""
    idx, planes = diff.mesh_tensors(mesh)
    inputs = [t.requires_grad_() for t in planes]
    inputs += [torch.tensor(light, requires_grad=True), torch.tensor([0.2, 3.0, 3.0, 32.0], requires_grad=True)]
    r = Renderer(64, 64)
    img = diff.render_views(r, [view], idx, *inputs, shader=shader)
    img.sum().backward()
    ids = r.batch_read(0)[2]
    r.close()
    return [t.grad.cpu().numpy() for t in inputs], int((ids != 0xFFFFFFFF).sum())


@pytest.mark.parametrize("shader", [L.SHADER_LAMBERT_ALBEDO, L.SHADER_BLINN_PHONG_REF, L.SHADER_VC_BLINN_PHONG])
def test_coincident_vertices(built, shader):
    rng = np.random.default_rng(1)
    n = 200000
    a = rng.uniform(-1.2, 1.2, (n, 3))
    v = np.stack([a, a, a + rng.normal(0.0, 3.0, (n, 3))], 1)
    v = np.concatenate([np.roll(v, k, 1)[:, ::s] for k in range(3) for s in (1, -1)]).reshape(-1, 3).astype(np.float32)
    c = rng.uniform(0.1, 0.9, (3, len(v))).astype(np.float32)
    nn = rng.normal(0.0, 1.0, (3, len(v))).astype(np.float32)
    mesh = Mesh(*v.T.copy(), *nn, *c, np.arange(len(v), dtype=np.uint32))
    view = configs.Workload("slivers", 400, 300, mesh, *configs.camera(400, 300, (0.0, 0.0, -3.0), (0.0, 0.0, 0.0)))
    grads, covered = gradients(mesh, view, (1.0, 1.0, -1.0), shader)
    assert covered >= 10
    for g in grads:
        assert not g.any()


def test_light_in_the_surface(built):
    mesh = Mesh.load_heightfield(20, 0.2, height_seed=3, color_seed=4)
    mesh.nx[:], mesh.ny[:], mesh.nz[:] = 0.7, -0.7, 0.0
    view = configs.Workload("plane", 150, 100, mesh, *configs.camera(150, 100, (0.0, 1.2, -1.6), (0.0, 0.0, 0.0)))
    grads, covered = gradients(mesh, view, (1.0, 1.0, 0.0), L.SHADER_LAMBERT_ALBEDO)
    assert covered > 3000
    for g in grads[3:6] + grads[9:10]:  # normals, light
        assert not g.any()
    assert grads[10][0] > 0.0  # the ambient term alone
