"""The backward pass reads the mesh again: it gets the mesh of the forward pass
where the caller has let go of it (temporaries, copies of strided tensors) and its
memory would be taken by other tensors."""
import numpy as np
import pytest
import torch

from edxraster_amd import configs, diff, Renderer

pytestmark = pytest.mark.gpu


def gradients(form, spoil):
    mesh, views = configs.diff_scene(2, 96, hf_n=12, sphere_segments=(12, 8))
    idx, planes = diff.mesh_tensors(mesh)
    leaves = [t.requires_grad_() for t in planes]
    light = torch.tensor([1.0, 1.0, -1.0], requires_grad=True)
    material = torch.tensor([0.2, 3.0, 3.0, 32.0], requires_grad=True)
    r = Renderer(64, 64)
    img = diff.render_views(r, views, form(idx), *[form(t) for t in leaves], light, material)
    others = [torch.full_like(t, 0.25) for t in planes * 4 for _ in range(4)] if spoil else []
    others += [torch.zeros_like(idx) for _ in range(8 if spoil else 0)]  # (indices in range)
    img.square().sum().backward()
    del others
    r.close()
    return [t.grad.cpu().numpy() for t in leaves + [light, material]]


FORMS = {
    "temporaries": lambda t: t * 1,
    "strided": lambda t: torch.stack([t, t], 1)[:, 0],
}


@pytest.mark.parametrize("name", list(FORMS))
def test_mesh_outlives_the_forward_pass(built, name):
    want = gradients(lambda t: t, False)
    got = gradients(FORMS[name], True)
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)
