"""Jobs of differentiable views, copied from a template: byte for byte those of
Renderer.make_job for every form of matrix that it takes, and what it refuses is
refused; the forms of light and material tensors; and what may be done with the
gradients."""
import numpy as np
import pytest
import torch

from edxraster_amd import configs, diff, Renderer
from edxraster_amd import _lib as L


def views(forms):
    out = []
    for k, form in enumerate(forms):
        v = configs.Workload("view", 40 + k, 30 + 2 * k, None, *configs.camera(40, 30, (0.1 * k, 1.0, -2.0), (0.0, 0.0, 0.0)))
        for name in ("mv", "proj", "raster"):
            setattr(v, name, form(np.asarray(getattr(v, name), np.float32)))
        out.append(v)
    return out


FORMS = {
    "matrix": lambda m: m.reshape(4, 4), "flat": lambda m: m.reshape(16), "list": lambda m: m.reshape(4, 4).tolist(),
    "double": lambda m: m.reshape(4, 4).astype(np.float64) * (1 + 1e-9), "transposed": lambda m: m.reshape(4, 4).T,
    "row": lambda m: m.reshape(1, 16), "tensor": lambda m: torch.from_numpy(m.reshape(4, 4).copy()),
}


LIGHT = (0.3, 1.0, -0.2)


def material():
    mat = L.Material()
    mat.ambient, mat.kd, mat.ks, mat.shininess = 0.2, 3.0, 1.0, 32.0
    return mat


@pytest.mark.parametrize("names", [[n] * 3 for n in FORMS] + [list(FORMS)], ids=lambda n: "-".join(sorted(set(n))))
def test_equal_make_job(built, names):
    vs, mesh, mat = views([FORMS[n] for n in names]), L.Mesh(), material()
    got = diff._view_jobs(mesh, vs, LIGHT, L.SHADER_VC_BLINN_PHONG, mat)
    assert len(got) == len(vs)
    for a, v in zip(got, vs):
        b = Renderer.make_job(mesh, v.width, v.height, v.mv, v.proj, v.raster, LIGHT, L.SHADER_VC_BLINN_PHONG, mat)
        assert bytes(a) == bytes(b)


@pytest.mark.parametrize("name", ["mv", "proj", "raster"])
@pytest.mark.parametrize("sizes", [(16, 15, 17), (16, 17, 15), (16, 16, 15), (12, 16, 20), (16, 0, 32)])
def test_matrices_of_other_sizes_are_refused(built, name, sizes):
    vs = views([FORMS["flat"]] * 3)
    for v, n in zip(vs, sizes):
        setattr(v, name, np.resize(getattr(v, name), n))
    with pytest.raises(ValueError):
        diff._view_jobs(L.Mesh(), vs, LIGHT, L.SHADER_VC_BLINN_PHONG, material())


@pytest.mark.parametrize("shape", [(3,), (3, 1), (3, 1, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.int32])
def test_light_and_material_forms(shape, dtype):
    t = torch.tensor([1.0, -2.0, 3.0]).to(dtype).reshape(shape).requires_grad_(dtype.is_floating_point)
    assert diff._floats(t) == [1.0, -2.0, 3.0]


@pytest.mark.parametrize("shape", [(), (1, 3), (3, 2)])
def test_other_forms_are_refused(shape):
    with pytest.raises((TypeError, ValueError, RuntimeError)):
        diff._floats(torch.ones(shape))


class _Gradients(torch.autograd.Function):
    @staticmethod
    def forward(ctx, *inputs):
        return sum(t.sum() for t in inputs)

    @staticmethod
    def backward(ctx, g):
        return tuple(diff._split_grads(torch.arange(9 * 5 + 7.0), 5, "cpu"))


@pytest.mark.parametrize("k,create_graph", [(0, True), (8, True), (9, False), (9, True), (10, False), (10, True)])
def test_gradients_change_in_place(k, create_graph):
    """With a graph of the gradients any of them, without one the light's and the
    material's (planes are then views made without one), take values that have a
    gradient themselves."""
    inputs = [torch.zeros(n, requires_grad=True) for n in [5] * 9 + [3, 4]]
    grads = torch.autograd.grad(_Gradients.apply(*inputs), inputs, create_graph=create_graph)
    assert torch.equal(torch.cat(grads), torch.arange(9 * 5 + 7.0))
    grads[k].add_(inputs[0].sum())
    assert grads[k].requires_grad
