"""Texture addressing at its edges: coordinates below 0 and far beyond 1,
sides of a power of two and not, of one texel, magnified (one mip level) and
minified, with every filter, against the oracle (colour within 1 LSB, as for
the other textured frames: log2f may differ by an ulp)."""
import numpy as np
import pytest

from edxraster_amd import configs
from test_textures import render_gpu_and_oracle
from test_gpu_parity import assert_frame_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0.02, 9.7], ids=["magnified", "minified"])
@pytest.mark.parametrize("tex_filter", range(6))
def test_sizes_and_coordinates(built, tex_filter, scale):
    w = configs.textured_scene(320, 240, n=40, tex_filter=tex_filter)
    m = w.mesh
    m.tu = (m.px * np.float32(scale) - np.float32(2.3)).astype(np.float32)
    m.tv = (m.pz * np.float32(scale) - np.float32(0.1)).astype(np.float32)
    sizes = [(1, 1), (3, 5), (64, 1), (1, 7), (128, 32), (100, 60)]
    m.tex_ids = (np.arange(m.num_triangles) % len(sizes)).astype(np.uint32)
    full = configs.checker_texture(128, 16, 5)
    w.textures = [np.ascontiguousarray(full[:h, :x]) for x, h in sizes]
    r, o = render_gpu_and_oracle(w)
    assert_frame_parity(r, o, "filter %d" % tex_filter)
    r.close()
