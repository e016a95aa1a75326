"""One-lane density work-groups stage the halos of quads of cells where all of
theirs fit, otherwise of single cells, and walk the rest from HBM (k_density,
csrc/sph.hip; states of more than 180,224 particles). Sums and lists keep one
order, so a scene gives the same bits there, with any work-group size, as by
sixteen lanes per particle in a state of its own."""
import numpy as np
import pytest

from libclsph_amd import native, scenes
from test_gpu_density_paths import CASES, FIELDS, beside, cloud, ctx  # noqa: F401

pytestmark = pytest.mark.gpu

ONE_LANE = 180225  # particles of a dam break beside the scene

# besides the stages' cases: densities at which all quads of a work-group fit,
# some do, none does, and cells don't either
MORE = {
    "thin": lambda: cloud(3000, 11, 0.1, 0.9),
    "rest": lambda: cloud(8192, 12, 0.3, 0.7),
    "dense2": lambda: cloud(9000, 13, 0.4, 0.66),
    "dense4": lambda: cloud(9000, 14, 0.4, 0.6),
    "dense9": lambda: cloud(9001, 15, 0.4, 0.55),
}


@pytest.fixture(scope="module")
def filler():
    return scenes.dam_break(ONE_LANE, seed=3)


@pytest.mark.parametrize("size", [64, 128, 256, 512])
@pytest.mark.parametrize("name", list(CASES) + list(MORE))
def test_units_agree_bit_for_bit(ctx, filler, name, size):  # noqa: F811
    sc = (CASES | MORE)[name]()
    alone = beside(ctx, sc, 0)
    b = native.Batch(ctx, [filler.n, sc.n])
    sizes = b.block_sizes()
    sizes[4] = size
    b.set_block_sizes(sizes)
    for i, s in enumerate((filler, sc)):
        b.set_scene_params(i, s.params, s.terms)
        b.mesh_scene(i, s.normals, s.vertices, s.indices)
        b.upload_scene(i, s.particles)
    b.step(1)
    got = b.download_scene(1)
    b.close()
    for f in FIELDS:
        assert np.array_equal(alone[f].view(np.uint32), got[f].view(np.uint32)), f
