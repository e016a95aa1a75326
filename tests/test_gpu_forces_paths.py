"""The forces stage takes 16 lanes or one per particle by the state's particle
count (launch_forces, csrc/sph.hip). Both add a particle's pair terms in list
order, so a scene's accelerations and what follows are the same bits in states
of every size; against the oracle they meet the stage's tolerance."""
import numpy as np
import pytest

import oracle
from libclsph_amd import native, scenes

pytestmark = pytest.mark.gpu

LANES_MAX = 57344
FIELDS = ("position", "velocity", "intermediate_velocity", "density", "pressure", "grid_index")


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def cloud(n, seed, lo, hi, dup=0, velocity=0.05):
    """n random particles in [lo, hi]^3 at h = 0.04, `dup` of them twice."""
    rng = np.random.default_rng(seed)
    sc = scenes.dam_break(max(n, 64), seed=seed)
    parts = sc.particles[:n].copy()
    parts["position"][:, :3] = rng.uniform(lo, hi, (n, 3)).astype(np.float32)
    v = rng.normal(0, velocity, (n, 3)).astype(np.float32)
    parts["velocity"][:, :3] = v
    parts["intermediate_velocity"][:, :3] = v
    if dup:
        parts[n - dup:] = parts[:dup]
    p = sc.params.copy()
    p["particles_count"] = n
    p["h"] = np.float32(0.04)
    p["max_velocity"] = np.float32(0.8) * p["h"] / p["time_delta"]
    return scenes.Scene(parts, p, native.kernel_terms(0.04), sc.normals, sc.vertices, sc.indices)


# no neighbours, counts either side of a round of 16 and of a list's groups of
# four, coincident particles, and lists that overflow (more than 128)
CASES = {
    "one": lambda: cloud(1, 1, 0.4, 0.5),
    "two_far": lambda: cloud(2, 8, 0.1, 0.9),
    **{f"clique{k}": (lambda k=k: cloud(k, k, 0.45, 0.465))
       for k in (2, 4, 5, 15, 16, 17, 18, 32, 33, 34, 128, 129, 130, 200)},
    "coincident": lambda: cloud(300, 3, 0.4, 0.5, dup=120),
    "spray": lambda: cloud(4097, 4, 0.2, 0.8),
    "dam": lambda: scenes.dam_break(6001, seed=7, jitter=0.1),
}


def step(ctx, scs):
    b = native.Batch(ctx, [s.n for s in scs])
    for i, s in enumerate(scs):
        b.set_scene_params(i, s.params, s.terms)
        b.mesh_scene(i, s.normals, s.vertices, s.indices)
        b.upload_scene(i, s.particles)
    b.step(1)
    out = b.download_scene(len(scs) - 1)
    b.close()
    return out


@pytest.mark.parametrize("name", CASES)
def test_lanes_agree_bit_for_bit(ctx, name):
    sc = CASES[name]()
    lanes = step(ctx, [sc])
    one = step(ctx, [scenes.dam_break(LANES_MAX + 1, seed=3), sc])
    for f in FIELDS:
        assert np.array_equal(lanes[f].view(np.uint32), one[f].view(np.uint32)), f


@pytest.mark.parametrize("n", [LANES_MAX, LANES_MAX + 1])
def test_forces_match_the_oracle(ctx, n):
    sc = scenes.dam_break(n, seed=5, jitter=0.1)
    ref = oracle.stages(sc.particles, sc.params, sc.terms, sc.normals, sc.vertices, sc.indices)
    st = native.State(ctx, n)
    st.set_params(sc.params, sc.terms)
    st.scene(sc.normals, sc.vertices, sc.indices)
    st.upload(sc.particles)
    for s in ("grid", "hash", "sort", "density", "forces"):
        st.stage(s)
    got = st.download_sorted()["acceleration"][:, :3]
    ra = ref.forces["acceleration"][:, :3]
    assert np.max(np.linalg.norm(got - ra, axis=1)) <= 1e-4 * np.max(np.linalg.norm(ra, axis=1))
    st.close()
