"""The density stage takes 16, 4 or 1 lanes per particle by the state's
particle count (launch_density, csrc/sph.hip), and walks particles outside
the staged halos by 4 lanes each. Sums and lists are in one order everywhere,
so a scene's results are the same bits in states of every size."""
import numpy as np
import pytest

import oracle
from libclsph_amd import native, scenes

pytestmark = pytest.mark.gpu

LANES16_MAX, LANES4_MAX = 40960, 147456
FIELDS = ("position", "velocity", "intermediate_velocity", "density", "pressure", "grid_index")


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def cloud(n, seed, lo=0.2, hi=0.8, dup=0):
    """n random particles in [lo, hi]^3 at h = 0.04, `dup` of them twice."""
    rng = np.random.default_rng(seed)
    sc = scenes.dam_break(max(n, 64), seed=seed)
    parts = sc.particles[:n].copy()
    parts["position"][:, :3] = rng.uniform(lo, hi, (n, 3)).astype(np.float32)
    parts["velocity"][:, :3] = rng.normal(0, 0.05, (n, 3)).astype(np.float32)
    if dup:
        parts[n - dup:] = parts[:dup]
    p = sc.params.copy()
    p["particles_count"] = n
    p["h"] = np.float32(0.04)
    p["max_velocity"] = np.float32(0.8) * p["h"] / p["time_delta"]
    return scenes.Scene(parts, p, native.kernel_terms(0.04), sc.normals, sc.vertices, sc.indices)


def beside(ctx, sc, filler):
    """One substep of `sc` in a batch with a dam break of `filler` particles
    before it."""
    scs = ([scenes.dam_break(filler, seed=3)] if filler else []) + [sc]
    b = native.Batch(ctx, [s.n for s in scs])
    for i, s in enumerate(scs):
        b.set_scene_params(i, s.params, s.terms)
        b.mesh_scene(i, s.normals, s.vertices, s.indices)
        b.upload_scene(i, s.particles)
    b.step(1)
    out = b.download_scene(len(scs) - 1)
    b.close()
    return out


# one particle, either side of a wave and of a list's groups of four, random
# and coincident particles, more neighbours than a list holds (300 within one
# h), and cells beyond every staging capacity (4,000 in one cell)
CASES = {
    "cloud1": lambda: cloud(1, 1),
    "cloud63": lambda: cloud(63, 2, 0.4, 0.5),
    "cloud65": lambda: cloud(65, 3, 0.4, 0.5),
    "cloud3001dup": lambda: cloud(3001, 4, 0.3, 0.6, dup=40),
    "dense300": lambda: cloud(300, 5, 0.49, 0.51),
    "dense4000": lambda: cloud(4000, 6, 0.49, 0.51),
    "dam4096": lambda: scenes.dam_break(4096, seed=7),
}


@pytest.mark.parametrize("case", list(CASES))
def test_scene_is_the_same_in_states_of_every_size(ctx, case):
    print(f"case {case}", flush=True)
    sc = CASES[case]()
    want = beside(ctx, sc, 0)
    for filler in (LANES16_MAX + 1, LANES4_MAX + 1):
        got = beside(ctx, sc, filler)
        for f in FIELDS:
            np.testing.assert_array_equal(got[f], want[f], err_msg=f"{f}, filler {filler}")


@pytest.mark.parametrize("n", [LANES16_MAX, LANES16_MAX + 1, LANES4_MAX, LANES4_MAX + 1])
def test_density_at_the_edges_of_the_rule(ctx, n):
    """Against the oracle's density stage: 1e-5 relative, the bound of the
    other parity tests (FP32 sums of about 35 terms in another order)."""
    print(f"case n {n}", flush=True)
    sc = scenes.dam_break(n, seed=9, jitter=0.1)
    p = sc.params.copy()
    assert oracle.grid_params(sc.particles, p) == 0
    srt = oracle.sort_particles(oracle.locate_in_grid(sc.particles, p))
    ref = oracle.density_pressure(srt, p, sc.terms,
                                  oracle.cell_table(srt, int(p["grid_cell_count"])))
    st = native.State(ctx, n)
    st.set_params(sc.params, sc.terms)
    st.upload(sc.particles)
    for name in ("grid", "hash", "sort", "density"):
        st.stage(name)
    got = st.download_sorted()
    st.close()
    rel = np.abs(got["density"] - ref["density"]) / ref["density"]
    assert rel.max() <= 1e-5
