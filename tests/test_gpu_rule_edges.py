"""The density stage against the oracle on either side of the particle counts
at which it takes another kernel, and one scene in states of each kind. The
counts are read from the source, so that they follow the rule (launch_density,
csrc/sph.hip)."""
import os
import re

import numpy as np
import pytest

import oracle
from libclsph_amd import build, native, scenes
from test_gpu_density_paths import CASES, FIELDS, beside

pytestmark = pytest.mark.gpu

SOURCE = open(os.path.join(build.CSRC, "sph.hip")).read()
LANES16, LANES4 = (int(re.search(rf"k{name}Max = (\d+)", SOURCE).group(1))
                   for name in ("Lanes16", "Lanes4"))


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [LANES16, LANES16 + 1, LANES4, LANES4 + 1])
def test_density_on_both_sides(ctx, n):
    """1e-5 relative, the bound of the other parity tests (FP32 sums of about
    35 terms in another order)."""
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
    assert (np.abs(got["density"] - ref["density"]) / ref["density"]).max() <= 1e-5


@pytest.mark.parametrize("case", list(CASES))
def test_a_scene_beside_one_lane_fillers(ctx, case):
    """The filler alone is past the rule's last count."""
    sc = CASES[case]()
    want = beside(ctx, sc, 0)
    got = beside(ctx, sc, LANES4 + 1)
    for f in FIELDS:
        np.testing.assert_array_equal(got[f], want[f], err_msg=f)
