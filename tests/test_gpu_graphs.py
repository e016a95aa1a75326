"""A state that has run 64 substeps replays 4 and 16 of them as one graph
(launch_steps, csrc/capi.cpp). Whatever the calls' lengths, and with
parameters, work-group sizes and particles changed in between, it is bit for
bit where single substeps leave it; every call is checked, with the program's
own work and a read-back in between."""
import numpy as np
import pytest

from libclsph_amd import native, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [1500, 20011])
def test_calls_of_any_length(ctx, n):
    sc = scenes.dam_break(n, seed=4)
    many, ones = (native.State(ctx, n) for _ in range(2))
    for st in (many, ones):
        st.set_params(sc.params, sc.terms)
        st.scene(sc.normals, sc.vertices, sc.indices)
        st.upload(sc.particles)
    p = sc.params.copy()
    p["dynamic_viscosity"] = np.float32(2) * p["dynamic_viscosity"]
    for k, steps in enumerate((3, 61, 1, 4, 5, 15, 16, 17, 36, 16, 21, 20, 70, 19)):
        if k == 8:  # parameters are read from the device: the graphs stay
            for st in (many, ones):
                st.set_params(p, sc.terms)
        if k == 10:  # new work-group sizes: captured anew
            for st in (many, ones):
                st.set_block_sizes([0, 128, 0, 0, 0, 0, 128])
        if k == 12:
            back = many.download()
            for st in (many, ones):
                st.upload(back)
        many.step(steps)
        for _ in range(steps):
            ones.step(1)
        assert many.download().tobytes() == ones.download().tobytes(), (k, steps)
        assert many.bounce_capped() == ones.bounce_capped()
    many.close()
    ones.close()


def test_identities_follow(ctx):
    sc = scenes.dam_break(5000, seed=6)
    many, ones = (native.State(ctx, sc.n) for _ in range(2))
    for st in (many, ones):
        st.set_params(sc.params, sc.terms)
        st.scene(sc.normals, sc.vertices, sc.indices)
        st.upload(sc.particles)
    many.step(80)
    for _ in range(80):
        ones.step(1)
    for st in (many, ones):  # the substep gains two kernels: captured anew
        st.track_ids(True)
    for steps in (64, 23, 40):
        many.step(steps)
        for _ in range(steps):
            ones.step(1)
        assert np.array_equal(many.ids(), ones.ids())
        assert many.download().tobytes() == ones.download().tobytes()
    many.close()
    ones.close()
