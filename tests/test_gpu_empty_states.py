"""The training evaluation of the corrective network on a state without
particles: no edges and no outputs, and no error."""
import pytest

from libclsph_amd import native, scenes

pytestmark = pytest.mark.gpu


def test_forward_of_an_empty_state():
    ctx = native.Context(0)
    sc = scenes.dam_break(64, seed=1)
    st = native.State(ctx, sc.n)
    st.set_params(sc.params, sc.terms)
    st.upload(sc.particles[:0])
    for name in ("grid", "hash", "sort", "density", "forces"):
        st.stage(name)
    net = native.Network(ctx, sc.n, e_cap=64 * sc.n)
    assert net.forward(st) == 0
    with pytest.raises(native.ClsphError):
        net.backward()
    # and the workspace serves the next state with particles
    st.upload(sc.particles)
    for name in ("grid", "hash", "sort", "density", "forces"):
        st.stage(name)
    assert net.forward(st) > 0
    net.close()
    st.close()
    ctx.close()
