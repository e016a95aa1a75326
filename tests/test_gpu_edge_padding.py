"""The fused edge rounds pad every particle's list to groups of four edges.
The padding takes part in no sum, whatever the rows that stand in for it
hold: a particle whose node term overflows reaches its neighbours only, not
the other particles of its wave's run."""
import numpy as np
import pytest

from libclsph_amd import native, scenes
from oracle import gnn as L

pytestmark = pytest.mark.gpu


def test_an_overflowing_node_term_reaches_its_neighbours_only():
    ctx = native.Context(0)
    sc = scenes.dam_break(9000, seed=4, jitter=0.1)
    parts = sc.particles.copy()
    # a cluster of coincident particles at the block's lowest corner (first in
    # the order, and so first of their runs): density several times the rest's
    x = parts["position"][:, :3]
    corner = np.argsort(x.sum(axis=1))[:12]
    x[corner] = x[corner[0]]
    st = native.State(ctx, sc.n)
    st.set_params(sc.params, sc.terms)
    st.upload(parts)
    for name in ("grid", "hash", "sort", "density"):
        st.stage(name)
    # H_0 = 2 silu(silu(rho / rho0 - 1)); PB_0 = 3e38 H_0, infinite in the
    # cluster only; PA = 0; the products of PB's rows are 0 unless it is infinite
    P = {name: np.zeros(shape) for name, shape in L.LAYOUT}
    P["n1.w1"][L.WIDTH, 0] = P["n1.w2"][0, 0] = 1.0
    P["n1.w3"][0, 0] = 2.0
    P["e2.wb"][0, 0] = 3e38
    P["e2.b2"][:] = 0.5
    P["e2.w3"][:] = P["n2.w2"][:] = np.eye(L.WIDTH)
    P["n2.w1"][L.WIDTH:] = np.eye(L.WIDTH)
    P["n2.w3"][:] = 0.01
    net = native.TwoRoundNetwork(ctx, st.n)
    net.set_params(L.pack(P).astype(np.float32))
    net.forward(st)
    ref = net.output().astype(np.float64)[:, :3]
    net.infer(st)
    got = net.output().astype(np.float64)[:, :3]
    ok = np.isfinite(ref).all(axis=1)
    print(f"{(~ok).sum()} particles not finite, {(~np.isfinite(got).all(axis=1)).sum()} fused",
          flush=True)
    assert 0 < (~ok).sum() < 1000
    assert (np.isfinite(got).all(axis=1) == ok).all()
    # the bounds of the same comparison with finite terms
    assert np.abs(got - ref)[ok].max() <= 1e-2 * np.abs(ref[ok]).max()
    net.close()
    st.close()
    ctx.close()
