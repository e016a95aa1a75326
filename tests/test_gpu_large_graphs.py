"""The two-round network's training forward on more rows than 65,536
work-groups of 256 threads cover with one item each: every row of its node and
edge arrays is written, so that its outputs agree with the fused inference's
on every particle, the last ones included."""
import numpy as np
import pytest

from libclsph_amd import native, scenes
from oracle import gnn as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def compare(ctx, n, spread, e_cap):
    """Outputs of forward and infer, and the edge count. Both round each
    layer's inputs to bf16 and sum in float32, in another order: the bounds of
    the same comparison at small sizes."""
    sc = scenes.dam_break(n, seed=5, jitter=0.1)
    parts = sc.particles.copy()
    parts["velocity"][:, :3] = np.random.default_rng(6).normal(0.0, 0.5, (n, 3))
    if spread > 1.0:
        shake = np.random.default_rng(5).normal(0.0, 0.25 * float(sc.params["h"]), (n, 3))
        parts["position"][:, :3] = parts["position"][:, :3] * spread + shake
    st = native.State(ctx, n)
    st.set_params(sc.params, sc.terms)
    st.upload(parts)
    for name in ("grid", "hash", "sort", "density"):
        st.stage(name)
    net = native.TwoRoundNetwork(ctx, n, e_cap=e_cap)
    flat = L.random_params(11)
    weights = L.unpack(flat)
    for name in ("e1.w1", "e2.w1"):  # outputs that depend on the edges' inputs
        weights[name][:] *= 16.0
    net.set_params(flat.astype(np.float32))
    edges = net.forward(st)
    ref = net.output().astype(np.float64)[:, :3]
    net.infer(st)
    got = net.output().astype(np.float64)[:, :3]
    net.close()
    st.close()
    rel = np.sqrt(((ref - got) ** 2).mean()) / np.sqrt((got ** 2).mean())
    print(f"n {n}, {edges} edges, rel.rms {rel:.2e}", flush=True)
    scale = np.abs(got).max()
    assert np.isfinite(got).all()
    for part in (slice(0, n), slice(n - 50000, n)):
        assert np.abs(ref - got)[part].max() <= 1e-2 * scale
        rms = np.sqrt(((ref - got)[part] ** 2).mean()) / np.sqrt((got[part] ** 2).mean())
        assert rms <= 1e-3
    return edges


def test_more_than_a_million_particles(ctx):
    """16 items of u2's H half per particle: 65,536 work-groups end at
    particle 1,048,576."""
    edges = compare(ctx, 1100000, 1.9, 16 * 1100000)
    assert edges < 16 * 1100000


def test_more_than_sixteen_million_edges(ctx):
    """One item of the edge inputs per edge: 65,536 work-groups end at edge
    16,777,216."""
    edges = compare(ctx, 700000, 1.0, 34 * 700000)
    assert edges > 65536 * 256
