"""The fused edge rounds' ways of cutting neighbour lists into tiles.

  one particle to many per wave, lists split over streams, particles without
  neighbours                          : the training forward's outputs
  a particle with a non-finite state  : the particles it reaches, no others
"""
import numpy as np
import pytest

from libclsph_amd import native, scenes
from oracle import gnn as L

pytestmark = pytest.mark.gpu

DENSITY_STAGES = ("grid", "hash", "sort", "cell_table", "density")


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def state(ctx, n, steps, seed, spread=1.0):
    sc = scenes.dam_break(n, seed=seed)
    st = native.State(ctx, sc.n)
    st.set_params(sc.params, sc.terms)
    st.scene(sc.normals, sc.vertices, sc.indices)
    p = sc.particles.copy()
    if spread > 1.0:
        jitter = np.random.default_rng(seed).normal(0.0, 0.25 * float(sc.params["h"]), (sc.n, 3))
        p["position"][:, :3] = p["position"][:, :3] * spread + jitter
    st.upload(p)
    st.step(steps)
    for name in DENSITY_STAGES:
        st.stage(name)
    return st


# both outputs round each layer's inputs to bf16 and sum in float32, in another
# order: the bounds of the same comparison at 4,000 particles
@pytest.mark.parametrize("n,steps,spread", [
    (1, 1, 1.0), (7, 2, 1.0), (300, 5, 1.0),      # a particle or none per wave
    (3071, 20, 1.0), (3073, 20, 1.0),             # about one per wave
    (9000, 30, 1.0), (60000, 20, 1.0),            # runs up to 16, last ones short
    (5000, 1, 1.6), (40000, 1, 1.9),              # short lists, particles without neighbours
])
def test_outputs_match_the_training_forward(ctx, n, steps, spread):
    st = state(ctx, n, steps, 3, spread)
    net = native.TwoRoundNetwork(ctx, st.n)
    net.set_params(L.random_params(11).astype(np.float32))
    net.forward(st)
    off, _ = net.graph()
    deg = np.diff(off.astype(np.int64))
    ref = net.output().astype(np.float64)[:, :3]
    net.infer(st)
    got = net.output().astype(np.float64)[:, :3]
    err = np.abs(got - ref)
    scale = np.abs(ref).max()
    rms = np.sqrt((err ** 2).mean()) / np.sqrt((ref ** 2).mean())
    print(f"n={st.n} neighbours {deg.min()}..{deg.max()}: max {err.max() / scale:.2e} of scale, "
          f"rel.rms {rms:.2e}", flush=True)
    assert np.isfinite(got).all()
    assert err.max() <= 1e-2 * scale
    assert rms <= 1e-3


def test_a_non_finite_particle_reaches_its_neighbours_only(ctx):
    sc = scenes.dam_break(9000, seed=4)
    st = native.State(ctx, sc.n)
    st.set_params(sc.params, sc.terms)
    st.scene(sc.normals, sc.vertices, sc.indices)
    p = sc.particles.copy()
    p["velocity"][4321, 1] = np.inf
    st.upload(p)
    for name in DENSITY_STAGES:
        st.stage(name)
    net = native.TwoRoundNetwork(ctx, st.n)
    net.set_params(L.random_params(11).astype(np.float32))
    net.forward(st)
    ref = net.output().astype(np.float64)[:, :3]
    net.infer(st)
    got = net.output().astype(np.float64)[:, :3]
    ok = np.isfinite(ref).all(axis=1)
    print(f"{(~ok).sum()} particles not finite", flush=True)
    assert 0 < (~ok).sum() < 500
    assert (np.isfinite(got).all(axis=1) == ok).all()
    assert np.abs(got - ref)[ok].max() <= 1e-2 * np.abs(ref[ok]).max()
