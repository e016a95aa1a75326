"""Particle records to and from the device go through page-locked buffers of
13,056 records (kTransferRecords, csrc/state.h): counts either side of a
work-group of 256 records and of one, two and three buffers come back whole,
in the state's order and in sorted order, alone and as a scene of a batch."""
import numpy as np
import pytest

from libclsph_amd import layout, native, scenes

pytestmark = pytest.mark.gpu

BUFFER = 13056
COUNTS = [1, 63, 255, 257, BUFFER - 1, BUFFER, BUFFER + 1, 2 * BUFFER, 2 * BUFFER + 1,
          3 * BUFFER + 77]
VECTORS = ("position", "velocity", "intermediate_velocity", "acceleration")


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def filled(n, seed):
    """A dam break whose every field holds something."""
    sc = scenes.dam_break(n, seed=seed, jitter=0.1)
    rng = np.random.default_rng(seed)
    for f in VECTORS[1:]:
        sc.particles[f][:, :3] = rng.normal(0, 0.05, (n, 3)).astype(np.float32)
    sc.particles["density"] = rng.uniform(900, 1100, n).astype(np.float32)
    sc.particles["pressure"] = rng.normal(0, 10, n).astype(np.float32)
    sc.particles["grid_index"] = rng.integers(0, 1 << 20, n)
    return sc


def state_of(ctx, sc):
    st = native.State(ctx, sc.n)
    st.set_params(sc.params, sc.terms)
    st.scene(sc.normals, sc.vertices, sc.indices)
    st.upload(sc.particles)
    return st


@pytest.mark.parametrize("n", COUNTS)
def test_records_come_back_as_uploaded(ctx, n):
    sc = filled(n, 5)
    st = state_of(ctx, sc)
    assert st.download().tobytes() == sc.particles.tobytes()
    part = layout.particles(max(1, n // 2))
    ctx.check(native.lib.clsph_download_aos(st.h, native._ptr(part), len(part)))
    assert part.tobytes() == sc.particles[:len(part)].tobytes()
    st.close()


@pytest.mark.parametrize("n", COUNTS)
def test_sorted_and_substep_records(ctx, n):
    """Sorted records are the uploaded ones in the stable order by cell id; a
    synchronous download after a substep is the asynchronous one's bytes."""
    sc = filled(n, 6)
    st = state_of(ctx, sc)
    for s in ("grid", "hash", "sort", "density", "forces"):
        st.stage(s)
    got = st.download_sorted()
    keys, perm = st.sorted()
    assert np.array_equal(got["grid_index"], keys)
    for f in VECTORS[:3]:
        assert np.array_equal(got[f], sc.particles[f][perm])
    st.upload(sc.particles)
    st.step(1)
    out = np.zeros(n, dtype=layout.PARTICLE)
    p = native._ptr(out)
    ctx.check(native.lib.clsph_download_begin(st.h, 0, p, n))
    ctx.check(native.lib.clsph_download_wait(st.h, 0, None))
    assert st.download().tobytes() == out.tobytes()
    assert np.array_equal(out["grid_index"], keys)
    st.close()


def test_batch_scenes_come_back_as_uploaded(ctx):
    scs = [filled(n, 10 + i) for i, n in enumerate((300, BUFFER + 5, 1, 2 * BUFFER + 3))]
    b = native.Batch(ctx, [s.n for s in scs])
    for i, s in enumerate(scs):
        b.set_scene_params(i, s.params, s.terms)
        b.mesh_scene(i, s.normals, s.vertices, s.indices)
        b.upload_scene(i, s.particles)
    for i, s in enumerate(scs):
        assert b.download_scene(i).tobytes() == s.particles.tobytes()
    b.step(1)
    for i, s in enumerate(scs):
        st = state_of(ctx, s)
        st.step(1)
        assert b.download_scene(i).tobytes() == st.download().tobytes()
        st.close()
    b.close()
