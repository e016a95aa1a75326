"""The learned step takes the particles whose lists overflow (more than 128
neighbours) from the forces kernel, sixteen lanes each, four at a time per
wave (k_forces_overflow, csrc/sph.hip). Without a network's correction they
move as in the plain substep, to the bit."""
import numpy as np
import pytest

from libclsph_amd import learned as lrn
from libclsph_amd import native, scenes

pytestmark = pytest.mark.gpu


def balls(sizes, h=0.04):
    """Balls far apart: of each, the particle in the middle sees all the
    others, on a sphere of 0.9 h, and they see less than a third of them; a
    negative size is a small ball whose particles all see each other."""
    rng = np.random.default_rng(5)
    x = []
    for q, size in enumerate(sizes):
        middle = np.array([0.1 + 0.1 * (q % 8), 0.2 + 0.1 * (q // 8), 0.3])
        d = rng.normal(size=(abs(size), 3))
        d /= np.linalg.norm(d, axis=1)[:, None]
        x.append(middle[None, :])
        x.append(middle + d * (0.9 * h if size > 0 else 0.2 * h))
    x = np.concatenate(x).astype(np.float32)
    sc = scenes.dam_break(max(len(x), 64), seed=1)
    parts = sc.particles[:len(x)].copy()
    parts["position"][:, :3] = x
    v = rng.normal(0, 0.05, (len(x), 3)).astype(np.float32)
    parts["velocity"][:, :3] = parts["intermediate_velocity"][:, :3] = v
    p = sc.params.copy()
    p["particles_count"] = len(x)
    p["h"] = np.float32(h)
    p["max_velocity"] = np.float32(0.8) * p["h"] / p["time_delta"]
    return scenes.Scene(parts, p, native.kernel_terms(h), sc.normals, sc.vertices, sc.indices)


# overflowing particles of a wave: none, one, several rounds of four
@pytest.mark.parametrize("sizes", [(100, 120), (200,), (200, 210, 220, 230, 240, 250),
                                   (-129, 150), (-128, -140, 200), (-700, 200, -300)])
def test_overflowing_particles_move_as_in_the_plain_substep(sizes):
    ctx = native.Context(0)
    sc = balls(sizes)
    print(f"sizes {sizes}, {sc.n} particles", flush=True)
    plain, learned = (lrn.make_state(ctx, sc) for _ in range(2))
    for st in (plain, learned):
        st.upload(sc.particles)
        st.track_ids(True)
    net = native.Network(ctx, sc.n, e_cap=64)
    net.set_params(np.zeros(net.count, np.float32))
    plain.step(1)
    learned.learned_step(net, 1)
    d = np.linalg.norm(sc.particles["position"][:, None, :3] -
                       sc.particles["position"][None, :, :3], axis=2)
    over = np.where((d < float(sc.params["h"])).sum(axis=1) - 1 > 128)[0]
    a, b = plain.download(), learned.download()
    a, b = a[np.argsort(plain.ids())][over], b[np.argsort(learned.ids())][over]
    assert (len(over) == 0) == (sizes == (100, 120))
    for f in ("position", "velocity", "intermediate_velocity"):
        assert np.array_equal(a[f].view(np.uint32), b[f].view(np.uint32)), f
    net.close()
    plain.close()
    learned.close()
    ctx.close()
