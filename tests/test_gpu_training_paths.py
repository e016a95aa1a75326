"""The training products at the edges of their tiles and splits, and both
networks' gradients where their kernels take another branch: neighbour lists
cut short at 128, particle counts that leave work-groups partly filled."""
import numpy as np
import pytest

from libclsph_amd import native, scenes
from oracle import gnn as oracle_gnn
from oracle import learned as oracle_nn
import test_gpu_gnn
import test_gpu_nn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("ta,tb,acc,m,n,k", [
    (False, False, False, 1, 8, 8),          # one row, one step not filled
    (False, True, False, 129, 128, 56),      # one row into the second tile
    (True, False, False, 120, 136, 64),      # a whole step
    (True, True, False, 136, 127, 72),       # a step and a remainder
    (False, False, True, 257, 40, 128),      # added without a split
    (True, False, True, 128, 128, 511),      # just below the first split of K
    (True, False, True, 144, 128, 520),      # two splits, the second almost empty
    (True, False, True, 32, 32, 70001),      # split over about 270 work-groups
    (True, True, True, 16, 33, 4096),
])
def test_gemm_at_tile_and_split_edges(ctx, ta, tb, acc, m, n, k):
    """1e-5 of sum |a||b| + 1 per entry: float32 sums of k exact products,
    in partial sums of at most 512 splits."""
    print(f"gemm ta={ta} tb={tb} acc={acc} {m}x{n}x{k}", flush=True)
    m, n, k = (m if not ta else -(-m // 8) * 8), (n if tb else -(-n // 8) * 8), (
        k if ta and not tb else -(-k // 8) * 8)
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    a = rng.normal(size=(k, m) if ta else (m, k)).astype(np.float32)
    b = rng.normal(size=(n, k) if tb else (k, n)).astype(np.float32)
    c0 = rng.normal(size=(m, n)).astype(np.float32) if acc else np.zeros((m, n), np.float32)
    bias = None if acc else rng.normal(size=n).astype(np.float32)
    ab, bb = oracle_nn.bf16_bits(a), oracle_nn.bf16_bits(b)
    got = native.nn_gemm(ctx, ab, bb, c0.copy(), m, n, k, ta, tb, acc, bias)
    A = oracle_nn.bits_to_float(ab).reshape(a.shape).astype(np.float64)
    B = oracle_nn.bits_to_float(bb).reshape(b.shape).astype(np.float64)
    A, B = (A.T if ta else A), (B.T if tb else B)
    ref = A @ B + (c0 if acc else bias[None, :])
    assert np.all(np.abs(got - ref) <= 1e-5 * (np.abs(A) @ np.abs(B) + 1.0))


def cloud(n, neighbours, seed):
    """n random particles in a unit cube at rest density, h such that an
    interior particle has `neighbours` others within h."""
    rng = np.random.default_rng(seed)
    sc = scenes.dam_break(max(n, 64), seed=seed)
    parts = sc.particles[:n].copy()
    parts["position"][:, :3] = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    parts["velocity"][:, :3] = rng.normal(0, 0.3, (n, 3)).astype(np.float32)
    p = sc.params.copy()
    p["particles_count"] = n
    p["h"] = np.float32((3.0 * neighbours / (4.0 * np.pi * n)) ** (1.0 / 3.0))
    p["particle_mass"] = np.float32(1000.0 / n)
    p["max_velocity"] = np.float32(0.8) * p["h"] / p["time_delta"]
    return scenes.Scene(parts, p, native.kernel_terms(float(p["h"])), sc.normals, sc.vertices,
                        sc.indices)


def state_of(ctx, sc, stages):
    st = native.State(ctx, sc.n)
    st.set_params(sc.params, sc.terms)
    st.upload(sc.particles)
    for name in stages:
        st.stage(name)
    return st


# n and neighbours: lists of at most 128 (rows gathered), most lists cut short
# (rows added), particles without neighbours, one particle
CASES = [(1501, 35, "whole"), (1500, 170, "cut"), (65, 0.5, "sparse"), (33, 6, "small"),
         (1, 1.0, "one")]


@pytest.mark.parametrize("n,neighbours,case", CASES)
@pytest.mark.parametrize("which", ["corrective", "two_round"])
def test_gradients(ctx, which, n, neighbours, case):
    """Each tensor's gradient within 5 % of the oracle's backward of the
    FP64 network (bf16 operands on the GPU), as in the networks' own tests."""
    print(f"case {which} {case}", flush=True)
    two = which == "two_round"
    helper, ref_net = (test_gpu_gnn, oracle_gnn) if two else (test_gpu_nn, oracle_nn)
    sc = cloud(n, neighbours, 11)
    stages = ("grid", "hash", "sort", "density") + (() if two else ("forces",))
    st = state_of(ctx, sc, stages)
    net = (native.TwoRoundNetwork if two else native.Network)(ctx, n, e_cap=128 * n)
    flat = ref_net.random_params(7).astype(np.float32).astype(np.float64)
    net.set_params(flat.astype(np.float32))
    e = net.forward(st)
    deg = np.diff(net.graph()[0].astype(np.int64))
    assert (deg.max() == 128) == (case == "cut")
    target = np.random.default_rng(1).normal(0, 0.5, (n, 3)).astype(np.float32)
    net.set_target(target)
    loss = net.backward()
    got = ref_net.unpack(net.grad().astype(np.float64))
    args = helper.oracle_inputs(sc, st, net)
    out, keep = ref_net.forward(flat, bf16_round=True, keep=True, **args)
    want_loss = ref_net.loss(out, target.astype(np.float64))
    assert abs(loss - want_loss) <= 1e-3 * want_loss
    want = ref_net.unpack(ref_net.backward(flat, keep, target.astype(np.float64), args["src"],
                                           args["dst"], args["deg"]))
    for name, _ in ref_net.LAYOUT:
        size = np.linalg.norm(want[name])
        if size == 0.0:
            assert np.all(got[name] == 0.0), name
        else:
            assert np.linalg.norm(got[name] - want[name]) <= 5e-2 * size, (name, e)
