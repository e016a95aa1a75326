"""Substeps of single scenes compute grid, keys and the first digit counts in
one kernel up to 655,360 particles, and scatters add up the tiles' counts
themselves up to 48 tiles of 2,048 keys (csrc/sort.hip). They leave what the
grid, hash and sort stages leave, bit for bit, and the cell table is the one
the sorted cell ids define, its long runs of empty keys included."""
import numpy as np
import pytest

from libclsph_amd import native, scenes

pytestmark = pytest.mark.gpu

TILE, FOLD, FUSED = 2048, 48 * 2048, 655360
GRID = ("min_point", "max_point", "grid_size_x", "grid_size_y", "grid_size_z", "grid_cell_count")


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def cloud(n, side, h=0.04, seed=1, corners=False):
    """n random particles in a box of `side`, a tenth of them coincident; with
    `corners` in two cells at opposite ends of the box's z axis."""
    rng = np.random.default_rng(seed)
    sc = scenes.dam_break(max(n, 64), seed=seed)
    parts = sc.particles[:n].copy()
    x = rng.uniform(0, 0.05 if corners else side, (n, 3)).astype(np.float32)
    if corners:
        x[n // 2:, 2] += np.float32(side)
    x[n - n // 10:] = x[0]
    parts["position"][:, :3] = x
    p = sc.params.copy()
    p["particles_count"] = n
    p["h"] = np.float32(h)
    p["max_velocity"] = np.float32(0.8) * p["h"] / p["time_delta"]
    return scenes.Scene(parts, p, native.kernel_terms(h), sc.normals, sc.vertices, sc.indices)


def state_of(ctx, sc, table_cap=0):
    st = native.State(ctx, sc.n, table_cap=table_cap)
    st.set_params(sc.params, sc.terms)
    st.scene(sc.normals, sc.vertices, sc.indices)
    st.upload(sc.particles)
    return st


def check(ctx, sc, steps=2, table_cap=0):
    """`steps` substeps, each against the stages one by one; the cell count."""
    one, stages = state_of(ctx, sc, table_cap), state_of(ctx, sc, table_cap)
    for _ in range(steps):
        before = stages.download()
        one.step(1)
        for s in ("grid", "hash", "sort", "density", "forces", "advect"):
            stages.stage(s)
        ga, gb = one.grid(), stages.grid()
        for f in GRID:
            assert np.array_equal(ga[f], gb[f]), f
        keys = one.keys()
        assert np.array_equal(keys, stages.keys())
        sk, perm = one.sorted()
        assert np.array_equal(perm, np.argsort(keys, kind="stable"))
        assert np.array_equal(sk, keys[perm])
        for x, y in zip(one.order(), stages.order()):
            assert np.array_equal(x, y)
        cells = int(ga["grid_cell_count"])
        table = np.searchsorted(sk, np.arange(cells, dtype=np.uint32)).astype(np.uint32)
        assert np.array_equal(one.cell_table(cells), table)
        got = one.download()
        assert got.tobytes() == stages.download().tobytes()
        assert len(before) == len(got)
    one.close()
    stages.close()
    return cells


@pytest.mark.parametrize("n", [1, 63, 64, 257, TILE - 1, TILE, TILE + 1, 16384, FOLD, FOLD + 1,
                               FUSED, FUSED + 1])
def test_counts(ctx, n):
    check(ctx, scenes.dam_break(n, seed=2, jitter=0.1), steps=2 if n < FUSED else 1)


# bits: of the Morton code of the grid's size, floor((side + 8 h) / 2 h) cells
# on each axis; with 21 bits a pass has 2,048 digits, more than the threads of
# a scatter, and most of the table is long runs of empty keys
@pytest.mark.parametrize("side,bits,cap", [(0.04, 9, 0), (0.5, 12, 0), (1.2, 15, 0),
                                           (9.5, 21, 1 << 22)])
@pytest.mark.parametrize("n", [700, 30001])
def test_cell_id_widths(ctx, n, side, bits, cap):
    cells = check(ctx, cloud(n, side), steps=1, table_cap=cap)
    assert cells.bit_length() == bits


@pytest.mark.parametrize("side", [1.0, 5.0, 20.0])
def test_runs_between_far_clusters(ctx, side):
    check(ctx, cloud(5000, side, corners=True), steps=1, table_cap=1 << 24)


def test_errors_are_reported(ctx):
    st = state_of(ctx, cloud(300, 500.0))  # 1,024 cells and more on an axis
    st.step(1)
    with pytest.raises(native.ClsphError):
        st.download()
    st.close()
