"""Times of stages against each other, where a work-group size or the state of
the fluid has once cost a multiple."""
import pytest

from libclsph_amd import learned as lrn
from libclsph_amd import native, scenes
from test_gpu_sort_paths import cloud, state_of

pytestmark = pytest.mark.gpu


def test_small_density_work_groups_in_settled_fluid():
    """Work-groups of 64 and 128 threads against the default of 512 after 1,800
    substeps: 1.80 and 2.06 times as long, 2.2 and 2.6 when four lanes took
    each particle outside the staged halos; bounds in between."""
    ctx = native.Context(0)
    sc = scenes.dam_break(207000, seed=1)
    st = lrn.make_state(ctx, sc)
    st.upload(sc.particles)
    for _ in range(36):
        st.step(50)
        ctx.sync()
    for name in ("grid", "hash", "sort", "density"):
        st.stage(name)
    us = {}
    for size in (64, 128, 512):
        st.set_block_sizes([0, 0, 0, 0, size, 0, 0])
        st.stage("density")
        us[size] = 1e3 * min(st.time_stage("density", 30) for _ in range(3))
    print({k: round(v, 1) for k, v in us.items()}, flush=True)
    st.close()
    ctx.close()
    assert us[64] <= 2.0 * us[512]
    assert us[128] <= 2.3 * us[512]


def test_a_wide_table_is_filled_by_the_whole_chip():
    """5,000 particles in two far corners: the cell table of 77 million keys
    takes 2.1 times as long as that of 8.4 million, 4.1 times when 128
    work-groups wrote its long runs of empty keys; a bound in between."""
    ctx = native.Context(0)
    us = []
    for side in (5.0, 20.0):
        st = state_of(ctx, cloud(5000, side, corners=True), 1 << 24)
        for name in ("grid", "hash", "sort", "cell_table"):
            st.stage(name)
        us.append(1e3 * min(st.time_stage("cell_table", 20) for _ in range(3)))
        st.close()
    ctx.close()
    print(["%.1f" % u for u in us], flush=True)
    assert us[1] <= 3.0 * us[0]


def test_digit_counts_of_a_wide_table_are_added_up_at_no_loss():
    """The LSD passes (the sort stage less its cell pass) in a table of 2.1
    million cells, whose digits have 2,048 values, on either side of the 48
    tiles up to which the scatter may add up the tiles' counts: as long, 3.3
    times when it did so whatever the digits; a bound in between."""
    ctx = native.Context(0)
    us = []
    for n in (98304, 98305):
        st = state_of(ctx, cloud(n, 9.5), 1 << 22)
        for name in ("grid", "hash", "sort", "cell_table"):
            st.stage(name)
        us.append(1e3 * min(st.time_stage("sort", 20) - st.time_stage("cell_table", 20)
                            for _ in range(5)))
        st.close()
    ctx.close()
    print(["%.1f" % u for u in us], flush=True)
    assert us[0] <= 1.6 * us[1]
