"""Forces in batches of small scenes, whose lists stay short: sixteen lanes per
particle up to 28,672 particles in all, one beyond (launch_forces,
csrc/sph.hip). Either way a scene is the same bits as by itself."""
import pytest

from libclsph_amd import autotune, native, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("count,size", [(57, 503), (58, 503), (3, 8192), (4, 8192), (4, 8193)])
def test_a_scene_is_the_same_alone(ctx, count, size):
    scs = [scenes.dam_break(size, seed=i, jitter=0.1) for i in range(count)]
    many = autotune.make_batch(ctx, scs)
    many.step(3)
    for i in (0, count // 2, count - 1):
        one = autotune.make_batch(ctx, [scs[i]])
        one.step(3)
        assert many.download_scene(i).tobytes() == one.download_scene(0).tobytes()
        one.close()
    many.close()


def test_many_small_scenes_take_a_lane_per_particle(ctx):
    """The forces stage of 100 scenes of 500 particles against 57 of them: as
    long, 1.4 times when sixteen lanes took each particle of both; a bound in
    between."""
    us = []
    for count in (57, 100):
        b = autotune.make_batch(ctx, [scenes.dam_break(500, seed=i) for i in range(count)])
        b.step(20)
        for name in ("grid", "hash", "sort", "density", "forces"):
            b.stage(name)
        us.append(1e3 * min(b.time_stage("forces", 30) for _ in range(5)))
        b.close()
    print(["%.1f" % u for u in us], flush=True)
    assert us[1] <= 1.22 * us[0]
