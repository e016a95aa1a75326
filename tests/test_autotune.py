"""The autotuner times work-group sizes only where a stage uses them."""
import os
import re

import pytest

from libclsph_amd import autotune, build


def constant(source, name):
    text = open(os.path.join(build.CSRC, source)).read()
    return int(re.search(rf"{name} = (\d+)", text).group(1))


def test_limits_are_the_kernels():
    assert autotune.OWN_UP_TO == {"density": constant("sph.hip", "kLanes4Max"),
                                  "forces": constant("sph.hip", "kForceLanesMax")}
    assert autotune.SMALL_SCENE == constant("sph.hip", "kSmallScene")
    assert autotune.OWN_SMALL_UP_TO == {"forces": constant("sph.hip", "kForceLanesSmallMax")}
    assert autotune.OWN_SINGLE_UP_TO == {"hash": constant("sort.hip", "kFusedMax")}


class Recorder:
    """A state whose substeps all take as long."""

    def __init__(self, counts):
        self.counts, self.n = counts, sum(counts)
        self.sizes, self.tried = list(autotune.DEFAULT), set()

    def block_sizes(self):
        return list(self.sizes)

    def set_block_sizes(self, sizes):
        self.tried |= {k for k, (a, b) in enumerate(zip(autotune.DEFAULT, sizes)) if a != b}
        self.sizes = list(sizes)

    def step(self, steps):
        pass

    def time_steps(self, steps):
        return float(steps)


@pytest.mark.parametrize("counts,stages", [
    ([4096], {"advect"}), ([65536], {"forces", "advect"}),
    ([262144], {"density", "forces", "advect"}),
    ([1048576], {"hash", "density", "forces", "advect"}),
    ([2048] * 14, {"hash", "advect"}), ([2048] * 15, {"hash", "forces", "advect"}),
    ([8193] * 6, {"hash", "advect"}), ([4096] * 16, {"hash", "forces", "advect"}),
    ([16384] * 16, {"hash", "density", "forces", "advect"})])
def test_stages_that_choose_their_own_are_left_out(counts, stages):
    state = Recorder(counts)
    assert autotune.tune_state(state, log=lambda m: None) == autotune.DEFAULT
    assert state.tried == {autotune.TUNED[s] for s in stages}
