"""The full sort (first substep, and every substep with hooks) in tables from exactly full
(one particle, its eight blocks) over the sizes at which its scan changes (a slot per
thread, four at a time) to both sides of the four- and eight-launch variants (16384 slots):
active blocks and cell counts bit-exact with the oracle's, and the state after hooked
substeps the oracle's (relative L2 1e-5 per substep)."""
import numpy as np
import pytest

from oracle import oracle as O
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from tests.parity import assert_blocks_equal, rel_l2

pytestmark = pytest.mark.gpu


class Observer(P.MpmPipelineHooks):
    def after_particle_sort(self, data, stream):
        pass


@pytest.mark.parametrize("n,side,cap", [(1, 0.5, 8), (3, 0.5, 16), (70, 1.0, 128), (500, 2.0, 256), (500, 2.0, 512),
                                        (4000, 3.0, 1024), (9000, 5.0, 16384), (9000, 5.0, 32768)])
def test_full_sort_is_exact(gpu_pipeline, n, side, cap):
    pl, st = gpu_pipeline
    dx = 1.0 / 64
    rng = np.random.RandomState(n)
    ext = side * 4 * dx
    pos = (0.5 + 0.6 * dx + rng.uniform(0.0, ext, (n, 3))).astype(np.float32)
    vel = rng.uniform(-0.4, 0.4, (n, 3)).astype(np.float32) * np.float32(dx / 1.0e-4) * (n > 3)
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3), vel.astype(np.float32))
    bodies, mats = scenes.box_walls(M.STICK)
    sc = scenes.Scene("sort", parts, 1.0e-4, dx, cap, bodies, mats, gravity=(0.0, 0.0, 0.0))
    data, orc = P.MpmData.from_scene(pl, sc), O.Oracle(sc)
    pl.launch_step(data, st)
    data.check_errors(st)
    orc.step(1)
    assert_blocks_equal(data.blocks(st), orc.blocks())
    hooked, orc = P.MpmData.from_scene(pl, sc), O.Oracle(sc)
    hooks = Observer()
    for k in range(3):
        pl.launch_step(hooked, st, hooks=hooks)
        orc.step(1)
        hooked.check_errors(st)
        assert rel_l2(hooked.positions(st)[:, :3], orc.positions()[:, :3]) <= 1.0e-5 * (k + 1)
        assert rel_l2(hooked.kinematics(st)["velocity"], orc.kinematics()["velocity"]) <= 1.0e-5 * (k + 1) or n <= 3
        assert rel_l2(hooked.def_grad(st), orc.def_grad()) <= 1.0e-5 * (k + 1)
