"""Steady-state substeps of a scattered cloud: particles cross block faces in every
direction and blocks appear and vanish each substep, from a few particles a block to
several hundred, in tables from fewer slots than the block list has regions to many times
the blocks. After each run of substeps the active blocks and their cell counts must be
those of the oracle's sort of the same positions (bit-exact), and the state after one more
substep the oracle's from the same start (relative L2 1e-5, the bound of one substep)."""
import copy

import numpy as np
import pytest

from oracle import oracle as O
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from tests.parity import assert_blocks_equal, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,side,cap", [(1, 1.0, 32), (5, 1.5, 64), (63, 1.0, 128), (640, 4.0, 1024),
                                        (3000, 6.0, 16384), (13000, 6.0, 131072), (40000, 5.0, 1024),
                                        (98304, 5.0, 1024), (98305, 7.0, 4096), (262145, 8.0, 4096)])
def test_moving_cloud_keeps_exact_blocks(gpu_pipeline, n, side, cap):
    pl, st = gpu_pipeline
    dx, dt = 1.0 / 64, 1.0e-4
    rng = np.random.RandomState(n)
    ext = side * 4 * dx  # `side` blocks along an axis
    pos = rng.uniform(0.5 - ext / 2, 0.5 + ext / 2, (n, 3)).astype(np.float32)
    vel = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32) * np.float32(dx / dt)
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3), vel)
    bodies, mats = scenes.box_walls(M.STICK)
    sc = scenes.Scene("cloud", parts, dt, dx, cap, bodies, mats, gravity=(0.0, 0.0, 0.0))
    data = P.MpmData.from_scene(pl, sc)
    for run in (1, 1, 2, 3) if n < 90000 else (2,):
        for _ in range(run):
            pl.launch_step(data, st)
        data.check_errors(st)
        pos = data.positions(st)
        pos[:, 3] = 0.0
        at = copy.copy(sc)
        at.particles = {"pos4": pos, "kin": data.kinematics(st), "def_grad": data.def_grad(st),
                        "props": data.properties(st), "models": data.models(st)}
        orc = O.Oracle(at)
        pl.launch_step(data, st)
        orc.step(1)
        assert_blocks_equal(data.blocks(st), orc.blocks())
        assert rel_l2(data.positions(st)[:, :3], orc.positions()[:, :3]) <= 1.0e-5
        assert rel_l2(data.kinematics(st)["velocity"], orc.kinematics()["velocity"]) <= 1.0e-5
        assert rel_l2(data.def_grad(st), orc.def_grad()) <= 1.0e-5
