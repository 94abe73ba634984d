"""Readbacks after a grid overflow, in which particles were lost: they read as zeros, and
not as bytes that an earlier readback left in the staging. A cluster that flies apart until
its blocks no longer fit the table."""
import numpy as np
import pytest

from slosh_amd import _lib
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes

pytestmark = pytest.mark.gpu


def test_lost_particles_read_as_zeros(gpu_pipeline):
    pl, st = gpu_pipeline
    n, dx, dt = 200, 1.0 / 64, 1.0e-4
    rng = np.random.RandomState(2)
    away = rng.normal(size=(n, 3))
    away /= np.linalg.norm(away, axis=1, keepdims=True)
    pos = (0.5 + 0.6 * dx + away * dx).astype(np.float32)
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0, 0.3),
                              (away * 0.9 * dx / dt).astype(np.float32))
    bodies, mats = scenes.box_walls(M.SLIP)
    sc = scenes.Scene("apart", parts, dt, dx, 64, bodies, mats, gravity=(0.0, 0.0, 0.0))
    data = P.MpmData.from_scene(pl, sc)
    for _ in range(4):  # both particle buffers hold every particle
        pl.launch_step(data, st)
    data.check_errors(st)
    whole = data.kinematics(st)
    assert (whole["mass"] > 0).all() and (np.abs(data.positions(st)[:, :3]).max(1) > 0).all()
    for _ in range(30):
        pl.launch_step(data, st)
    with pytest.raises(_lib.SloshError):
        data.check_errors(st)
    first = {"x": data.positions(st), "k": data.kinematics(st), "f": data.def_grad(st)}
    again = {"f": data.def_grad(st), "x": data.positions(st), "k": data.kinematics(st)}
    for key in first:
        assert np.array_equal(first[key].view(np.uint8), again[key].view(np.uint8)), key
    lost = ~first["x"].any(1)
    assert lost.any() and not lost.all()
    assert np.array_equal(lost, ~first["f"].reshape(n, -1).any(1))
    assert np.array_equal(lost, first["k"]["mass"] == 0)
