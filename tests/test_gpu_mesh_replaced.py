"""A collision mesh replaced between substeps: the steps after it are those of a data that
had the new mesh from the start, and a refused replacement (its links point backward)
leaves the one that is there, for the direct launch and for captured runs."""
import numpy as np
import pytest

from slosh_amd import _lib
from slosh_amd import pipeline as P
from slosh_amd import scenes
from tests.parity import rel_l2

pytestmark = pytest.mark.gpu


def raised(vertices, by):
    """The same mesh a little higher (boxes and vertices; the normals stay)."""
    shape = scenes.heightfield_test_scene(12).bodies[-1]["shape"]
    a, b = np.asarray(shape["a"]).view(np.uint32), np.asarray(shape["b"]).view(np.uint32)
    out = vertices.copy()
    first, count = int(a[0]), 2 * int(a[2]) + int(b[1])
    out[first:first + count, 1] += np.float32(by)
    return out


def state(data, st):
    return data.positions(st)[:, :3], data.kinematics(st)["velocity"]


@pytest.mark.parametrize("graph", [False, True])
def test_replaced_mesh_is_the_one_stepped_with(gpu_pipeline, graph):
    pl, st = gpu_pipeline
    sc = scenes.heightfield_test_scene(12)
    vtx, idx = sc.collision_vertices, sc.collision_indices
    high = raised(vtx, 0.02)
    step = (lambda d: pl.launch_steps_graph(d, 4, st)) if graph else (lambda d: [pl.launch_step(d, st) for _ in range(4)])
    data = P.MpmData.from_scene(pl, sc, collision_mesh=(high, idx))
    data.set_collision_mesh(vtx, idx)
    data.set_collision_mesh(high, idx)
    want = {}
    for key, mesh in (("low", vtx), ("high", high)):
        d = P.MpmData.from_scene(pl, sc, collision_mesh=(mesh, idx))
        step(d)
        d.check_errors(st)
        want[key] = state(d, st)
    assert rel_l2(want["low"][1], want["high"][1]) > 1.0e-3
    bad = idx.copy()
    bad[0] = 0
    with pytest.raises(_lib.SloshError):
        data.set_collision_mesh(vtx, bad)
    step(data)
    data.check_errors(st)
    for got, ref in zip(state(data, st), want["high"]):
        assert rel_l2(got, ref) <= 4.0e-5
