"""Device memory of readbacks: a scene's is gathered in buffers the data has, so reading
scenes takes none (a server fills its budget with particles and grid); a whole state's is
staged, in at most 64 MiB."""
import ctypes as C

import numpy as np
import pytest

from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_reading_scenes_takes_no_device_memory(gpu_pipeline):
    pl, st = gpu_pipeline
    n, dx = 1100000, 1.0 / 128
    pos = scenes.lattice((104,) * 3, dx / 2, (0.05, 0.05, 0.05), 0.1 * dx, 1)[:n]
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3))
    bodies, mats = scenes.box_walls(M.SLIP)
    sc = scenes.Scene("memory", parts, 1.0e-4, dx, 16384, bodies, mats)
    data = P.MpmData.from_scene(pl, sc, scene_ids=np.zeros(n, np.uint32))
    pl.launch_step(data, st)
    data.read_scene(0, st, positions_only=True)[0]  # (the stream's own first use)
    small = scenes.Scene("small", {k: v[:1000] for k, v in parts.items()}, 1.0e-4, dx, 16384, bodies, mats)
    one = P.MpmData.from_scene(pl, small, scene_ids=np.zeros(1000, np.uint32))
    one.positions(st)
    one.close()
    st.synchronize()
    before = free_bytes()
    again = P.MpmData.from_scene(pl, sc, scene_ids=np.zeros(n, np.uint32))
    pl.launch_step(again, st)
    st.synchronize()
    held = free_bytes()
    x, k, f = again.read_scene(0, st)
    assert free_bytes() == held
    assert np.array_equal(again.positions(st), x)
    assert np.array_equal(again.kinematics(st).view(np.uint8), k.view(np.uint8))
    assert 0 <= held - free_bytes() <= 72 << 20  # the 64 MiB staging and its alignment
    again.close()
    assert abs(before - free_bytes()) <= 4 << 20
