"""Readbacks of the particle state: the device writes the reference records in id order
and they come through pinned staging in pieces. After substeps that reorder the storage,
positions, kinematics and deformation gradients must be the very bits of the device
buffers at the particle's slot, at sizes around the kernel's workgroup, the pieces of a
copy (1 MiB) and the staging of a pass (64 MiB)."""
import ctypes as C

import numpy as np
import pytest

from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes

pytestmark = pytest.mark.gpu


def device_array(ptr, shape, dtype):
    a = np.empty(shape, dtype)
    hip = C.CDLL("libamdhip64.so")
    assert hip.hipMemcpy(C.c_void_p(a.ctypes.data), C.c_void_p(ptr), C.c_size_t(a.nbytes), 2) == 0
    return a


# 1 MiB holds 65536 positions, 10922 kinematics; 64 MiB 699050 kinematics.
@pytest.mark.parametrize("n", [1, 255, 257, 10923, 65537, 140003, 699051])
def test_readback_is_the_device_state_in_id_order(gpu_pipeline, n):
    pl, st = gpu_pipeline
    side = int(np.ceil(n ** (1.0 / 3.0)))
    dx = 1.0 / 128
    pos = scenes.lattice((side,) * 3, dx / 2, (0.25, 0.3, 0.25), 0.1 * dx, n)[:n]
    rng = np.random.RandomState(n)
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3),
                              rng.uniform(-20.0, 20.0, (n, 3)).astype(np.float32))
    parts["kin"]["force_dt"] = rng.uniform(-1.0e-9, 1.0e-9, (n, 3))
    bodies, mats = scenes.box_walls(M.SLIP)
    sc = scenes.Scene("readback", parts, 1.0e-4, dx, 32768, bodies, mats)
    data = P.MpmData.from_scene(pl, sc)
    assert np.array_equal(data.kinematics(st)["force_dt"], parts["kin"]["force_dt"])
    for _ in range(3):
        pl.launch_step(data, st)
    data.check_errors(st)
    got_x, got_k, got_f = data.positions(st), data.kinematics(st), data.def_grad(st)
    v = data.device_view()
    ids = device_array(v.particle_ids, n, np.uint32)
    assert np.array_equal(np.sort(ids), np.arange(n))
    x = device_array(v.positions, (n, 4), np.float32)
    vm = device_array(v.vel_mass, (n, 4), np.float32)
    aff = device_array(v.affine, (9, n), np.float32).T.reshape(n, 3, 3)
    f = device_array(v.def_grad, (9, n), np.float32).T.reshape(n, 3, 3)
    vgd = device_array(v.vel_grad_det, n, np.float32)
    assert np.array_equal(got_x[ids, :3], x[:, :3]) and not got_x[:, 3].any()
    assert np.array_equal(got_k["velocity"][ids], vm[:, :3]) and np.array_equal(got_k["mass"][ids], vm[:, 3])
    assert np.array_equal(got_k["affine"][ids][..., :3], aff) and not got_k["affine"][..., 3].any()
    assert np.array_equal(got_k["vel_grad_det"][ids], vgd) and not got_k["force_dt"].any()
    assert np.array_equal(got_k["enabled"][ids], x[:, 3].view(np.uint32) & 1)
    assert np.array_equal(got_f[ids][..., :3], f) and not got_f[..., 3].any()
