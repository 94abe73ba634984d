"""Small meshes whose leaves the grid update tests without a walk (at most 8192 BVH nodes,
every inner box holding what is below it), against the same mesh with one inner box a
micron short of its triangles, which is walked: few and many (above the 2048 that a block
shares) triangles in reach of a block, and a mesh over many blocks. Both must meet the
oracle after one substep at the parity gate, with bit-exact blocks."""
import numpy as np
import pytest

from oracle import oracle as O
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from slosh_amd import trimesh as TM
from tests.parity import assert_blocks_equal, state_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("short", [False, True])
@pytest.mark.parametrize("samples,extent", [(2, 0.3), (12, 0.03), (44, 0.03), (46, 0.03), (40, 0.4)])
def test_flat_and_walked_meshes_match_oracle(gpu_pipeline, samples, extent, short):
    pl, st = gpu_pipeline
    dx, side = 1.0 / 64, 14
    pos = scenes.lattice((side,) * 3, dx / 2, (0.5 - side * dx / 4,) * 3, 0.1 * dx, 5)
    vel = np.cross(np.array([0.7, -0.4, 1.1]), pos.astype(np.float64) - 0.5) - np.array([0.0, 1.0, 0.0])
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(3.0e4, 0.3), vel.astype(np.float32))
    bodies, mats = scenes.box_walls(M.SLIP)
    buf = TM.CollisionBuffers()
    i, j = np.meshgrid(np.arange(samples), np.arange(samples), indexing="ij")
    shape = TM.convert(*TM.heightfield(np.sin(i / 3.0) * np.cos(j / 2.5), (extent, 0.004, extent)), buf)
    bodies.append(M.body(shape, (0.51, 0.49, 0.5), M.quat_from_scaled_axis((0.05, 0.3, -0.04))))
    mats.append(M.boundary_condition(M.STICK))
    sc = scenes.Scene("flat_mesh", parts, 1.0e-4, dx, 1024, bodies, mats)
    sc.collision_vertices, sc.collision_indices = buf.vertex_array(), buf.index_array()
    if short and samples > 2:
        sc.collision_vertices[3, 0] -= np.float32(1.0e-6)  # the second node's upper corner
    data, orc = P.MpmData.from_scene(pl, sc), O.Oracle(sc)
    pl.launch_step(data, st)
    data.check_errors(st)
    orc.step(1)
    assert_blocks_equal(data.blocks(st), orc.blocks())
    errs = state_errors((data.positions(st), data.kinematics(st), data.def_grad(st)),
                        (orc.positions(), orc.kinematics(), orc.def_grad()), sc.particles["pos4"])
    assert errs["enabled_diff"] == 0
    for k in ("x", "v", "affine", "F"):
        assert errs[k] <= 1.0e-5, f"{k}: {errs[k]:.3e}"
