"""Triangle-mesh colliders of growing density under one block: the grid update shares a
block's triangles between waves while they fit its candidate list (512 leaves in reach)
and its BVH levels (256 nodes), and walks the BVH per node beyond. Spheres of 80 to
20480 triangles, smaller than a block and spanning several, fixed and moving, against
the oracle after one substep (the parity gate) and with bit-exact blocks."""
import numpy as np
import pytest

from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from slosh_amd import trimesh as TM
from oracle import oracle as O
from tests.parity import assert_blocks_equal, state_errors

pytestmark = pytest.mark.gpu


def sphere_scene(subdivisions, radius, moving):
    dx, side = 1.0 / 64, 14
    pos = scenes.lattice((side,) * 3, dx / 2, (0.5 - side * dx / 4,) * 3, 0.1 * dx, 11)
    rel = pos.astype(np.float64) - 0.5
    vel = np.cross(np.array([0.9, -0.5, 1.3]), rel) - 1.5 * rel
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(3.0e4, 0.3),
                              vel.astype(np.float32))
    bodies, mats = scenes.box_walls(M.SLIP)
    buf = TM.CollisionBuffers()
    # A box first, so that the sphere's nodes do not start the shared buffers.
    bodies.append(M.body(TM.convert(*TM.box_mesh((0.03, 0.01, 0.02)), buf), (0.45, 0.47, 0.52),
                         M.quat_from_scaled_axis((0.3, 0.1, 0.6))))
    mats.append(M.boundary_condition(M.SEPARATE, 0.2))
    sphere = TM.convert(*TM.icosphere(radius, subdivisions), buf)
    bodies.append(M.body(sphere, (0.51, 0.5, 0.49), M.quat_from_scaled_axis((0.0, 0.4, 0.2)),
                         linvel=(0.1, 0.0, 0.05) if moving else (0, 0, 0), mass=0.4 if moving else None,
                         inv_inertia_diag=(800.0,) * 3 if moving else None))
    mats.append(M.boundary_condition(M.STICK))
    sc = scenes.Scene("mesh", parts, 1.0e-4, dx, 1024, bodies, mats)
    sc.collision_vertices, sc.collision_indices = buf.vertex_array(), buf.index_array()
    return sc


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("subdivisions,radius", [(1, 0.012), (2, 0.012), (3, 0.012), (4, 0.012), (3, 0.05), (5, 0.05)])
def test_dense_mesh_matches_oracle(gpu_pipeline, subdivisions, radius, moving):
    pl, st = gpu_pipeline
    sc = sphere_scene(subdivisions, radius, moving)
    data, orc = P.MpmData.from_scene(pl, sc), O.Oracle(sc)
    pl.launch_step(data, st)
    data.check_errors(st)
    orc.step(1)
    assert_blocks_equal(data.blocks(st), orc.blocks())
    errs = state_errors((data.positions(st), data.kinematics(st), data.def_grad(st)),
                        (orc.positions(), orc.kinematics(), orc.def_grad()), sc.particles["pos4"])
    print(errs)
    assert errs["enabled_diff"] == 0
    for k in ("x", "v", "affine", "F"):
        assert errs[k] <= 1.0e-5, f"{k}: {errs[k]:.3e}"
