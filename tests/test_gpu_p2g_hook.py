"""A program that does P2G itself (a run_p2g hook writing the grid's momenta through the
device view, with the built-in grid update or one of its own): the state after each of three
substeps is the oracle's (relative L2 1e-5 per substep), and the built-in G2P after it is
the fused one, which leaves the particles stored block by block. Clouds from one particle to
several items (64 particles) a block, uploaded in an order that has nothing to do with the
blocks."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from tests.parity import rel_l2

pytestmark = pytest.mark.gpu

DX = 1.0 / 64


class HostP2G(P.MpmPipelineHooks):
    """P2G in FP64 on the host; with `velocities`, the grid's velocities instead (no gravity
    and no collider in reach: what the grid update would make of the momenta)."""

    def __init__(self, stream, velocities):
        self.stream, self.velocities, self.sorted_blocks = stream, velocities, None
        self.hip = C.CDLL("libamdhip64.so")
        self.hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]

    def fetch(self, ptr, shape, dtype):
        a = np.empty(shape, dtype)
        assert self.hip.hipMemcpy(a.ctypes.data, ptr, a.nbytes, 2) == 0
        return a

    def run_p2g(self, data, stream):
        blocks = data.blocks(self.stream)  # waits for the sort
        v = data.device_view()
        n, cap = int(v.num_particles), int(v.particle_capacity)
        x = self.fetch(v.positions, (n, 4), np.float32)[:, :3].astype(np.float64)
        vm = self.fetch(v.vel_mass, (n, 4), np.float32).astype(np.float64)
        c = self.fetch(v.affine, (9, cap), np.float32)[:, :n].T.reshape(n, 3, 3).astype(np.float64)
        hids = self.fetch(v.block_list, len(blocks), np.uint32)
        slot = {tuple(b["vid"]): int(h) for b, h in zip(blocks, hids)}
        grid = np.zeros((int(v.grid_capacity) * 64, 4))
        cell = np.rint(x / DX) - 1
        t = (x - cell * DX) / DX
        w = np.stack([0.5 * (1.5 - t) ** 2, 0.75 - (t - 1) ** 2, 0.5 * (t - 0.5) ** 2], 2)
        for i in range(3):
            for j in range(3):
                for k in range(3):
                    node = cell + (i, j, k)
                    d = node * DX - x
                    wt = w[:, 0, i] * w[:, 1, j] * w[:, 2, k]
                    mom = vm[:, :3] * vm[:, 3:] + np.einsum("na,nac->nc", d, c)
                    b = np.floor(node / 4).astype(int)
                    at = (node - 4 * b).astype(int)
                    idx = [slot[tuple(q)] * 64 + a[0] + 4 * a[1] + 16 * a[2] for q, a in zip(b, at)]
                    np.add.at(grid, idx, np.concatenate([mom, vm[:, 3:]], 1) * wt[:, None])
        if self.velocities:
            grid[:, :3] /= np.maximum(grid[:, 3:], 1e-30)
        g = grid.astype(np.float32)
        assert self.hip.hipMemcpy(v.nodes, g.ctypes.data, g.nbytes, 1) == 0
        return True


def blocks_in_storage(hook, data):
    v = data.device_view()
    ids = hook.fetch(v.particle_ids, int(v.num_particles), np.uint32)
    return ids


@pytest.mark.parametrize("grid_update", [True, False])
@pytest.mark.parametrize("n,side", [(1, 1.0), (64, 1.0), (65, 1.0), (900, 2.0), (1500, 1.0)])
def test_hooked_p2g_matches_oracle_and_keeps_blocks_together(gpu_pipeline, n, side, grid_update):
    _, st = gpu_pipeline
    pl = P.MpmPipeline(P.MpmPipelineKernels(grid_update=grid_update))
    rng = np.random.RandomState(n)
    pos = (0.5 + 0.6 * DX + rng.uniform(0.0, side * 4 * DX, (n, 3))).astype(np.float32)
    vel = (rng.uniform(-0.1, 0.1, (n, 3)) * DX / 1.0e-4).astype(np.float32)
    parts = M.particle_arrays(pos, np.float32(DX / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3), vel)
    bodies, mats = scenes.box_walls(M.STICK)
    sc = scenes.Scene("p2g hook", parts, 1.0e-4, DX, 1024, bodies, mats, gravity=(0.0, 0.0, 0.0))
    data, orc = P.MpmData.from_scene(pl, sc), O.Oracle(sc)
    hook = HostP2G(st, not grid_update)
    for k in range(3):
        before = data.positions(st)[:, :3].astype(np.float64)
        pl.launch_step(data, st, hooks=hook)
        data.check_errors(st)
        orc.step(1)
        assert rel_l2(data.positions(st)[:, :3], orc.positions()[:, :3]) <= 1.0e-5 * (k + 1)
        assert rel_l2(data.kinematics(st)["velocity"], orc.kinematics()["velocity"]) <= 1.0e-5 * (k + 1)
        assert rel_l2(data.def_grad(st), orc.def_grad()) <= 1.0e-5 * (k + 1)
        block = np.floor((np.rint(before / DX) - 1) / 4).astype(int)[blocks_in_storage(hook, data)]
        runs = 1 + int((np.diff(block, axis=0) != 0).any(1).sum())
        assert runs == len(np.unique(block, axis=0)), "a block's particles lie apart"
