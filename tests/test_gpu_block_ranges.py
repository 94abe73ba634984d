"""Where a block's particles begin (first_particle), after substeps without hooks: the ranges
of the blocks with particles tile [0, n), in the order in which the particles are stored,
and a block without particles begins somewhere in [0, n] as well. Clouds whose blocks fall
into one region of the table, a few, and all of them, in memory that held other numbers."""
import ctypes as C

import numpy as np
import pytest

from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes

pytestmark = pytest.mark.gpu


def dirty_memory(nbytes, count):
    """Leaves `count` freed allocations of `nbytes` all ones for what is allocated next."""
    hip = C.CDLL("libamdhip64.so")
    ptrs = [C.c_void_p() for _ in range(count)]
    for p in ptrs:
        assert hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
        assert hip.hipMemset(p, 0xff, C.c_size_t(nbytes)) == 0
    for p in ptrs:
        assert hip.hipFree(p) == 0


@pytest.mark.parametrize("n,side,cap", [(1, 1.0, 16), (300, 2.0, 128), (9000, 4.0, 1024), (9000, 4.0, 65536)])
def test_block_ranges_tile_the_storage(gpu_pipeline, n, side, cap):
    pl, st = gpu_pipeline
    dx, dt = 1.0 / 64, 1.0e-4
    rng = np.random.RandomState(n)
    pos = (0.5 + rng.uniform(0.0, side * 4 * dx, (n, 3))).astype(np.float32)
    vel = (rng.uniform(-0.5, 0.5, (n, 3)) * dx / dt).astype(np.float32)
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3), vel)
    bodies, mats = scenes.box_walls(M.SLIP)
    sc = scenes.Scene("ranges", parts, dt, dx, cap, bodies, mats, gravity=(0.0, 0.0, 0.0))
    dirty_memory(4 * cap, 64)
    data = P.MpmData.from_scene(pl, sc)
    for run in (1, 1, 2, 5):
        for _ in range(run):
            pl.launch_step(data, st)
        data.check_errors(st)
        blocks = data.blocks(st)
        first, count = blocks["first_particle"].astype(np.int64), blocks["num_particles"].astype(np.int64)
        assert (count == 0).any() and ((first >= 0) & (first <= n)).all()
        order = np.argsort(first[count > 0])
        assert np.array_equal(first[count > 0][order], np.concatenate([[0], np.cumsum(count[count > 0][order])[:-1]]))
        assert count.sum() == n
