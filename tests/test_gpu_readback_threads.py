"""Host threads that read the same data at once, each on a stream of its own: positions,
kinematics, deformation gradients and one scene of the batch, of a size whose readbacks go
through the staging in one piece and one that takes several (1 MiB each), every result the
bits of a lone readback. Records of three sizes share the staging, so that it also grows
under the other readers."""
import threading

import numpy as np
import pytest

from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [700, 150001])
def test_threads_read_the_same_data(gpu_pipeline, n):
    pl, st = gpu_pipeline
    side = int(np.ceil(n ** (1.0 / 3.0)))
    dx = 1.0 / 128
    pos = scenes.lattice((side,) * 3, dx / 2, (0.05, 0.05, 0.05), 0.1 * dx, n)[:n]
    vel = np.random.RandomState(n).uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    parts = M.particle_arrays(pos, np.float32(dx / 4), 1000.0, M.elastic_neo_hookean(1.0e5, 0.3), vel)
    bodies, mats = scenes.box_walls(M.SLIP)
    sc = scenes.Scene("threads", parts, 1.0e-4, dx, 16384, bodies, mats)
    one = P.MpmData.from_scene(pl, sc, scene_ids=(np.arange(n) >= n // 3).astype(np.uint32))
    for _ in range(2):
        pl.launch_step(one, st)
    one.check_errors(st)
    st.synchronize()
    twin = {"positions": one.positions(st), "kinematics": one.kinematics(st), "def_grad": one.def_grad(st)}
    twin["scene"] = one.read_scene(1, st, positions_only=True)
    # The same state again, whose staging is not yet made when the threads begin.
    parts2 = dict(parts, pos4=np.concatenate([twin["positions"][:, :3], np.zeros((n, 1), np.float32)], 1),
                  kin=twin["kinematics"], def_grad=twin["def_grad"])
    data = P.MpmData(pl, sc.params, parts2, bodies, mats, dx, 16384, scene_ids=(np.arange(n) >= n // 3).astype(np.uint32))
    reads = {"positions": lambda s: data.positions(s), "def_grad": lambda s: data.def_grad(s),
             "kinematics": lambda s: data.kinematics(s), "scene": lambda s: data.read_scene(1, s, positions_only=True)}
    start, wrong = threading.Barrier(len(reads)), []

    def work(kind):
        mine = P.Stream()
        start.wait()
        try:
            for k in range(25):
                if not np.array_equal(reads[kind](mine).view(np.uint8), twin[kind].view(np.uint8)):
                    wrong.append((kind, k))
        finally:
            mine.close()

    workers = [threading.Thread(target=work, args=(kind,)) for kind in reads]
    for w in workers:
        w.start()
    for w in workers:
        w.join()
    assert not wrong, wrong
