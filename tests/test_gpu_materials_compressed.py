"""The Drucker-Prager projection (FP64 steps) of strongly compressed and stretched particles:
singular values down to 1e-6 of the largest, and gradients uniformly small or large, against
the return mapping in numpy FP64 on the same FP32 gradients (an SVD, whose absolute error of
1e-16 of the largest singular value leaves 1e-10 of the smallest one here).

Tolerances: a projected gradient is an FP32 number (a few round-offs of its largest entry,
3e-7), and its singular values are exponentials of strains that carry the cone's slope, which
the kernel takes from FP32 sine and divisions (five round-offs, 3e-7 of the slope's term)."""
import math

import numpy as np
import pytest

from slosh_amd import layouts as L
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from tests.test_gpu_materials import rotations

pytestmark = pytest.mark.gpu

N = 130


def gradients(kind, rng):
    one = np.ones(N)
    if kind == "flat":      # one direction crushed, the others nearly free
        s = np.stack([one, rng.uniform(0.8, 1.2, N), 10.0 ** rng.uniform(-6, -2, N)], 1)
    elif kind == "needle":  # two directions crushed
        s = np.stack([one, 10.0 ** rng.uniform(-4, -1, N), 10.0 ** rng.uniform(-4, -1, N)], 1)
    elif kind == "tiny":
        s = 10.0 ** rng.uniform(-8, -4, (N, 1)) * rng.uniform(0.5, 1.0, (N, 3))
    else:                   # stretched
        s = np.stack([10.0 ** rng.uniform(0.5, 2, N), one, 10.0 ** rng.uniform(-4, -1, N)], 1)
    return np.einsum("nij,nj,nkj->nik", rotations(rng, N), s, rotations(rng, N))


def project(f, state, h, lam, mu):
    """(F', state', the slope's share of gamma) of the return mapping (Klar et al. 2016)."""
    u, s, vt = np.linalg.svd(f)
    if np.linalg.det(f) <= 0.0:
        return None
    angle = h[0] + (h[1] * state[1] - h[3]) * math.exp(-h[2] * state[1])
    alpha = math.sqrt(2.0 / 3.0) * 2.0 * math.sin(angle) / (3.0 - math.sin(angle))
    strain = np.log(s) + state[2] / 3.0
    tr = strain.sum()
    dev = strain - tr / 3.0
    dn = np.linalg.norm(dev)
    slope = (3.0 * lam + 2.0 * mu) / (2.0 * mu) * tr * alpha
    if tr > 0.0:
        ns, hard, slope = np.ones(3), np.linalg.norm(strain), 0.0
    else:
        gamma = dn + slope
        if gamma <= 0.0:
            return None
        ns, hard = np.exp(strain - dev * gamma / dn), gamma
    logs = np.log(s).sum() - np.log(ns).sum()
    return (u * ns) @ vt, np.array([state[0] * math.exp(logs), state[1] + hard, state[2] + logs]), abs(slope)


@pytest.mark.parametrize("tag", [2, 3])
@pytest.mark.parametrize("kind", ["flat", "needle", "tiny", "stretched"])
def test_projection_of_extreme_gradients(gpu_pipeline, tag, kind):
    pl, st = gpu_pipeline
    dx, dt = np.float32(1.0 / 64), np.float32(1.0e-4)
    rng = np.random.RandomState(11)
    f = gradients(kind, rng).astype(np.float32)
    model = M.sand(5.0e4, 0.1, 25.0, neo_hookean=tag == 3)
    pos = rng.uniform(0.3, 0.7, (N, 3)).astype(np.float32)
    parts = M.particle_arrays(pos, dx / 4, 1000.0, model)
    if kind == "tiny":  # a log volume gain that has them in tension
        parts["models"][:, 3] = np.float32(64.0).view(np.uint32)
    parts["def_grad"] = L.mat_to_slang(f)
    bodies, mats = scenes.box_walls(M.STICK)
    sc = scenes.Scene("compressed", parts, dt, dx, 4096, bodies, mats, gravity=(0.0, 0.0, 0.0))
    data = P.MpmData.from_scene(pl, sc)
    pl.launch_step(data, st)
    data.check_errors(st)
    got_f, got_m, enabled = data.def_grad(st)[..., :3], data.models(st), data.kinematics(st)["enabled"]
    par = parts["models"][:, 1:].view(np.float32).astype(np.float64)
    projected = 0
    for i in range(N):
        want = project(f[i].astype(np.float64), par[i, 0:3], par[i, 3:7], par[i, 7], par[i, 8])
        if want is None:
            continue
        projected += 1
        want_f, want_s, slope = want
        assert enabled[i], (i, np.linalg.svd(f[i].astype(np.float64))[1])
        tol = 3.0e-7 * (1.0 + slope)
        assert np.abs(got_f[i] - want_f).max() <= tol * np.abs(want_f).max(), (i, got_f[i], want_f)
        state = got_m[i, 1:4].view(np.float32).astype(np.float64)
        assert np.abs(state - want_s).max() <= tol + 2.0e-6 * np.abs(want_s).max(), (i, state, want_s)
        assert abs(state[0] / want_s[0] - 1.0) <= 2.0e-6 + 2.0e-7 * abs(want_s[2]), (i, state, want_s)
    assert projected >= N // 2
