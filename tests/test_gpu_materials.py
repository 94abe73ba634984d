"""The SVD-based material steps (FP64 path) at chosen deformation gradients, against
the oracle's model_update: every material tag at rotations (exact and perturbed below
FP32 round-off), small and large strains, volume changes, repeated singular values and
non-positive determinants.

One substep of particles at rest without gravity leaves every deformation gradient as
given, so that the projected gradient, the plastic state and the stress (the affine
matrix over -V0 (4 / h^2) dt) are the material model's alone.

Tolerances: the results are FP32 numbers from FP64 steps, so a gradient may differ by a
few FP32 round-offs (6e-8) of its entries, and a stress by those of its own value plus
what round-off of the gradient is worth (6e-8 (lambda + 2 mu) per unit entry, several
entries each); plastic states carry the FP32 exponential and sine of the hardening rule.
"""
import numpy as np
import pytest

from slosh_amd import layouts as L
from slosh_amd import models as M
from slosh_amd import pipeline as P
from slosh_amd import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu

N = 70  # one wave and a remainder


def rotations(rng, n):
    q, r = np.linalg.qr(rng.randn(n, 3, 3))
    q = q * np.sign(np.einsum("nii->ni", r))[:, None, :]
    q[np.linalg.det(q) < 0, :, 0] *= -1
    return q


def gradients(kind, n):
    rng = np.random.RandomState(7)
    eye = np.eye(3)
    a = rng.randn(n, 3, 3)
    if kind == "identity":
        return np.broadcast_to(eye, (n, 3, 3)).copy()
    if kind == "tiny_rotation":  # antisymmetric parts far below the FP32 spacing of 1
        return eye + (a - a.transpose(0, 2, 1)) * 10.0 ** rng.uniform(-14, -6, (n, 1, 1))
    if kind == "rotation":
        return rotations(rng, n)
    if kind == "small":
        return rotations(rng, n) @ (eye + 10.0 ** rng.uniform(-6, -2, (n, 1, 1)) * a)
    if kind == "large":
        return rotations(rng, n) @ (eye + 0.15 * a)
    if kind == "volume":  # isotropic compression and expansion
        return rotations(rng, n) * rng.uniform(0.4, 1.6, (n, 1, 1))
    if kind == "repeated":  # two equal singular values
        s = np.stack([np.diag(v) for v in np.stack([rng.uniform(0.9, 1.1, n)] * 2 + [rng.uniform(0.5, 1.5, n)], 1)])
        return rotations(rng, n) @ s @ rotations(rng, n)
    assert kind == "inverted"
    f = rotations(rng, n) @ (eye + 0.1 * a)
    f[:, :, 0] *= -1
    return f


@pytest.mark.parametrize("tag", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", ["identity", "tiny_rotation", "rotation", "small", "large", "volume", "repeated",
                                  "inverted"])
def test_material_step_at_gradients(gpu_pipeline, tag, kind):
    pl, st = gpu_pipeline
    dx, dt = np.float32(1.0 / 64), np.float32(1.0e-4)
    f = gradients(kind, N).astype(np.float32)
    model = [M.elastic(2.0e4, 0.3), M.elastic_neo_hookean(3.0e4, 0.25), M.sand(5.0e4, 0.3, 30.0),
             M.sand(4.0e4, 0.35, 25.0, neo_hookean=True)][tag]
    pos = np.random.RandomState(3).uniform(0.3, 0.7, (N, 3)).astype(np.float32)
    parts = M.particle_arrays(pos, dx / 4, 1000.0, model)
    if tag >= 2:
        parts["models"][::3, 3] = np.float32(2.0e-3).view(np.uint32)  # a log volume gain
    parts["def_grad"] = L.mat_to_slang(f)
    bodies, mats = scenes.box_walls(M.STICK)
    sc = scenes.Scene("gradients", parts, dt, dx, 4096, bodies, mats, gravity=(0.0, 0.0, 0.0))
    data = P.MpmData.from_scene(pl, sc)
    pl.launch_step(data, st)
    data.check_errors(st)
    kin, got_f, got_m = data.kinematics(st), data.def_grad(st)[..., :3], data.models(st)
    if kind == "inverted":
        assert not kin["enabled"].any() and not kin["mass"].any()
        assert np.array_equal(got_f, np.broadcast_to(np.eye(3, dtype=np.float32), f.shape))
        assert not kin["affine"].any()
        return
    assert kin["enabled"].all()
    sk = float(parts["props"]["init_volume"][0]) * 4.0 / float(dx) ** 2 * float(dt)
    lam, mu = np.float32(model[10:12].view(np.float32) if tag >= 2 else model[1:3].view(np.float32))
    for i in range(N):
        m, want_f, want_s = O.model_update(parts["models"][i], f[i])
        size = max(1.0, np.abs(f[i]).max())
        assert np.abs(got_f[i] - want_f).max() <= 3.0e-7 * size, (i, got_f[i], want_f)
        tol = 2.0e-6 * np.abs(want_s).max() + 4.0e-7 * (lam + 2.0 * mu) * size ** 2
        stress = -kin["affine"][i][:, :3].astype(np.float64) / sk
        assert np.abs(stress - want_s).max() <= tol, (i, stress, want_s, tol)
        if tag >= 2:
            assert np.allclose(got_m[i, 1:4].view(np.float32), m[1:4].view(np.float32), rtol=2.0e-6, atol=1.0e-6)
