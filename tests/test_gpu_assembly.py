"""Assembly through staged element blocks (engine.hip, at most 32,768 elements) against the colour by
colour kernel, which the same mesh takes with one more, detached element.

Tolerance: both add the same at most eight element blocks per entry (at most 64 nodal terms per force
component) in other orders, with rounding below 64 eps of the largest of a row's values: 1e-13 of the
largest of all; FP32, rounded up to eight times in the coloured kernel: 1e-6."""
import numpy as np
import pytest

import neon_amd
from neon_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [(neon_amd.PRECISION_FP64, 1e-13), (neon_amd.PRECISION_MIXED, 1e-6)])
@pytest.mark.parametrize("model,params,scale", [(neon_amd.MODEL_NEOHOOKE, (10.0, 1.0), 0.01),
                                                (neon_amd.MODEL_MICROSPHERE_NONAFFINE | neon_amd.SPHERE_BO33,
                                                 (3.0, 1.0, 8.0, 2.0), 0.01),
                                                (neon_amd.MODEL_J2, (166666.0, 76923.0, 250.0, 2000.0), 1e-3),
                                                (neon_amd.MODEL_J2_DAMAGE, (111667.0, 51538.0, 85.0, 0.0), 1e-3)])
def test_staged_assembly_agrees_with_the_coloured(ctx, model, params, scale, precision, tol):
    X, conn, _ = problems.box_mesh(32, 32, 32, jitter=0.1)
    rng = np.random.default_rng(5)
    new = rng.permutation(len(X)).astype(np.int32)
    Xp = np.empty_like(X)
    Xp[new] = X
    conn = new[conn]
    u = scale * Xp[:, [1, 2, 0]] ** 2 + rng.uniform(-1, 1, X.shape) * scale / 320
    out = []
    for extra in (False, True):
        Xe, ce, ue = Xp, conn, u
        if extra:
            cube = Xp[conn[0]] - Xp[conn[0]].mean(0)
            Xe = np.vstack([Xp, cube + 5.0])
            ce = np.vstack([conn, len(Xp) + np.arange(8, dtype=np.int32)])
            ue = np.vstack([u, np.zeros((8, 3))])
        p = np.zeros((len(ce), 4))
        p[:, : len(params)] = params
        mesh = neon_amd.DeviceMesh(Xe, ce, p, model=model, context=ctx,
                                   damage=problems.DAMAGE_CONSTANTS if model == neon_amd.MODEL_J2_DAMAGE else None)
        mesh.set_displacement(ue.reshape(-1))
        mesh.update_internal_variables()
        mesh.assemble(precision)
        rp, _ = mesh.pattern()
        val, f = mesh.download()
        n = 3 * len(Xp)
        out.append((val[: rp[n]].copy(), f[:n].copy()))
        del mesh
    (k0, f0), (k1, f1) = out
    assert np.abs(k0 - k1).max() <= tol * np.abs(k1).max()
    assert np.abs(f0 - f1).max() <= 1e-13 * np.abs(f1).max()
