"""Shifted BiCGStab: one and 32 shifts, check intervals of 1 and 3 steps (the scalar stages carry over from one
recorded group of steps to the next), vectors smaller than one workgroup and larger than the grid."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2, 4), (5, 4, 6, 8), (16, 16, 16, 32)])
@pytest.mark.parametrize("nshift,every", [(1, 3), (32, 1), (7, 10)])
@pytest.mark.parametrize("prec,acc,bar", [(clg.F64, 1e-10, 2e-10), (clg.F32, 1e-4, 1e-3)])
def test_residuals(dims, nshift, every, prec, acc, bar):
    two_am, shifts = 0.4, np.logspace(-3, 1, nshift)
    U, b = orc.gauge_random(dims, 0.3, 1), orc.ks_gaussian(dims, 2)
    with clg.Context(0) as ctx:
        g, f = clg.Field(ctx, clg.GAUGE, clg.F64, dims), clg.Field(ctx, clg.KS, clg.F64, dims, bc=orc.BC_FERMION)
        g.upload(U)
        f.upload(b)
        xs = [clg.Field(ctx, clg.KS, clg.F64, dims, bc=orc.BC_FERMION) for _ in shifts]
        p = clg.solver_params(kind=clg.KS, max_step=2000, deviation_step=every, accuracy=acc, absolute_accuracy=1)
        for _ in range(2):  # the second solve replays the recorded steps
            st, _ = clg.multishift_solve(ctx, p, xs, shifts, f, g, two_am, clg.EFO_F_DDdagger, clg.MS_BICGSTAB, prec)
            assert st == clg.OK
        for k in {0, nshift // 2, nshift - 1}:
            x = xs[k].download()
            r = orc.ks_op(dims, orc.BC_FERMION, two_am, U, x, orc.DDDAG) + shifts[k] * x - b
            # the recurrence's |s_k| < acc, plus its drift from the true residual: rounding of vectors of norm |b|
            drift = np.linalg.norm(b) * (1e-12 if prec == clg.F64 else 3e-5)
            assert np.linalg.norm(r) < bar + drift, (k, np.linalg.norm(r))
