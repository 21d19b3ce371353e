"""Fermion force kernels in 64-site blocks: lattices whose planes leave partly idle blocks or fill them exactly,
odd extents, and pole counts at the edges of the two-pole rounds."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu

LATTICES = [(5, 3, 4, 4), (4, 6, 10, 14), (3, 9, 8, 16)]


def put(ctx, kind, dims, data):
    f = clg.Field(ctx, kind, clg.F64, dims, bc=None if kind == clg.GAUGE else orc.BC_FERMION)
    f.upload(data)
    return f


def close(got, want):
    # a few hundred FP64 products a link, in another order
    return np.abs(got - want).max() < 1e-13 * np.abs(want).max()


@pytest.mark.parametrize("dims", LATTICES)
def test_wilson(dims):
    U, x, y = orc.gauge_random(dims, 0.4, 1), orc.wilson_gaussian(dims, 2), orc.wilson_gaussian(dims, 3)
    F0 = np.random.default_rng(4).standard_normal(U.size)
    with clg.Context(0) as ctx:
        f = put(ctx, clg.GAUGE, dims, F0)
        clg.wilson_force_kernel(ctx, f, put(ctx, clg.GAUGE, dims, U), put(ctx, clg.WILSON, dims, x),
                                put(ctx, clg.WILSON, dims, y), 0.1355)
        assert close(f.download(), orc.wilson_force(dims, orc.BC_FERMION, 0.1355, U, y, x, F0.copy()))


@pytest.mark.parametrize("dims", LATTICES)
@pytest.mark.parametrize("poles", [1, 2, 3, 32])
def test_staggered(dims, poles):
    U = orc.gauge_random(dims, 0.4, 1)
    phis, ds = ([orc.ks_gaussian(dims, 10 * k + i) for k in range(poles)] for i in (2, 3))
    w = np.linspace(-0.4, 1.3, poles)
    F0 = np.random.default_rng(4).standard_normal(U.size)
    with clg.Context(0) as ctx:
        f = put(ctx, clg.GAUGE, dims, F0)
        clg.ks_force_kernel(ctx, f, put(ctx, clg.GAUGE, dims, U), [put(ctx, clg.KS, dims, v) for v in phis],
                            [put(ctx, clg.KS, dims, v) for v in ds], w)
        assert close(f.download(), orc.ks_force(dims, orc.BC_FERMION, U, phis, ds, w, F0.copy()))
