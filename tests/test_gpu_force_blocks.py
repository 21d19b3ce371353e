"""Fermion force kernels in 64-site blocks, in both work orders: XCD slabs, and the tiled order over (x, y) planes
that lattices take where it leaves at most one lane in eight idle; pole counts at the edges of the two-pole rounds."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu

# slabs: small planes, planes of 70 sites of a parity, odd extents; then tiles: eight full ones, one empty, of one
# and two rows, and planes of 63 and 60 sites, whose blocks are not full
SLABS = [(5, 3, 4, 4), (4, 6, 10, 14), (3, 9, 8, 16)]
TILES = [(2, 8, 8, 16), (2, 7, 8, 16), (3, 15, 8, 16), (3, 8, 9, 14), (2, 16, 10, 12)]
LATTICES = SLABS + TILES


def busy(dims):
    """share of the lanes that the tiled order (eight tiles along y, planes in blocks of 64 sites) keeps busy"""
    plane = dims[2] * dims[3] // 2
    return dims[0] * dims[1] * plane / (8 * dims[0] * -(-dims[1] // 8) * -(-plane // 64) * 64)


@pytest.mark.parametrize("dims", LATTICES)
def test_orders(dims):
    assert (busy(dims) >= 7 / 8) == (dims in TILES)


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
