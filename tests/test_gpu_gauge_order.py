"""Gauge force and plaquette energy in 64-site blocks, in both work orders: XCD slabs, and the tiled order over
(x, y) planes that lattices take where it leaves at most one lane in eight idle."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu


# small planes, planes of 70 sites of a parity, odd extents, tiles far from full
SLABS = [(5, 3, 4, 4), (4, 6, 10, 14), (3, 9, 8, 16), (2, 2, 16, 8), (2, 11, 8, 16)]
# eight full tiles; one tile empty; tiles of one and two rows; planes of 63 and 60 sites, whose blocks are not full
TILES = [(2, 8, 8, 16), (2, 7, 8, 16), (3, 15, 8, 16), (3, 8, 9, 14), (2, 16, 10, 12)]


def busy(dims):
    """share of the lanes that the tiled order (eight tiles along y, planes in blocks of 64 sites) keeps busy"""
    plane = dims[2] * dims[3] // 2
    return dims[0] * dims[1] * plane / (8 * dims[0] * -(-dims[1] // 8) * -(-plane // 64) * 64)


@pytest.mark.parametrize("dims", SLABS + TILES)
def test_force_and_energy(dims):
    assert (busy(dims) >= 7 / 8) == (dims in TILES)
    U = orc.gauge_random(dims, 0.4, 1)
    rng = np.random.default_rng(2)
    F0 = rng.standard_normal(U.size)
    with clg.Context(0) as ctx:
        g, f = (clg.Field(ctx, clg.GAUGE, clg.F64, dims) for _ in range(2))
        g.upload(U)
        f.upload(F0)
        clg.gauge_force(ctx, f, g, 5.5)
        want = F0 + orc.gauge_force(dims, U, 5.5)
        # sums of 6 products of 4 unitary matrices in FP64: some tens of 2^-53 of the largest entry
        assert np.abs(f.download() - want).max() < 1e-13 * np.abs(want).max()
        e = 5.5 / 3 * orc.plaquette_sum(dims, U)
        assert abs(clg.plaquette_energy(ctx, g, 5.5) - e) < 1e-12 * abs(e)
