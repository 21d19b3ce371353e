"""Gauge force and plaquette energy in 64-site blocks, on lattices whose planes leave partly idle blocks (slab
order), fill them exactly (tiled order), or whose extents are odd, 2 or 1 tile short."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 3, 4, 4), (4, 6, 10, 14), (3, 9, 8, 16), (2, 2, 16, 8), (2, 11, 8, 16)])
def test_force_and_energy(dims):
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
