"""The partial-sum buffer of the reductions grows with the call; recorded graphs keep the one they were recorded with."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg

pytestmark = pytest.mark.gpu
DIMS = (8, 8, 8, 8)


def record(ctx, y, x, energy_of):
    """y += x, and the launches that a refused energy call leaves in an open recording"""
    clg.Graph.begin(ctx)
    clg.axpy(ctx, y, 1.0, x)
    with pytest.raises(clg.CLGError):
        clg.plaquette_energy(ctx, energy_of, 5.5)
    return clg.Graph.end(ctx)


def fields(ctx):
    x, y = (clg.Field(ctx, clg.WILSON, clg.F64, DIMS) for _ in range(2))
    x.gaussian(1)
    y.zero()
    return x, y


def test_replay_after_the_buffer_has_grown():
    with clg.Context(0) as ctx:
        g = clg.Field(ctx, clg.GAUGE, clg.F64, DIMS)
        g.gauge_random(0.4, 1)
        x, y = fields(ctx)
        graph = record(ctx, y, x, g)
        clg.gram_matrix(ctx, [x, x], [x])  # asks for a larger buffer than the recorded one
        # fields that would take the place of a freed one (2048 x 33 doubles)
        taken = [clg.Field(ctx, clg.WILSON, clg.F64, (4, 4, 4, 2 * n)) for n in (2, 4, 8, 11) for _ in range(4)]
        for f in taken:
            f.zero()
        for k in range(1, 4):
            graph.launch()
            ctx.sync()
            assert np.allclose(y.download(), k * x.download(), rtol=1e-15)
            assert clg.norm2(ctx, x) > 0  # eager reductions between replays
            assert all(not f.download().any() for f in taken), k
        graph.close()


def test_growth_while_recording():
    # more 64-site blocks (69120) than the buffer reserved when recording begins holds
    with clg.Context(0) as ctx:
        big = clg.Field(ctx, clg.GAUGE, clg.F64, (40, 48, 48, 48))
        big.gauge_unit()
        x, y = fields(ctx)
        graph = record(ctx, y, x, big)
        for k in range(1, 4):
            graph.launch()
            ctx.sync()
            assert np.allclose(y.download(), k * x.download(), rtol=1e-15)
            assert clg.plaquette_energy(ctx, big, 5.5) == 0.0
        graph.close()
