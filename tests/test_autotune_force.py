"""Every launch shape that the Wilson hop tuner can list can also be forced; shapes that no launch takes are refused.
No device is needed to set or clear one."""
import pytest

import cudalatticegauge_amd as clg

TILED = (20, 21, 40, 41, 80, 81)


@pytest.fixture(autouse=True)
def cleared():
    yield
    clg.autotune_force(0)


def test_listed_shapes():
    shapes = [(pin, block, xcd, spt) for pin in range(1, 9) for block in (64, 128, 256) for xcd in (0, 1, 8) + TILED
              for spt in (1, 2, 4)]
    shapes += [(pin, 64, xcd, spt) for pin in (9, 10) for xcd in (0, 8) + TILED for spt in (0, 1)]
    shapes += [(pin, 64, 100 + xcd, 1) for pin in (1, 2, 3, 4) for xcd in TILED]
    for shape in shapes:
        clg.autotune_force(*shape)


@pytest.mark.parametrize("shape", [(9, 256, 8, 1), (9, 64, 8, 2), (10, 64, 1, 1), (9, 64, 120, 1), (5, 64, 120, 1),
                                   (1, 128, 120, 1), (1, 64, 120, 2), (1, 64, 100, 1), (11, 64, 8, 1), (1, 64, 22, 1)])
def test_other_shapes(shape):
    with pytest.raises(clg.CLGError):
        clg.autotune_force(*shape)


@pytest.mark.gpu
def test_forced_launches_agree():
    dims = (4, 6, 10, 14)
    with clg.Context(0) as ctx:
        g = clg.Field(ctx, clg.GAUGE, clg.F64, dims)
        g.gauge_random(0.4, 1)
        x, y = (clg.Field(ctx, clg.WILSON, clg.F64, dims) for _ in range(2))
        x.gaussian(2)
        want = None
        for shape in ((1, 64, 0, 1), (9, 64, 0, 1), (10, 64, 81, 1), (4, 64, 181, 1)):
            clg.autotune_force(*shape)
            y.zero()
            clg.wilson_apply(ctx, y, x, g, 0.13)
            got = y.download()
            want = got if want is None else want
            # the eight terms of a site in another order
            assert abs(got - want).max() < 1e-14 * abs(want).max(), shape
