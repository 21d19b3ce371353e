"""Batched hops and solves of systems that share a gauge field but not the boundary signs of their spinors."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu
DIMS = (4, 6, 4, 8)
# anti-periodic in t, periodic, anti-periodic in x, and the first twice again
BCS = [(1, 1, 1, -1), (1, 1, 1, 1), (-1, 1, 1, 1), (1, 1, 1, -1), (1, 1, 1, -1)]


def put(ctx, kind, prec, data, bc=None):
    f = clg.Field(ctx, kind, prec, DIMS, bc=bc)
    f.upload(data)
    return f


@pytest.fixture(autouse=True)
def untuned():
    """the default launch takes two right-hand sides per thread; the tuner may settle on one"""
    clg.autotune_enable(0)
    yield
    clg.autotune_enable(-1)


@pytest.mark.parametrize("prec,tile", [(p, t) for p in (clg.F64, clg.F32, clg.F16) for t in (0, 1, 2, 4)
                                       if not (p == clg.F64 and t == 4)])
def test_hop(prec, tile):
    links = {clg.F64: (clg.GAUGE, clg.F64), clg.F32: (clg.GAUGE, clg.F32), clg.F16: (clg.GAUGE12, clg.F16)}[prec]
    with clg.Context(0) as ctx:
        g = put(ctx, *links, orc.gauge_random(DIMS, 0.3, 1))
        ins = [put(ctx, clg.WILSON, prec, orc.wilson_gaussian(DIMS, 2 + i), bc) for i, bc in enumerate(BCS)]
        outs = [clg.Field(ctx, clg.WILSON, prec, DIMS, bc=bc) for bc in BCS]
        clg.wilson_hop_batch(ctx, outs, ins, [g] * len(BCS), 0.7, tile=tile)
        got = [o.download() for o in outs]
        for i in range(len(BCS)):
            clg.wilson_hop_batch(ctx, outs[i:i + 1], ins[i:i + 1], [g], 0.7, tile=tile)
            want = outs[i].download()
            # the same sums per site; another tile size may contract them differently: a few units of the type
            err = np.abs(got[i] - want).max() / np.abs(want).max()
            assert err <= {clg.F64: 1e-14, clg.F32: 2e-6, clg.F16: 1.1e-3}[prec], (i, err)


@pytest.mark.parametrize("inner", [clg.F64, clg.F32, clg.INNER_F16_VECTORS])
def test_solve(inner):
    U, kappa, acc = orc.gauge_random(DIMS, 0.3, 1), 0.12, 1e-10
    bs = [orc.wilson_gaussian(DIMS, 2 + i) for i in range(len(BCS))]
    with clg.Context(0) as ctx:
        g = put(ctx, clg.GAUGE, clg.F64, U)
        xs = [clg.Field(ctx, clg.WILSON, clg.F64, DIMS, bc=bc) for bc in BCS]
        p = clg.solver_params(max_dim=10, restart=100, accuracy=acc, stop_rule=clg.STOP_TRUE_RESIDUAL, even_odd=1,
                              inner_prec=inner, inner_accuracy=1e-2, max_outer=60)
        fb = [put(ctx, clg.WILSON, clg.F64, b, bc) for b, bc in zip(bs, BCS)]
        st, _ = clg.solve_batch(ctx, p, xs, fb, [g] * len(BCS), kappa)
        assert st == clg.OK
        for i, (x, b, bc) in enumerate(zip(xs, bs, BCS)):
            r = orc.wilson_op(DIMS, bc, kappa, U, x.download()) - b
            assert np.linalg.norm(r) < 1.01 * acc * np.linalg.norm(b), i
