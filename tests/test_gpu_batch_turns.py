"""Batched hops whose segments of one gauge field take turns workgroup by workgroup: every system as a launch of its
own gives it (with one right-hand side per thread bit for bit: a site's sum does not depend on the order of the
sites), for one to several segments per gauge field, gauge fields in mixed order, lattices that end in part of a
workgroup, and different coefficients."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu
A, B, ODD = (6, 4, 10, 14), (4, 4, 4, 4), (5, 3, 7, 4)


@pytest.mark.parametrize("lattices", [[A], [A] * 5, [A, B] * 4 + [A] * 2, [ODD] * 3 + [B] * 13])
@pytest.mark.parametrize("prec", [clg.F64, clg.F32, clg.F16])
def test_turns(lattices, prec):
    ctx = clg.Context(0)
    links = {clg.F64: (clg.GAUGE, clg.F64), clg.F32: (clg.GAUGE, clg.F32), clg.F16: (clg.GAUGE12, clg.F16)}[prec]
    gauges, fields = {}, []

    def put(kind, p, dims, data):
        f = clg.Field(ctx, kind, p, dims, bc=orc.BC_FERMION if kind == clg.WILSON else None)
        f.upload(data)
        return f

    for dims in set(lattices):
        gauges[dims] = put(*links, dims, orc.gauge_random(dims, 0.3, 1))
    for i, dims in enumerate(lattices):
        fields.append([put(clg.WILSON, prec, dims, orc.wilson_gaussian(dims, 2 * i + k)) for k in (0, 1)]
                      + [clg.Field(ctx, clg.WILSON, prec, dims, bc=orc.BC_FERMION)])
    ins, xs, outs = ([f[k] for f in fields] for k in range(3))
    gs = [gauges[d] for d in lattices]
    for coef in ([0.7] * len(ins), [0.7 if i % 3 else 0.4 for i in range(len(ins))]):
        for x in (None, xs):
            want = []
            for i in range(len(ins)):
                clg.wilson_hop_batch(ctx, outs[i:i + 1], ins[i:i + 1], gs[i:i + 1], coef[i:i + 1],
                                     xs=x and x[i:i + 1], b=0.3, tile=1)
                want.append(outs[i].download())
            for tile in (1, 2) if prec == clg.F64 else (1, 2, 4):
                for o in outs:
                    o.zero()
                clg.wilson_hop_batch(ctx, outs, ins, gs, coef, xs=x, b=0.3, tile=tile)
                for i, o in enumerate(outs):
                    err = np.abs(o.download() - want[i]).max() / np.abs(want[i]).max()
                    # the compiler may contract the sums of another tile size differently: a few units of the type
                    assert err <= {clg.F64: 1e-14, clg.F32: 2e-6, clg.F16: 1.1e-3}[prec], (i, tile, err)
                    assert tile != 1 or err == 0, (i, err)
    ctx.close()
