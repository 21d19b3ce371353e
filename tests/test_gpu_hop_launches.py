"""The hop kernels in 64-site blocks: the direction-split form (one direction per wave, summed in LDS) of the
Wilson and the staggered hop, and the tiled order over (x, y) planes, on lattices whose planes leave partly
idle blocks, whose extents the tiles do not divide, or that are smaller than one block."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu

KAPPA = 0.1355
# planes of 8 (odd extents), 70 (a block and 6 lanes more), 64 (exactly one block) and 32 sites of a parity
LATTICES = [(5, 3, 4, 4), (4, 6, 10, 14), (9, 2, 8, 16), (2, 2, 8, 8)]
SPLIT = ["9,64,0", "9,64,8", "10,64,8", "9,64,20,1,1", "9,64,41", "10,64,80", "10,64,81,1,1"]
TILED = ["1,64,120", "2,64,141,1,1", "3,64,180", "4,64,121"]


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.fixture(scope="module")
def ctx():
    c = clg.Context(0)
    yield c
    c.close()


def put(ctx, kind, prec, dims, data):
    f = clg.Field(ctx, kind, prec, dims, bc=None if kind in (clg.GAUGE, clg.GAUGE12) else orc.BC_FERMION)
    f.upload(data)
    return f


@pytest.mark.parametrize("dims", LATTICES)
def test_wilson_launches(ctx, dims, monkeypatch):
    U, psi, chi = orc.gauge_random(dims, 0.3, 1), orc.wilson_gaussian(dims, 2), orc.wilson_gaussian(dims, 3)
    even = all(d % 2 == 0 for d in dims)
    for prec, links, bar in ((clg.F64, (clg.GAUGE, clg.F64), 1e-12), (clg.F64, (clg.GAUGE12, clg.F64), 1e-12),
                             (clg.F32, (clg.GAUGE, clg.F32), 1e-6), (clg.F32, (clg.GAUGE12, clg.F16), 3e-6),
                             (clg.F16, (clg.GAUGE12, clg.F16), 1.1e-3)):
        g, f, x = put(ctx, *links, dims, U), put(ctx, clg.WILSON, prec, dims, psi), put(ctx, clg.WILSON, prec, dims, chi)
        out = clg.Field(ctx, clg.WILSON, prec, dims, bc=orc.BC_FERMION)

        def results(launch):
            monkeypatch.setenv("CLG_TUNE_FORCE", launch)
            got = []
            for op in (clg.EFO_F_D, clg.EFO_F_Ddagger):
                out.zero()
                clg.wilson_apply(ctx, out, f, g, KAPPA, op)
                got.append(out.download())
            for dag in (False, True) if even else ():
                for a, b, xx in ((0.7 - 0.2j, 0.0, None), (-0.3, 0.5 + 0.1j, x.parity(clg.ODD))):
                    out.zero()
                    clg.wilson_hop(ctx, out.parity(clg.ODD), f.parity(clg.EVEN), g, dag, a, xx, b)
                    got.append(out.download())
            return got

        # FP64 and FP32 (same-precision links): D and D^dagger against the oracle; everything against one
        # site per thread in hardware order.  FP32 sums in another order differ by a few 2^-24 of the largest
        # term; FP16 storage rounds each to one unit of 2^-10 of the site's largest component at most
        ref = results("1,64,0")
        if links[1] == prec and prec != clg.F16:
            for got, op in zip(ref, (orc.D, orc.DDAG)):
                assert rel(got, orc.wilson_op(dims, orc.BC_FERMION, KAPPA, U, psi, op)) < bar
        for launch in SPLIT + TILED:
            for got, want in zip(results(launch), ref):
                assert rel(got, want) < bar, (launch, prec, links)


@pytest.mark.parametrize("dims", LATTICES)
def test_staggered_launches(ctx, dims, monkeypatch):
    U, chi, phi = orc.gauge_random(dims, 0.3, 1), orc.ks_gaussian(dims, 2), orc.ks_gaussian(dims, 3)
    even = all(d % 2 == 0 for d in dims)
    for prec, links, bar in ((clg.F64, (clg.GAUGE, clg.F64), 1e-12), (clg.F32, (clg.GAUGE12, clg.F32), 1e-6),
                             (clg.F32, (clg.GAUGE12, clg.F16), 3e-6), (clg.F16, (clg.GAUGE12, clg.F16), 1.1e-3)):
        g, f, x = put(ctx, *links, dims, U), put(ctx, clg.KS, prec, dims, chi), put(ctx, clg.KS, prec, dims, phi)
        out = clg.Field(ctx, clg.KS, prec, dims, bc=orc.BC_FERMION)

        def results(launch):
            monkeypatch.setenv("CLG_TUNE_FORCE_KS", launch)
            got = []
            for op in (clg.EFO_F_D, clg.EFO_F_Ddagger):
                out.zero()
                clg.ks_apply(ctx, out, f, g, 0.3, op, clg.EOCT_Complex, 0.8, -0.4)
                got.append(out.download())
            if even:
                for xx, b in ((None, 0.0), (x.parity(clg.EVEN), 0.6)):
                    out.zero()
                    clg.ks_hop(ctx, out.parity(clg.EVEN), f.parity(clg.ODD), g, -0.7, xx, b)
                    got.append(out.download())
            return got

        ref = results("64,0,2")
        if links[1] == prec and prec != clg.F16:
            for got, op in zip(ref, (orc.D, orc.DDAG)):
                assert rel(got, orc.ks_op(dims, orc.BC_FERMION, 0.3, U, chi, op, 3, 0.8, -0.4)) < bar
        for launch in ("64,0,9", "64,8,9", "64,20,9", "64,41,9", "64,80,9", "64,81,9"):
            for got, want in zip(results(launch), ref):
                assert rel(got, want) < bar, (launch, prec, links)
