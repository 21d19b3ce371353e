"""Krylov spaces that close after one vector: on the unit field D acts on a constant spinor field as a number.  The
basis then ends in zero vectors, whatever the rounding leaves of the next one (nothing, or noise), in the bases of up
to 64 vectors, the shifted solvers, the deflated and the batched solver as in the short single-system ones."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg

pytestmark = pytest.mark.gpu
DIMS, PERIODIC = (4, 4, 4, 4), (1, 1, 1, 1)


@pytest.fixture(scope="module")
def ctx():
    c = clg.Context(0)
    yield c
    c.close()


def unit(ctx):
    g = clg.Field(ctx, clg.GAUGE, clg.F64, DIMS)
    g.gauge_unit()
    return g


def spinor(ctx, site, even_only=False):
    """the same 24 numbers at every site (or every even one)"""
    v = np.tile(np.asarray(site, dtype=float), (int(np.prod(DIMS)), 1))
    if even_only:
        v[np.indices(DIMS).sum(axis=0).ravel() % 2 == 1] = 0
    f = clg.Field(ctx, clg.WILSON, clg.F64, DIMS, bc=PERIODIC)
    f.upload(v.ravel())
    return f


def empty(ctx):
    return clg.Field(ctx, clg.WILSON, clg.F64, DIMS, bc=PERIODIC)


def residual(ctx, x, b, g, kappa):
    r = empty(ctx)
    clg.wilson_apply(ctx, r, x, g, kappa)
    clg.axpy(ctx, r, -1.0, b)
    return np.sqrt(clg.norm2(ctx, r) / clg.norm2(ctx, b))


EXACT = [1.0, 0.0, 0.0, 1.0] + [0.0] * 20  # 256 equal terms in every sum: the next vector is exactly zero
NOISY = np.arange(1, 25)                   # rounding leaves something of it


@pytest.mark.parametrize("site", [EXACT, NOISY])
@pytest.mark.parametrize("inner", [clg.F64, clg.F32])
@pytest.mark.parametrize("max_dim", [4, 16, 17, 40])
def test_single(ctx, site, inner, max_dim):
    g = unit(ctx)
    for eo in (0, 1):
        b, x = spinor(ctx, site, even_only=eo == 1), empty(ctx)
        p = clg.solver_params(max_dim=max_dim, restart=20, accuracy=1e-12, stop_rule=clg.STOP_TRUE_RESIDUAL,
                              even_odd=eo, inner_prec=inner, inner_accuracy=1e-3, max_outer=20)
        st, _ = clg.solve(ctx, p, x, b, g, 0.0625, clg.EFO_F_D)
        res = residual(ctx, x, b, g, 0.0625)
        assert st == clg.OK and res < 1e-12, (eo, res)


@pytest.mark.parametrize("site", [EXACT, NOISY])
@pytest.mark.parametrize("inner", [clg.F64, clg.F32, clg.INNER_F16_VECTORS])
def test_batch(ctx, site, inner):
    g = unit(ctx)
    bs = [spinor(ctx, site, even_only=True), spinor(ctx, site)]
    xs = [empty(ctx) for _ in bs]
    p = clg.solver_params(max_dim=8, restart=20, accuracy=1e-12, stop_rule=clg.STOP_TRUE_RESIDUAL, even_odd=1,
                          inner_prec=inner, inner_accuracy=1e-2, max_outer=40)
    st, _ = clg.solve_batch(ctx, p, xs, bs, [g, g], 0.0625)
    res = [residual(ctx, x, b, g, 0.0625) for x, b in zip(xs, bs)]
    assert st == clg.OK and max(res) < 1e-12, res


@pytest.mark.parametrize("site", [EXACT, NOISY])
@pytest.mark.parametrize("solver", [clg.MS_FOM, clg.MS_GMRES])
def test_shifted(ctx, site, solver):
    g, b, kappa = unit(ctx), spinor(ctx, site), 0.0625
    shifts = [0.25, 0.5, 1.0]
    xs = [empty(ctx) for _ in shifts]
    p = clg.solver_params(kind=clg.WILSON, max_dim=20, restart=20, accuracy=1e-12, absolute_accuracy=0)
    st, _ = clg.multishift_solve(ctx, p, xs, shifts, b, g, kappa, clg.EFO_F_D, kind=solver)
    want = b.download()
    for s, x in zip(shifts, xs):
        # D b = (1 - 8 kappa) b, so x = b / (1/2 + s)
        err = np.abs(x.download() * (0.5 + s) - want).max() / np.abs(want).max()
        assert st == clg.OK and err < 1e-12, (s, err)


@pytest.mark.parametrize("site", [EXACT, NOISY])
@pytest.mark.parametrize("m_dim", [8, 24])
@pytest.mark.parametrize("deflate", [clg.DEFLATE_REV, clg.DEFLATE_HEV, clg.DEFLATE_SVD])
def test_deflated(ctx, site, m_dim, deflate):
    g, b, x = unit(ctx), spinor(ctx, site), empty(ctx)
    s = clg.Gcrodr(ctx, m_dim=m_dim, k_dim=4, restart=20, accuracy=1e-22, deflate=deflate)
    st, _ = s.solve(x, b, g, 0.0625, clg.EFO_F_D)
    res = residual(ctx, x, b, g, 0.0625)
    s.close()
    assert st == clg.OK and res < 1e-12, res
