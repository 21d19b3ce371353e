"""GMRES on both sides of the size up to which the Gram-Schmidt passes total the projections themselves, through
the fast form (Wilson D, whose steps run on 1 - D) and the general one without and with its second pass (staggered D
of a small and a large mass), and Krylov dimensions at the edges of the least-squares kernel."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu

# 49152, 65520 and 73728 complex numbers of a spinor: up to 65536 packets (a complex number in FP64, two in FP32) the
# passes run one packet a lane, beyond that 256 workgroups take several
LATTICES = [(8, 8, 8, 8), (5, 6, 13, 14), (8, 8, 8, 12)]


def put(ctx, kind, prec, dims, data):
    f = clg.Field(ctx, kind, prec, dims, bc=None if kind == clg.GAUGE else orc.BC_FERMION)
    f.upload(data)
    return f


@pytest.fixture(scope="module")
def ctx():
    c = clg.Context(0)
    yield c
    c.close()


# both sides of 262144 packets, up to which a pass has 256 workgroups and the next one totals their partials
EDGES = {(clg.WILSON, clg.F64): [(12, 12, 12, 12), (12, 12, 12, 14)],
         (clg.WILSON, clg.F32): [(24, 12, 12, 12), (24, 12, 12, 14)],
         (clg.KS, clg.F64): [(16, 16, 18, 18), (16, 16, 18, 20)],
         (clg.KS, clg.F32): [(20, 20, 20, 20), (20, 20, 20, 24)]}
ACCURACY = {clg.F64: 1e-11, clg.F32: 2e-6}
# kind, kappa or 2am, operator; the last one's steps keep about 8 / (100 + 8) of |A v|^2 and take the second pass
SYSTEMS = [(clg.WILSON, 0.13, clg.EFO_F_D, orc.D), (clg.WILSON, 0.05, clg.EFO_F_DDdagger, orc.DDDAG),
           (clg.KS, 1.5, clg.EFO_F_D, orc.D), (clg.KS, 10.0, clg.EFO_F_D, orc.D)]


def solves(ctx, dims, prec, systems):
    U, acc = orc.gauge_random(dims, 0.3, 1), ACCURACY[prec]
    g = put(ctx, clg.GAUGE, prec, dims, U)
    for kind, m, op, oop in systems:
        b = orc.wilson_gaussian(dims, 2) if kind == clg.WILSON else orc.ks_gaussian(dims, 4)
        apply = orc.wilson_op if kind == clg.WILSON else orc.ks_op
        x = clg.Field(ctx, kind, prec, dims, bc=orc.BC_FERMION)
        for max_dim in (1, 12, 16):
            p = clg.solver_params(kind=kind, max_dim=max_dim, restart=2000, accuracy=acc,
                                  stop_rule=clg.STOP_TRUE_RESIDUAL, even_odd=0)
            st, rep = clg.solve(ctx, p, x, put(ctx, kind, prec, dims, b), g, m, op)
            r = apply(dims, orc.BC_FERMION, m, U, x.download(), oop) - b
            res = np.linalg.norm(r) / np.linalg.norm(b)
            # the solver's own residual, plus the rounding of x and U to FP32 (2^-24 times |D||x|/|b| < 8)
            assert st == clg.OK and res < acc * 1.01 + (1e-6 if prec == clg.F32 else 1e-14), (kind, op, max_dim, res)


@pytest.mark.parametrize("dims", LATTICES)
@pytest.mark.parametrize("prec", [clg.F64, clg.F32])
def test_solves(ctx, dims, prec):
    solves(ctx, dims, prec, SYSTEMS)


@pytest.mark.parametrize("kind,prec", EDGES)
@pytest.mark.parametrize("side", [0, 1])
def test_merge_edge(ctx, kind, prec, side):
    dims = EDGES[kind, prec][side]
    packets = int(np.prod(dims)) * (12 if kind == clg.WILSON else 3) // (1 if prec == clg.F64 else 2)
    assert (packets > 262144) == (side == 1)
    solves(ctx, dims, prec, [s for s in SYSTEMS if s[0] == kind and s[2] == clg.EFO_F_D])


@pytest.mark.parametrize("max_dim", [17, 64])
def test_long_bases(ctx, max_dim):
    dims = (4, 4, 4, 6)
    U, b = orc.gauge_random(dims, 0.3, 1), orc.wilson_gaussian(dims, 2)
    g, x = put(ctx, clg.GAUGE, clg.F64, dims, U), clg.Field(ctx, clg.WILSON, clg.F64, dims, bc=orc.BC_FERMION)
    p = clg.solver_params(max_dim=max_dim, restart=20, accuracy=1e-11, stop_rule=clg.STOP_TRUE_RESIDUAL, even_odd=0)
    st, _ = clg.solve(ctx, p, x, put(ctx, clg.WILSON, clg.F64, dims, b), g, 0.13, clg.EFO_F_D)
    r = orc.wilson_op(dims, orc.BC_FERMION, 0.13, U, x.download()) - b
    assert st == clg.OK and np.linalg.norm(r) < 1.01e-11 * np.linalg.norm(b)


def repeats(rep, max_dim):
    """cycles run again in the general form, from the applications of the operator: max_dim a cycle and one for each
    residual between them (in mixed precision the outer ones take the place of the inner solves' first), one for the
    last, and max_dim for each repeat"""
    n, rest = divmod(rep.operator_applies - (max_dim + 1) * rep.cycles - 1, max_dim)
    assert rest == 0, rep.operator_applies
    return n


def gmres12(inner, eo):
    return clg.solver_params(max_dim=12, restart=50, accuracy=1e-10, stop_rule=clg.STOP_TRUE_RESIDUAL, even_odd=eo,
                             inner_prec=inner, inner_accuracy=1e-2, max_outer=60)


@pytest.mark.parametrize("inner", [clg.F64, clg.F32, clg.INNER_F16_VECTORS])
@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (16, 16, 16, 16)])
@pytest.mark.parametrize("noise", [0.0, 1e-12, 1e-3])
def test_refused_fast_steps(ctx, inner, dims, noise):
    """On the unit field a constant source spans an invariant subspace of D, and one with some noise nearly so: K V_j
    lies in the span of the basis after a few steps, the fast Gram-Schmidt step is refused and the cycle repeated in
    the general form, once a solve (without noise in every precision)."""
    g, b = clg.Field(ctx, clg.GAUGE, clg.F64, dims), clg.Field(ctx, clg.WILSON, clg.F64, dims, bc=(1, 1, 1, 1))
    g.gauge_unit()
    src = np.tile(np.arange(1, 25, dtype=float), int(np.prod(dims)))
    src += noise * np.random.default_rng(1).standard_normal(src.size)
    b.upload(src)
    x, r = (clg.Field(ctx, clg.WILSON, clg.F64, dims, bc=(1, 1, 1, 1)) for _ in range(2))
    for eo in (0, 1):
        st, rep = clg.solve(ctx, gmres12(inner, eo), x, b, g, 0.11, clg.EFO_F_D)
        assert repeats(rep, 12) in ((1,) if noise == 0 else (0, 1)), eo
        clg.wilson_apply(ctx, r, x, g, 0.11)
        clg.axpy(ctx, r, -1.0, b)
        res = np.sqrt(clg.norm2(ctx, r) / clg.norm2(ctx, b))
        assert st == clg.OK and res < 1e-10, (eo, rep.cycles, rep.true_residual, res)


@pytest.mark.parametrize("inner", [clg.F64, clg.F32, clg.INNER_F16_VECTORS])
def test_no_repeat_on_a_random_field(ctx, inner):
    dims = (8, 8, 8, 8)
    g, b, x = clg.Field(ctx, clg.GAUGE, clg.F64, dims), *(clg.Field(ctx, clg.WILSON, clg.F64, dims) for _ in range(2))
    g.gauge_random(0.4, 1)
    b.gaussian(2)
    for eo in (0, 1):
        st, rep = clg.solve(ctx, gmres12(inner, eo), x, b, g, 0.13, clg.EFO_F_D)
        assert st == clg.OK and rep.true_residual < 1e-10 and repeats(rep, 12) == 0, eo
