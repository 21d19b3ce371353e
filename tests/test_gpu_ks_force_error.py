"""The staggered force's error against long double does not grow with the number of poles."""
import numpy as np
import pytest

import cudalatticegauge_amd as clg
import orc

pytestmark = pytest.mark.gpu
DIMS = (5, 4, 6, 8)


def complex_of(values, *shape):
    v = values.astype(np.longdouble).reshape(*DIMS, *shape, 2)
    return v[..., 0] + 1j * v[..., 1]


def exact(U, phis, ds, a):
    """-sum_i a_i eta s Ta[(U phi_i(x+mu)) d_i(x)^dagger + phi_i(x) (U d_i(x+mu))^dagger] in long double"""
    u, at = complex_of(U, 4, 3, 3), np.indices(DIMS)
    out = np.zeros((*DIMS, 4, 3, 3), dtype=np.clongdouble)
    for mu in range(4):
        sign = np.where(at[mu] == DIMS[mu] - 1, orc.BC_FERMION[mu], 1) * (1 - 2 * (at[:mu].sum(axis=0) % 2))
        t = np.zeros((*DIMS, 3, 3), dtype=np.clongdouble)
        for phi, d, w in zip(phis, ds, a):
            phi, d = complex_of(phi, 3), complex_of(d, 3)
            up, ud = ((u[..., mu, :, :] * np.roll(v, -1, axis=mu)[..., None, :]).sum(-1) for v in (phi, d))
            t += w * (up[..., :, None] * d.conj()[..., None, :] + phi[..., :, None] * ud.conj()[..., None, :])
        t = (t - t.conj().swapaxes(-1, -2)) / 2
        t -= np.trace(t, axis1=-2, axis2=-1)[..., None, None] / 3 * np.eye(3)
        out[..., mu, :, :] = -sign[..., None, None] * t
    return np.stack([out.real, out.imag], -1).ravel()


@pytest.mark.parametrize("poles", [1, 2, 5, 12, 32])
@pytest.mark.parametrize("alike", [False, True])
def test_error(poles, alike):
    U = orc.gauge_random(DIMS, 0.4, 1)
    phis, ds = ([orc.ks_gaussian(DIMS, 100 * k + i) for i in range(poles)] for k in (1, 2))
    a = np.linspace(0.1, 1.0, poles)
    if alike:  # solutions of one source at growing shifts
        size = 1 / (0.05 + np.logspace(-4, 1, poles))
        phis, ds = ([s * (orc.ks_gaussian(DIMS, 98 + k) + 0.3 * v) for s, v in zip(size, vs)]
                    for k, vs in enumerate((phis, ds)))
        a = 0.01 * np.logspace(0, 2, poles)
    with clg.Context(0) as ctx:
        def put(kind, data):
            f = clg.Field(ctx, kind, clg.F64, DIMS, bc=None if kind == clg.GAUGE else orc.BC_FERMION)
            f.upload(data)
            return f
        f = clg.Field(ctx, clg.GAUGE, clg.F64, DIMS)
        f.zero()
        clg.ks_force_kernel(ctx, f, put(clg.GAUGE, U), [put(clg.KS, v) for v in phis], [put(clg.KS, v) for v in ds], a)
        want = exact(U, phis, ds, a)
        err = float(np.linalg.norm((f.download() - want).astype(float)) / np.linalg.norm(want.astype(float)))
        # the roundings of one product of 3x3 matrices (six terms an entry) and of Ta, each at most 2^-53 of a partial
        # sum: their mean square comes to about 1.3 of that unit, whatever the number of poles
        assert err < 1.6e-16, err
