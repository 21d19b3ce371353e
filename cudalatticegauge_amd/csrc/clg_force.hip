// clg_force.hip -- HMC fermion forces and pseudofermion energies.
//
// Conventions (reference CIntegrator / CFieldGaugeSU3): momenta P are traceless anti-Hermitian,
// the kinetic energy is sum ReTr P^dagger P, P <- P + eps F and U <- exp(eps P) U.  A force F is
// therefore consistent with an action S when dS/deps = -2 Re sum Tr(F^dagger T) along U -> exp(eps T) U,
// which tests/test_oracle_forces.py checks by finite differences on the oracle.
//
// Wilson (CFieldFermionWilsonSquareSU3.cu:170-231, driver :1016-1100):
//   X = (D D^dagger)^-1 phi, Y = D^dagger X,
//   F_mu(x) += s kappa Ta[ U_mu(x) ( sum_s ((1-g_mu) Y(x+mu))_s X(x)_s^dagger + (X(x+mu))_s ((1+g_mu) Y(x))_s^dagger ) ]
// with s the boundary sign of the forward hop.
// Staggered (CFieldFermionKSSU3.cu:216-264, driver :412-497), over the MD rational poles:
//   phi_i = (D D^dagger + b_i)^-1 phi, d_i = D0 phi_i (massless),
//   F_mu(x) -= Ta[ a_i eta_mu(x) s ( (U phi_i(x+mu)) d_i(x)^dagger + phi_i(x) (U d_i(x+mu))^dagger ) ]
#include "clg_internal.h"
#include "clg_wilson_common.h"

#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

using namespace clg;
using namespace clgd;

namespace clg {
int blas_dot_dev(clg_context, const clg_field_s*, const clg_field_s*, double*);
int blas_norm2_dev(clg_context, const clg_field_s*, double*);
int fetch_doubles(clg_context, const double*, int, double*);
int wilson_full(clg_context, clg_field_s*, const clg_field_s*, const clg_field_s*, double, bool, double, double);
int ks_full(clg_context, clg_field_s*, const clg_field_s*, const clg_field_s*, double, bool, double, double);
}  // namespace clg

namespace {

typedef C2<double> cx;

// F(e) += f m, F read and written past L2: no other workgroup reads it
__device__ __forceinline__ void add_link(char* F, int Vh, unsigned e, const cx* m, double f) {
    cx cur[9];
    LinkIO<CLG_F64, 18>::load<true>(F, Vh, e, cur);
#pragma unroll
    for (int k = 0; k < 9; ++k) cur[k] = cx{cur[k].x + f * m[k].x, cur[k].y + f * m[k].y};
    LinkIO<CLG_F64, 18>::store<true>(F, Vh, e, cur);
}
// m += a b^dagger on colour vectors
__device__ __forceinline__ void outer_add(const cx* a, const cx* b, cx* m) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) cfmac(m[3 * i + j], b[j], a[i]);
}

// The force kernels run in 64-site blocks, wave mu of a workgroup on direction mu (clg::site_order): the
// site's own vectors, which all four waves read, come from L1, and there are four times the waves of one
// thread per site.

// half-spinor (1 + s g_mu) psi, rows 0 and 1
template <int MU, int SG>
__device__ __forceinline__ void load_half(const char* f, int Vh, int p, int h, cx* hh) {
    cx psi[12];
    WilsonIO<CLG_F64>::load(f, nullptr, Vh, (unsigned)(p * 12 * Vh + h), 0u, psi);
    project<MU, SG>(psi, hh);
}
// Wilson force kernel; X = (DD^dagger)^-1 phi, Y = D^dagger X, FULL FP64 fields.  (1 -+ g_mu) has rank 2 and is
// twice a projector, so the spin sum over four rows of ((1-g_mu) Y(x+mu)) X(x)^dagger is the sum over rows 0
// and 1 of both vectors' half-spinors, and the same for the other term: half the products, and 24 complex
// numbers a lane instead of 48.  Bound by HBM: measured at 32^3x16 215 us, 5.1 TB/s of the 1.1 GB compulsory
// bytes (one thread per site, four rows, everything through L2: 304 us).
template <int MU>
__device__ __forceinline__ void wilson_force_mu(const Geo& g, const Site& s, int p, int h, const char* X, const char* Y,
                                                const char* U, char* F, double kappa) {
    const int Vh = g.Vh;
    const Nbr n = fwd_nbr<MU>(g, s, p);
    const unsigned el = (unsigned)((p * 4 + MU) * 9 * Vh + h);
    cx a[6], b[6], mid[9], u[9], f[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) mid[k] = cx{0.0, 0.0};
    load_half<MU, 2>(Y, Vh, n.p, n.h, a);
    load_half<MU, 2>(X, Vh, p, h, b);
    outer_add(a, b, mid);
    outer_add(a + 3, b + 3, mid);
    load_half<MU, 0>(X, Vh, n.p, n.h, a);
    load_half<MU, 0>(Y, Vh, p, h, b);
    outer_add(a, b, mid);
    outer_add(a + 3, b + 3, mid);
    LinkIO<CLG_F64, 18>::load<true>(U, Vh, el, u);
    su3_mm(u, mid, f);
    su3_ta(f);
    add_link(F, Vh, el, f, n.sign < 0 ? -kappa : kappa);
}
__global__ __launch_bounds__(256) void k_wilson_force(Geo g, const char* X, const char* Y, const char* U, char* F,
                                                      double kappa, int tile_y) {
    const int mu = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int p, h;
    if (!order_site(g, tile_y, (int)threadIdx.x & 63, p, h)) return;
    const Site s = site_of(g, p, h);
    switch (mu) {
        case 0: wilson_force_mu<0>(g, s, p, h, X, Y, U, F, kappa); break;
        case 1: wilson_force_mu<1>(g, s, p, h, X, Y, U, F, kappa); break;
        case 2: wilson_force_mu<2>(g, s, p, h, X, Y, U, F, kappa); break;
        default: wilson_force_mu<3>(g, s, p, h, X, Y, U, F, kappa); break;
    }
}

// staggered force kernel over npole (phi_i, d_i) pairs with numerators a_i.  The link does not depend on the
// pole, and Ta[X^dagger] = -Ta[X], so the poles are summed first,
//   sum_i a_i Ta[ (U phi_i(x+mu)) d_i(x)^dagger + phi_i(x) (U d_i(x+mu))^dagger ] = Ta[ U M ],
//   M = sum_i a_i ( phi_i(x+mu) d_i(x)^dagger - d_i(x+mu) phi_i(x)^dagger ),
// and U and Ta are applied once: 144 instead of 210 FP64 operations per pole and link, half of them to keep what
// the sum over the poles rounds off, without which the error grows with their number.  Relative error (2-norm,
// against long double) at 1 / 5 / 12 / 32 poles of equal size: 1.4 / 1.4 / 1.4 / 1.4e-16, of one direction and sizes
// over two decades 1.4 / 1.3 / 1.2 / 1.2e-16; the whole expression per pole in turn 1.3 / 1.5 / 1.6 / 2.0 and
// 1.3 / 1.2 / 1.4 / 2.0e-16, numerators on the vectors and plain sums of both outer products 1.5 / 1.6 / 1.9 / 2.4
// and 1.5 / 1.8 / 2.2 / 3.1e-16.
// Bound by the loads in flight (184 VGPRs, two waves per SIMD) and by L2: the site's own vectors are read once
// per workgroup, two poles a round, through LDS (straight from L1/L2 by all four waves a third slower), the next
// round's in flight during this one.  Measured, us a launch among others: 24^3x8, 12 poles 132 -> 70; 12x10x14x16,
// 3 poles 29 -> 12; 19x21x15x18, 1 pole 43 -> 39 (one thread per site, the four directions and the whole expression
// per pole in turn before); plain sums take 69, 12 and 39.
// m += a t; lost takes what the sum rounds off (exact for |m| >= |a t|)
__device__ __forceinline__ void add_kept(double& m, double& lost, double a, double t) {
    const double y = fma(a, t, m);
    lost += fma(a, t, m - y);
    m = y;
}
struct PolePtrs {
    const char* phi[32];
    const char* d[32];
    double a[32];
};
__global__ __launch_bounds__(256) void k_ks_force(Geo g, PolePtrs pp, int npole, const char* U, char* F, int tile_y) {
    // two poles a round: own vectors [buffer][pole, phi or d][colour][site]
    __shared__ double2 own[2][4][3][64];
    const int mu = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int Vh = g.Vh;
    int p, h;
    const bool valid = order_site(g, tile_y, lane, p, h);
    if (!valid) {  // idle lanes follow along on a site
        p = 0;
        h = 0;
    }
    const Site s = site_of(g, p, h);
    Nbr n;
    int sum = 0;
    switch (mu) {
        case 0: n = fwd_nbr<0>(g, s, p); break;
        case 1: n = fwd_nbr<1>(g, s, p); sum = s.c[0]; break;
        case 2: n = fwd_nbr<2>(g, s, p); sum = s.c[0] + s.c[1]; break;
        default: n = fwd_nbr<3>(g, s, p); sum = s.c[0] + s.c[1] + s.c[2]; break;
    }
    const unsigned el = (unsigned)((p * 4 + mu) * 9 * Vh + h);
    const unsigned en = (unsigned)(n.p * 3 * Vh + n.h), ex = (unsigned)(p * 3 * Vh + h);
    cx m[9], lost[9], mine[3] = {};  // M, and what rounding dropped from its sum over the poles
#pragma unroll
    for (int k = 0; k < 9; ++k) m[k] = lost[k] = cx{0.0, 0.0};
    // wave w brings vector w & 1 of pole r + w / 2
    auto fetch = [&](int r) {
        const int rr = r + (mu >> 1);
        if (rr >= npole) return;
        KSIO<CLG_F64>::load((mu & 1) ? pp.d[rr] : pp.phi[rr], nullptr, Vh, ex, 0u, mine);
    };
    fetch(0);
    for (int r = 0, buf = 0; r < npole; r += 2, buf ^= 1) {
#pragma unroll
        for (int c = 0; c < 3; ++c) own[buf][mu][c][lane] = make_double2(mine[c].x, mine[c].y);
        cx phin[2][3], dn[2][3];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (i > 0 && r + i >= npole) continue;
            KSIO<CLG_F64>::load(pp.phi[r + i], nullptr, Vh, en, 0u, phin[i]);
            KSIO<CLG_F64>::load(pp.d[r + i], nullptr, Vh, en, 0u, dn[i]);
        }
        if (r + 2 < npole) fetch(r + 2);
        __syncthreads();  // one a round: the next one writes the other buffer
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (r + i < npole) {
                const double ai = pp.a[r + i];
                cx dx[3], nphix[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double2 v = own[buf][2 * i][c][lane], w = own[buf][2 * i + 1][c][lane];
                    nphix[c] = cx{-v.x, -v.y};
                    dx[c] = cx{w.x, w.y};
                }
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    cx t = cmulc(dx[k % 3], phin[i][k / 3]);
                    cfmac(t, nphix[k % 3], dn[i][k / 3]);
                    add_kept(m[k].x, lost[k].x, ai, t.x);
                    add_kept(m[k].y, lost[k].y, ai, t.y);
                }
            }
        }
    }
    if (!valid) return;
    cx u[9], f[9];
    LinkIO<CLG_F64, 18>::load<true>(U, Vh, el, u);
#pragma unroll
    for (int k = 0; k < 9; ++k) m[k] = cadd(m[k], lost[k]);
    su3_mm(u, m, f);
    su3_ta(f);
    add_link(F, Vh, el, f, ((sum & 1) != 0) == (n.sign < 0) ? -1.0 : 1.0);  // F -= eta sign f
}

int check_force_args(const clg_field_s* force, const clg_field_s* gauge) {
    CLG_CHECK_ARG(force && gauge, "null field");
    CLG_CHECK_ARG(force->kind == CLG_GAUGE && force->prec == CLG_F64, "force must be an FP64 18-real gauge-shaped field");
    CLG_CHECK_ARG(gauge->kind == CLG_GAUGE && gauge->prec == CLG_F64, "gauge must be the FP64 18-real field");
    return check_same_lattice(force, gauge);
}

}  // namespace

extern "C" {

int clg_wilson_force_kernel(clg_context ctx, clg_field force, clg_field gauge, clg_field inv_dddag, clg_field inv_d,
                            double kappa) {
    CLG_CHECK_ARG(ctx && inv_dddag && inv_d, "null argument");
    CLG_TRY(check_force_args(force, gauge));
    CLG_CHECK_ARG(inv_dddag->kind == CLG_WILSON && inv_d->kind == CLG_WILSON && inv_dddag->prec == CLG_F64 &&
                      inv_d->prec == CLG_F64 && inv_dddag->subset == CLG_FULL && inv_d->subset == CLG_FULL,
                  "need FULL FP64 Wilson fields");
    Geo g = make_geo(inv_dddag);
    (void)hipSetDevice(ctx->device);
    const SiteOrder o = site_order(g);
    k_wilson_force<<<o.grid, 256, 0, ctx->stream>>>(g, (const char*)inv_dddag->data, (const char*)inv_d->data,
                                                     (const char*)gauge->data, (char*)force->data, kappa, o.tile_y);
    CLG_HIP(hipGetLastError());
    return CLG_OK;
}

int clg_ks_force_kernel(clg_context ctx, clg_field force, clg_field gauge, const clg_field* phis, const clg_field* dphis,
                        const double* numerators, int npole) {
    CLG_CHECK_ARG(ctx && phis && dphis && numerators, "null argument");
    CLG_CHECK_ARG(npole >= 1 && npole <= 32, "npole must be in [1, 32]");
    CLG_TRY(check_force_args(force, gauge));
    PolePtrs pp;
    std::memset(&pp, 0, sizeof(pp));
    for (int r = 0; r < npole; ++r) {
        CLG_CHECK_ARG(phis[r] && dphis[r] && phis[r]->kind == CLG_KS && dphis[r]->kind == CLG_KS &&
                          phis[r]->prec == CLG_F64 && dphis[r]->prec == CLG_F64 && phis[r]->subset == CLG_FULL &&
                          dphis[r]->subset == CLG_FULL,
                      "pole fields must be FULL FP64 staggered fields");
        pp.phi[r] = (const char*)phis[r]->data;
        pp.d[r] = (const char*)dphis[r]->data;
        pp.a[r] = numerators[r];
    }
    Geo g = make_geo(phis[0]);
    (void)hipSetDevice(ctx->device);
    const SiteOrder o = site_order(g);
    k_ks_force<<<o.grid, 256, 0, ctx->stream>>>(g, pp, npole, (const char*)gauge->data, (char*)force->data, o.tile_y);
    CLG_HIP(hipGetLastError());
    return CLG_OK;
}

// CFieldFermionWilsonSquareSU3::CalculateForceS (CFieldFermionWilsonSquareSU3.cu:1016-1100):
// X = (DD^dagger)^-1 phi with the configured solver (start may be the cached previous X),
// Y = D^dagger X, F += kernel.  x_out (nullable) receives X for the caller's cache.
int clg_wilson_force(clg_context ctx, const clg_solver_params* params, clg_field force, clg_field phi, clg_field gauge,
                     double kappa, clg_field start, clg_field x_out, clg_solve_report* rep) {
    CLG_CHECK_ARG(ctx && params && phi, "null argument");
    CLG_TRY(check_force_args(force, gauge));
    (void)hipSetDevice(ctx->device);
    clg_field_s *X, *Y;
    CLG_TRY(scratch_field(ctx, phi, CLG_WILSON, CLG_F64, CLG_FULL, 200, &X));
    CLG_TRY(scratch_field(ctx, phi, CLG_WILSON, CLG_F64, CLG_FULL, 201, &Y));
    for (int i = 0; i < 4; ++i) { X->bc[i] = phi->bc[i]; Y->bc[i] = phi->bc[i]; }
    const int st = clg_solve(ctx, params, X, phi, gauge, kappa, EFO_F_InverseDDdagger, start, rep);
    if (st != CLG_OK && st != CLG_NOT_CONVERGED) return st;
    CLG_TRY(wilson_full(ctx, Y, X, gauge, kappa, true, 1.0, 0.0));
    CLG_TRY(clg_wilson_force_kernel(ctx, force, gauge, X, Y, kappa));
    if (x_out) CLG_TRY(clg_field_copy(x_out, X));
    return st;
}

// CFieldFermionKSSU3::CalculateForceS (CFieldFermionKSSU3.cu:412-497) with the MD rational
// coefficients [c, a_1..a_n, b_1..b_n]
int clg_ks_force(clg_context ctx, const clg_solver_params* params, int ms_kind, int prec, clg_field force, clg_field phi,
                 clg_field gauge, double two_am, const double* coeffs, int degree, clg_solve_report* rep) {
    CLG_CHECK_ARG(ctx && params && phi && coeffs, "null argument");
    CLG_CHECK_ARG(degree >= 1 && degree <= 32, "degree must be in [1, 32]");
    CLG_TRY(check_force_args(force, gauge));
    (void)hipSetDevice(ctx->device);
    std::vector<clg_field_s*> P(degree), Dp(degree);
    std::vector<double> sh(2 * degree), a(degree);
    for (int k = 0; k < degree; ++k) {
        CLG_TRY(scratch_field(ctx, phi, CLG_KS, CLG_F64, CLG_FULL, 6000 + k, &P[k]));
        CLG_TRY(scratch_field(ctx, phi, CLG_KS, CLG_F64, CLG_FULL, 7000 + k, &Dp[k]));
        for (int i = 0; i < 4; ++i) { P[k]->bc[i] = phi->bc[i]; Dp[k]->bc[i] = phi->bc[i]; }
        a[k] = coeffs[1 + k];
        sh[2 * k] = coeffs[1 + degree + k];
        sh[2 * k + 1] = 0.0;
    }
    std::vector<clg_field> xs(P.begin(), P.end());
    const int st = clg_multishift_solve(ctx, params, ms_kind, prec, xs.data(), sh.data(), degree, phi, gauge, two_am,
                                        EFO_F_DDdagger, rep);
    if (st != CLG_OK && st != CLG_NOT_CONVERGED) return st;
    for (int k = 0; k < degree; ++k) CLG_TRY(ks_full(ctx, Dp[k], P[k], gauge, 0.0, false, 1.0, 0.0));  // D0 phi_i
    std::vector<clg_field> ps(P.begin(), P.end()), ds(Dp.begin(), Dp.end());
    CLG_TRY(clg_ks_force_kernel(ctx, force, gauge, ps.data(), ds.data(), a.data(), degree));
    return st;
}

// CActionFermionWilsonNf2::Energy (CActionFermionWilsonNf2.cpp:53-68): |D^-1 phi|^2 = phi^dagger (DD^dagger)^-1 phi
int clg_wilson_pf_energy(clg_context ctx, const clg_solver_params* params, clg_field phi, clg_field gauge, double kappa,
                         double* energy, clg_solve_report* rep) {
    CLG_CHECK_ARG(ctx && params && phi && gauge && energy, "null argument");
    (void)hipSetDevice(ctx->device);
    clg_field_s* X;
    CLG_TRY(scratch_field(ctx, phi, CLG_WILSON, CLG_F64, CLG_FULL, 202, &X));
    for (int i = 0; i < 4; ++i) X->bc[i] = phi->bc[i];
    const int st = clg_solve(ctx, params, X, phi, gauge, kappa, EFO_F_InverseD, nullptr, rep);
    if (st != CLG_OK && st != CLG_NOT_CONVERGED) return st;
    CLG_TRY(blas_norm2_dev(ctx, X, ctx->red_result + 32));
    CLG_TRY(fetch_doubles(ctx, ctx->red_result + 32, 1, energy));
    return st;
}

// CActionFermionKS::Energy (CActionFermionKS.cpp:52-71): Re phi^dagger r_MD(DD^dagger) phi
int clg_ks_pf_energy(clg_context ctx, const clg_solver_params* params, int ms_kind, int prec, clg_field phi,
                     clg_field gauge, double two_am, const double* coeffs, int degree, double* energy,
                     clg_solve_report* rep) {
    CLG_CHECK_ARG(ctx && params && phi && gauge && coeffs && energy, "null argument");
    (void)hipSetDevice(ctx->device);
    clg_field_s* T;
    CLG_TRY(scratch_field(ctx, phi, CLG_KS, CLG_F64, CLG_FULL, 203, &T));
    for (int i = 0; i < 4; ++i) T->bc[i] = phi->bc[i];
    const int st = clg_rational_apply(ctx, params, ms_kind, prec, T, phi, gauge, two_am, EFO_F_DDdagger, coeffs, degree,
                                      rep);
    if (st != CLG_OK && st != CLG_NOT_CONVERGED) return st;
    CLG_TRY(blas_dot_dev(ctx, T, phi, ctx->red_result + 32));
    double z[2];
    CLG_TRY(fetch_doubles(ctx, ctx->red_result + 32, 2, z));
    *energy = z[0];
    return st;
}

}  // extern "C"
