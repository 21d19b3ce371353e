// clg_wilson.hip -- Wilson-square SU(3) hopping kernels (D, D^dagger, even-odd hops, Schur).
//
// Operator (reference _kernelDFermionWilsonSquareSU3, CFieldFermionWilsonSquareSU3.cu:32-163):
//   (D psi)(x) = psi(x) - kappa sum_mu [ (1-g_mu) U_mu(x) s+ psi(x+mu) + (1+g_mu) U_mu(x-mu)^dag s- psi(x-mu) ]
//   D^dagger = g5 D g5, i.e. the same sum with the two projectors exchanged.
// The reference applies full 4x4 gamma products to 4-spinors.  Here each hop is spin
// projected: (1 -+ g_mu) has rank 2, so psi(x+-mu) is projected to a 2-spinor, the link is
// applied to 2 colour vectors instead of 4, and the other two spin rows are rebuilt from
// the gamma table's phases: 1320 flops per site instead of ~2700.
//
// Chiral gamma table (GammaMatrix.h:447-475): (g_mu psi)[r] = i^z[r] psi[idx[r]].  For a
// projector (1 + s g_mu), s = +-1:  h_j = psi_j + s i^z_j psi_idx_j (j = 0,1) and the full
// 4-spinor is (h_0, h_1, s i^z_2 h_idx_2, s i^z_3 h_idx_3), because g_mu^2 = 1.
#include "clg_internal.h"
#include "clg_wilson_common.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <iterator>
#include <map>
#include <mutex>
#include <vector>

using namespace clg;
using namespace clgd;

namespace {

struct HopArgs {
    Geo g;
    const char* in;      // input field base (parity-0 block of a FULL field, or the half field)
    const float* inn;
    char* out;
    float* outn;
    const char* x;       // optional b*x term (same layout as out)
    const float* xn;
    const char* gauge;   // 8 (parity, mu) blocks
    int in_full, out_full;  // 1 if the field holds both parity blocks
    double ar, ai, br, bi;
    int pbase, nblk;     // output parities handled
    int xcd, pinter;     // work decomposition (clgd::map_site)
    int spt;             // logical blocks (sites per thread) per workgroup
    int tile_y, tile_ymaj;  // tiled plane schedule (clgd::tile_block) when tile_y > 0
    int nt_out;             // output written with the non-temporal policy
};

// Neighbour spinors come from the input field, or (STAGED, z and t only) from the copy of this
// (x,y) plane's other-parity sites in LDS: `st`/`stn` hold NPL planes of blockDim.x 16-byte chunks
// (and the FP16 site scales); the site with index h sits at local index h - hbase.

template <int MU, bool DAG, int PM, bool STAGED, typename R, class SIO, class LIO>
__device__ __forceinline__ void hop_mu(const HopArgs& a, const Site& s, int p, int h, C2<R>* acc, const char* st,
                                       const float* stn, int hbase) {
    C2<R> psi[12], hh[6], uh[6], u[9];
    const int Vh = a.g.Vh;
    constexpr bool LDS = STAGED && MU >= 2;
    // forward: (1 - g_mu) U_mu(x) psi(x+mu)  [dagger: (1 + g_mu)]
    {
        const Nbr n = fwd_nbr<MU>(a.g, s, p);
        const unsigned pe = a.in_full ? (unsigned)n.p : 0u;
        if constexpr (LDS)
            load_projected<SIO, MU, DAG ? 0 : 2>(st, stn, (int)blockDim.x, (unsigned)(n.h - hbase), (unsigned)(n.h - hbase), n.sign, psi, hh);
        else
            load_projected<SIO, MU, DAG ? 0 : 2>(a.in, a.inn, Vh, pe * SIO::NPL * Vh + n.h, pe * Vh + n.h, n.sign, psi, hh);
        LIO::template load<(PM >= 3)>(a.gauge, Vh, (unsigned)(p * 4 + MU) * LIO::NPL * Vh + h, u);
        su3_mv(u, hh, uh);
        su3_mv(u, hh + 3, uh + 3);
        reconstruct_add<MU, DAG ? 0 : 2>(acc, uh);
    }
    if constexpr (PM == 1 || PM == 3) pin_acc(acc);
    // backward: (1 + g_mu) U_mu(x-mu)^dag psi(x-mu)  [dagger: (1 - g_mu)]
    {
        const Nbr n = bwd_nbr<MU>(a.g, s, p);
        const unsigned pe = a.in_full ? (unsigned)n.p : 0u;
        if constexpr (LDS)
            load_projected<SIO, MU, DAG ? 2 : 0>(st, stn, (int)blockDim.x, (unsigned)(n.h - hbase), (unsigned)(n.h - hbase), n.sign, psi, hh);
        else
            load_projected<SIO, MU, DAG ? 2 : 0>(a.in, a.inn, Vh, pe * SIO::NPL * Vh + n.h, pe * Vh + n.h, n.sign, psi, hh);
        LIO::template load<(PM >= 3)>(a.gauge, Vh, (unsigned)(n.p * 4 + MU) * LIO::NPL * Vh + n.h, u);
        su3_mdv(u, hh, uh);
        su3_mdv(u, hh + 3, uh + 3);
        reconstruct_add<MU, DAG ? 2 : 0>(acc, uh);
    }
    if constexpr (PM >= 1) pin_acc(acc);
}

// PM 1..4: register pinning and link cache policy (hop_mu); PM 5..8: PM 1..4 with the z and t
// neighbours staged in LDS.  A staged launch needs one workgroup per (x,y) plane of
// one parity (blockDim = L2*L3/2, L3 even, no padded workgroups): a plane's z and t neighbours
// then all lie in the same plane of the other parity, which the workgroup copies into LDS with
// one coalesced read before any hop (stage_bytes of dynamic LDS).
template <typename R, int SP, int GP, int RECON, bool DAG, bool HASX, int PM>
__global__ __launch_bounds__(256) void k_wilson_hop(HopArgs a) {
    typedef WilsonIO<SP> SIO;
    typedef LinkIO<GP, RECON> LIO;
    constexpr bool STAGED = PM >= 5;
    constexpr int PMH = STAGED ? PM - 4 : PM;
    const unsigned lw = STAGED && a.tile_y > 0 ? tile_block(a.g, a.nblk, a.tile_y, a.tile_ymaj) : logical_wg(a.xcd);
    for (int vs = 0; vs < a.spt; ++vs) {
    int p, h;
    const bool valid = !STAGED && a.tile_y > 0
                           ? tile64_site(a.g, a.nblk, a.pbase, a.tile_y, a.tile_ymaj, (int)threadIdx.x, p, h)
                           : block_site(lw * (unsigned)a.spt + (unsigned)vs, a.g.Vh, a.nblk, a.pbase, a.pinter, p, h);
    const char* st = nullptr;
    const float* stn = nullptr;
    int hbase = 0;
    const unsigned po = a.out_full ? (unsigned)p : 0u;
    const unsigned eo = po * SIO::NPL * a.g.Vh + h, no = po * a.g.Vh + h;
    C2<R> xv[12];
    if constexpr (STAGED) {
        extern __shared__ uint4 stage[];
        const int B = (int)blockDim.x;
        float* stage_n = reinterpret_cast<float*>(stage + SIO::NPL * B);
        // padded blocks (xcd remap, spt) are whole: every lane of a workgroup agrees on valid,
        // and blocks past the end stay past it
        if (!valid) break;
        // a staged workgroup's own-parity sites have usually left L2 by the end of its hops (its
        // other reads all go to the stage or to other planes): read the x term first, in flight
        // together with the stage loads
        if constexpr (HASX) SIO::load(a.x, a.xn, a.g.Vh, eo, no, xv);
        hbase = h - (int)threadIdx.x;
        const unsigned pe = a.in_full ? (unsigned)(1 - p) : 0u;
#pragma unroll
        for (int k = 0; k < SIO::NPL; ++k) stage[k * B + threadIdx.x] = ldp<uint4>(a.in, a.g.Vh, k, pe * SIO::NPL * a.g.Vh + h);
        if constexpr (SIO::SCALED) stage_n[threadIdx.x] = a.inn[pe * a.g.Vh + h];
        __syncthreads();
        st = reinterpret_cast<const char*>(stage);
        stn = stage_n;
    } else {
        if (!valid) continue;
    }
    const Site s = site_of(a.g, p, h);
    C2<R> acc[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) acc[k] = cmk<R>(0, 0);
    hop_mu<0, DAG, PMH, STAGED, R, SIO, LIO>(a, s, p, h, acc, st, stn, hbase);
    hop_mu<1, DAG, PMH, STAGED, R, SIO, LIO>(a, s, p, h, acc, st, stn, hbase);
    hop_mu<2, DAG, PMH, STAGED, R, SIO, LIO>(a, s, p, h, acc, st, stn, hbase);
    hop_mu<3, DAG, PMH, STAGED, R, SIO, LIO>(a, s, p, h, acc, st, stn, hbase);
    const C2<R> ca = cmk<R>((R)a.ar, (R)a.ai);
    C2<R> o[12];
    if constexpr (HASX) {
        const C2<R> cb = cmk<R>((R)a.br, (R)a.bi);
        if constexpr (!STAGED) SIO::load(a.x, a.xn, a.g.Vh, eo, no, xv);
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            o[k] = cmul(cb, xv[k]);
            cfma(o[k], ca, acc[k]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 12; ++k) o[k] = cmul(ca, acc[k]);
    }
    if (a.nt_out) SIO::template store<R, true>(a.out, a.outn, a.g.Vh, eo, no, o);
    else SIO::store(a.out, a.outn, a.g.Vh, eo, no, o);
    if constexpr (STAGED) __syncthreads();  // the next block rewrites the stage
    }
}

// ---- direction-split form
// One site per thread walks a serial chain of eight dependent load-multiply groups, and a small lattice has
// less than a wave per SIMD to hide it.  Here a workgroup of 8 waves takes 64 sites, one direction (mu,
// forward or backward) per wave: the eight groups of a site run side by side, each wave leaves its
// link-multiplied half-spinor (6 complex numbers a site) in LDS, and after one barrier waves 0..2 sum 4
// spinor components each, rebuild the spin rows, add the x term and store.  All neighbours of a 64-site
// block are then requested within one workgroup at one time, so what they share is still in the CU's L1 and
// the XCD's L2: with the tiled order (tile64_site) it also leads on lattices that fill the chip.  Measured
// (us, one site per thread -> split): FP64 D 8^4 7.6 -> 5.0, 24^3x24 101 -> 66, 32^4 311 -> 256; FP32 D
// 24^3x48 95 -> 67; half hops FP64 16^4 11.7 -> 9.7, 32^4 154 -> 143 (non-temporal links), FP32 16^4 7.9 ->
// 5.9, 24^3x48 49 -> 38; FP16 storage, D 12^4 7.3 -> 4.5, half hops 16^4 6.7 -> 4.7, 24^3x16 11.3 -> 10.7.  It
// loses where one thread per site is already bound by memory with little state: FP16 storage on larger lattices
// (half hop 32^3x16 18.6 against 22.0, 32^4 33 against 40; D from 16^3x32 on, 11.5 against 11.8), and is level
// with the staged launches for FP64 D at 32^3x16 (122 against 124).  The tuner times both.
constexpr int kSplitSites = 64;

// U h (forward) or U^dagger h (backward) of the neighbour in direction MU
template <int MU, bool FWD, bool DAG, bool NTL, typename R, class SIO, class LIO>
__device__ __forceinline__ void split_dir(const HopArgs& a, const Site& s, int p, int h, C2<R>* uh) {
    C2<R> psi[12], hh[6], u[9];
    const int Vh = a.g.Vh;
    const Nbr n = FWD ? fwd_nbr<MU>(a.g, s, p) : bwd_nbr<MU>(a.g, s, p);
    const unsigned pe = a.in_full ? (unsigned)n.p : 0u;
    load_projected<SIO, MU, FWD != DAG ? 2 : 0>(a.in, a.inn, Vh, pe * SIO::NPL * Vh + n.h, pe * Vh + n.h, n.sign, psi, hh);
    if constexpr (FWD) {
        LIO::template load<NTL>(a.gauge, Vh, (unsigned)(p * 4 + MU) * LIO::NPL * Vh + h, u);
        su3_mv(u, hh, uh);
        su3_mv(u, hh + 3, uh + 3);
    } else {
        LIO::template load<NTL>(a.gauge, Vh, (unsigned)(n.p * 4 + MU) * LIO::NPL * Vh + n.h, u);
        su3_mdv(u, hh, uh);
        su3_mdv(u, hh + 3, uh + 3);
    }
}
// spinor component K (spin K / 3, colour K % 3) of the hop in one direction, from its half-spinor in LDS
template <int MU, int SG, int K, typename R>
__device__ __forceinline__ C2<R> split_term(const C2<R>* half, int lane) {
    constexpr int S = K / 3, C = K % 3;
    constexpr int row = S == 2 ? G<MU, 2>::idx : S == 3 ? G<MU, 3>::idx : S;
    constexpr int z = S == 2 ? G<MU, 2>::z + SG : S == 3 ? G<MU, 3>::z + SG : 0;
    return mulz4<z>(half[(row * 3 + C) * kSplitSites + lane]);
}
template <int K, bool DAG, typename R>
__device__ __forceinline__ C2<R> split_sum(const C2<R>* sm, int lane) {
    constexpr int F = DAG ? 0 : 2, B = DAG ? 2 : 0, D = 6 * kSplitSites;
    C2<R> v = split_term<0, F, K>(sm, lane);
    v = cadd(v, split_term<0, B, K>(sm + D, lane));
    v = cadd(v, split_term<1, F, K>(sm + 2 * D, lane));
    v = cadd(v, split_term<1, B, K>(sm + 3 * D, lane));
    v = cadd(v, split_term<2, F, K>(sm + 4 * D, lane));
    v = cadd(v, split_term<2, B, K>(sm + 5 * D, lane));
    v = cadd(v, split_term<3, F, K>(sm + 6 * D, lane));
    return cadd(v, split_term<3, B, K>(sm + 7 * D, lane));
}
template <int W, bool DAG, typename R>
__device__ __forceinline__ void split_sum4(const C2<R>* sm, int lane, C2<R>* v) {
    v[0] = split_sum<4 * W, DAG>(sm, lane);
    v[1] = split_sum<4 * W + 1, DAG>(sm, lane);
    v[2] = split_sum<4 * W + 2, DAG>(sm, lane);
    v[3] = split_sum<4 * W + 3, DAG>(sm, lane);
}

template <typename R, int SP, int GP, int RECON, bool DAG, bool HASX, bool NTL>
__global__ __launch_bounds__(8 * kSplitSites) void k_wilson_hop_split(HopArgs a) {
    typedef WilsonIO<SP> SIO;
    typedef LinkIO<GP, RECON> LIO;
    __shared__ C2<R> sm[8 * 6 * kSplitSites];
    __shared__ float smax[SIO::SCALED ? 3 * kSplitSites : 1];
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int p, h;
    const bool valid = a.tile_y > 0 ? tile64_site(a.g, a.nblk, a.pbase, a.tile_y, a.tile_ymaj, lane, p, h)
                                    : block_site(logical_wg(a.xcd), kSplitSites, (unsigned)lane, a.g.Vh, a.nblk, a.pbase,
                                                 a.pinter, p, h);
    const unsigned po = a.out_full ? (unsigned)p : 0u;
    const unsigned eo = po * SIO::NPL * a.g.Vh + h, no = po * a.g.Vh + h;
    C2<R> xv[4];
    if (valid) {
        if constexpr (HASX)
            if (w < 3) SIO::load4(a.x, a.xn, a.g.Vh, eo, no, w, xv);  // in flight beside the neighbour loads
        const Site s = site_of(a.g, p, h);
        C2<R> uh[6];
        switch (w) {
            case 0: split_dir<0, true, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            case 1: split_dir<0, false, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            case 2: split_dir<1, true, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            case 3: split_dir<1, false, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            case 4: split_dir<2, true, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            case 5: split_dir<2, false, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            case 6: split_dir<3, true, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
            default: split_dir<3, false, DAG, NTL, R, SIO, LIO>(a, s, p, h, uh); break;
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) sm[(w * 6 + k) * kSplitSites + lane] = uh[k];
    }
    __syncthreads();
    C2<R> o[4];
    if (w < 3 && valid) {
        C2<R> acc[4];
        if (w == 0) split_sum4<0, DAG>(sm, lane, acc);
        else if (w == 1) split_sum4<1, DAG>(sm, lane, acc);
        else split_sum4<2, DAG>(sm, lane, acc);
        const C2<R> ca = cmk<R>((R)a.ar, (R)a.ai);
        const C2<R> cb = cmk<R>((R)a.br, (R)a.bi);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if constexpr (HASX) {
                o[k] = cmul(cb, xv[k]);
                cfma(o[k], ca, acc[k]);
            } else {
                o[k] = cmul(ca, acc[k]);
            }
        }
    }
    if constexpr (SIO::SCALED) {  // the site scale is the largest of the three waves' components
        if (w < 3 && valid) {
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) m = fmaxf(m, fmaxf(fabsf((float)o[k].x), fabsf((float)o[k].y)));
            smax[w * kSplitSites + lane] = m;
        }
        __syncthreads();
        if (w < 3 && valid) {
            const float m = fmaxf(smax[lane], fmaxf(smax[kSplitSites + lane], smax[2 * kSplitSites + lane]));
            const float inv = m > 0.f ? 1.0f / m : 0.f;
            if (w == 0) a.outn[no] = m;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = cscale(o[k], (R)inv);
        }
    }
    if (w < 3 && valid) {
        if (a.nt_out) SIO::template store4<R, true>(a.out, a.g.Vh, eo, w, o);
        else SIO::store4(a.out, a.g.Vh, eo, w, o);
    }
}

struct HopCfg {
    int pm;     // pin mode: 1 after each half of a direction, 2 after each direction; 3 / 4 the same
                // with non-temporal link loads (links read once per launch stream past the caches);
                // 5..8 as 1..4 with the z and t neighbours staged in LDS (block = L2*L3/2);
                // kSplitPm the direction-split kernel (block = kSplitSites sites, xcd 0 or 8)
    int block;  // threads per workgroup
    int xcd;    // 0: hardware order; 8: XCD-contiguous slabs, for full D with the two parities
                // interleaved block by block; 1: XCD-contiguous slabs, parities one after the other;
                // 10*TY + m (TY in 2, 4, 8; m = 0 x-major, 1 y-major): tiled plane schedule, staged
                // launches only (clgd::tile_block), parities interleaved; kSplitPm and kSplitNtPm take the same
                // codes for the schedule in 64-site blocks (clgd::tile64_site), pm 1..4 take them + 100
    int spt = 1;  // sites per thread: consecutive logical blocks per workgroup (1, 2 or 4)
    int nt = 0;   // 1: the output spinor is stored with the non-temporal policy (it is not read again by
                  // the launch, so it need not take L2 space from the neighbour spinors and links)
};
constexpr int kTile64 = 100;  // tile64_site for one site per thread (pm 1..4, block 64)
inline bool tiled_xcd(int xcd) { return xcd >= 20 && xcd <= 81 && (xcd / 10 == 2 || xcd / 10 == 4 || xcd / 10 == 8) && xcd % 10 <= 1; }

template <typename R, int SP, int GP, int RECON, int PM>
void launch_pm(const HopArgs& a0, bool dag, bool hasx, hipStream_t st, int block, int xcd, int spt, int nt) {
    HopArgs a = a0;
    a.nt_out = nt;
    unsigned grid;
    if (tiled_xcd(xcd)) {
        a.xcd = 0;
        a.pinter = 1;
        a.spt = 1;
        a.tile_y = xcd / 10;
        a.tile_ymaj = xcd % 10;
        grid = (unsigned)(a.nblk * a.g.L[0] * a.g.L[1]);
    } else if (tiled_xcd(xcd - kTile64)) {
        a.xcd = 0;
        a.spt = 1;
        a.tile_y = (xcd - kTile64) / 10;
        a.tile_ymaj = (xcd - kTile64) % 10;
        grid = tile64_grid(a.g, a.nblk, a.tile_y);
    } else {
        a.xcd = xcd ? 8 : 0;
        a.pinter = xcd == 8 ? 1 : 0;
        a.spt = spt;
        a.tile_y = 0;
        a.tile_ymaj = 0;
        grid = sched_grid(a.g.Vh, a.nblk, block, a.xcd, a.pinter, spt);
    }
    // staged launches: NPL 16-byte chunks per site of the plane, plus the FP16 site scales
    const size_t shm = PM >= 5 ? (size_t)block * (16 * WilsonIO<SP>::NPL + (WilsonIO<SP>::SCALED ? 4 : 0)) : 0;
    if (dag) {
        if (hasx) k_wilson_hop<R, SP, GP, RECON, true, true, PM><<<grid, block, shm, st>>>(a);
        else k_wilson_hop<R, SP, GP, RECON, true, false, PM><<<grid, block, shm, st>>>(a);
    } else {
        if (hasx) k_wilson_hop<R, SP, GP, RECON, false, true, PM><<<grid, block, shm, st>>>(a);
        else k_wilson_hop<R, SP, GP, RECON, false, false, PM><<<grid, block, shm, st>>>(a);
    }
}

constexpr int kSplitPm = 9;    // the direction-split kernel
constexpr int kSplitNtPm = 10;  // the same with non-temporal link loads
inline bool split_pm(int pm) { return pm == kSplitPm || pm == kSplitNtPm; }
template <typename R, int SP, int GP, int RECON, bool NTL>
void launch_split(const HopArgs& a0, bool dag, bool hasx, hipStream_t st, int xcd, int nt) {
    HopArgs a = a0;
    a.nt_out = nt;
    unsigned grid;
    if (tiled_xcd(xcd)) {
        a.tile_y = xcd / 10;
        a.tile_ymaj = xcd % 10;
        grid = tile64_grid(a.g, a.nblk, a.tile_y);
    } else {
        a.xcd = xcd ? 8 : 0;
        a.pinter = xcd ? 1 : 0;
        grid = sched_grid(a.g.Vh, a.nblk, kSplitSites, a.xcd, a.pinter);
    }
    if (dag) {
        if (hasx) k_wilson_hop_split<R, SP, GP, RECON, true, true, NTL><<<grid, 8 * kSplitSites, 0, st>>>(a);
        else k_wilson_hop_split<R, SP, GP, RECON, true, false, NTL><<<grid, 8 * kSplitSites, 0, st>>>(a);
    } else {
        if (hasx) k_wilson_hop_split<R, SP, GP, RECON, false, true, NTL><<<grid, 8 * kSplitSites, 0, st>>>(a);
        else k_wilson_hop_split<R, SP, GP, RECON, false, false, NTL><<<grid, 8 * kSplitSites, 0, st>>>(a);
    }
}

template <typename R, int SP, int GP, int RECON>
int launch_t(const HopArgs& a, bool dag, bool hasx, hipStream_t st, HopCfg c) {
    if (c.pm == kSplitPm) launch_split<R, SP, GP, RECON, false>(a, dag, hasx, st, c.xcd, c.nt);
    else if (c.pm == kSplitNtPm) launch_split<R, SP, GP, RECON, true>(a, dag, hasx, st, c.xcd, c.nt);
    else if (c.pm == 8) launch_pm<R, SP, GP, RECON, 8>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else if (c.pm == 7) launch_pm<R, SP, GP, RECON, 7>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else if (c.pm == 6) launch_pm<R, SP, GP, RECON, 6>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else if (c.pm == 5) launch_pm<R, SP, GP, RECON, 5>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else if (c.pm == 4) launch_pm<R, SP, GP, RECON, 4>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else if (c.pm == 3) launch_pm<R, SP, GP, RECON, 3>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else if (c.pm == 2) launch_pm<R, SP, GP, RECON, 2>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    else launch_pm<R, SP, GP, RECON, 1>(a, dag, hasx, st, c.block, c.xcd, c.spt, c.nt);
    CLG_HIP(hipGetLastError());
    return CLG_OK;
}

// the workgroup size of an LDS-staged launch on this lattice (one (x,y) plane of one parity), or 0
int staged_block(const Geo& g) {
    if (g.L[3] % 2) return 0;
    const int b = g.L[2] * g.L[3] / 2;
    return (b == 64 || b == 128 || b == 256) ? b : 0;
}
int launch_cfg(const HopArgs& a, int prec, int gprec, int recon, bool dag, bool hasx, hipStream_t st, HopCfg c) {
    // a staged launch needs one workgroup per (x,y) plane of one parity; the tuner only proposes
    // fitting ones, so a misfit comes from a forced configuration and is refused, not replaced
    if (c.pm >= 5 && c.pm <= 8) {
        const int sb = staged_block(a.g);
        CLG_CHECK_ARG(sb != 0 && c.block == sb,
                      "LDS-staged pin mode %d needs block = L2*L3/2 in {64,128,256} (lattice %dx%dx%dx%d gives %d), "
                      "asked for block %d",
                      c.pm, a.g.L[0], a.g.L[1], a.g.L[2], a.g.L[3], a.g.L[2] * a.g.L[3] / 2, c.block);
    }
    if (tiled_xcd(c.xcd) && !split_pm(c.pm)) {
        const int TY = c.xcd / 10, TX = 8 / TY;
        CLG_CHECK_ARG(c.pm >= 5 && c.spt == 1 && a.g.L[0] % TX == 0 && a.g.L[1] % TY == 0,
                      "tiled schedule %d needs an LDS-staged pin mode, one site per thread, L0 %% %d == 0 and "
                      "L1 %% %d == 0 (lattice %dx%dx%dx%d)",
                      c.xcd, TX, TY, a.g.L[0], a.g.L[1], a.g.L[2], a.g.L[3]);
    }
    if (prec == CLG_F64) {
        return recon == 12 ? launch_t<double, CLG_F64, CLG_F64, 12>(a, dag, hasx, st, c)
                           : launch_t<double, CLG_F64, CLG_F64, 18>(a, dag, hasx, st, c);
    } else if (prec == CLG_F32 && gprec == CLG_F32) {
        return recon == 12 ? launch_t<float, CLG_F32, CLG_F32, 12>(a, dag, hasx, st, c)
                           : launch_t<float, CLG_F32, CLG_F32, 18>(a, dag, hasx, st, c);
    } else if (prec == CLG_F32) {  // FP16 links, FP32 spinors
        return recon == 12 ? launch_t<float, CLG_F32, CLG_F16, 12>(a, dag, hasx, st, c)
                           : launch_t<float, CLG_F32, CLG_F16, 18>(a, dag, hasx, st, c);
    }
    return recon == 12 ? launch_t<float, CLG_F16, CLG_F16, 12>(a, dag, hasx, st, c)
                       : launch_t<float, CLG_F16, CLG_F16, 18>(a, dag, hasx, st, c);
}

// ---- autotuner: the first launch of a (precision, recon, dagger, x, shape) key times each
//      candidate with HIP events on the launch stream and keeps the fastest.  Outputs are
//      rewritten identically by every candidate, so tuning is invisible to the caller unless
//      out aliases x (then the default is used).  CLG_TUNE=0 disables tuning.
struct TuneKey {
    int prec, gprec, recon, dag, hasx, nblk, L0, L1, L2, L3;
    bool operator<(const TuneKey& o) const {
        return std::memcmp(this, &o, sizeof(TuneKey)) < 0;
    }
};
std::map<TuneKey, HopCfg>& tune_table() {
    static std::map<TuneKey, HopCfg> t;
    return t;
}
std::mutex& tune_mutex() {
    static std::mutex m;
    return m;
}
// the tuning-cache file whose entries are in tune_table() (under tune_mutex)
std::string& tune_loaded() {
    static std::string p;
    return p;
}
std::vector<long> key_vec(const TuneKey& k) {
    return {k.prec, k.gprec, k.recon, k.dag, k.hasx, k.nblk, k.L0, k.L1, k.L2, k.L3};
}
bool valid_cfg(int pm, int blk, int xcd, int spt) {
    return pm >= 1 && pm <= 8 && (blk == 64 || blk == 128 || blk == 256) &&
           (xcd == 0 || xcd == 1 || xcd == 8 || tiled_xcd(xcd)) && (spt == 1 || spt == 2 || spt == 4);
}
// the configurations in 64-site blocks (the tuner's, its cache file's and forced ones): the
// direction-split kernel, and one site per thread in the tiled order
bool valid_split(int pm, int blk, int xcd, int spt) {
    if (blk != kSplitSites || spt != 1) return false;
    if (pm >= 1 && pm <= 4) return tiled_xcd(xcd - kTile64);
    return split_pm(pm) && (xcd == 0 || xcd == 8 || tiled_xcd(xcd));
}
// process-wide overrides set through clg_autotune_enable / clg_autotune_force
std::atomic<int> g_tune_mode{-1};  // -1: CLG_TUNE environment (default on), 0 off, 1 on
std::atomic<int> g_forced{0};      // packed pin | block << 4 | xcd << 16 | spt << 24 | nt << 28, 0 = none
// CLG_TUNE_FORCE="pin,block,xcd[,spt[,nt]]" (or clg_autotune_force) fixes the launch configuration of
// every hop launch (used to profile one configuration under counters, where event timings are
// not representative)
bool forced_cfg(HopCfg& c) {
    const int f = g_forced.load();
    if (f) {
        c = HopCfg{f & 15, (f >> 4) & 4095, (f >> 16) & 255, (f >> 24) & 7, (f >> 28) & 1};
        return true;
    }
    const char* e = std::getenv("CLG_TUNE_FORCE");
    if (!e) return false;
    int pm = 0, blk = 0, xcd = 0, spt = 1, nt = 0;
    const int got = std::sscanf(e, "%d,%d,%d,%d,%d", &pm, &blk, &xcd, &spt, &nt);
    if (got < 3 || !(valid_cfg(pm, blk, xcd, spt) || valid_split(pm, blk, xcd, spt)) || (nt != 0 && nt != 1)) return false;
    c = HopCfg{pm, blk, xcd, spt, nt};
    return true;
}

// Untuned launches (tuning off, small lattices, graph capture) take the direction split up to this many
// sites: measured, it is ahead of one site per thread for FP64 and FP32 spinors in the XCD-slab order up to
// here (FP64 D at 24^3x16 48.6 against 61.2 us, FP32 26.7 against 27.7).  In FP16 it is well ahead up to
// 12^3x24 (D 5.9 against 7.9 us), less so at 16^4 (7.0 against 8.1), level at 16^3x32 (11.9) and behind at
// 32^3x16 (half hop 21.8 against 18.8, D 40 against 35): the line lies where the gain is still large.
inline long split_default_max(int prec) { return prec == CLG_F16 ? 32768 : 262144; }

int launch_hop(const HopArgs& a, int prec, int gprec, int recon, bool dag, bool hasx, hipStream_t st) {
    const long nsite = (long)a.nblk * a.g.Vh;
    const HopCfg dflt = nsite <= split_default_max(prec) ? HopCfg{kSplitPm, kSplitSites, 8} : HopCfg{1, 256, 8};
    TuneKey k;
    std::memset(&k, 0, sizeof(k));
    k.prec = prec; k.gprec = gprec; k.recon = recon; k.dag = dag; k.hasx = hasx; k.nblk = a.nblk;
    k.L0 = a.g.L[0]; k.L1 = a.g.L[1]; k.L2 = a.g.L[2]; k.L3 = a.g.L[3];
    HopCfg cfg = dflt;
    if (forced_cfg(cfg)) return launch_cfg(a, prec, gprec, recon, dag, hasx, st, cfg);
    bool need_tune = false;
    const std::string cpath = tune_cache_path();
    {
        std::lock_guard<std::mutex> lk(tune_mutex());
        auto it = tune_table().find(k);
        if (it == tune_table().end() && !cpath.empty() && cpath != tune_loaded()) {
            std::vector<std::pair<std::vector<long>, std::vector<long>>> ent;
            tune_cache_read(cpath, "wilson_hop", ent);
            for (const auto& e : ent) {
                const std::vector<long>& v = e.first;
                const std::vector<long>& c = e.second;
                if (v.size() != 10 || (c.size() != 4 && c.size() != 5) ||
                    !(valid_cfg((int)c[0], (int)c[1], (int)c[2], (int)c[3]) ||
                      valid_split((int)c[0], (int)c[1], (int)c[2], (int)c[3])))
                    continue;
                TuneKey t;
                std::memset(&t, 0, sizeof(t));
                t.prec = (int)v[0]; t.gprec = (int)v[1]; t.recon = (int)v[2]; t.dag = (int)v[3]; t.hasx = (int)v[4];
                t.nblk = (int)v[5]; t.L0 = (int)v[6]; t.L1 = (int)v[7]; t.L2 = (int)v[8]; t.L3 = (int)v[9];
                tune_table()[t] = HopCfg{(int)c[0], (int)c[1], (int)c[2], (int)c[3], c.size() == 5 ? (int)(c[4] != 0) : 0};
            }
            tune_loaded() = cpath;
            it = tune_table().find(k);
        }
        if (it != tune_table().end()) cfg = it->second;
        else need_tune = true;
    }
    const bool aliased = hasx && a.x == a.out;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(st, &cs);
    if (need_tune && tuning_enabled() && !aliased && cs == hipStreamCaptureStatusNone && (long)a.nblk * a.g.Vh >= 4096) {
        const HopCfg cands[] = {{1, 64, 0}, {1, 128, 0}, {1, 256, 0}, {2, 64, 0}, {2, 128, 0}, {2, 256, 0},
                                {1, 64, 8}, {1, 128, 8}, {1, 256, 8}, {2, 64, 8}, {2, 128, 8}, {2, 256, 8},
                                {3, 64, 8}, {3, 128, 8}, {3, 256, 8}, {4, 64, 8}, {4, 128, 8}, {4, 256, 8}};
        std::vector<HopCfg> all(std::begin(cands), std::end(cands));
        // several sites per thread for the XCD-slab launches
        for (int spt : {2, 4})
            for (int pm : {2, 4})
                for (int blk : {128, 256}) all.push_back(HopCfg{pm, blk, 8, spt});
        for (int pm : {kSplitPm, kSplitNtPm}) {
            all.push_back(HopCfg{pm, kSplitSites, 8});
            if (pm == kSplitPm) all.push_back(HopCfg{pm, kSplitSites, 0});
            for (int TY : {2, 4, 8})
                if (tile64_fits(a.g, TY))
                    for (int m : {0, 1})
                        for (int nt : {0, 1}) all.push_back(HopCfg{pm, kSplitSites, 10 * TY + m, 1, nt});
        }
        for (int TY : {2, 4, 8})
            if (tile64_fits(a.g, TY))
                for (int pm = 1; pm <= 4; ++pm)
                    for (int nt : {0, 1}) all.push_back(HopCfg{pm, kSplitSites, kTile64 + 10 * TY, 1, nt});
        if (const int sb = staged_block(a.g)) {
            for (int pm = 5; pm <= 8; ++pm) all.push_back(HopCfg{pm, sb, 8});
            for (int pm : {6, 8}) all.push_back(HopCfg{pm, sb, 8, 2});
            // tiled plane schedules where the plane grid divides
            for (int TY : {2, 4, 8})
                for (int m : {0, 1})
                    if (a.g.L[0] % (8 / TY) == 0 && a.g.L[1] % TY == 0)
                        for (int pm = 5; pm <= 8; ++pm) {
                            all.push_back(HopCfg{pm, sb, 10 * TY + m});
                            if (m == 0 && TY >= 4) all.push_back(HopCfg{pm, sb, 10 * TY + m, 1, 1});
                        }
        }
        // Links that fit the 32 MB of L2 are read from there by the next hops: no non-temporal loads of them.  Best
        // cached against best non-temporal launch, us, each repeated: FP64 D 12^3x16 (15 MB) 6.7 / 8.1, 16^3x12
        // (27 MB) 11.5 / 13.7, half hop 7.4 / 8.6; FP32 D 16^4 (18 MB) 8.6 / 11.0, 16^3x24 (27 MB) 12.8 / 16.1, half
        // hop 7.1 / 8.0; FP16 D 24^3x16 (20 MB) 18.1 / 19.7; level where everything is small (8^4).  Between the
        // other kernels of a solve the gap is wider (FP32 half hops at 16^4 6.6 / 9.4) than a candidate's few
        // launches show.
        if (8L * a.g.Vh * (recon == 12 ? 12 : 18) * (gprec == CLG_F64 ? 8 : gprec == CLG_F32 ? 4 : 2) <= (32L << 20))
            all.erase(std::remove_if(all.begin(), all.end(),
                                     [](const HopCfg& c) {
                                         return c.pm == 3 || c.pm == 4 || c.pm == 7 || c.pm == 8 || c.pm == kSplitNtPm;
                                     }),
                      all.end());
        float best = 0.f;
        const char* v2 = std::getenv("CLG_TUNE_VERBOSE");
        const bool each = v2 && v2[0] == '2';
        CLG_TRY(tune_pick(
            st, all, [&](const HopCfg& c) { return launch_cfg(a, prec, gprec, recon, dag, hasx, st, c); },
            [&](const HopCfg& c, float ms) {
                if (each)
                    std::fprintf(stderr, "[clg tune]   candidate pin=%d block=%d xcd=%d spt=%d nt=%d: %.1f us\n", c.pm,
                                 c.block, c.xcd, c.spt, c.nt, ms * 1e3);
            },
            cfg, best));
        const char* verbose = std::getenv("CLG_TUNE_VERBOSE");
        if (verbose && (verbose[0] == '1' || verbose[0] == '2'))
            std::fprintf(stderr, "[clg tune] wilson hop prec=%d gprec=%d recon=%d dag=%d x=%d nblk=%d L=%dx%dx%dx%d -> pin=%d block=%d xcd=%d spt=%d nt=%d (%.1f us)\n",
                         prec, gprec, recon, (int)dag, (int)hasx, a.nblk, a.g.L[0], a.g.L[1], a.g.L[2], a.g.L[3],
                         cfg.pm, cfg.block, cfg.xcd, cfg.spt, cfg.nt, best * 1e3);
        std::lock_guard<std::mutex> lk(tune_mutex());
        tune_table()[k] = cfg;
        tune_cache_append(cpath, "wilson_hop", key_vec(k), {cfg.pm, cfg.block, cfg.xcd, cfg.spt, cfg.nt});
    }
    return launch_cfg(a, prec, gprec, recon, dag, hasx, st, cfg);
}

int check_gauge(const clg_field_s* f, const clg_field_s* gauge) {
    CLG_CHECK_ARG(gauge && is_gauge(gauge->kind), "need a gauge field");
    CLG_TRY(check_same_lattice(f, gauge));
    CLG_CHECK_ARG(gauge->prec == f->prec || (f->prec == CLG_F32 && gauge->prec == CLG_F16),
                  "gauge precision must match the fermion precision (or FP16 links with FP32 spinors)");
    return CLG_OK;
}

HopArgs base_args(const clg_field_s* out, const clg_field_s* gauge) {
    HopArgs a;
    std::memset(&a, 0, sizeof(a));
    a.g = make_geo(out);
    a.gauge = (const char*)gauge->data;
    return a;
}

}  // namespace

namespace clg {

bool tuning_enabled() {
    const int m = g_tune_mode.load();
    if (m >= 0) return m != 0;
    const char* e = std::getenv("CLG_TUNE");
    return !(e && e[0] == '0');
}

// out(full) = coeff * (in - kappa H in) with dagger projectors when dag
int wilson_full(clg_context ctx, clg_field_s* out, const clg_field_s* in, const clg_field_s* gauge, double kappa,
                bool dag, double cre, double cim) {
    HopArgs a = base_args(out, gauge);
    a.in = (const char*)in->data;
    a.inn = in->norm;
    a.x = (const char*)in->data;
    a.xn = in->norm;
    a.out = (char*)out->data;
    a.outn = out->norm;
    a.in_full = 1;
    a.out_full = 1;
    a.br = cre;
    a.bi = cim;
    a.ar = -kappa * cre;
    a.ai = -kappa * cim;
    a.pbase = 0;
    a.nblk = 2;
    return launch_hop(a, out->prec, gauge->prec, gauge->kind == CLG_GAUGE12 ? 12 : 18, dag, true, ctx->stream);
}

// out(full) = a H in (no diagonal term): the K of D = 1 - kappa H when a = kappa
int wilson_full_hop(clg_context ctx, clg_field_s* out, const clg_field_s* in, const clg_field_s* gauge, double a_re,
                    bool dag) {
    HopArgs a = base_args(out, gauge);
    a.in = (const char*)in->data;
    a.inn = in->norm;
    a.out = (char*)out->data;
    a.outn = out->norm;
    a.in_full = 1;
    a.out_full = 1;
    a.ar = a_re;
    a.pbase = 0;
    a.nblk = 2;
    return launch_hop(a, out->prec, gauge->prec, gauge->kind == CLG_GAUGE12 ? 12 : 18, dag, false, ctx->stream);
}

// out(parity p) = b x + a H_{p,1-p} in
int wilson_hop_half(clg_context ctx, clg_field_s* out, const clg_field_s* in, const clg_field_s* gauge, bool dag,
                    double ar, double ai, const clg_field_s* x, double br, double bi) {
    const int p = field_parity(out);
    HopArgs a = base_args(out, gauge);
    a.in = (const char*)in->data;
    a.inn = in->norm;
    a.out = (char*)out->data;
    a.outn = out->norm;
    if (x) {
        a.x = (const char*)x->data;
        a.xn = x->norm;
    }
    a.ar = ar;
    a.ai = ai;
    a.br = br;
    a.bi = bi;
    a.pbase = p;
    a.nblk = 1;
    return launch_hop(a, out->prec, gauge->prec, gauge->kind == CLG_GAUGE12 ? 12 : 18, dag, x != nullptr, ctx->stream);
}

int check_hop_fields(const clg_field_s* out, const clg_field_s* in, const clg_field_s* gauge) {
    CLG_CHECK_ARG(out && in, "null field");
    CLG_CHECK_ARG(out->kind == CLG_WILSON && in->kind == CLG_WILSON, "need Wilson fields");
    CLG_CHECK_ARG(out->subset != CLG_FULL && in->subset != CLG_FULL, "hop needs half-lattice fields");
    CLG_CHECK_ARG(out->subset != in->subset, "hop maps one parity to the other");
    CLG_CHECK_ARG(out->prec == in->prec, "precision mismatch");
    CLG_TRY(check_same_lattice(out, in));
    for (int i = 0; i < 4; ++i) CLG_CHECK_ARG((out->dims[i] & 1) == 0, "even-odd operators need even extents");
    CLG_TRY(check_gauge(out, gauge));
    return CLG_OK;
}

// Schur complement on even sites: Mhat = 1 - kappa^2 H_eo H_oe (dag: projectors swapped)
int wilson_schur_once(clg_context ctx, clg_field_s* out, const clg_field_s* in, const clg_field_s* gauge,
                      double kappa, bool dag, clg_field_s* tmp_odd) {
    CLG_TRY(wilson_hop_half(ctx, tmp_odd, in, gauge, dag, 1.0, 0.0, nullptr, 0.0, 0.0));
    return wilson_hop_half(ctx, out, tmp_odd, gauge, dag, -kappa * kappa, 0.0, in, 1.0, 0.0);
}

}  // namespace clg

extern "C" {

int clg_wilson_apply(clg_context ctx, clg_field out, clg_field in, clg_field gauge, double kappa, int op,
                     int coeff_type, double cre, double cim) {
    CLG_CHECK_ARG(ctx && out && in, "null argument");
    CLG_CHECK_ARG(out != in && out->data != in->data, "out and in must be distinct fields");
    CLG_CHECK_ARG(out->kind == CLG_WILSON && in->kind == CLG_WILSON, "need Wilson fields");
    CLG_CHECK_ARG(out->subset == CLG_FULL && in->subset == CLG_FULL, "need FULL fields");
    CLG_CHECK_ARG(out->prec == in->prec, "precision mismatch");
    CLG_TRY(check_same_lattice(out, in));
    CLG_TRY(check_gauge(out, gauge));
    CLG_CHECK_ARG(op >= EFO_F_D && op <= EFO_F_DDdagger, "operator %d not supported here", op);
    double fr = 1.0, fi = 0.0;
    switch (coeff_type) {
        case EOCT_None: break;
        case EOCT_Minus: fr = -1.0; break;
        case EOCT_Real: fr = cre; break;
        case EOCT_Complex: fr = cre; fi = cim; break;
        default: CLG_CHECK_ARG(false, "bad coefficient type %d", coeff_type);
    }
    (void)hipSetDevice(ctx->device);
    for (int i = 0; i < 4; ++i) out->bc[i] = in->bc[i];
    if (op == EFO_F_D || op == EFO_F_Ddagger) return wilson_full(ctx, out, in, gauge, kappa, op == EFO_F_Ddagger, fr, fi);
    // DD = D(D psi), DD^dagger = D(D^dagger psi); the coefficient is applied by the second D
    // (CFieldFermionWilsonSquareSU3.cu:962-1014)
    clg_field_s* tmp = nullptr;
    CLG_TRY(scratch_field(ctx, in, CLG_WILSON, in->prec, CLG_FULL, 0, &tmp));
    CLG_TRY(wilson_full(ctx, tmp, in, gauge, kappa, op == EFO_F_DDdagger, 1.0, 0.0));
    return wilson_full(ctx, out, tmp, gauge, kappa, false, fr, fi);
}

int clg_wilson_hop(clg_context ctx, clg_field out, clg_field in, clg_field gauge, int dagger, double a_re,
                   double a_im, clg_field x, double b_re, double b_im) {
    CLG_CHECK_ARG(ctx, "null context");
    CLG_TRY(check_hop_fields(out, in, gauge));
    if (x) {
        CLG_CHECK_ARG(x->kind == CLG_WILSON && x->subset == out->subset && x->prec == out->prec,
                      "x must match out");
    }
    CLG_CHECK_ARG(out->data != in->data, "out and in must be distinct");
    (void)hipSetDevice(ctx->device);
    return wilson_hop_half(ctx, out, in, gauge, dagger != 0, a_re, a_im, x, b_re, b_im);
}

int clg_wilson_schur(clg_context ctx, clg_field out, clg_field in, clg_field gauge, double kappa, int op) {
    CLG_CHECK_ARG(ctx && out && in, "null argument");
    CLG_CHECK_ARG(out->subset == CLG_EVEN && in->subset == CLG_EVEN, "Schur operator acts on EVEN fields");
    CLG_CHECK_ARG(out->kind == CLG_WILSON && in->kind == CLG_WILSON && out->prec == in->prec, "need Wilson fields");
    CLG_CHECK_ARG(out->data != in->data, "out and in must be distinct");
    CLG_TRY(check_same_lattice(out, in));
    for (int i = 0; i < 4; ++i) CLG_CHECK_ARG((out->dims[i] & 1) == 0, "even-odd operators need even extents");
    CLG_TRY(check_gauge(out, gauge));
    CLG_CHECK_ARG(op >= EFO_F_D && op <= EFO_F_DDdagger, "operator %d not supported", op);
    (void)hipSetDevice(ctx->device);
    clg_field_s* todd = nullptr;
    CLG_TRY(scratch_field(ctx, in, CLG_WILSON, in->prec, CLG_ODD, 0, &todd));
    for (int i = 0; i < 4; ++i) { out->bc[i] = in->bc[i]; todd->bc[i] = in->bc[i]; }
    if (op == EFO_F_D || op == EFO_F_Ddagger)
        return wilson_schur_once(ctx, out, in, gauge, kappa, op == EFO_F_Ddagger, todd);
    clg_field_s* teven = nullptr;
    CLG_TRY(scratch_field(ctx, in, CLG_WILSON, in->prec, CLG_EVEN, 0, &teven));
    for (int i = 0; i < 4; ++i) teven->bc[i] = in->bc[i];
    CLG_TRY(wilson_schur_once(ctx, teven, in, gauge, kappa, op == EFO_F_DDdagger, todd));
    return wilson_schur_once(ctx, out, teven, gauge, kappa, false, todd);
}

int clg_time_wilson(clg_context ctx, clg_field out, clg_field in, clg_field gauge, double kappa, int variant,
                    int reps, double* ms_avg) {
    CLG_CHECK_ARG(ctx && ms_avg && reps > 0, "bad arguments");
    (void)hipSetDevice(ctx->device);
    auto one = [&]() -> int {
        if (variant == 0) return clg_wilson_apply(ctx, out, in, gauge, kappa, EFO_F_D, EOCT_None, 1.0, 0.0);
        if (variant == 1) return clg_wilson_hop(ctx, out, in, gauge, 0, 1.0, 0.0, nullptr, 0.0, 0.0);
        return clg_wilson_schur(ctx, out, in, gauge, kappa, EFO_F_D);
    };
    CLG_TRY(one());  // validates arguments, warms up
    CLG_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    for (int r = 0; r < reps; ++r) CLG_TRY(one());
    CLG_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    CLG_HIP(hipEventSynchronize(ctx->ev1));
    float ms = 0.f;
    CLG_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    *ms_avg = (double)ms / reps;
    return CLG_OK;
}

// ---- launch autotuner control
int clg_autotune_enable(int mode) {
    CLG_CHECK_ARG(mode >= -1 && mode <= 1, "mode must be -1 (environment), 0 or 1");
    g_tune_mode.store(mode);
    return CLG_OK;
}

int clg_autotune_force(int pin_mode, int block, int xcd, int sites_per_thread) {
    if (pin_mode == 0) {
        g_forced.store(0);
        return CLG_OK;
    }
    if (sites_per_thread == 0) sites_per_thread = 1;
    CLG_CHECK_ARG(valid_cfg(pin_mode, block, xcd, sites_per_thread) || valid_split(pin_mode, block, xcd, sites_per_thread),
                  "pin_mode 1..8, block 64|128|256, xcd 0|1|8 or a tiled plane schedule 20|21|40|41|80|81, "
                  "sites_per_thread 1|2|4; or, with block 64 and one site per thread, pin_mode 9|10, xcd 0|8 or a tiled "
                  "schedule, and pin_mode 1..4, xcd 100 + a tiled schedule");
    g_forced.store(pin_mode | block << 4 | xcd << 16 | sites_per_thread << 24);
    return CLG_OK;
}

int clg_autotune_reset(void) {
    {
        std::lock_guard<std::mutex> lk(tune_mutex());
        tune_table().clear();
        tune_loaded().clear();
    }
    batch_tune_reset();
    ks_tune_reset();
    return CLG_OK;
}

int clg_autotune_count(void) {
    int n = 0;
    {
        std::lock_guard<std::mutex> lk(tune_mutex());
        n = (int)tune_table().size();
    }
    return n + batch_tune_count() + ks_tune_count();
}

int clg_autotune_entry(int index, char* buf, int len) {
    CLG_CHECK_ARG(buf && len > 0 && index >= 0, "bad arguments");
    {
        std::lock_guard<std::mutex> lk(tune_mutex());
        if (index < (int)tune_table().size()) {
            auto it = tune_table().begin();
            std::advance(it, index);
            const TuneKey& k = it->first;
            const HopCfg& c = it->second;
            std::snprintf(buf, (size_t)len,
                          "wilson_hop prec=%d gauge_prec=%d recon=%d dagger=%d x=%d parities=%d dims=%dx%dx%dx%d "
                          "-> pin=%d block=%d xcd=%d spt=%d nt=%d",
                          k.prec, k.gprec, k.recon, k.dag, k.hasx, k.nblk, k.L0, k.L1, k.L2, k.L3, c.pm, c.block, c.xcd,
                          c.spt, c.nt);
            return CLG_OK;
        }
        index -= (int)tune_table().size();
    }
    const int nb = batch_tune_count();
    if (index < nb) return batch_tune_entry(index, buf, len);
    return ks_tune_entry(index - nb, buf, len);
}

}  // extern "C"
