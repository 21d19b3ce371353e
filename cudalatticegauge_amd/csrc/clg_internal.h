// clg_internal.h -- shared definitions of libclg_hip.so (not installed, not part of the ABI).
//
// Data layout in HBM (all fields):
//   * Sites are split by parity.  The e-th site of parity p is the lexicographic site
//     2e or 2e+1 with parity p (the reference's even/odd numbering, CLGLib_Private.h:72-116),
//     so a half-lattice index h maps to coordinates with one division chain and Lt even.
//   * A FULL fermion field is [parity-0 block | parity-1 block]; an EVEN/ODD field is one
//     block.  A block is structure-of-arrays: `nplane` planes of Vh 16-byte (or 8/4-byte)
//     chunks, so lane i of a wavefront reads chunk i of a plane: every load is a contiguous
//     64-lane burst.
//   * Gauge fields hold 8 blocks, (parity, mu), each a set of link planes over Vh sites:
//     U_mu(x) for x of that parity.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <functional>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../../include/clg_hip.h"

namespace clg {

// ------------------------------------------------------------------ errors
void set_error(const char* fmt, ...);
const char* last_error();

#define CLG_CHECK_ARG(cond, ...)              \
    do {                                      \
        if (!(cond)) {                        \
            ::clg::set_error(__VA_ARGS__);    \
            return CLG_BAD_ARG;               \
        }                                     \
    } while (0)

#define CLG_HIP(call)                                                                  \
    do {                                                                               \
        hipError_t _e = (call);                                                        \
        if (_e != hipSuccess) {                                                        \
            ::clg::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(_e),   \
                             __FILE__, __LINE__);                                      \
            return CLG_HIP_ERROR;                                                      \
        }                                                                              \
    } while (0)

#define CLG_TRY(call)                 \
    do {                              \
        int _s = (call);              \
        if (_s != CLG_OK) return _s;  \
    } while (0)

// ------------------------------------------------------------------ geometry
struct Geo {
    int L[4];       // x, y, z, t extents
    int stride[4];  // lexicographic strides (t fastest)
    int sgn[4];     // fermion boundary sign per direction
    int Vh;         // half volume
};

// ------------------------------------------------------------------ handles
}  // namespace clg

struct clg_field_s;

struct clg_context_s {
    int device = 0;
    hipStream_t stream = nullptr;
    int num_cu = 0;
    char arch[64] = {0};
    // reduction scratch: per-block partials, device results
    double* red_partial = nullptr;
    size_t red_partial_cap = 0;  // doubles
    std::vector<double*> red_outgrown;  // earlier, smaller ones: recorded graphs may still write to them
    double* red_result = nullptr;  // 4096 doubles of device-resident results
    double* host_result = nullptr;  // pinned
    // solver workspace (Hessenberg, Givens, scalars), grow-only
    double* ws = nullptr;
    size_t ws_cap = 0;
    // scratch fields keyed by shape (owned)
    std::vector<clg_field_s*> scratch;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // objects made on this context (GCRO-DR solvers, graphs) with their destroy functions:
    // clg_finalize destroys those the caller has not
    std::vector<std::pair<void*, void (*)(void*)>> owned;
    // recorded solver cycles (clg::cycle_graph_run): key -> instantiated graph
    std::map<std::vector<unsigned long long>, hipGraphExec_t> cycle_graphs;
};

struct clg_field_s {
    clg_context ctx = nullptr;
    int kind = 0, prec = 0, subset = 0;
    int dims[4] = {0, 0, 0, 0};
    int bc[4] = {1, 1, 1, -1};
    long V = 0;
    long Vh = 0;
    long nsites = 0;       // V (FULL) or Vh
    void* data = nullptr;  // device storage
    float* norm = nullptr; // FP16 fields: per-site scale, [parity block][Vh]
    size_t bytes = 0;
    bool owns = true;
    clg_field_s* parent = nullptr;  // views
    // size of one parity block in bytes (fermions) or one (parity,mu) block (gauge)
    size_t block_bytes = 0;
    int scratch_slot = -1;  // context-owned scratch fields: the slot id they were created for
};

namespace clg {

// ------------------------------------------------------------------ layout sizes
// bytes of one site's worth of a fermion parity block / one link of a gauge block
inline size_t site_bytes(int kind, int prec) {
    switch (kind) {
        case CLG_WILSON: return prec == CLG_F64 ? 192 : prec == CLG_F32 ? 96 : 48;
        case CLG_KS: return prec == CLG_F64 ? 48 : prec == CLG_F32 ? 24 : 12;
        case CLG_GAUGE: return prec == CLG_F64 ? 144 : prec == CLG_F32 ? 72 : 36;
        case CLG_GAUGE12: return prec == CLG_F64 ? 96 : prec == CLG_F32 ? 48 : 24;
    }
    return 0;
}
inline bool is_gauge(int kind) { return kind == CLG_GAUGE || kind == CLG_GAUGE12; }
inline bool is_fermion(int kind) { return kind == CLG_WILSON || kind == CLG_KS; }
inline int parity_of_subset(int subset) { return subset == CLG_ODD ? 1 : 0; }

Geo make_geo(const clg_field_s* f);
int check_same_lattice(const clg_field_s* a, const clg_field_s* b);
// device pointer of parity block p of a fermion field (FULL: p in {0,1}; half: p must match)
inline char* block_ptr(const clg_field_s* f, int p) {
    if (f->subset == CLG_FULL) return (char*)f->data + (size_t)p * f->block_bytes;
    return (char*)f->data;
}
inline float* norm_ptr(const clg_field_s* f, int p) {
    if (!f->norm) return nullptr;
    if (f->subset == CLG_FULL) return f->norm + (size_t)p * f->Vh;
    return f->norm;
}
inline int field_parity(const clg_field_s* f) { return f->subset == CLG_ODD ? 1 : 0; }
// true when the device storage of a and b overlaps (data bytes or FP16 site scales); parity views
// of one FULL field overlap it, and the two parity views of one field do not overlap each other
inline size_t data_bytes(const clg_field_s* f) {
    return f->block_bytes * (size_t)(is_gauge(f->kind) ? 8 : (f->subset == CLG_FULL ? 2 : 1));
}
inline bool fields_overlap(const clg_field_s* a, const clg_field_s* b) {
    if (!a || !b) return false;
    const char *a0 = (const char*)a->data, *b0 = (const char*)b->data;
    if (a0 < b0 + data_bytes(b) && b0 < a0 + data_bytes(a)) return true;
    if (a->norm && b->norm) {
        const size_t na = (size_t)a->nsites, nb = (size_t)b->nsites;
        if (a->norm < b->norm + nb && b->norm < a->norm + na) return true;
    }
    return false;
}
inline void ctx_adopt(clg_context c, void* obj, void (*destroy)(void*)) { c->owned.emplace_back(obj, destroy); }
inline void ctx_release(clg_context c, void* obj) {
    for (auto it = c->owned.begin(); it != c->owned.end(); ++it)
        if (it->first == obj) {
            c->owned.erase(it);
            return;
        }
}

// reductions (clg_blas.hip)
int ensure_reduction_scratch(clg_context ctx, size_t doubles);
// allocates the partial-sum buffer every reduction kernel uses (its final size)
int reduction_ready(clg_context ctx);
// looks up, once per device, the device address of clg_multidot_noalloc's static partial-sum array
int noalloc_scratch_init(int device);
// device scratch (doubles) one Arnoldi orthogonalisation step (arn_step, clg_arnoldi.hip) needs
constexpr int kArnScratch = 264;
// up to this many workgroups of partials the pass after a small reduction totals them itself
constexpr long kMergeGrid = 256;
// within that scratch, of the fast Gram-Schmidt steps: whether one was refused, and the projections
constexpr int kGsBad = 39, kGsH = 40;
// scratch field of the same shape as `like` (kind/prec/subset/dims), index slot
int scratch_field(clg_context ctx, const clg_field_s* like, int kind, int prec, int subset,
                  int slot, clg_field_s** out);
// true while the context stream records a graph (blocking calls are refused then)
bool stream_capturing(clg_context ctx);
// Runs the device work of one solver cycle as a recorded graph: the first call with a key records
// what `record` launches on the context stream (it must neither block nor allocate) and instantiates
// it; every call (the first included) then replays it.  The key names every pointer and scalar the
// recorded launches take.  CLG_GRAPHS=0 runs `record` directly instead.
int cycle_graph_run(clg_context ctx, const std::vector<unsigned long long>& key, const std::function<int()>& record);
// the bits of a double, for graph keys
inline unsigned long long key_bits(double v) {
    unsigned long long u;
    static_assert(sizeof(u) == sizeof(v), "64-bit double");
    __builtin_memcpy(&u, &v, sizeof(u));
    return u;
}

// launch autotuner (clg_wilson.hip, clg_batch.hip): process-wide switch and tuned-shape tables
bool tuning_enabled();
int batch_tune_count();
int batch_tune_entry(int index, char* buf, int len);
void batch_tune_reset();
// Persistent tuning cache (CLG_TUNE_CACHE=<file>): one text line per tuned key,
//   "<device arch> <tuner> <key integers> : <configuration integers>".
// A tuner reads the lines of its name and of the current device's architecture the first time it
// misses a key under a cache path (again after clg_autotune_reset), and appends every key it tunes.
std::string tune_cache_path();
std::string device_arch();
int tune_cache_read(const std::string& path, const char* tuner,
                    std::vector<std::pair<std::vector<long>, std::vector<long>>>& out);
void tune_cache_append(const std::string& path, const char* tuner, const std::vector<long>& key,
                       const std::vector<long>& cfg);
int ks_tune_count();
int ks_tune_entry(int index, char* buf, int len);
void ks_tune_reset();

// Times the candidate launches of one operator call on its stream (every candidate writes the same output) and
// returns the fastest in `best`, its time in `best_ms` (milliseconds a launch).  A first round of a warm-up and
// three launches each; then those within 15 % of the fastest, six at most, are timed in turn three times over 20
// launches or about 1 ms, and the sum counts: three launches are within the noise of the clocks and of what ran
// before them.
template <class C, class L, class V>
int tune_pick(hipStream_t st, const std::vector<C>& cands, L launch, V report, C& best, float& best_ms) {
    hipEvent_t e0, e1;
    CLG_HIP(hipEventCreate(&e0));
    CLG_HIP(hipEventCreate(&e1));
    auto timed = [&](const C& c, int reps, float& ms) -> int {
        CLG_HIP(hipEventRecord(e0, st));
        for (int r = 0; r < reps; ++r) CLG_TRY(launch(c));
        CLG_HIP(hipEventRecord(e1, st));
        CLG_HIP(hipEventSynchronize(e1));
        CLG_HIP(hipEventElapsedTime(&ms, e0, e1));
        ms /= (float)reps;
        return CLG_OK;
    };
    std::vector<std::pair<float, size_t>> t;
    int status = CLG_OK;
    for (size_t i = 0; i < cands.size() && status == CLG_OK; ++i) {
        float ms = 0.f;
        status = launch(cands[i]);  // warm
        if (status == CLG_OK) status = timed(cands[i], 3, ms);
        t.emplace_back(ms, i);
        report(cands[i], ms);
    }
    std::sort(t.begin(), t.end());
    size_t near = 0;
    while (near < t.size() && near < 6 && t[near].first <= 1.15f * t[0].first) ++near;
    std::vector<float> sum(near, 0.f);
    for (int round = 0; round < 3 && near > 1; ++round)
        for (size_t q = 0; q < near && status == CLG_OK; ++q) {
            float ms = 0.f;
            const int reps = std::max(3, std::min(20, (int)(1.f / std::max(t[0].first, 1e-4f))));
            status = timed(cands[t[q].second], reps, ms);
            sum[q] += ms / 3.f;
        }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    CLG_TRY(status);
    size_t q = 0;
    for (size_t k = 1; k < near && near > 1; ++k)
        if (sum[k] < sum[q]) q = k;
    best = cands[t[q].second];
    best_ms = near > 1 ? sum[q] : t[q].first;
    return CLG_OK;
}

// launch helpers
inline unsigned grid_for(long n, int block) { return (unsigned)((n + block - 1) / block); }
// grid for clgd::map_site: nblk parity blocks of Vh sites, optional parity interleave, spt logical
// blocks per workgroup and XCD padding
inline unsigned sched_grid(long Vh, int nblk, int block, int xcd, int pinter, int spt = 1) {
    long g = (nblk == 2 && pinter) ? 2 * ((Vh + block - 1) / block) : (nblk * Vh + block - 1) / block;
    g = (g + spt - 1) / spt;
    if (xcd > 1) g = (g + xcd - 1) / xcd * xcd;
    return (unsigned)g;
}

// grid of clgd::tile64_site: 8 tiles of at most ceil(L0 / TX) x ceil(L1 / TY) planes
inline unsigned tile64_grid(const Geo& g, int nblk, int TY) {
    const int plane = g.L[2] * g.L[3] / 2, TX = 8 / TY;
    return 8u * (unsigned)(nblk * ((plane + 63) / 64) * ((g.L[0] + TX - 1) / TX) * ((g.L[1] + TY - 1) / TY));
}
// whether that schedule keeps at least 7/8 of its lanes busy
inline bool tile64_fits(const Geo& g, int TY) {
    const long lanes = 64L * tile64_grid(g, 1, TY);
    return 8L * g.Vh >= 7L * lanes;
}

// work order of the site kernels in 64-site blocks: the tiled plane order where it keeps the lanes busy
// (neighbour planes then meet in one XCD's L2), else XCD slabs.  Gauge force at 32^3x16: eight tiles along y
// 322 us, 2 x 4 tiles 341, 4 x 2 tiles 346, slabs 344; at 21x19x25x18, where a plane of 225 sites fills 3.5 of 4
// blocks and the tiles at most 0.80 of the lanes, all within 1 %.
struct SiteOrder {
    int tile_y;  // 0: slabs
    unsigned grid;
};
inline SiteOrder site_order(const Geo& g) {
    if (tile64_fits(g, 8)) return SiteOrder{8, tile64_grid(g, 2, 8)};
    return SiteOrder{0, sched_grid(g.Vh, 2, 64, 8, 1)};
}
}  // namespace clg

// ======================================================================= device side
namespace clgd {

template <typename R> struct C2 { R x, y; };
typedef C2<double> cd;
typedef C2<float> cf;

template <typename R> __device__ __forceinline__ C2<R> cmk(R a, R b) { return C2<R>{a, b}; }
template <typename R> __device__ __forceinline__ C2<R> cadd(C2<R> a, C2<R> b) { return {a.x + b.x, a.y + b.y}; }
template <typename R> __device__ __forceinline__ C2<R> csub(C2<R> a, C2<R> b) { return {a.x - b.x, a.y - b.y}; }
template <typename R> __device__ __forceinline__ C2<R> cmul(C2<R> a, C2<R> b) {
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// conj(a) * b
template <typename R> __device__ __forceinline__ C2<R> cmulc(C2<R> a, C2<R> b) {
    return {a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x};
}
template <typename R> __device__ __forceinline__ C2<R> cconj(C2<R> a) { return {a.x, -a.y}; }
template <typename R> __device__ __forceinline__ C2<R> cscale(C2<R> a, R s) { return {a.x * s, a.y * s}; }
// acc += a*b
template <typename R> __device__ __forceinline__ void cfma(C2<R>& acc, C2<R> a, C2<R> b) {
    acc.x = fma(a.x, b.x, fma(-a.y, b.y, acc.x));
    acc.y = fma(a.x, b.y, fma(a.y, b.x, acc.y));
}
// acc += conj(a)*b
template <typename R> __device__ __forceinline__ void cfmac(C2<R>& acc, C2<R> a, C2<R> b) {
    acc.x = fma(a.x, b.x, fma(a.y, b.y, acc.x));
    acc.y = fma(a.x, b.y, fma(-a.y, b.x, acc.y));
}
// i^k * a for compile-time k
template <int K, typename R> __device__ __forceinline__ C2<R> mulz4(C2<R> a) {
    if constexpr ((K & 3) == 1) return {-a.y, a.x};
    else if constexpr ((K & 3) == 2) return {-a.x, -a.y};
    else if constexpr ((K & 3) == 3) return {a.y, -a.x};
    else return a;
}

// ------------------------------------------------------------------ site geometry
struct Site {
    int c[4];
    int lex;
};
// coordinates of half-index h of parity p (Lt even)
__device__ __forceinline__ Site site_of(const clg::Geo& g, int p, int h) {
    Site s;
    const int lex0 = 2 * h;
    const int t0 = lex0 % g.L[3];
    int r = lex0 / g.L[3];
    s.c[2] = r % g.L[2];
    r /= g.L[2];
    s.c[1] = r % g.L[1];
    s.c[0] = r / g.L[1];
    const int b = (p ^ (s.c[0] + s.c[1] + s.c[2])) & 1;
    s.c[3] = t0 + b;
    s.lex = lex0 + b;
    return s;
}
struct Nbr {
    int p, h, sign;
};
template <int MU>
__device__ __forceinline__ Nbr fwd_nbr(const clg::Geo& g, const Site& s, int p) {
    Nbr n;
    int lex;
    const bool wrap = s.c[MU] == g.L[MU] - 1;
    if (wrap) {
        lex = s.lex - (g.L[MU] - 1) * g.stride[MU];
        n.sign = g.sgn[MU];
        n.p = p ^ 1 ^ (g.L[MU] & 1);
    } else {
        lex = s.lex + g.stride[MU];
        n.sign = 1;
        n.p = p ^ 1;
    }
    n.h = lex >> 1;
    return n;
}
template <int MU>
__device__ __forceinline__ Nbr bwd_nbr(const clg::Geo& g, const Site& s, int p) {
    Nbr n;
    int lex;
    const bool wrap = s.c[MU] == 0;
    if (wrap) {
        lex = s.lex + (g.L[MU] - 1) * g.stride[MU];
        n.sign = g.sgn[MU];
        n.p = p ^ 1 ^ (g.L[MU] & 1);
    } else {
        lex = s.lex - g.stride[MU];
        n.sign = 1;
        n.p = p ^ 1;
    }
    n.h = lex >> 1;
    return n;
}

// ------------------------------------------------------------------ work decomposition
// Workgroups are handed to the 8 XCDs round-robin (wg -> XCD wg % 8), and each XCD has its
// own L2.  With xcd = 8 the hardware id is remapped so that XCD k sweeps the contiguous
// logical range [k*n/8, (k+1)*n/8): neighbouring sites, whose spinors and links are shared,
// then meet in one L2.  With pinter = 1 a two-parity launch alternates parities block by
// block, so a link's forward user (parity p) and backward user (parity 1-p) are co-resident.
// The grid must be padded to a multiple of xcd (sched_grid) for the remap to be a bijection.
// A launch with spt logical blocks per workgroup (sites per thread) gives workgroup w the
// logical blocks w*spt .. w*spt+spt-1 after the remap, so each XCD still sweeps one range.
__device__ __forceinline__ unsigned logical_wg(int xcd) {
    unsigned wg = blockIdx.x;
    if (xcd > 1) {
        const unsigned per = gridDim.x / (unsigned)xcd;
        wg = (wg % (unsigned)xcd) * per + wg / (unsigned)xcd;
    }
    return wg;
}
// site (p, h) of lane `tid` in logical block lb of `bs` sites
__device__ __forceinline__ bool block_site(unsigned lb, unsigned bs, unsigned tid, int Vh, int nblk, int pbase, int pinter,
                                           int& p, int& h) {
    if (nblk == 2 && pinter) {
        p = (int)(lb & 1u);
        h = (int)((lb >> 1) * bs + tid);
        return h < Vh;
    }
    const long gid = (long)lb * bs + tid;
    if (gid >= (long)nblk * Vh) return false;
    const int blk = (int)(gid / Vh);
    h = (int)(gid - (long)blk * Vh);
    p = nblk == 2 ? blk : pbase;
    return true;
}
// the same for one site per thread: logical block lb of blockDim.x sites
__device__ __forceinline__ bool block_site(unsigned lb, int Vh, int nblk, int pbase, int pinter, int& p, int& h) {
    return block_site(lb, blockDim.x, threadIdx.x, Vh, nblk, pbase, pinter, p, h);
}
// Tiled plane schedule for launches of one workgroup per (x,y) plane (blockDim = L2*L3/2 sites of one
// parity; nblk = 2 interleaves the parities plane by plane): the L0 x L1 grid of planes is cut into
// 8 tiles, 8/TY along x and TY along y, and XCD k (hardware workgroups k, k+8, ...) sweeps tile k,
// x-major (y fastest) or y-major.  A plane's x+-1 and y+-1 neighbour planes then come up within
// 2*L1/TY (x-major) workgroups of it in the same XCD's L2, instead of a whole x-slab later.  Needs
// L0 % (8/TY) == 0, L1 % TY == 0 and a grid of exactly nblk*L0*L1 workgroups.
__device__ __forceinline__ unsigned tile_block(const clg::Geo& g, int nblk, int TY, int ymajor) {
    const unsigned wg = blockIdx.x;
    const unsigned k = wg & 7u, j = wg >> 3;
    const int TX = 8 / TY;
    const int tx = g.L[0] / TX, ty = g.L[1] / TY;
    const int ix = (int)k / TY, iy = (int)k % TY;
    const unsigned par = nblk == 2 ? (j & 1u) : 0u;
    const int q = (int)(nblk == 2 ? (j >> 1) : j);
    int xl, yl;
    if (ymajor) {
        yl = q / tx;
        xl = q - yl * tx;
    } else {
        xl = q / ty;
        yl = q - xl * ty;
    }
    const unsigned P = (unsigned)((ix * tx + xl) * g.L[1] + iy * ty + yl);
    return nblk == 2 ? 2u * P + par : P;
}
// The same schedule in blocks of 64 sites for any lattice: a plane's L2*L3/2 sites of one parity are
// ceil(plane / 64) blocks (the last one partly idle), the tile borders are rounded where the extents do not
// divide, and an XCD with a smaller tile leaves its last blocks idle.  Grid: tile64_grid.  What it buys
// over XCD slabs is the reuse distance in x: at 24^3x48 a slab step is 10.6 MB of FP32 links and spinors,
// past the 4 MB L2, a tile step 2.6 MB (direction-split FP32 half hop 46 -> 38 us, FP64 D 200 -> 158 us).
__device__ __forceinline__ bool tile64_site(const clg::Geo& g, int nblk, int pbase, int TY, int ymajor, int lane, int& p,
                                            int& h) {
    const int plane = g.L[2] * g.L[3] / 2, nsub = (plane + 63) / 64, TX = 8 / TY;
    const int k = (int)(blockIdx.x & 7u), j = (int)(blockIdx.x >> 3);
    const int ix = k / TY, iy = k % TY;
    const int x0 = ix * g.L[0] / TX, y0 = iy * g.L[1] / TY;
    const int tx = (ix + 1) * g.L[0] / TX - x0, ty = (iy + 1) * g.L[1] / TY - y0;
    const int sub = j % nsub;
    int q = j / nsub;
    p = pbase;
    if (nblk == 2) {
        p = q & 1;
        q >>= 1;
    }
    h = 0;
    if (q >= tx * ty) return false;
    const int major = q / (ymajor ? tx : ty), minor = q - major * (ymajor ? tx : ty);
    const int x = x0 + (ymajor ? minor : major), y = y0 + (ymajor ? major : minor);
    h = (x * g.L[1] + y) * plane + sub * 64 + lane;
    return sub * 64 + lane < plane;
}
// site of a full-lattice launch in clg::site_order
__device__ __forceinline__ bool order_site(const clg::Geo& g, int tile_y, int lane, int& p, int& h) {
    return tile_y ? tile64_site(g, 2, 0, tile_y, 0, lane, p, h) : block_site(logical_wg(8), 64, (unsigned)lane, g.Vh, 2, 0, 1, p, h);
}
__device__ __forceinline__ bool map_site(int Vh, int nblk, int pbase, int xcd, int pinter, int& p, int& h) {
    return block_site(logical_wg(xcd), Vh, nblk, pbase, pinter, p, h);
}

// ------------------------------------------------------------------ storage traits
// Every field is a uniform base pointer plus a set of planes.  An element index e selects
// one site inside the planes (e = block * NPL * Vh + h for a field of several blocks), and
// plane k of that site sits at base + k*Vh*CH + e*CH.  The element index is 32-bit; the byte
// offset is formed in 64 bits, so a field may exceed 4 GiB.
__device__ __forceinline__ size_t plane_off(int Vh, int k, unsigned e, size_t ch) {
    return ((size_t)k * (size_t)Vh + (size_t)e) * ch;
}
template <typename T>
__device__ __forceinline__ T ldp(const char* base, int Vh, int k, unsigned e) {
    return *reinterpret_cast<const T*>(base + plane_off(Vh, k, e, sizeof(T)));
}
template <typename T>
__device__ __forceinline__ void stp(char* base, int Vh, int k, unsigned e, T v) {
    *reinterpret_cast<T*>(base + plane_off(Vh, k, e, sizeof(T))) = v;
}

// Non-temporal form of ldp (the "nt" cache policy: the line is marked for early eviction), for data
// a kernel reads exactly once, so it does not displace data that is read again (neighbour spinors).
template <typename T> struct NtVec;
template <> struct NtVec<double2> { typedef double V __attribute__((ext_vector_type(2))); };
template <> struct NtVec<float2> { typedef float V __attribute__((ext_vector_type(2))); };
template <> struct NtVec<float4> { typedef float V __attribute__((ext_vector_type(4))); };
template <> struct NtVec<uint2> { typedef unsigned V __attribute__((ext_vector_type(2))); };
template <> struct NtVec<uint4> { typedef unsigned V __attribute__((ext_vector_type(4))); };
template <> struct NtVec<unsigned> { typedef unsigned V; };
template <typename T, bool NT>
__device__ __forceinline__ T ldq(const char* base, int Vh, int k, unsigned e) {
    if constexpr (NT) {
        typedef typename NtVec<T>::V V;
        const V* p = reinterpret_cast<const V*>(base + plane_off(Vh, k, e, sizeof(T)));
        const V v = __builtin_nontemporal_load(p);
        T out;
        __builtin_memcpy(&out, &v, sizeof(T));
        return out;
    } else {
        return ldp<T>(base, Vh, k, e);
    }
}

// store form of ldq: with NT the line is written with the non-temporal policy (streamed towards memory
// and marked for early eviction), for outputs no later read of the same launch wants in the cache
template <typename T, bool NT>
__device__ __forceinline__ void stq(char* base, int Vh, int k, unsigned e, T v) {
    if constexpr (NT) {
        typedef typename NtVec<T>::V V;
        V* p = reinterpret_cast<V*>(base + plane_off(Vh, k, e, sizeof(T)));
        V x;
        __builtin_memcpy(&x, &v, sizeof(T));
        __builtin_nontemporal_store(x, p);
    } else {
        stp<T>(base, Vh, k, e, v);
    }
}

// FP16 storage helpers
__device__ __forceinline__ unsigned pack_h2(float a, float b) {
    __half2 h = __floats2half2_rn(a, b);
    return *reinterpret_cast<unsigned*>(&h);
}
__device__ __forceinline__ float2 unpack_h2(unsigned u) {
    __half2 h = *reinterpret_cast<__half2*>(&u);
    return __half22float2(h);
}

// FP16-storage Wilson sites as flat BLAS sees them: site i of a field of Vh-site parity blocks has
// its three 16-byte chunks at chunk index (3 * (i / Vh) + k) * Vh + i % Vh and its scale at s[i].
__device__ __forceinline__ size_t h16_chunk(unsigned i, unsigned Vh, int k) {
    const unsigned b = i / Vh, h = i - b * Vh;
    return (size_t)(3 * b + k) * Vh + h;
}
__device__ __forceinline__ void h16_unpack8(uint4 a, float s, float* v) {
    float2 f;
    f = unpack_h2(a.x); v[0] = f.x * s; v[1] = f.y * s;
    f = unpack_h2(a.y); v[2] = f.x * s; v[3] = f.y * s;
    f = unpack_h2(a.z); v[4] = f.x * s; v[5] = f.y * s;
    f = unpack_h2(a.w); v[6] = f.x * s; v[7] = f.y * s;
}
// all 24 components of site i
__device__ __forceinline__ void h16_load_site(const uint4* c, const float* s, unsigned Vh, unsigned i, float* v) {
    const float sc = s[i];
#pragma unroll
    for (int k = 0; k < 3; ++k) h16_unpack8(c[h16_chunk(i, Vh, k)], sc, v + 8 * k);
}
// stores site i with a new scale; v is left holding the stored (rounded) values
__device__ __forceinline__ void h16_store_site(uint4* c, float* s, unsigned Vh, unsigned i, float* v) {
    float m = 0.f;
#pragma unroll
    for (int q = 0; q < 24; ++q) m = fmaxf(m, fabsf(v[q]));
    const float inv = m > 0.f ? 1.0f / m : 0.f;
    s[i] = m;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint4 a;
        a.x = pack_h2(v[8 * k + 0] * inv, v[8 * k + 1] * inv);
        a.y = pack_h2(v[8 * k + 2] * inv, v[8 * k + 3] * inv);
        a.z = pack_h2(v[8 * k + 4] * inv, v[8 * k + 5] * inv);
        a.w = pack_h2(v[8 * k + 6] * inv, v[8 * k + 7] * inv);
        c[h16_chunk(i, Vh, k)] = a;
        h16_unpack8(a, m, v + 8 * k);
    }
}


// Wilson spinor: 12 complex numbers per site.
//   F64: 12 planes of double2; F32: 6 planes of float4 (two complex); F16: 3 planes of 8
//   halves plus a per-site float scale (max |component|), element index ne for the scale.
template <int PREC> struct WilsonIO;

template <> struct WilsonIO<CLG_F64> {
    static constexpr int NPL = 12;
    static constexpr bool SCALED = false;
    template <typename R>
    __device__ __forceinline__ static void load(const char* b, const float*, int Vh, unsigned e, unsigned, C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            const double2 a = ldp<double2>(b, Vh, k, e);
            v[k] = C2<R>{(R)a.x, (R)a.y};
        }
    }
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store(char* b, float*, int Vh, unsigned e, unsigned, const C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 12; ++k) stq<double2, NT>(b, Vh, k, e, make_double2((double)v[k].x, (double)v[k].y));
    }
    // components 4 w .. 4 w + 3 only (a third of the site)
    template <typename R>
    __device__ __forceinline__ static void load4(const char* b, const float*, int Vh, unsigned e, unsigned, int w, C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double2 a = ldp<double2>(b, Vh, 4 * w + k, e);
            v[k] = C2<R>{(R)a.x, (R)a.y};
        }
    }
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store4(char* b, int Vh, unsigned e, int w, const C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 4; ++k) stq<double2, NT>(b, Vh, 4 * w + k, e, make_double2((double)v[k].x, (double)v[k].y));
    }
};

template <> struct WilsonIO<CLG_F32> {
    static constexpr int NPL = 6;
    static constexpr bool SCALED = false;
    template <typename R>
    __device__ __forceinline__ static void load(const char* b, const float*, int Vh, unsigned e, unsigned, C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const float4 a = ldp<float4>(b, Vh, k, e);
            v[2 * k] = C2<R>{(R)a.x, (R)a.y};
            v[2 * k + 1] = C2<R>{(R)a.z, (R)a.w};
        }
    }
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store(char* b, float*, int Vh, unsigned e, unsigned, const C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 6; ++k)
            stq<float4, NT>(b, Vh, k, e,
                            make_float4((float)v[2 * k].x, (float)v[2 * k].y, (float)v[2 * k + 1].x, (float)v[2 * k + 1].y));
    }
    template <typename R>
    __device__ __forceinline__ static void load4(const char* b, const float*, int Vh, unsigned e, unsigned, int w, C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float4 a = ldp<float4>(b, Vh, 2 * w + k, e);
            v[2 * k] = C2<R>{(R)a.x, (R)a.y};
            v[2 * k + 1] = C2<R>{(R)a.z, (R)a.w};
        }
    }
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store4(char* b, int Vh, unsigned e, int w, const C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            stq<float4, NT>(b, Vh, 2 * w + k, e,
                        make_float4((float)v[2 * k].x, (float)v[2 * k].y, (float)v[2 * k + 1].x, (float)v[2 * k + 1].y));
    }
};

template <> struct WilsonIO<CLG_F16> {
    static constexpr int NPL = 3;
    static constexpr bool SCALED = true;
    // the stored halves without the site scale, which is returned (a hop scales the projected
    // half-spinor instead: 12 products instead of 24)
    template <typename R>
    __device__ __forceinline__ static float load_unscaled(const char* b, const float* nb, int Vh, unsigned e, unsigned ne,
                                                          C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint4 a = ldp<uint4>(b, Vh, k, e);
            float2 f;
            f = unpack_h2(a.x); v[4 * k + 0] = C2<R>{(R)f.x, (R)f.y};
            f = unpack_h2(a.y); v[4 * k + 1] = C2<R>{(R)f.x, (R)f.y};
            f = unpack_h2(a.z); v[4 * k + 2] = C2<R>{(R)f.x, (R)f.y};
            f = unpack_h2(a.w); v[4 * k + 3] = C2<R>{(R)f.x, (R)f.y};
        }
        return nb[ne];
    }
    template <typename R>
    __device__ __forceinline__ static void load(const char* b, const float* nb, int Vh, unsigned e, unsigned ne, C2<R>* v) {
        const float s = nb[ne];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint4 a = ldp<uint4>(b, Vh, k, e);
            float2 f;
            f = unpack_h2(a.x); v[4 * k + 0] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
            f = unpack_h2(a.y); v[4 * k + 1] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
            f = unpack_h2(a.z); v[4 * k + 2] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
            f = unpack_h2(a.w); v[4 * k + 3] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
        }
    }
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store(char* b, float* nb, int Vh, unsigned e, unsigned ne, const C2<R>* v) {
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < 12; ++k) m = fmaxf(m, fmaxf(fabsf((float)v[k].x), fabsf((float)v[k].y)));
        const float inv = m > 0.f ? 1.0f / m : 0.f;
        nb[ne] = m;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            uint4 a;
            a.x = pack_h2((float)v[4 * k + 0].x * inv, (float)v[4 * k + 0].y * inv);
            a.y = pack_h2((float)v[4 * k + 1].x * inv, (float)v[4 * k + 1].y * inv);
            a.z = pack_h2((float)v[4 * k + 2].x * inv, (float)v[4 * k + 2].y * inv);
            a.w = pack_h2((float)v[4 * k + 3].x * inv, (float)v[4 * k + 3].y * inv);
            stq<uint4, NT>(b, Vh, k, e, a);
        }
    }
    template <typename R>
    __device__ __forceinline__ static void load4(const char* b, const float* nb, int Vh, unsigned e, unsigned ne, int w,
                                                 C2<R>* v) {
        const float s = nb[ne];
        const uint4 a = ldp<uint4>(b, Vh, w, e);
        float2 f;
        f = unpack_h2(a.x); v[0] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
        f = unpack_h2(a.y); v[1] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
        f = unpack_h2(a.z); v[2] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
        f = unpack_h2(a.w); v[3] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
    }
    // v already divided by the site scale, which the caller stores
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store4(char* b, int Vh, unsigned e, int w, const C2<R>* v) {
        uint4 a;
        a.x = pack_h2((float)v[0].x, (float)v[0].y);
        a.y = pack_h2((float)v[1].x, (float)v[1].y);
        a.z = pack_h2((float)v[2].x, (float)v[2].y);
        a.w = pack_h2((float)v[3].x, (float)v[3].y);
        stq<uint4, NT>(b, Vh, w, e, a);
    }
};

// Staggered vector: 3 complex per site, one complex per plane (16 / 8 / 4 bytes)
template <int PREC> struct KSIO;
template <> struct KSIO<CLG_F64> {
    static constexpr int NPL = 3;
    template <typename R>
    __device__ __forceinline__ static void load(const char* b, const float*, int Vh, unsigned e, unsigned, C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 3; ++k) { const double2 a = ldp<double2>(b, Vh, k, e); v[k] = C2<R>{(R)a.x, (R)a.y}; }
    }
    template <typename R>
    __device__ __forceinline__ static void store(char* b, float*, int Vh, unsigned e, unsigned, const C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 3; ++k) stp<double2>(b, Vh, k, e, make_double2((double)v[k].x, (double)v[k].y));
    }
    // colour k only
    template <typename R>
    __device__ __forceinline__ static void load1(const char* b, int Vh, int k, unsigned e, C2<R>& v) {
        const double2 a = ldp<double2>(b, Vh, k, e);
        v = C2<R>{(R)a.x, (R)a.y};
    }
    template <typename R>
    __device__ __forceinline__ static void store1(char* b, int Vh, int k, unsigned e, C2<R> v) {
        stp<double2>(b, Vh, k, e, make_double2((double)v.x, (double)v.y));
    }
};
template <> struct KSIO<CLG_F32> {
    static constexpr int NPL = 3;
    template <typename R>
    __device__ __forceinline__ static void load(const char* b, const float*, int Vh, unsigned e, unsigned, C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 3; ++k) { const float2 a = ldp<float2>(b, Vh, k, e); v[k] = C2<R>{(R)a.x, (R)a.y}; }
    }
    template <typename R>
    __device__ __forceinline__ static void store(char* b, float*, int Vh, unsigned e, unsigned, const C2<R>* v) {
#pragma unroll
        for (int k = 0; k < 3; ++k) stp<float2>(b, Vh, k, e, make_float2((float)v[k].x, (float)v[k].y));
    }
    // colour k only
    template <typename R>
    __device__ __forceinline__ static void load1(const char* b, int Vh, int k, unsigned e, C2<R>& v) {
        const float2 a = ldp<float2>(b, Vh, k, e);
        v = C2<R>{(R)a.x, (R)a.y};
    }
    template <typename R>
    __device__ __forceinline__ static void store1(char* b, int Vh, int k, unsigned e, C2<R> v) {
        stp<float2>(b, Vh, k, e, make_float2((float)v.x, (float)v.y));
    }
};
template <> struct KSIO<CLG_F16> {
    static constexpr int NPL = 3;
    template <typename R>
    __device__ __forceinline__ static void load(const char* b, const float* nb, int Vh, unsigned e, unsigned ne, C2<R>* v) {
        const float s = nb[ne];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float2 f = unpack_h2(ldp<unsigned>(b, Vh, k, e));
            v[k] = C2<R>{(R)(f.x * s), (R)(f.y * s)};
        }
    }
    template <typename R, bool NT = false>
    __device__ __forceinline__ static void store(char* b, float* nb, int Vh, unsigned e, unsigned ne, const C2<R>* v) {
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < 3; ++k) m = fmaxf(m, fmaxf(fabsf((float)v[k].x), fabsf((float)v[k].y)));
        const float inv = m > 0.f ? 1.0f / m : 0.f;
        nb[ne] = m;
#pragma unroll
        for (int k = 0; k < 3; ++k) stp<unsigned>(b, Vh, k, e, pack_h2((float)v[k].x * inv, (float)v[k].y * inv));
    }
};

// Gauge links: 8 blocks (parity, mu) of Vh links each; element index e = (p*4+mu)*NPL*Vh + h.
// 18-real: 9 planes of one complex; 12-real: rows 0,1 only, row 2 = conj(r0 x r1) as
// SU3::Norm builds it (SU3.h:1083-1085).
template <typename R>
__device__ __forceinline__ void rebuild_row2(C2<R>* m) {
    m[6] = cconj(csub(cmul(m[1], m[5]), cmul(m[2], m[4])));
    m[7] = cconj(csub(cmul(m[2], m[3]), cmul(m[0], m[5])));
    m[8] = cconj(csub(cmul(m[0], m[4]), cmul(m[1], m[3])));
}

template <int PREC, int RECON> struct LinkIO;
template <> struct LinkIO<CLG_F64, 18> {
    static constexpr int NPL = 9;
    template <bool NT = false, typename R>
    __device__ __forceinline__ static void load(const char* b, int Vh, unsigned e, C2<R>* m) {
#pragma unroll
        for (int k = 0; k < 9; ++k) { const double2 a = ldq<double2, NT>(b, Vh, k, e); m[k] = C2<R>{(R)a.x, (R)a.y}; }
    }
    template <bool NT = false>
    __device__ __forceinline__ static void store(char* b, int Vh, unsigned e, const cd* m) {
#pragma unroll
        for (int k = 0; k < 9; ++k) stq<double2, NT>(b, Vh, k, e, make_double2(m[k].x, m[k].y));
    }
};
template <> struct LinkIO<CLG_F64, 12> {
    static constexpr int NPL = 6;
    template <bool NT = false, typename R>
    __device__ __forceinline__ static void load(const char* b, int Vh, unsigned e, C2<R>* m) {
#pragma unroll
        for (int k = 0; k < 6; ++k) { const double2 a = ldq<double2, NT>(b, Vh, k, e); m[k] = C2<R>{(R)a.x, (R)a.y}; }
        rebuild_row2(m);
    }
    __device__ __forceinline__ static void store(char* b, int Vh, unsigned e, const cd* m) {
#pragma unroll
        for (int k = 0; k < 6; ++k) stp<double2>(b, Vh, k, e, make_double2(m[k].x, m[k].y));
    }
};
template <> struct LinkIO<CLG_F32, 18> {
    static constexpr int NPL = 9;
    template <bool NT = false, typename R>
    __device__ __forceinline__ static void load(const char* b, int Vh, unsigned e, C2<R>* m) {
#pragma unroll
        for (int k = 0; k < 9; ++k) { const float2 a = ldq<float2, NT>(b, Vh, k, e); m[k] = C2<R>{(R)a.x, (R)a.y}; }
    }
    __device__ __forceinline__ static void store(char* b, int Vh, unsigned e, const cd* m) {
#pragma unroll
        for (int k = 0; k < 9; ++k) stp<float2>(b, Vh, k, e, make_float2((float)m[k].x, (float)m[k].y));
    }
};
template <> struct LinkIO<CLG_F32, 12> {
    static constexpr int NPL = 3;
    template <bool NT = false, typename R>
    __device__ __forceinline__ static void load(const char* b, int Vh, unsigned e, C2<R>* m) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float4 a = ldq<float4, NT>(b, Vh, k, e);
            m[2 * k] = C2<R>{(R)a.x, (R)a.y};
            m[2 * k + 1] = C2<R>{(R)a.z, (R)a.w};
        }
        rebuild_row2(m);
    }
    __device__ __forceinline__ static void store(char* b, int Vh, unsigned e, const cd* m) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            stp<float4>(b, Vh, k, e,
                        make_float4((float)m[2 * k].x, (float)m[2 * k].y, (float)m[2 * k + 1].x, (float)m[2 * k + 1].y));
    }
};
template <> struct LinkIO<CLG_F16, 18> {
    static constexpr int NPL = 9;
    template <bool NT = false, typename R>
    __device__ __forceinline__ static void load(const char* b, int Vh, unsigned e, C2<R>* m) {
#pragma unroll
        for (int k = 0; k < 9; ++k) { const float2 f = unpack_h2(ldq<unsigned, NT>(b, Vh, k, e)); m[k] = C2<R>{(R)f.x, (R)f.y}; }
    }
    __device__ __forceinline__ static void store(char* b, int Vh, unsigned e, const cd* m) {
#pragma unroll
        for (int k = 0; k < 9; ++k) stp<unsigned>(b, Vh, k, e, pack_h2((float)m[k].x, (float)m[k].y));
    }
};
template <> struct LinkIO<CLG_F16, 12> {
    static constexpr int NPL = 3;
    template <bool NT = false, typename R>
    __device__ __forceinline__ static void load(const char* b, int Vh, unsigned e, C2<R>* m) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint2 a = ldq<uint2, NT>(b, Vh, k, e);
            const float2 f0 = unpack_h2(a.x), f1 = unpack_h2(a.y);
            m[2 * k] = C2<R>{(R)f0.x, (R)f0.y};
            m[2 * k + 1] = C2<R>{(R)f1.x, (R)f1.y};
        }
        rebuild_row2(m);
    }
    __device__ __forceinline__ static void store(char* b, int Vh, unsigned e, const cd* m) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            stp<uint2>(b, Vh, k, e,
                       make_uint2(pack_h2((float)m[2 * k].x, (float)m[2 * k].y),
                                  pack_h2((float)m[2 * k + 1].x, (float)m[2 * k + 1].y)));
    }
};

// y = U x and y = U^dagger x on colour 3-vectors
template <typename R>
__device__ __forceinline__ void su3_mv(const C2<R>* u, const C2<R>* x, C2<R>* y) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        C2<R> a = cmul(u[3 * i], x[0]);
        cfma(a, u[3 * i + 1], x[1]);
        cfma(a, u[3 * i + 2], x[2]);
        y[i] = a;
    }
}
template <typename R>
__device__ __forceinline__ void su3_mdv(const C2<R>* u, const C2<R>* x, C2<R>* y) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        C2<R> a = cmulc(u[i], x[0]);
        cfmac(a, u[3 + i], x[1]);
        cfmac(a, u[6 + i], x[2]);
        y[i] = a;
    }
}

// ------------------------------------------------------------------ SU(3) helpers
// r = a b
template <typename R>
__device__ __forceinline__ void su3_mm(const C2<R>* a, const C2<R>* b, C2<R>* r) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            C2<R> acc = cmul(a[3 * i], b[j]);
            cfma(acc, a[3 * i + 1], b[3 + j]);
            cfma(acc, a[3 * i + 2], b[6 + j]);
            r[3 * i + j] = acc;
        }
}
// traceless anti-Hermitian part (SU3::Ta, SU3.h:953-984)
__device__ __forceinline__ void su3_ta(cd* m) {
    const cd n1 = csub(m[1], cconj(m[3]));
    const cd n2 = csub(m[2], cconj(m[6]));
    const cd n5 = csub(m[5], cconj(m[7]));
    m[1] = cscale(n1, 0.5);
    m[3] = cd{-m[1].x, m[1].y};
    m[2] = cscale(n2, 0.5);
    m[6] = cd{-m[2].x, m[2].y};
    m[5] = cscale(n5, 0.5);
    m[7] = cd{-m[5].x, m[5].y};
    const double tr = (m[0].y + m[4].y + m[8].y) / 3.0;
    m[0] = cd{0.0, m[0].y - tr};
    m[4] = cd{0.0, m[4].y - tr};
    m[8] = cd{0.0, m[8].y - tr};
}
// re-unitarisation as SU3::Norm does it (SU3.h:1058-1088): Gram-Schmidt on rows 0 and 1,
// row 2 = conj(r0 x r1)
__device__ __forceinline__ void su3_reunit(cd* m) {
    const double d1 = 1.0 / sqrt(m[0].x * m[0].x + m[0].y * m[0].y + m[1].x * m[1].x + m[1].y * m[1].y +
                                 m[2].x * m[2].x + m[2].y * m[2].y);
    m[0] = cscale(m[0], d1); m[1] = cscale(m[1], d1); m[2] = cscale(m[2], d1);
    cd sp = cadd(cadd(cmul(m[0], cconj(m[3])), cmul(m[1], cconj(m[4]))), cmul(m[2], cconj(m[5])));
    sp = cconj(sp);
    m[3] = csub(m[3], cmul(sp, m[0])); m[4] = csub(m[4], cmul(sp, m[1])); m[5] = csub(m[5], cmul(sp, m[2]));
    const double d2 = 1.0 / sqrt(m[3].x * m[3].x + m[3].y * m[3].y + m[4].x * m[4].x + m[4].y * m[4].y +
                                 m[5].x * m[5].x + m[5].y * m[5].y);
    m[3] = cscale(m[3], d2); m[4] = cscale(m[4], d2); m[5] = cscale(m[5], d2);
    rebuild_row2(m);
}

// ------------------------------------------------------------------ random numbers
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11), counter = (index, draw, stream, c3),
// key = (seed, 0x434C4721); two uniforms of 53 bits -> one Box-Muller pair of N(0,1)
__device__ __forceinline__ void philox(unsigned c0, unsigned c1, unsigned c2, unsigned c3, unsigned k0,
                                       unsigned k1, unsigned out[4]) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const unsigned hi0 = __umulhi(0xD2511F53u, c0), lo0 = 0xD2511F53u * c0;
        const unsigned hi1 = __umulhi(0xCD9E8D57u, c2), lo1 = 0xCD9E8D57u * c2;
        const unsigned n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}
__device__ __forceinline__ double u53(unsigned a, unsigned b) {
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6) + 0.5) * (1.0 / 9007199254740992.0);
}
__device__ __forceinline__ void gauss2(unsigned idx, unsigned draw, unsigned stream, unsigned seed, double g[2],
                                       unsigned c3 = 0u) {
    unsigned w[4];
    philox(idx, draw, stream, c3, seed, 0x434C4721u, w);
    const double u1 = u53(w[0], w[1]), u2 = u53(w[2], w[3]);
    const double r = sqrt(-2.0 * log(u1));
    double s, c;
    sincos(6.283185307179586476925286766559 * u2, &s, &c);
    g[0] = r * c;
    g[1] = r * s;
}
enum { STREAM_GAUGE = 0, STREAM_WILSON = 1, STREAM_KS = 2, STREAM_MOMENTUM = 3, STREAM_GAUGE_TRANSFORM = 4 };

// reunitarise(exp(i eps H)) for H traceless Hermitian with Gaussian entries drawn from stream `stream`
// at counter `idx`, by Taylor scaling-and-squaring (the same recipe as the oracle's generator)
__device__ inline void random_su3(unsigned idx, double eps, unsigned seed, unsigned stream, cd* out) {
    double g[10];
    for (int d = 0; d < 5; ++d) gauss2(idx, (unsigned)d, stream, seed, g + 2 * d);
    const double tr = (g[0] + g[1] + g[2]) / 3.0;
    const double is2 = 0.70710678118654752440084436210485;
    cd H[9];
    H[0] = cd{g[0] - tr, 0.0};
    H[4] = cd{g[1] - tr, 0.0};
    H[8] = cd{g[2] - tr, 0.0};
    H[1] = cd{g[3] * is2, g[4] * is2};
    H[2] = cd{g[5] * is2, g[6] * is2};
    H[5] = cd{g[7] * is2, g[8] * is2};
    H[3] = cconj(H[1]);
    H[6] = cconj(H[2]);
    H[7] = cconj(H[5]);
    cd A[9];
    double nrm = 0;
    for (int i = 0; i < 9; ++i) {
        A[i] = cd{-eps * H[i].y, eps * H[i].x};
        nrm += A[i].x * A[i].x + A[i].y * A[i].y;
    }
    nrm = sqrt(nrm);
    int s = 0;
    while (nrm > 0.5) { nrm *= 0.5; ++s; }
    const double f = ldexp(1.0, -s);
    for (int i = 0; i < 9; ++i) A[i] = cscale(A[i], f);
    cd T[9], S[9], tmp[9];
    for (int i = 0; i < 9; ++i) T[i] = cd{0.0, 0.0};
    T[0] = T[4] = T[8] = cd{1.0, 0.0};
    for (int i = 0; i < 9; ++i) S[i] = T[i];
    for (int k = 1; k <= 20; ++k) {
        su3_mm(T, A, tmp);
        for (int i = 0; i < 9; ++i) { T[i] = cscale(tmp[i], 1.0 / k); S[i] = cadd(S[i], T[i]); }
    }
    for (int k = 0; k < s; ++k) {
        su3_mm(S, S, tmp);
        for (int i = 0; i < 9; ++i) S[i] = tmp[i];
    }
    su3_reunit(S);
    for (int i = 0; i < 9; ++i) out[i] = S[i];
}


// ------------------------------------------------------------------ grid reductions
constexpr int kRedBlock = 256;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Totals of N per-lane FP64 values over the 64 lanes, written to dst[0..N) (LDS, this wave's row).  N butterflies
// would take 6 N shuffles; folding halves the values a lane carries at every step (lanes on either side of the
// exchange keep half of them each), about N + 5 shuffles, after which each lane holds one total.
template <int N, int OFF>
__device__ __forceinline__ void wave_fold_step(double* v, int lane, int first, int count, double* dst) {
    if constexpr (OFF == 0) {
        if (count > 0) dst[first] = v[0];
    } else if constexpr (N == 1) {
        v[0] += __shfl_xor(v[0], OFF, 64);
        wave_fold_step<1, OFF / 2>(v, lane, first, count, dst);
    } else {
        constexpr int H = (N + 1) / 2;
        const bool up = (lane & OFF) != 0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const double lo = v[i], hi = i + H < N ? v[i + H] : 0.0;
            v[i] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, OFF, 64);
        }
        wave_fold_step<H, OFF / 2>(v, lane, up ? first + H : first, up ? max(count - H, 0) : min(count, H), dst);
    }
}
template <int N>
__device__ __forceinline__ void wave_fold(double (&v)[N], double* dst) {
    wave_fold_step<N, 32>(v, (int)(threadIdx.x & 63), 0, N, dst);
}

// Block-level stage of a two-kernel grid reduction: sums NR per-lane FP64 values over the
// workgroup (blockDim.x <= kRedBlock, a multiple of 64) and writes them to
// partial[blockIdx.x * NR + r].  No fence or counter: the finishing kernel launched after it on the
// same stream sees every partial.  (A device-scope release fence per workgroup costs a
// cross-XCD L2 write-back on gfx950: tens of microseconds over a 1024-block grid.)
template <int NR>
__device__ void block_partial(double (&v)[NR], double* partial) {
    __shared__ double sm[kRedBlock / 64][NR];
    const int nw = blockDim.x >> 6;
    wave_fold<NR>(v, sm[threadIdx.x >> 6]);
    __syncthreads();
    for (int r = threadIdx.x; r < NR; r += blockDim.x) {
        double s = 0;
        for (int w = 0; w < nw; ++w) s += sm[w][r];
        partial[(size_t)blockIdx.x * NR + r] = s;
    }
}

// Totals tot[0..nr) (LDS) of nblk x nr row-major partials by one workgroup of BLOCK threads, in a fixed order:
// thread (q, r) sums value r of blocks q, q + G, ..., neighbouring threads reading neighbouring values, then
// up to 32 strands (never more than G) and one fold the G rows.  nr <= kFinMax.  Measured for 25 values of 24
// blocks: the finish 5.5 -> 3.8 us (a thread per block with nr strided accumulators and nr wave butterflies before).
constexpr int kFinBlock = 1024, kFinMax = 33;
template <int BLOCK>
__device__ __forceinline__ void partial_totals(const double* __restrict__ partial, int nblk, int nr, double* tot) {
    __shared__ double rows[BLOCK];
    __shared__ double strands[8 * kFinMax];
    const int G = BLOCK / nr, S = min(G, nr <= 2 ? 32 : nr <= 8 ? 16 : 8), r = (int)threadIdx.x % nr, q = (int)threadIdx.x / nr;
    double a = 0.0;
    if (q < G) {
#pragma unroll 8
        for (int b = q; b < nblk; b += G) a += partial[(size_t)b * nr + r];
        rows[threadIdx.x] = a;
    }
    __syncthreads();
    if (q < S) {
        double t = 0.0;
        for (int i = q; i < G; i += S) t += rows[i * nr + r];
        strands[threadIdx.x] = t;
    }
    __syncthreads();
    if ((int)threadIdx.x < nr) {
        double t = 0.0;
        for (int i = 0; i < S; ++i) t += strands[i * nr + threadIdx.x];
        tot[threadIdx.x] = t;
    }
    __syncthreads();
}

// Least-squares solution of the (m+1) x m Hessenberg system H y = sqrt(beta2) e_1 by one wave (m <= 64): Givens
// rotations and back substitution as RotateH / SolveY (CSolverGMRES.cpp:262-358), FP64.  H is column-major with
// leading dimension ld; sm holds m * ld complex numbers of LDS.  Lane j carries column j: a rotation is one
// broadcast and four products a lane, and the back substitution eliminates column by column.  A column of
// zeros (the vectors after an invariant subspace) gets y = 0.  dev[0] = |g_m|^2, dev[1] = |g_m|.  Measured for
// m = 12: 7.7 us (one thread on global memory: 28).
__device__ __forceinline__ cd lane_bcast(cd a, int src) { return cd{__shfl(a.x, src, 64), __shfl(a.y, src, 64)}; }
// With *bad set (a refused fast Gram-Schmidt step in the cycle) y is zero; dev[2] passes it on.
__device__ __forceinline__ void gmres_lsq_wave(const double* __restrict__ H, int ld, int m, double beta2, double* y,
                                               double* dev, cd* sm, const double* bad = nullptr) {
    const int lane = (int)(threadIdx.x & 63), col = min(lane, m - 1);
    for (int i = lane; i < m * ld; i += 64) sm[i] = cd{H[2 * i], H[2 * i + 1]};
    __syncthreads();
    cd cur = sm[col * ld], g = cd{sqrt(beta2), 0.0}, z = cd{0.0, 0.0};
    for (int k = 0; k < m; ++k) {
        const cd nxt = sm[col * ld + k + 1];  // below the subdiagonal of columns < k: not used
        const cd hkk = lane_bcast(cur, k), hk1 = lane_bcast(nxt, k);
        const double n2 = hkk.x * hkk.x + hkk.y * hkk.y + hk1.x * hk1.x + hk1.y * hk1.y;
        const double den = n2 == 0.0 ? 0.0 : 1.0 / sqrt(n2);
        const cd cs = n2 == 0.0 ? cd{1.0, 0.0} : cscale(hkk, den), sn = cscale(hk1, den);
        const cd gk = cmul(cconj(cs), g);
        g = cmul(sn, cd{-g.x, -g.y});
        if (lane == k) z = gk;
        if (lane >= k && lane < m) {
            sm[col * ld + k] = cadd(cmul(cconj(cs), cur), cmul(cconj(sn), nxt));
            cur = csub(cmul(cs, nxt), cmul(sn, cur));
        }
    }
    if (lane == 0) {
        dev[0] = g.x * g.x + g.y * g.y;
        dev[1] = sqrt(dev[0]);
        if (bad) dev[2] = *bad;
    }
    if (bad && *bad != 0.0) {
        if (lane < m) y[2 * lane] = y[2 * lane + 1] = 0.0;
        return;
    }
    __syncthreads();
    for (int k = m - 1; k >= 0; --k) {
        const cd d = sm[k * ld + k], acc = lane_bcast(z, k);
        const double dd = d.x * d.x + d.y * d.y;
        const cd yk = dd == 0.0 ? cd{0.0, 0.0}
                                : cd{(acc.x * d.x + acc.y * d.y) / dd, (acc.y * d.x - acc.x * d.y) / dd};
        if (lane == k) z = yk;
        else if (lane < k) z = csub(z, cmul(sm[k * ld + lane], yk));
    }
    if (lane < m) {
        y[2 * lane] = z.x;
        y[2 * lane + 1] = z.y;
    }
}

// ---- Gram-Schmidt steps of GMRES: Hessenberg column hcol (column j, interleaved complex) from the projections
// the column of the fast form from the projections h
template <int K>
__device__ __forceinline__ void gs_fast_column(const double* h, double w2, double* hcol, int j, int shifted) {
    const int i = threadIdx.x;
    if (i < K) {
        hcol[2 * i] = shifted ? (i == j ? 1.0 : 0.0) - h[2 * i] : h[2 * i];
        hcol[2 * i + 1] = shifted ? -h[2 * i + 1] : h[2 * i + 1];
    }
    if (i == 0) {
        const double f = sqrt(w2);
        hcol[2 * (j + 1)] = shifted ? -f : f;
        hcol[2 * (j + 1) + 1] = 0.0;
    }
}
// the step's scalars from h and |w|^2: the scale of w' (0 where the fast form does not hold); workgroup 0 writes
// the column and notes in sc[clg::kGsBad] whether any fast step of the cycle (j = 1 is its first) was refused
template <int K>
__device__ __forceinline__ double gs_fast_scalars(const double* h, double w2, double* hcol, int j, double* sc) {
    double b2 = w2;
#pragma unroll
    for (int k = 0; k < 2 * K; ++k) b2 -= h[k] * h[k];
    const bool ok = b2 >= 0.5 * w2 && b2 > 1e-300;
    if (blockIdx.x == 0) {
        gs_fast_column<K>(h, ok ? b2 : 0.0, hcol, j, 1);
        if (threadIdx.x == 0) {
            if (!ok) sc[clg::kGsBad] = 1.0;
            else if (j == 1) sc[clg::kGsBad] = 0.0;
        }
    }
    return ok ? 1.0 / sqrt(b2) : 0.0;
}

}  // namespace clgd

