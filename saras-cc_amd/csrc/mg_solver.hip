// mg_solver.hip -- device-resident multigrid hierarchy and the C-ABI of
// include/saras_hip.h.
//
// The host drives the reference's V-cycle (lib/poisson/poisson.cc:203-279)
// level by level on one HIP stream; all level arrays stay in HBM between
// calls, as the reference's poisson object keeps its hierarchy between time
// steps (timestep.h:142).  Two arithmetic modes:
//   SARAS_PREC_FP64  - the reference algorithm in FP64, bit-exact with the
//                      FP64 CPU build for the L-inf residual type;
//   SARAS_PREC_MIXED - FP64 residual and iterative refinement around FP32
//                      V-cycles on the correction equation A e = r.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <array>
#include <vector>

#include "grid_host.hpp"
#include "mg_fused.hpp"
#include "mg_internal.hpp"
#include "mg_kernels.hpp"
#include "mg_split.hpp"
#include "mg_tail.hpp"
#include "mg_tile.hpp"
#include "saras_hip.h"

namespace {

thread_local std::string g_last_error;

void set_error(const std::string &s) { g_last_error = s; }

#define HIP_TRY(expr)                                                                   \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess) {                                                         \
            set_error(std::string(#expr) + ": " + hipGetErrorString(e_));               \
            return e_ == hipErrorOutOfMemory ? SARAS_OOM : SARAS_HIP_ERROR;             \
        }                                                                               \
    } while (0)

constexpr int kThreads = 256;
inline unsigned blocks_for(long n) { return (unsigned)std::max<long>(1, (n + kThreads - 1) / kThreads); }

template <typename T>
long row_pitch(int nz) {
    const long a = 128 / (long)sizeof(T);
    return (nz + a - 1) / a * a;
}

template <typename T>
struct DevLevel {
    int n[3] = {0, 0, 0};
    long sx = 0, sy = 0;
    size_t elems = 0;  // allocation size in elements
    T *x = nullptr, *b = nullptr;
    T *xalt = nullptr;  // second iterate buffer: fused sweeps and tiles run out of place
    // the visits of a V-cycle by tiles (k_tile): pre-smoothing from a zero
    // iterate (and, level 0, from any) with the restriction, post-smoothing
    // with the prolongation; no launches: by separate passes
    saras::TilePlan pre, pre0, post;
    long hz = 0;        // colour-split rows when > 0 (offset of the odd half)
    T *c2zs = nullptr, *c1zs = nullptr;  // z coefficients in split order
    bool uniform = false;                // every axis has one value of c2 and one of c1
    T *c2[3] = {nullptr, nullptr, nullptr}, *c1[3] = {nullptr, nullptr, nullptr};
    T *rlo[3] = {nullptr, nullptr, nullptr}, *rhi[3] = {nullptr, nullptr, nullptr}, *rwd[3] = {nullptr, nullptr, nullptr};
};

// The small constant arrays of a hierarchy, gathered on the host and sent in one
// allocation and one transfer (each pair of them takes about 10 us; a 32^3 mixed
// handle has some 170 arrays: making one took 1.8 ms with a pair for each).
template <typename T>
struct ConstImage {
    std::vector<T> data;
    std::vector<std::pair<T **, size_t>> at;   // array pointers to set and their places
    // every array starts at a multiple of 256 bytes, as an allocation does
    void add(T **dst, const std::vector<double> &src) {
        at.emplace_back(dst, data.size());
        data.insert(data.end(), src.begin(), src.end());
        constexpr size_t kAlign = 256 / sizeof(T);
        data.resize((data.size() + kAlign - 1) / kAlign * kAlign);
    }
    saras_status send(T **base) {
        HIP_TRY(hipMalloc((void **)base, std::max<size_t>(1, data.size()) * sizeof(T)));
        HIP_TRY(hipMemcpy(*base, data.data(), data.size() * sizeof(T), hipMemcpyHostToDevice));
        for (auto &p : at) *p.first = *base + p.second;
        return SARAS_OK;
    }
};

template <typename T>
struct Hierarchy {
    int dim = 3;
    std::vector<DevLevel<T>> lv;
    T *image = nullptr;   // the levels' constant arrays and `wall`
    T *wall[3] = {nullptr, nullptr, nullptr};   // DIRICHLET_TEST level-0 wall values
    T *coarse_scratch = nullptr;
    bool coarse_lds = true;
    size_t coarse_lds_bytes = 0;
    bool split_rows = false;   // store levels whose rows split into whole vectors colour-split
    // host copies of the metric coefficients (c2, c1) and restriction
    // factors (lo, hi, wd) per level and axis, for the tail's packed image
    std::vector<std::array<std::vector<double>, 3>> hc2, hc1, hlo, hhi, hwd;
    // the tail kernel's levels tail_first..D (D + 1: no tail), its arguments
    // and LDS size, and the packed images of its coefficients and cell tables
    int tail_first = -1;
    saras::TailArgs<T> tail_args{};
    size_t tail_bytes = 0;
    unsigned *tail_image = nullptr;

    // a level takes split rows when each half-row is a whole number of 16-byte vectors
    static bool splittable(int nz) {
        constexpr int W = 16 / (int)sizeof(T);
        return nz >= 2 * W && nz % (2 * W) == 0;
    }

    ~Hierarchy() {
        for (auto &L : lv) {
            (void)hipFree(L.x); (void)hipFree(L.b); (void)hipFree(L.xalt);
        }
        (void)hipFree(image);
        (void)hipFree(coarse_scratch);
        (void)hipFree(tail_image);
    }

    saras_status build(const saras::GridLevels &G, const std::vector<std::vector<double>> &walls) {
        dim = G.dim;
        const int D = G.depth;
        lv.resize(D + 1);
        ConstImage<T> img;
        hc2.assign(D + 1, {});
        hc1.assign(D + 1, {});
        hlo.assign(D + 1, {});
        hhi.assign(D + 1, {});
        hwd.assign(D + 1, {});
        for (int l = 0; l <= D; ++l) {
            DevLevel<T> &L = lv[l];
            for (int a = 0; a < 3; ++a) L.n[a] = G.axes[l][a].n;
            if (dim == 2) L.n[1] = 1;
            L.sy = row_pitch<T>(L.n[2]);
            L.sx = L.sy * (long)L.n[1];
            L.elems = (size_t)L.sx * L.n[0];
            L.hz = split_rows && splittable(L.n[2]) ? L.sy / 2 : 0;
            HIP_TRY(hipMalloc((void **)&L.x, L.elems * sizeof(T)));
            HIP_TRY(hipMalloc((void **)&L.b, L.elems * sizeof(T)));
            HIP_TRY(hipMemset(L.x, 0, L.elems * sizeof(T)));
            if (l < D && dim == 3 && L.hz == 0) {
                HIP_TRY(hipMalloc((void **)&L.xalt, L.elems * sizeof(T)));
                HIP_TRY(hipMemset(L.xalt, 0, L.elems * sizeof(T)));
            }
            HIP_TRY(hipMemset(L.b, 0, L.elems * sizeof(T)));
            L.uniform = true;
            for (int a = 0; a < 3; ++a) {
                if (dim == 2 && a == 1) {
                    std::vector<double> z(1, 0.0);
                    img.add(&L.c2[a], z);
                    img.add(&L.c1[a], z);
                    hc2[l][a] = z;
                    hc1[l][a] = z;
                    continue;
                }
                const saras::AxisLevel &A = G.axes[l][a];
                // poisson::setCoefficients (poisson.cc:463-482)
                const int hInc = 1 << l;
                const double dxi = 1.0 / double(G.axes[0][a].n);
                const double h = hInc * dxi;
                const double h2 = std::pow(h, 2);
                const double i2h = 0.5 / h, ih2 = 1.0 / h2;
                std::vector<double> c2(A.n), c1(A.n);
                for (int i = 0; i < A.n; ++i) {
                    c2[i] = A.xix2[i + 1] * ih2;
                    c1[i] = A.xixx[i + 1] * i2h;
                }
                for (int i = 1; i < A.n; ++i) L.uniform = L.uniform && c2[i] == c2[0] && c1[i] == c1[0];
                img.add(&L.c2[a], c2);
                img.add(&L.c1[a], c1);
                hc2[l][a] = c2;
                hc1[l][a] = c1;
                if (a == 2 && L.hz) {
                    const int half = A.n / 2;
                    std::vector<double> c2s(A.n), c1s(A.n);
                    for (int hh = 0; hh < 2; ++hh)
                        for (int mm = 0; mm < half; ++mm) {
                            c2s[hh * half + mm] = c2[2 * mm + hh];
                            c1s[hh * half + mm] = c1[2 * mm + hh];
                        }
                    img.add(&L.c2zs, c2s);
                    img.add(&L.c1zs, c1s);
                }
                if (l > 0) {
                    // restriction factors of coarse index I (poisson_d3.cc:494-502)
                    const saras::AxisLevel &Fa = G.axes[l - 1][a];
                    std::vector<double> lo(A.n), hi(A.n), wd(A.n);
                    for (int I = 0; I < A.n; ++I) {
                        const double X = A.coord[I + 1];
                        const double f0 = Fa.coord[2 * I + 1], f1 = Fa.coord[2 * I + 2];
                        lo[I] = X - f0;
                        hi[I] = f1 - X;
                        wd[I] = f1 - f0;
                    }
                    img.add(&L.rlo[a], lo);
                    img.add(&L.rhi[a], hi);
                    img.add(&L.rwd[a], wd);
                    hlo[l][a] = lo;
                    hhi[l][a] = hi;
                    hwd[l][a] = wd;
                }
            }
        }
        for (int a = 0; a < 3; ++a)
            if (!walls[a].empty()) img.add(&wall[a], walls[a]);
        saras_status st = img.send(&image);
        if (st) return st;
        // coarsest-level workspace
        const DevLevel<T> &C = lv[D];
        const size_t padded = dim == 3 ? (size_t)(C.n[0] + 2) * (C.n[1] + 2) * (C.n[2] + 2)
                                       : (size_t)(C.n[0] + 2) * (C.n[2] + 2);
        const size_t need = (padded + (size_t)C.n[0] * C.n[1] * C.n[2]) * sizeof(T);
        // a workgroup may hold up to 64 KB of dynamic LDS without opting in
        // (k_coarse's static LDS is 128 bytes): 14^3 in FP64 fits
        coarse_lds = need <= 64 * 1024 - 256;
        coarse_lds_bytes = coarse_lds ? need : 0;
        if (!coarse_lds) HIP_TRY(hipMalloc((void **)&coarse_scratch, std::max(need, C.elems * sizeof(T))));
        return SARAS_OK;
    }
};

int bc_code(const saras_mg_params &p, const saras_grid_desc &g, int axis, int level, bool inhom_allowed, bool hi) {
    if (g.periodic[axis]) return saras::BC_PER;
    switch (p.bc) {
        // multigrid_d2::imposeBC, all-Neumann branch: probType 9 turns the
        // top wall Dirichlet (poisson_d2.cc:641-647)
        case SARAS_BC_NEUMANN: return (hi && axis == 2 && p.top_dirichlet) ? saras::BC_DIR : saras::BC_NEU;
        case SARAS_BC_DIRICHLET: return saras::BC_DIR;
        default: return (level == 0 && inhom_allowed) ? saras::BC_DIRV : saras::BC_DIR;
    }
}

}  // namespace

struct saras_mg {
    saras_grid_desc g{};
    saras_mg_params p{};
    saras::GridLevels G;
    int depth = 0;
    int max_count = 0;
    Hierarchy<double> h64;
    std::unique_ptr<Hierarchy<float>> h32;
    double *x64b = nullptr;            // second FP64 iterate buffer (MIXED)
    double *partial = nullptr;         // norm partials
    // The norm's last reduction and the coarse solves write these pinned,
    // host-coherent words directly, with no copy kernel in between: the host
    // reads the norm once its ticket shows it written, and a coarse count
    // once a later norm has been read (kernels of a stream run in order).
    double *norm_host = nullptr;       // [numerator, denominator] of computeError
    unsigned *norm_seq = nullptr;      // ticket stored after norm_host (see wait_ticket)
    unsigned norm_ticket = 0;          // ticket of the last norm launched
    int *iters_host = nullptr;         // coarse iteration count of the last coarse solve
    double *stage_x = nullptr, *stage_b = nullptr;  // device staging for host pointers
    size_t stage_elems = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int coarse_iters_max = 0;
    int coarse_capped = 0;
    bool fused_off = false;            // SARAS_NO_FUSED_SWEEP=1 forces the two-pass smoother
    bool tail_off = false;             // SARAS_NO_TAIL=1 runs every level with multi-block kernels
    int march_wgs = 0;                 // target workgroups of a march sweep (SARAS_MARCH_WGS; 0 = per type)
    bool march_tj8 = false;            // FP32 march with 64 x 8 tiles (SARAS_MARCH_TJ8=1)
    bool split_off = false;            // SARAS_NO_SPLIT=1 keeps every level z-contiguous
    size_t tail_lds = saras::kTailLds;  // dynamic LDS budget of the tail kernel (SARAS_TAIL_LDS_KB lowers it)
    bool red_fold = true;              // SARAS_NO_RED_FOLD=1: the restriction leaves the first red pass to the sweep
    bool coarse_one = false;           // SARAS_COARSE_ONE=1 smooths every coarsest level in one workgroup
    bool rb_general = false;           // SARAS_RB_GENERAL=1 runs every split colour pass in the general form
    bool rb_wide = false;              // SARAS_RB_WIDE=1 runs every split colour pass and restriction as in arrays of 4 GB and more
    bool tile_off = false;             // SARAS_NO_TILE=1 runs every pass as a launch of its own
    bool rr_lane = false;              // SARAS_RR_LANE=1: 3-D split restriction with all eight children in one lane
    // V-cycles replayed from captured hipGraphs (saras_mg_set_graphs).  A
    // graph bakes in the level buffers, and out-of-place sweeps swap them, so
    // graphs are cached per buffer state (at most two states per precision).
    bool graphs = false;
    struct GraphEntry {
        std::vector<void *> key;    // (x, xalt) of every level before the cycle
        std::vector<void *> post;   // ... and after it
        hipGraphExec_t exec;
        hipStream_t stream;
    };
    std::vector<GraphEntry> graph_cache[2];   // [0] FP64 cycles, [1] FP32 cycles

    ~saras_mg() {
        for (auto &c : graph_cache)
            for (auto &e : c) (void)hipGraphExecDestroy(e.exec);
        (void)hipFree(x64b); (void)hipFree(partial);
        (void)hipHostFree(norm_host); (void)hipHostFree(iters_host);
        (void)hipHostFree(norm_seq);
        (void)hipFree(stage_x); (void)hipFree(stage_b);
        if (ev0) (void)hipEventDestroy(ev0);
        if (ev1) (void)hipEventDestroy(ev1);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

template <typename T>
saras::LevelArgs<T> level_args(const saras_mg *m, const Hierarchy<T> &H, int l, bool inhom) {
    const DevLevel<T> &L = H.lv[l];
    saras::LevelArgs<T> a{};
    for (int q = 0; q < 3; ++q) {
        a.n[q] = L.n[q];
        a.c2[q] = L.c2[q];
        a.c1[q] = L.c1[q];
        a.bc_lo[q] = bc_code(m->p, m->g, q, l, inhom, false);
        a.bc_hi[q] = bc_code(m->p, m->g, q, l, inhom, true);
        a.wall[q] = H.wall[q];
    }
    a.sx = L.sx;
    a.sy = L.sy;
    a.hz = L.hz;
    a.c2zs = L.c2zs;
    a.c1zs = L.c1zs;
    a.rtile = 0;
    // A colour pass reads row (i+1, j) again two i-planes after its first
    // read.  Where those two planes of x and b exceed half of an XCD's 4 MB
    // L2, the rows run in j-tiles of about 256 KB of such reuse instead.
    if (L.hz && H.dim == 3) {
        const size_t half = (size_t)L.n[2] / 2 * sizeof(T);
        if (4 * (size_t)L.n[1] * half > (2u << 20)) {
            int jt = 1;
            while (jt < 256 && (size_t)(2 * jt) * 4 * half <= (256u << 10)) jt *= 2;
            while (jt > 1 && L.n[1] % jt) jt /= 2;
            if (jt >= 8) a.rtile = jt;
        }
    }
    return a;
}

// The tail's LDS layout for levels S..D (the offsets of A.L) and its bytes;
// 0 where the levels do not fit or the tail does not take them.
template <typename T>
size_t tail_layout(const saras_mg *m, const Hierarchy<T> &H, int S, saras::TailArgs<T> &A) {
    const int D = (int)H.lv.size() - 1;
    if (D - S + 1 > saras::kTailMaxLevels) return 0;
    // inhomogeneous walls (the finest level of the reference's test problem) are
    // left to the multi-workgroup kernels
    if (S == 0 && m->p.bc == SARAS_BC_DIRICHLET_TEST) return 0;
    int n[saras::kTailMaxLevels][3];
    for (int l = S; l <= D; ++l)
        for (int a = 0; a < 3; ++a) n[l - S][a] = H.lv[l].n[a];
    const int per[3] = {m->g.periodic[0] != 0, m->g.periodic[1] != 0, m->g.periodic[2] != 0};
    const saras::TailPlan P = saras::plan_tail(sizeof(T), H.dim, n, D - S + 1, per, m->p.solve_flag != 0, m->tail_lds);
    if (!P.bytes) return 0;
    A = saras::TailArgs<T>{};
    A.first = S;
    A.last = D;
    A.res = P.res;
    A.coff = P.coff;
    A.ncoef = P.ncoef;
    A.cellw = P.cellw;
    A.ncellw = P.ncellw;
    for (int l = S; l <= D; ++l) {
        const saras::TailPlan::Level &Q = P.L[l - S];
        saras::TailLevel &V = A.L[l - S];
        for (int a = 0; a < 3; ++a) V.n[a] = Q.n[a];
        V.hz = Q.hz;
        V.half = Q.half;
        V.x = Q.x;
        V.b = Q.b;
        V.old = Q.old;
        V.cell4 = Q.cell4;
        V.cell1 = Q.cell1;
        V.odd = Q.odd;
        for (int a = 0; a < 3; ++a) {
            if (H.dim == 2 && a == 1) continue;
            V.neg |= bc_code(m->p, m->g, a, l, false, false) == saras::BC_DIR ||
                     bc_code(m->p, m->g, a, l, false, true) == saras::BC_DIR;
        }
    }
    return P.bytes;
}

// The plan of one visit of level l by tiles (none: by separate passes).
template <typename T>
saras::TilePlan plan_visit(const saras_mg *m, const Hierarchy<T> &H, int l, int count, bool zero, bool pro, bool restr) {
    const DevLevel<T> &L = H.lv[l];
    if (m->tile_off || l + 1 >= (int)H.lv.size()) return {};
    for (int a = 0; a < 3; ++a)
        if (m->g.periodic[a] && !(H.dim == 2 && a == 1) && (L.n[a] & 1)) return {};
    if (l == 0 && m->p.bc == SARAS_BC_DIRICHLET_TEST) return {};
    return saras::plan_tile(sizeof(T), H.dim, L.n, L.hz > 0, count, zero, pro, restr);
}

// plans of every level, and the second iterate buffer of those that tile
template <typename T>
saras_status plan_tiles(const saras_mg *m, Hierarchy<T> &H) {
    const int D = (int)H.lv.size() - 1;
    for (int l = 0; l < std::min(H.tail_first, D); ++l) {
        DevLevel<T> &L = H.lv[l];
        L.pre = plan_visit(m, H, l, m->p.pre_smooth, true, false, true);
        if (l == 0) L.pre0 = plan_visit(m, H, l, m->p.pre_smooth, false, false, true);
        L.post = plan_visit(m, H, l, m->p.post_smooth, false, true, false);
        if ((L.pre.sweeps || L.pre0.sweeps || L.post.sweeps) && !L.xalt) {
            HIP_TRY(hipMalloc((void **)&L.xalt, L.elems * sizeof(T)));
            HIP_TRY(hipMemset(L.xalt, 0, L.elems * sizeof(T)));
        }
    }
    return SARAS_OK;
}

// The tail of a hierarchy: the levels from the finest one that fits its LDS
// budget to the coarsest (none when even that does not fit), with the images
// the kernel copies to LDS -- the coefficients as pairs (c2, c1) per level and
// axis (a pair of zeros for the planar y axis), the restriction factors lo,
// hi, wd of levels S+1..D of a 3-D hierarchy, and the cell tables.
template <typename T>
saras_status pack_tail(const saras_mg *m, Hierarchy<T> &H) {
    const int D = (int)H.lv.size() - 1;
    H.tail_first = D + 1;
    for (int S = D; S >= 0; --S) {
        saras::TailArgs<T> A;
        const size_t bytes = tail_layout(m, H, S, A);
        if (!bytes) break;
        H.tail_first = S;
        H.tail_args = A;
        H.tail_bytes = bytes;
    }
    const int S = H.tail_first;
    if (S > D) return SARAS_OK;
    saras::TailArgs<T> &A = H.tail_args;
    std::vector<double> flat;
    int coff[saras::kTailMaxLevels][3];
    for (int l = S; l <= D; ++l)
        for (int a = 0; a < 3; ++a) {
            coff[l - S][a] = A.coff + (int)flat.size();
            for (size_t q = 0; q < H.hc2[l][a].size(); ++q) {
                flat.push_back(H.hc2[l][a][q]);
                flat.push_back(H.hc1[l][a][q]);
            }
        }
    if (H.dim == 3)
        for (int l = S + 1; l <= D; ++l)
            for (int a = 0; a < 3; ++a) {
                saras::TailLevel &V = A.L[l - S];
                V.lo[a] = A.coff + (int)flat.size();
                flat.insert(flat.end(), H.hlo[l][a].begin(), H.hlo[l][a].end());
                V.hi[a] = A.coff + (int)flat.size();
                flat.insert(flat.end(), H.hhi[l][a].begin(), H.hhi[l][a].end());
                V.wd[a] = A.coff + (int)flat.size();
                flat.insert(flat.end(), H.hwd[l][a].begin(), H.hwd[l][a].end());
            }
    // host-side guard: the kernel copies ncoef elements
    if ((int)flat.size() != A.ncoef) {
        set_error("internal error: tail coefficients do not match their layout");
        return SARAS_HIP_ERROR;
    }
    // the LDS image of the cell tables, then the tables of larger levels
    std::vector<unsigned> img((size_t)A.ncellw, 0u);
    size_t gn = 0;   // entries of the tables in global memory
    for (int l = S; l <= D; ++l) {
        saras::TailLevel &V = A.L[l - S];
        if (V.cell1 >= 0) continue;
        V.cell4 = (int)gn;
        gn += (2 * (size_t)V.half + 3) / 4 * 4;
    }
    const size_t nimg = img.size();
    img.resize(nimg + 5 * gn, 0u);
    for (int l = S; l <= D; ++l) {
        const saras::TailLevel &V = A.L[l - S];
        int lo[3], hi[3];
        for (int a = 0; a < 3; ++a) {
            lo[a] = bc_code(m->p, m->g, a, l, false, false);
            hi[a] = bc_code(m->p, m->g, a, l, false, true);
        }
        std::vector<saras::TailCell> t(2 * (size_t)V.half);
        if (H.dim == 3) saras::tail_cells<3>(V, coff[l - S], lo, hi, t.data());
        else saras::tail_cells<2>(V, coff[l - S], lo, hi, t.data());
        unsigned *w4 = V.cell1 >= 0 ? img.data() + (V.cell4 - A.cellw) : img.data() + nimg + 4 * V.cell4;
        unsigned *w1 = V.cell1 >= 0 ? img.data() + (V.cell1 - A.cellw) : img.data() + nimg + 4 * gn + V.cell4;
        for (size_t q = 0; q < t.size(); ++q) {
            w4[4 * q] = t[q].a[0];
            w4[4 * q + 1] = t[q].a[1];
            w4[4 * q + 2] = t[q].a[2];
            w4[4 * q + 3] = t[q].cxy;
            w1[q] = t[q].czf;
        }
    }
    // one allocation: the cell tables, the coefficients (each at a multiple of 256
    // bytes) and the right-hand side by colour where LDS has no room for it
    const size_t cells = (img.size() + 63) / 64 * 64, words = sizeof(T) / 4;
    const std::vector<T> coef(flat.begin(), flat.end());
    const size_t ncoef = (coef.size() * words + 63) / 64 * 64;
    img.resize(cells + ncoef, 0u);
    std::memcpy(img.data() + cells, coef.data(), coef.size() * sizeof(T));
    const size_t nb = A.L[0].b < 0 ? 2 * (size_t)A.L[0].half * words : 0;
    HIP_TRY(hipMalloc((void **)&H.tail_image, (img.size() + nb) * sizeof(unsigned)));
    HIP_TRY(hipMemcpy(H.tail_image, img.data(), img.size() * sizeof(unsigned), hipMemcpyHostToDevice));
    A.coef = reinterpret_cast<const T *>(H.tail_image + cells);
    if (nb) A.bcol = reinterpret_cast<T *>(H.tail_image + cells + ncoef);
    A.cellimg = H.tail_image;
    A.cells4 = reinterpret_cast<const uint4 *>(H.tail_image + nimg);
    A.cells1 = H.tail_image + nimg + 4 * gn;
    return SARAS_OK;
}

// Level operations for one precision.  `inhom0` selects the inhomogeneous
// DIRICHLET_TEST wall values on level 0 (false for the correction equation
// of the mixed-precision refinement, whose walls are homogeneous).
template <typename T>
struct Ops {
    saras_mg *m;
    Hierarchy<T> &H;
    hipStream_t s;
    bool inhom0;
    T w;

    int pend_level = -1;  // level whose next sweep also applies the prolongation
    // level 0's iterate is zero and has not been written: set by the mixed
    // solve instead of clearing it, for a V-cycle whose first operation is a
    // split-row sweep of level 0 (the conditions are its `zero_start`)
    bool zero0 = false;
    int skip_red = -1;    // level whose next sweep's red pass the restriction already applied
    // a host-side guard that refused a launch: the caller returns this status
    // (with the message in saras_last_error) instead of the process aborting
    saras_status err = SARAS_OK;

    bool refuse(const char *what) {
        if (err == SARAS_OK) set_error(std::string("internal error: ") + what);
        err = SARAS_HIP_ERROR;
        return false;
    }

    bool inhom(int l, bool zero_bc) const { return inhom0 && l == 0 && !zero_bc; }

    // FP32 cycles solve the coarsest level to max(mgTolerance, kCoarseFp32Rel
    // max|b| of that level): the FP32 residual of a level of up to a few
    // thousand cells stalls near 1e-5 of its right-hand side
    static constexpr double kCoarseFp32Rel = 1e-4;
    double coarse_rel_floor() const { return sizeof(T) == 4 ? kCoarseFp32Rel : 0.0; }

    // one RB-SOR sweep at level l: the fused out-of-place march kernel where
    // the level tiles exactly, else the two in-place colour passes
    template <int NP, int TJ>
    void march(int l, const saras::LevelArgs<T> &a) {
        DevLevel<T> &L = H.lv[l];
        const int ntk = L.n[2] / (2 * NP), ntj = L.n[1] / TJ;
        const int tiles2d = ntk * ntj;
        const int target = m->march_wgs > 0 ? m->march_wgs : (sizeof(T) == 4 ? 512 : 2048);
        int nchunks = (target + tiles2d - 1) / tiles2d;
        nchunks = std::max(1, std::min(nchunks, L.n[0] / 8));
        const int chunk = (L.n[0] + nchunks - 1) / nchunks;
        nchunks = (L.n[0] + chunk - 1) / chunk;
        const int ntiles = nchunks * tiles2d;
        const int grid = (ntiles + saras::kXcds - 1) / saras::kXcds * saras::kXcds;
        const T *e = nullptr;
        long esx = 0, esy = 0;
        if (pend_level == l) {  // prolongation folded into this first post-smoothing sweep
            const DevLevel<T> &C = H.lv[l + 1];
            e = C.x;
            esx = C.sx;
            esy = C.sy;
            pend_level = -1;
        }
        if (l == 0)
            hipLaunchKernelGGL((saras::k_sweep_march<T, NP, TJ, true>), dim3(grid), dim3(NP * TJ), 0, s, a, L.x, L.b,
                               L.xalt, w, chunk, ntk, ntj, ntiles, e, esx, esy);
        else
            hipLaunchKernelGGL((saras::k_sweep_march<T, NP, TJ, false>), dim3(grid), dim3(NP * TJ), 0, s, a, L.x,
                               L.b, L.xalt, w, chunk, ntk, ntj, ntiles, e, esx, esy);
        std::swap(L.x, L.xalt);
    }

    bool march_ok(int l) const {
        const DevLevel<T> &L = H.lv[l];
        if (H.dim != 3 || !L.xalt || m->fused_off || L.hz) return false;
        for (int q = 0; q < 3; ++q)
            if (m->g.periodic[q] && (L.n[q] & 1)) return false;
        // the march needs many tiles and planes to pay off; smaller levels use
        // the two colour passes
        return L.n[1] % 16 == 0 && L.n[2] % 64 == 0 && (long)L.n[0] * L.n[1] * L.n[2] >= (8L << 20);
    }

    // One colour pass of a split level, in the form that plan_pass chooses (the
    // levels above the coarsest have even row counts, so all but a
    // DIRICHLET_TEST level 0 go by row pairs).
    // Time of a pass, one row per lane with branches around each load / now:
    // FP32 256^3 19.6 / 16.8 us (after the prolongation: red 33 / 20, black
    // 20 / 16.4), 512^3 180 / 150 us (279 / 197, 183 / 147), tanh z 256^3 20.1 /
    // 17.7 us; FP64 256^3 38.9 / 32.0 us (red 58 / 47.8).  512^3 FP32 moves its
    // 1.5 words per cell at 5.4 TB/s.
    template <int DIM, int MODE>
    void rb_pass(int l, const saras::LevelArgs<T> &a, int colour, const T *e, long esx, long esy, long ehz) {
        using namespace saras;
        DevLevel<T> &L = H.lv[l];
        const bool dirv = a.bc_lo[0] == BC_DIRV || a.bc_lo[2] == BC_DIRV;
        const PassPlan P = plan_pass(sizeof(T), DIM, L.n, L.elems, a.rtile, dirv, w == T(1), m->rb_general, m->rb_wide);
        // host-side guard: a launch's vector numbers
        if (!P.ok) {
            refuse("a level too large for one pass");
            return;
        }
        RowMap M;
        const unsigned q = (unsigned)(L.n[2] / 2 / Vec16<T>::W);
        const unsigned wj = DIM == 3 ? (unsigned)((a.rtile ? a.rtile : L.n[1]) / P.rows) : 1u;
        M.q = FastDiv::of(q);
        M.tile = FastDiv::of((unsigned)L.n[0] * wj);
        M.wj = FastDiv::of(wj);
        M.total = P.total;
        M.div64 = P.div64;
        const unsigned nb = (unsigned)(((size_t)P.total + kSplitThreads - 1) / kSplitThreads);
        const dim3 g((nb + kXcds - 1) / kXcds * kXcds), bl(kSplitThreads);
        if (P.rows == 1)
            hipLaunchKernelGGL((k_rb_split<T, DIM, MODE, false, false, RB_GENERAL>), g, bl, 0, s, a, M, L.x, L.b, colour, w, e, esx, esy, ehz);
        else if (P.off64)
            hipLaunchKernelGGL((k_rb_split<T, DIM, MODE, true, false, RB_PAIR64>), g, bl, 0, s, a, M, L.x, L.b, colour, w, e, esx, esy, ehz);
        else if (w != T(1))
            hipLaunchKernelGGL((k_rb_split<T, DIM, MODE, false, false, RB_PAIR>), g, bl, 0, s, a, M, L.x, L.b, colour, w, e, esx, esy, ehz);
        else if (L.uniform)
            hipLaunchKernelGGL((k_rb_split<T, DIM, MODE, true, true, RB_PAIR>), g, bl, 0, s, a, M, L.x, L.b, colour, w, e, esx, esy, ehz);
        else
            hipLaunchKernelGGL((k_rb_split<T, DIM, MODE, true, false, RB_PAIR>), g, bl, 0, s, a, M, L.x, L.b, colour, w, e, esx, esy, ehz);
    }

    template <int DIM>
    void rb_pass(int l, const saras::LevelArgs<T> &a, int colour, bool pro, bool zero, const T *e, long esx, long esy,
                 long ehz) {
        using namespace saras;
        if (zero) rb_pass<DIM, RB_ZERO>(l, a, colour, e, esx, esy, ehz);
        else if (!pro) rb_pass<DIM, RB_PLAIN>(l, a, colour, e, esx, esy, ehz);
        else if (colour == 0) rb_pass<DIM, RB_RED>(l, a, colour, e, esx, esy, ehz);
        else rb_pass<DIM, RB_BLACK>(l, a, colour, e, esx, esy, ehz);
    }

    void rb_sweep(int l, bool zero_bc) {
        DevLevel<T> &L = H.lv[l];
        auto a = level_args(m, H, l, inhom(l, zero_bc));
        if (L.hz) {
            // the first sweep after the prolongation applies it (see k_rb_split)
            const bool pro = pend_level == l;
            const T *e = nullptr;
            long esx = 0, esy = 0, ehz = 0;
            if (pro) {
                const DevLevel<T> &C = H.lv[l + 1];
                e = C.x;
                esx = C.sx;
                esy = C.sy;
                ehz = C.hz;
                pend_level = -1;
            }
            const int first = skip_red == l ? 1 : 0;
            if (first) skip_red = -1;
            // the finest level's iterate is known to be zero: its first red
            // pass reads no x and clears the black half itself
            const bool z = l == 0 && zero0 && first == 0 && !pro;
            if (l == 0) zero0 = false;
            for (int colour = first; colour < 2; ++colour) {
                const bool zc = z && colour == 0;
                if (H.dim == 3) rb_pass<3>(l, a, colour, pro, zc, e, esx, esy, ehz);
                else rb_pass<2>(l, a, colour, pro, zc, e, esx, esy, ehz);
            }
            return;
        }
        if (march_ok(l)) {
            // FP32: 64 x 16 tiles (512 lanes); FP64: 64 x 8 tiles to keep LDS per workgroup ~50 KB
            constexpr int TJ = sizeof(T) == 4 ? 16 : 8;
            if (sizeof(T) == 4 && m->march_tj8) march<32, 8>(l, a);
            else if (L.n[2] % 64 == 0 && L.n[1] % TJ == 0) march<32, TJ>(l, a);
            else if (L.n[2] % 32 == 0) march<16, 8>(l, a);
            else march<8, 8>(l, a);
            return;
        }
        const long n = (long)L.n[0] * L.n[1] * ((L.n[2] + 1) / 2);
        for (int colour = 0; colour < 2; ++colour) {
            if (H.dim == 3) {
                if (l == 0)
                    hipLaunchKernelGGL((saras::k_rb_pass<T, 3, true>), dim3(blocks_for(n)), dim3(kThreads), 0, s, a, L.x, L.b, colour, w);
                else
                    hipLaunchKernelGGL((saras::k_rb_pass<T, 3, false>), dim3(blocks_for(n)), dim3(kThreads), 0, s, a, L.x, L.b, colour, w);
            } else {
                if (l == 0)
                    hipLaunchKernelGGL((saras::k_rb_pass<T, 2, true>), dim3(blocks_for(n)), dim3(kThreads), 0, s, a, L.x, L.b, colour, w);
                else
                    hipLaunchKernelGGL((saras::k_rb_pass<T, 2, false>), dim3(blocks_for(n)), dim3(kThreads), 0, s, a, L.x, L.b, colour, w);
            }
        }
    }

    // The coarsest level, solved (mode 0) or smoothed (mode 1), by one workgroup;
    // a level too large for its LDS is smoothed by colour passes of the whole
    // chip instead.  Three sweeps in FP64, one workgroup / six passes: 14k and
    // 31k cells 257 (mean) / 25 us, 8.8k in 2-D 78 / 21 us (a pass is its launch).
    void coarse(int l, bool zero_bc, int mode, int sweeps) {
        DevLevel<T> &L = H.lv[l];
        auto a = level_args(m, H, l, inhom(l, zero_bc));
        const size_t total = (size_t)L.n[0] * L.n[1] * L.n[2];
        if (mode == 1 && !H.coarse_lds && total < 0x7fffffffull && !m->coarse_one) {
            const dim3 gr((unsigned)((total + 255) / 256)), bl(256);
            for (int c = 0; c < 2 * sweeps; ++c) {
                T *from = c & 1 ? H.coarse_scratch : L.x, *to = c & 1 ? L.x : H.coarse_scratch;
                if (H.dim == 3)
                    hipLaunchKernelGGL((saras::k_coarse_pass<T, 3>), gr, bl, 0, s, a, from, to, L.b, c & 1, w);
                else
                    hipLaunchKernelGGL((saras::k_coarse_pass<T, 2>), gr, bl, 0, s, a, from, to, L.b, c & 1, w);
            }
            return;
        }
        saras::CoarseCtl ctl{mode, sweeps, m->max_count, m->p.mg_tol, m->iters_host, coarse_rel_floor()};
        const long cells = (long)L.n[0] * L.n[1] * L.n[2];
        int threads = 64;  // power of two: the kernel's tree reduction relies on it
        while (threads < cells && threads < 1024) threads <<= 1;
        if (H.dim == 3)
            hipLaunchKernelGGL((saras::k_coarse<T, 3>), dim3(1), dim3(threads), H.coarse_lds_bytes, s, a, L.x, L.b,
                               H.coarse_scratch, H.coarse_lds ? 1 : 0, w, ctl);
        else
            hipLaunchKernelGGL((saras::k_coarse<T, 2>), dim3(1), dim3(threads), H.coarse_lds_bytes, s, a, L.x, L.b,
                               H.coarse_scratch, H.coarse_lds ? 1 : 0, w, ctl);
    }

    // poisson smooth(count) at level l (coarsest level: literal kernel)
    void smooth(int l, int count, bool zero_bc) {
        if (count <= 0) return;
        if (l == (int)H.lv.size() - 1) {
            coarse(l, zero_bc, 1, count);
            return;
        }
        for (int c = 0; c < count; ++c) rb_sweep(l, zero_bc);
    }

    // Residual and restriction of a split 3-D level.  Time of a launch, one
    // row per lane with branches around each load / now: FP32 256^3 36 / 29 us,
    // 512^3 351 / 278 us (290 without the j-tiles); FP64 256^3 75 / 53 us.
    template <bool RED>
    void rr_pair(const DevLevel<T> &F, const saras::LevelArgs<T> &fa, const saras::LevelArgs<T> &ca, DevLevel<T> &C,
                 const saras::RestrictArgs<T> &r) {
        using namespace saras;
        const unsigned q = (unsigned)(F.n[2] / 2 / Vec16<T>::W);
        const size_t total = (size_t)C.n[0] * C.n[1] * q;
        // host-side guard: task numbers stay below 2^31
        if (total + kRrTasks * kXcds > 0x7fffffffull) {
            refuse("a level too large for one restriction");
            return;
        }
        const unsigned ntask = (unsigned)total, nb = (ntask + kRrTasks - 1) / kRrTasks;
        const dim3 g((nb + kXcds - 1) / kXcds * kXcds), bl(kSplitThreads);
        // The next coarse row reads two of the four x-planes again: where those
        // and b's exceed half of an XCD's 4 MB L2, the coarse rows run in
        // j-tiles whose share of them is 512 KB at most (a power of two that
        // divides the rows).
        unsigned wj = (unsigned)C.n[1];
        const size_t plane = 4 * (size_t)F.n[2] * sizeof(T);   // of one fine row of x and b, two planes
        if (plane * F.n[1] >= (2u << 20)) {
            unsigned t = 1;
            while (t < 256 && plane * 4 * t <= (512u << 10)) t *= 2;
            while (t > 1 && C.n[1] % t) t /= 2;
            if (t >= 4) wj = t;
        }
        RowMap M;
        M.q = FastDiv::of(q);
        M.tile = FastDiv::of((unsigned)C.n[0] * wj);
        M.wj = FastDiv::of(wj);
        M.total = ntask;
        const bool dirv = fa.bc_lo[0] == BC_DIRV || fa.bc_lo[2] == BC_DIRV;
        if (dirv || m->rb_general)
            hipLaunchKernelGGL((k_rr_pair<T, RED, false, RB_GENERAL>), g, bl, 0, s, fa, F.x, F.b, ca, C.b, C.x, r, M, w);
        else if (F.elems * sizeof(T) > 0xffffffffull || m->rb_wide)
            hipLaunchKernelGGL((k_rr_pair<T, RED, false, RB_PAIR64>), g, bl, 0, s, fa, F.x, F.b, ca, C.b, C.x, r, M, w);
        else if (F.uniform)
            hipLaunchKernelGGL((k_rr_pair<T, RED, true, RB_PAIR>), g, bl, 0, s, fa, F.x, F.b, ca, C.b, C.x, r, M, w);
        else
            hipLaunchKernelGGL((k_rr_pair<T, RED, false, RB_PAIR>), g, bl, 0, s, fa, F.x, F.b, ca, C.b, C.x, r, M, w);
    }

    // red_next: the restriction also applies the coarse level's first
    // pre-smoothing red pass (split levels; see k_rr_split)
    void resid_restrict(int l, bool red_next = false) {
        // host-side guard: never launch past the hierarchy
        if (l < 0 || l + 1 >= (int)H.lv.size()) {
            refuse("restriction from a level outside the hierarchy");
            return;
        }
        DevLevel<T> &F = H.lv[l], &C = H.lv[l + 1];
        auto fa = level_args(m, H, l, inhom(l, false));
        auto ca = level_args(m, H, l + 1, false);
        saras::RestrictArgs<T> r{};
        for (int q = 0; q < 3; ++q) {
            r.lo[q] = C.rlo[q];
            r.hi[q] = C.rhi[q];
            r.wd[q] = C.rwd[q];
        }
        const long n = (long)C.n[0] * C.n[1] * C.n[2];
        if (F.hz && H.dim == 3 && !m->rr_lane) {
            const bool red = red_next && C.hz;
            if (red) skip_red = l + 1;
            if (red) rr_pair<true>(F, fa, ca, C, r);
            else rr_pair<false>(F, fa, ca, C, r);
            return;
        }
        if (F.hz) {
            constexpr int W = saras::rr_width<T>();
            const long total = (long)C.n[0] * C.n[1] * (F.n[2] / 2 / W);
            const int nb = (int)((total + saras::kSplitThreads - 1) / saras::kSplitThreads);
            const int grid = (nb + saras::kXcds - 1) / saras::kXcds * saras::kXcds;
            const bool red = red_next && C.hz;
            if (red) skip_red = l + 1;
            if (H.dim == 3) {
                if (red)
                    hipLaunchKernelGGL((saras::k_rr_split<T, 3, true>), dim3(grid), dim3(saras::kSplitThreads), 0, s,
                                       fa, F.x, F.b, ca, C.b, C.x, r, nb, w);
                else
                    hipLaunchKernelGGL((saras::k_rr_split<T, 3, false>), dim3(grid), dim3(saras::kSplitThreads), 0, s,
                                       fa, F.x, F.b, ca, C.b, C.x, r, nb, w);
            } else {
                if (red)
                    hipLaunchKernelGGL((saras::k_rr_split<T, 2, true>), dim3(grid), dim3(saras::kSplitThreads), 0, s,
                                       fa, F.x, F.b, ca, C.b, C.x, r, nb, w);
                else
                    hipLaunchKernelGGL((saras::k_rr_split<T, 2, false>), dim3(grid), dim3(saras::kSplitThreads), 0, s,
                                       fa, F.x, F.b, ca, C.b, C.x, r, nb, w);
            }
            return;
        }
        if (H.dim == 3)
            hipLaunchKernelGGL((saras::k_resid_restrict<T, 3>), dim3(blocks_for(n)), dim3(kThreads), 0, s, fa, F.x, F.b,
                               ca, C.b, C.x, r);
        else
            hipLaunchKernelGGL((saras::k_resid_restrict<T, 2>), dim3(blocks_for(n)), dim3(kThreads), 0, s, fa, F.x, F.b,
                               ca, C.b, C.x, r);
    }

    void prolong_correct(int l) {
        // host-side guard: never launch past the hierarchy
        if (l < 0 || l + 1 >= (int)H.lv.size()) {
            refuse("prolongation onto a level outside the hierarchy");
            return;
        }
        DevLevel<T> &F = H.lv[l], &C = H.lv[l + 1];
        const long n = (long)F.n[0] * F.n[1] * F.n[2];
        if (F.hz) {
            constexpr int W = saras::Vec16<T>::W;
            const long total = (long)F.n[0] * F.n[1] * (F.n[2] / 2 / W);
            const int nb = (int)((total + saras::kSplitThreads - 1) / saras::kSplitThreads);
            const int grid = (nb + saras::kXcds - 1) / saras::kXcds * saras::kXcds;
            hipLaunchKernelGGL((saras::k_prolong_split<T>), dim3(grid), dim3(saras::kSplitThreads), 0, s, F.n[0],
                               F.n[1], F.n[2], F.sx, F.sy, F.hz, F.x, C.x, C.sx, C.sy, C.hz, nb);
            return;
        }
        hipLaunchKernelGGL((saras::k_prolong_correct<T>), dim3(blocks_for(n)), dim3(kThreads), 0, s, F.n[0], F.n[1],
                           F.n[2], F.sx, F.sy, F.hz, F.x, C.x, C.sx, C.sy, C.hz);
    }

    int tail_start() const { return H.tail_first; }

    template <int DIM, bool HZ, int MODE>
    void tile_launch(int grid, size_t bytes, const saras::TileArgs<T> &A) {
        hipLaunchKernelGGL((saras::k_tile<T, DIM, HZ, MODE>), dim3(grid), dim3(saras::kTileThreads), bytes, s, A);
    }
    template <int DIM>
    void tile_launch(int grid, size_t bytes, const saras::TileArgs<T> &A) {
        using namespace saras;
        if (A.L.hz) {
            if (A.zero) tile_launch<DIM, true, TILE_ZERO>(grid, bytes, A);
            else if (A.pro) tile_launch<DIM, true, TILE_PRO>(grid, bytes, A);
            else tile_launch<DIM, true, TILE_PLAIN>(grid, bytes, A);
        } else {
            if (A.zero) tile_launch<DIM, false, TILE_ZERO>(grid, bytes, A);
            else if (A.pro) tile_launch<DIM, false, TILE_PRO>(grid, bytes, A);
            else tile_launch<DIM, false, TILE_PLAIN>(grid, bytes, A);
        }
    }

    // `count` sweeps of level l by tiles of plan t, at most t.sweeps of them a
    // launch: the first launch takes `zero` or `pro`, the last one `restr`
    void tile(int l, const saras::TilePlan &t, int count, bool zero, bool pro, bool restr) {
        DevLevel<T> &L = H.lv[l];
        const int ntj = H.dim == 3 ? (L.n[1] + t.tj - 1) / t.tj : 1;
        for (int done = 0; done < count; done += t.sweeps) {
            const bool first = done == 0, last = done + t.sweeps >= count;
            saras::TileArgs<T> A{};
            A.L = level_args(m, H, l, false);
            A.x = L.x;
            A.y = L.xalt;
            A.b = L.b;
            A.ti = t.ti;
            A.tj = t.tj;
            A.nti = (L.n[0] + t.ti - 1) / t.ti;
            A.ntj = ntj;
            A.sweeps = std::min(t.sweeps, count - done);
            A.zero = zero && first;
            A.pro = pro && first;
            A.restr = restr && last;
            A.halo = saras::tile_halo(A.sweeps, A.zero, A.restr);
            A.w = w;
            if (A.pro) {
                const DevLevel<T> &C = H.lv[l + 1];
                A.e = C.x;
                A.esx = C.sx;
                A.esy = C.sy;
                A.ehz = C.hz;
            }
            if (A.restr) {
                DevLevel<T> &C = H.lv[l + 1];
                A.C = level_args(m, H, l + 1, false);
                A.cb = C.b;
                A.cx = C.x;
                for (int q = 0; q < 3; ++q) {
                    A.R.lo[q] = C.rlo[q];
                    A.R.hi[q] = C.rhi[q];
                    A.R.wd[q] = C.rwd[q];
                }
            }
            const size_t bytes = saras::tile_bytes(sizeof(T), H.dim, L.n[2], t.ti, t.tj, A.halo);
            // host-side guards of what the kernel assumes
            if (!L.xalt || bytes > saras::kTileLds || (L.n[2] & 1) || saras::tile_vecs(sizeof(T), L.n[2]) > saras::kTileThreads ||
                A.halo > L.n[0] || (H.dim == 3 && A.halo > L.n[1])) {
                refuse("a level that does not tile");
                return;
            }
            const int ntile = A.nti * A.ntj, grid = (ntile + saras::kXcds - 1) / saras::kXcds * saras::kXcds;
            if (H.dim == 3) tile_launch<3>(grid, bytes, A);
            else tile_launch<2>(grid, bytes, A);
            std::swap(L.x, L.xalt);
        }
    }

    // pre-smoothing of level l < D and the residual's restriction; `zero`: the iterate is zero
    void descend(int l, bool zero, bool red_next) {
        const auto &t = zero ? H.lv[l].pre : H.lv[l].pre0;
        if (t.sweeps) {
            tile(l, t, m->p.pre_smooth, zero, false, true);
            return;
        }
        smooth(l, m->p.pre_smooth, l != 0);
        resid_restrict(l, red_next);
    }

    void tail(int S) {
        const int D = (int)H.lv.size() - 1;
        // host-side guard: the tail packed for this hierarchy
        if (S != H.tail_first || S > D || H.tail_bytes > m->tail_lds || (H.tail_args.bcol && S != D)) {
            refuse("tail levels not packed");
            return;
        }
        saras::TailArgs<T> A = H.tail_args;
        A.x = H.lv[S].x;
        A.b = H.lv[S].b;
        A.sx = H.lv[S].sx;
        A.sy = H.lv[S].sy;
        A.hz = H.lv[S].hz;
        A.pre = m->p.pre_smooth;
        A.post = m->p.post_smooth;
        A.solve_flag = m->p.solve_flag;
        A.max_count = m->max_count;
        A.w = w;
        A.tol = m->p.mg_tol;
        A.rel_floor = coarse_rel_floor();
        A.iters_out = m->iters_host;
        if (H.dim == 3) tail_launch<3>(A);
        else tail_launch<2>(A);
    }
    template <int DIM>
    void tail_launch(const saras::TailArgs<T> &A) {
        const dim3 g(1), bl(saras::kTailThreads);
        if (A.bcol) hipLaunchKernelGGL((saras::k_tail<T, DIM, true>), g, bl, H.tail_bytes, s, A);
        else hipLaunchKernelGGL((saras::k_tail<T, DIM, false>), g, bl, H.tail_bytes, s, A);
    }

    // poisson::vCycle (poisson.cc:203-279); levels S..D run in the tail kernel
    void vcycle() {
        const int D = (int)H.lv.size() - 1;
        const int S = m->tail_off ? D + 1 : tail_start();
        if (S == 0) {
            tail(0);
            return;
        }
        if (D == 0) smooth(0, m->p.pre_smooth, false);
        for (int l = 0; l < D; ++l) {
            // the restriction also takes the coarse level's first red pass where that level runs by passes
            const bool red = m->red_fold && l + 1 < S && l + 1 < D && m->p.pre_smooth > 0 && !H.lv[l + 1].pre.sweeps;
            const bool zero = l > 0 || zero0;
            if (l == 0 && H.lv[0].pre.sweeps) zero0 = false;
            descend(l, zero, red);
            if (l + 1 == S) break;
            if (l + 1 == D) {
                if (m->p.solve_flag) coarse(D, true, 0, 0);
                else smooth(D, m->p.pre_smooth, true);
            }
        }
        if (S <= D) tail(S);
        for (int l = std::min(S, D) - 1; l >= 0; --l) {
            if (H.lv[l].post.sweeps) {
                tile(l, H.lv[l].post, m->p.post_smooth, false, true, false);
                continue;
            }
            if (m->p.post_smooth > 0 && (march_ok(l) || H.lv[l].hz)) pend_level = l;
            else prolong_correct(l);
            smooth(l, m->p.post_smooth, l != 0);
        }
    }
};

// One V-cycle of `ops`, eager or replayed from the handle's graph cache.
template <typename T>
saras_status run_vcycle(saras_mg *m, Ops<T> &ops) {
    if (!m->graphs) {
        ops.vcycle();
        return ops.err;
    }
    auto &cache = m->graph_cache[sizeof(T) == 4 ? 1 : 0];
    std::vector<void *> key;
    for (auto &L : ops.H.lv) {
        key.push_back((void *)L.x);
        key.push_back((void *)L.xalt);
    }
    for (auto &e : cache)
        if (e.key == key && e.stream == ops.s) {
            HIP_TRY(hipGraphLaunch(e.exec, ops.s));
            // the replayed cycle's buffer swaps, applied on the host side
            for (size_t l = 0; l < ops.H.lv.size(); ++l) {
                ops.H.lv[l].x = (T *)e.post[2 * l];
                ops.H.lv[l].xalt = (T *)e.post[2 * l + 1];
            }
            return SARAS_OK;
        }
    hipGraph_t g = nullptr;
    std::lock_guard<std::recursive_mutex> lk(saras::alloc_mutex());
    HIP_TRY(hipStreamBeginCapture(ops.s, hipStreamCaptureModeThreadLocal));
    ops.vcycle();
    hipError_t ce = hipStreamEndCapture(ops.s, &g);
    if (ops.err) {
        if (g) (void)hipGraphDestroy(g);
        return ops.err;
    }
    if (ce != hipSuccess) {
        set_error(std::string("hipStreamEndCapture: ") + hipGetErrorString(ce));
        return SARAS_HIP_ERROR;
    }
    hipGraphExec_t exec = nullptr;
    hipError_t ie = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ie != hipSuccess) {
        set_error(std::string("hipGraphInstantiate: ") + hipGetErrorString(ie));
        return SARAS_HIP_ERROR;
    }
    std::vector<void *> post;
    for (auto &L : ops.H.lv) {
        post.push_back((void *)L.x);
        post.push_back((void *)L.xalt);
    }
    cache.push_back({key, post, exec, ops.s});
    HIP_TRY(hipGraphLaunch(exec, ops.s));
    return SARAS_OK;
}

// Whether the FP64 residual passes of level 0 take k_refine_march: split rows,
// homogeneous walls, and arrays (the caller's padded one the largest) and
// vector numbers within 32 bits.
bool refine_marches(const saras_mg *m, const saras::LevelArgs<double> &a) {
    const size_t full = (size_t)(a.n[0] + 2 * m->g.pad) * (a.n[1] + 2 * m->g.pad) * (a.n[2] + 2 * m->g.pad) * 8;
    const size_t own = (size_t)a.sx * a.n[0] * 8, vecs = (size_t)a.n[0] * a.n[1] * (a.n[2] / 4);
    return a.hz && a.bc_lo[0] != saras::BC_DIRV && a.bc_lo[2] != saras::BC_DIRV && std::max(full, own) <= 0xffffffffull &&
           vecs + saras::kNormBlocks * saras::kNormThreads <= 0x7fffffffull && !m->rb_general;
}

// One FP64 residual pass (see k_refine_split for what the flags mean).  Times,
// k_refine_split / k_refine_march (us), 256^3 and 512^3: the norm alone 63 / 44
// (6.1 TB/s) at 256^3; the initial residual of a mixed solve 104 / 75, 914 / 658;
// the refinement from the caller's iterate 144 / 114, 1235 / 944, between
// split arrays 142 / 113, 1193 / 928, into the caller's iterate 166 / 126,
// 1414 / 1010.  (Issuing all loads of k_refine_split first, without the march,
// gave 133 and 1240 for the third: its re-reads bound it.)
template <int TYPE, int DIM, bool NORM_ONLY, bool E, bool CX, bool CB, bool CXO, bool NOXW>
void launch_refine_march(saras_mg *m, const saras::LevelArgs<double> &a, const double *x, const float *e, long esx,
                        long esy, long ehz, const double *b, float *r32, const saras::FullRows &fr, hipStream_t s) {
    using namespace saras;
    MarchMap M;
    const unsigned q = (unsigned)(a.n[2] / 4);
    M.plane = (DIM == 3 ? (unsigned)a.n[1] : 1u) * q;
    const unsigned pb = (M.plane + kNormThreads - 1) / kNormThreads;
    // as many chunks of planes as there are blocks for: a chunk reads two
    // planes more than it owns, but on the levels where chunks get that short
    // (single planes up to about 160 x 64 x 96) the pass is bound by latency
    const unsigned chunks = std::max(1u, std::min((unsigned)kNormBlocks / std::min(pb, (unsigned)kNormBlocks), (unsigned)a.n[0]));
    M.len = (int)((a.n[0] + chunks - 1) / chunks);
    M.q = FastDiv::of(q);
    M.pb = FastDiv::of(pb);
    M.items = pb * (unsigned)((a.n[0] + M.len - 1) / M.len);
    const dim3 g(kNormBlocks), bl(kNormThreads);
    if (TYPE == 0 && m->h64.lv[0].uniform)
        hipLaunchKernelGGL((k_refine_march<TYPE, DIM, NORM_ONLY, E, CX, CB, CXO, NOXW, TYPE == 0>), g, bl, 0, s, a, M, x, e,
                           esx, esy, ehz, b, m->x64b, r32, m->partial, fr);
    else
        hipLaunchKernelGGL((k_refine_march<TYPE, DIM, NORM_ONLY, E, CX, CB, CXO, NOXW, false>), g, bl, 0, s, a, M, x, e, esx,
                           esy, ehz, b, m->x64b, r32, m->partial, fr);
}

template <int DIM>
void launch_norm(int type, saras_mg *m, const saras::LevelArgs<double> &a, const double *x, const double *b,
                 hipStream_t s) {
    if (a.hz) {
        // split rows: the vectorised residual pass, norms only
        const unsigned nb = saras::kNormBlocks, nt = saras::kNormThreads;
        const saras::FullRows none{};
        if (refine_marches(m, a)) {
            if (type == 0) launch_refine_march<0, DIM, true, false, false, false, false, false>(m, a, x, nullptr, 0, 0, 0, b, nullptr, none, s);
            else if (type == 1) launch_refine_march<1, DIM, true, false, false, false, false, false>(m, a, x, nullptr, 0, 0, 0, b, nullptr, none, s);
            else launch_refine_march<2, DIM, true, false, false, false, false, false>(m, a, x, nullptr, 0, 0, 0, b, nullptr, none, s);
        } else if (type == 0)
            hipLaunchKernelGGL((saras::k_refine_split<0, DIM, true>), dim3(nb), dim3(nt), 0, s, a, x, nullptr, 0L, 0L,
                               0L, b, nullptr, nullptr, m->partial, saras::FullRows{});
        else if (type == 1)
            hipLaunchKernelGGL((saras::k_refine_split<1, DIM, true>), dim3(nb), dim3(nt), 0, s, a, x, nullptr, 0L, 0L,
                               0L, b, nullptr, nullptr, m->partial, saras::FullRows{});
        else
            hipLaunchKernelGGL((saras::k_refine_split<2, DIM, true>), dim3(nb), dim3(nt), 0, s, a, x, nullptr, 0L, 0L,
                               0L, b, nullptr, nullptr, m->partial, saras::FullRows{});
        if (type == 0)
            hipLaunchKernelGGL((saras::k_norm_final<0>), dim3(1), dim3(nt), 0, s, m->partial, saras::kNormBlocks,
                               m->norm_host, m->norm_seq, ++m->norm_ticket);
        else if (type == 1)
            hipLaunchKernelGGL((saras::k_norm_final<1>), dim3(1), dim3(nt), 0, s, m->partial, saras::kNormBlocks,
                               m->norm_host, m->norm_seq, ++m->norm_ticket);
        else
            hipLaunchKernelGGL((saras::k_norm_final<2>), dim3(1), dim3(nt), 0, s, m->partial, saras::kNormBlocks,
                               m->norm_host, m->norm_seq, ++m->norm_ticket);
        return;
    }
    switch (type) {
        case 0:
            hipLaunchKernelGGL((saras::k_norm_partial<0, DIM>), dim3(saras::kNormBlocks), dim3(saras::kNormThreads), 0,
                               s, a, x, b, m->partial);
            hipLaunchKernelGGL((saras::k_norm_final<0>), dim3(1), dim3(saras::kNormThreads), 0, s, m->partial,
                               saras::kNormBlocks, m->norm_host, m->norm_seq, ++m->norm_ticket);
            break;
        case 1:
            hipLaunchKernelGGL((saras::k_norm_partial<1, DIM>), dim3(saras::kNormBlocks), dim3(saras::kNormThreads), 0,
                               s, a, x, b, m->partial);
            hipLaunchKernelGGL((saras::k_norm_final<1>), dim3(1), dim3(saras::kNormThreads), 0, s, m->partial,
                               saras::kNormBlocks, m->norm_host, m->norm_seq, ++m->norm_ticket);
            break;
        default:
            hipLaunchKernelGGL((saras::k_norm_partial<2, DIM>), dim3(saras::kNormBlocks), dim3(saras::kNormThreads), 0,
                               s, a, x, b, m->partial);
            hipLaunchKernelGGL((saras::k_norm_final<2>), dim3(1), dim3(saras::kNormThreads), 0, s, m->partial,
                               saras::kNormBlocks, m->norm_host, m->norm_seq, ++m->norm_ticket);
            break;
    }
}

// the norm of the last k_norm_final launched on s, once it is on the host
static hipError_t wait_norm(saras_mg *m, hipStream_t s) {
    return saras::wait_ticket(m->norm_seq, m->norm_ticket, s);
}

// computeError (poisson_d3.cc:563-663): ratio formed on the host exactly as
// the reference does.
saras_status compute_error(saras_mg *m, int type, const double *x, hipStream_t s, double *out) {
    auto a = level_args(m, m->h64, 0, true);
    if (m->G.dim == 3) launch_norm<3>(type, m, a, x, m->h64.lv[0].b, s);
    else launch_norm<2>(type, m, a, x, m->h64.lv[0].b, s);
    HIP_TRY(wait_norm(m, s));
    const double num = m->norm_host[0], den = m->norm_host[1];
    const auto &L = m->h64.lv[0];
    const int pointCount = L.n[0] * L.n[1] * L.n[2];
    double r;
    if (type == 0) r = den != 0.0 ? num / den : num;
    else if (type == 1) r = den != 0.0 ? num / den : num / pointCount;
    else r = den != 0.0 ? std::sqrt(num / pointCount) / std::sqrt(den / pointCount) : std::sqrt(num / pointCount);
    *out = r;
    return SARAS_OK;
}

// the last coarse solve's iteration count, once a norm launched after it has
// been read
void note_coarse_iters(saras_mg *m) {
    const int it = *m->iters_host;
    m->coarse_iters_max = std::max(m->coarse_iters_max, it);
    if (it > m->max_count) m->coarse_capped = 1;
}


long full_elems(const saras_grid_desc &g) {
    const long p = g.pad;
    if (g.dim == 3) return (g.n[0] + 2 * p) * (long)(g.n[1] + 2 * p) * (g.n[2] + 2 * p);
    return (g.n[0] + 2 * p) * (long)(g.n[2] + 2 * p);
}

template <typename T>
void load_core(saras_mg *m, const double *full, const DevLevel<T> &L, T *dst, hipStream_t s) {
    const long n = (long)L.n[0] * L.n[1] * L.n[2];
    hipLaunchKernelGGL((saras::k_load_core<T>), dim3(blocks_for(n)), dim3(kThreads), 0, s, full, m->g.pad, m->g.dim,
                       L.n[0], L.n[1], L.n[2], L.sx, L.sy, L.hz, dst);
}

// core + the [-1, n] ghost shell, phased as the reference's final imposeBC;
// core == nullptr: the core is in `full` already, only the shell is written
void store_full(saras_mg *m, double *full, const double *core, hipStream_t s) {
    const auto &L = m->h64.lv[0];
    const long n = (long)L.n[0] * L.n[1] * L.n[2];
    if (core)
        hipLaunchKernelGGL(saras::k_store_core, dim3(blocks_for(n)), dim3(kThreads), 0, s, full, m->g.pad, m->g.dim,
                           L.n[0], L.n[1], L.n[2], L.sx, L.sy, L.hz, core);
    const int ext[3] = {L.n[0] + 2, m->g.dim == 3 ? L.n[1] + 2 : 1, L.n[2] + 2};
    for (int op = 0; op < 2; ++op)
        for (int a = 0; a < 3; ++a) {
            if (m->g.dim == 2 && a == 1) continue;
            const bool per = m->g.periodic[a] != 0;
            if ((op == 0) != per) continue;
            const int o1 = a == 0 ? 1 : 0, o2 = a == 2 ? 1 : 2;
            const long cnt = (long)ext[o1] * ext[o2];
            const int bc_lo = bc_code(m->p, m->g, a, 0, true, false), bc_hi = bc_code(m->p, m->g, a, 0, true, true);
            hipLaunchKernelGGL(saras::k_ghost_phase, dim3(blocks_for(cnt)), dim3(kThreads), 0, s, full, m->g.pad,
                               m->g.dim, L.n[0], L.n[1], L.n[2], a, op, bc_lo, bc_hi, (const double *)m->h64.wall[a]);
        }
}

std::vector<std::vector<double>> make_walls(const saras_grid_desc &g, const saras_mg_params &p) {
    std::vector<std::vector<double>> w(3);
    if (p.bc != SARAS_BC_DIRICHLET_TEST) return w;
    // initDirichlet (poisson_d3.cc:824-873, poisson_d2.cc:514-543): r^2/6 on
    // the walls from the field-grid cell centres; zero on the ghost shell
    std::vector<double> fx, fy, fz, t1, t2, t3;
    saras::field_axis(g, 0, fx, t1, t2, t3);
    saras::field_axis(g, 2, fz, t1, t2, t3);
    const int p0 = g.pad;
    const int nx = g.n[0], nz = g.n[2];
    if (g.dim == 3) {
        saras::field_axis(g, 1, fy, t1, t2, t3);
        const int ny = g.n[1];
        w[0].assign((size_t)(ny + 2) * (nz + 2), 0.0);
        w[1].assign((size_t)(nx + 2) * (nz + 2), 0.0);
        w[2].assign((size_t)(nx + 2) * (ny + 2), 0.0);
        double xD, yD, zD;
        xD = g.len[0] / 2.0;
        for (int j = 0; j < ny; ++j) {
            yD = fy[j + p0] - 0.5;
            for (int k = 0; k < nz; ++k) {
                zD = fz[k + p0] - 0.5;
                w[0][(size_t)(j + 1) * (nz + 2) + k + 1] = (xD * xD + yD * yD + zD * zD) / 6.0;
            }
        }
        yD = g.len[1] / 2.0;
        for (int i = 0; i < nx; ++i) {
            xD = fx[i + p0] - 0.5;
            for (int k = 0; k < nz; ++k) {
                zD = fz[k + p0] - 0.5;
                w[1][(size_t)(i + 1) * (nz + 2) + k + 1] = (xD * xD + yD * yD + zD * zD) / 6.0;
            }
        }
        zD = g.len[2] / 2.0;
        for (int i = 0; i < nx; ++i) {
            xD = fx[i + p0] - 0.5;
            for (int j = 0; j < ny; ++j) {
                yD = fy[j + p0] - 0.5;
                w[2][(size_t)(i + 1) * (ny + 2) + j + 1] = (xD * xD + yD * yD + zD * zD) / 6.0;
            }
        }
    } else {
        w[0].assign((size_t)(nz + 2), 0.0);
        w[2].assign((size_t)(nx + 2), 0.0);
        double xD = g.len[0] / 2.0, zD;
        for (int k = 0; k < nz; ++k) {
            zD = fz[k + p0] - 0.5;
            w[0][k + 1] = (xD * xD + zD * zD) / 4.0;
        }
        zD = g.len[2] / 2.0;
        for (int i = 0; i < nx; ++i) {
            xD = fx[i + p0] - 0.5;
            w[2][i + 1] = (xD * xD + zD * zD) / 4.0;
        }
    }
    return w;
}

hipStream_t pick_stream(saras_mg *m, void *stream) { return stream ? (hipStream_t)stream : m->stream; }


}  // namespace

// ===========================================================================
// C-ABI
// ===========================================================================
extern "C" {

const char *saras_last_error(void) { return g_last_error.c_str(); }

int saras_vc_depth(const saras_grid_desc *grid) { return grid ? saras::vc_depth(*grid) : -1; }

saras_status saras_level_metrics(const saras_grid_desc *grid, int level, int axis, double *coord, double *xi,
                                 double *xi_x, double *xixx, double *xix2) {
    if (!grid || axis < 0 || axis > 2) return SARAS_BAD_ARG;
    saras::GridLevels G;
    if (!saras::build_levels(*grid, G)) {
        set_error("grid cannot be coarsened");
        return SARAS_BAD_SHAPE;
    }
    if (level < 0 || level > G.depth) return SARAS_BAD_ARG;
    const saras::AxisLevel &A = G.axes[level][axis];
    const size_t m = A.coord.size();
    if (coord) std::memcpy(coord, A.coord.data(), m * sizeof(double));
    if (xi) std::memcpy(xi, A.xi.data(), m * sizeof(double));
    if (xi_x) std::memcpy(xi_x, A.xi_x.data(), m * sizeof(double));
    if (xixx) std::memcpy(xixx, A.xixx.data(), m * sizeof(double));
    if (xix2) std::memcpy(xix2, A.xix2.data(), m * sizeof(double));
    return SARAS_OK;
}

saras_status saras_mg_create(const saras_grid_desc *grid, const saras_mg_params *params, saras_mg **out) {
    if (!grid || !params || !out) {
        set_error("null argument");
        return SARAS_BAD_ARG;
    }
    *out = nullptr;
    const saras_grid_desc &g = *grid;
    const saras_mg_params &p = *params;
    if (g.dim != 2 && g.dim != 3) { set_error("dim must be 2 or 3"); return SARAS_BAD_ARG; }
    for (int a = 0; a < 3; ++a) {
        if (g.dim == 2 && a == 1) continue;
        if (g.n[a] < 2) { set_error("every axis needs at least 2 cells"); return SARAS_BAD_SHAPE; }
        if (!(g.len[a] > 0)) { set_error("domain lengths must be positive"); return SARAS_BAD_ARG; }
    }
    if (p.res_type < 0 || p.res_type > 2) { set_error("Residual Type must be 0, 1 or 2"); return SARAS_BAD_ARG; }
    if (p.bc < 0 || p.bc > 2 || p.precision < 0 || p.precision > 1) { set_error("bad bc/precision"); return SARAS_BAD_ARG; }
    if (p.top_dirichlet && !(g.dim == 2 && p.bc == SARAS_BC_NEUMANN && !g.periodic[2])) {
        set_error("top_dirichlet: 2-D Neumann problems with z walls (poisson_d2.cc:641-647)");
        return SARAS_BAD_ARG;
    }
    if (p.vc_count < 0 || p.pre_smooth < 0 || p.post_smooth < 0) { set_error("negative counts"); return SARAS_BAD_ARG; }
    std::lock_guard<std::recursive_mutex> lk(saras::alloc_mutex());
    std::unique_ptr<saras_mg> m(new saras_mg());
    m->g = g;
    m->p = p;
    {
        const char *env = std::getenv("SARAS_NO_FUSED_SWEEP");
        m->fused_off = env && env[0] == '1';
        const char *env2 = std::getenv("SARAS_NO_TAIL");
        m->tail_off = env2 && env2[0] == '1';
        const char *env3 = std::getenv("SARAS_MARCH_WGS");
        if (env3 && std::atoi(env3) > 0) m->march_wgs = std::atoi(env3);
        const char *env4 = std::getenv("SARAS_MARCH_TJ8");
        m->march_tj8 = env4 && env4[0] == '1';
        const char *env5 = std::getenv("SARAS_NO_SPLIT");
        m->split_off = env5 && env5[0] == '1';
        const char *env11 = std::getenv("SARAS_RB_GENERAL");
        m->rb_general = env11 && env11[0] == '1';
        const char *env13 = std::getenv("SARAS_RB_WIDE");
        m->rb_wide = env13 && env13[0] == '1';
        const char *env12 = std::getenv("SARAS_COARSE_ONE");
        m->coarse_one = env12 && env12[0] == '1';
        const char *env10 = std::getenv("SARAS_NO_TILE");
        m->tile_off = env10 && env10[0] == '1';
        const char *env9 = std::getenv("SARAS_RR_LANE");
        m->rr_lane = env9 && env9[0] == '1';
        const char *env8 = std::getenv("SARAS_NO_RED_FOLD");
        m->red_fold = !(env8 && env8[0] == '1');
        const char *env6 = std::getenv("SARAS_TAIL_LDS_KB");
        if (env6 && std::atoi(env6) > 0) m->tail_lds = std::min(saras::kTailLds, (size_t)std::atoi(env6) * 1024);
    }
    if (m->p.inner_cycles <= 0) m->p.inner_cycles = 3;
    if (m->p.max_refine <= 0) m->p.max_refine = 20;
    if (!saras::build_levels(g, m->G)) {
        set_error("grid cannot be coarsened (setVCDepth gives a negative depth)");
        return SARAS_BAD_SHAPE;
    }
    m->depth = m->G.depth;
    {
        const auto &C = m->G.axes[m->depth];
        const int cx = C[0].n, cy = g.dim == 3 ? C[1].n : 1, cz = C[2].n;
        m->max_count = g.dim == 2 ? (int)(2.5 * cx * cz) : (int)(2.5 * cx * cy * cz);
    }
    const auto walls = make_walls(g, p);
    m->h64.split_rows = !m->split_off;
    saras_status st = m->h64.build(m->G, walls);
    if (st) return st;
    if (p.precision == SARAS_PREC_MIXED) {
        m->h32.reset(new Hierarchy<float>());
        m->h32->split_rows = !m->split_off;
        std::vector<std::vector<double>> nowall(3);
        st = m->h32->build(m->G, nowall);
        if (st) return st;
        HIP_TRY(hipMalloc((void **)&m->x64b, m->h64.lv[0].elems * sizeof(double)));
        st = pack_tail(m.get(), *m->h32);
        if (!st) st = plan_tiles(m.get(), *m->h32);
        if (st) return st;
    }
    st = pack_tail(m.get(), m->h64);
    // (the mixed solver's cycles run on the FP32 hierarchy alone)
    if (!st && p.precision == SARAS_PREC_FP64) st = plan_tiles(m.get(), m->h64);
    if (st) return st;
    HIP_TRY(hipMalloc((void **)&m->partial, 2 * saras::kNormBlocks * sizeof(double)));
    HIP_TRY(hipHostMalloc((void **)&m->norm_host, 2 * sizeof(double), hipHostMallocCoherent));
    HIP_TRY(hipHostMalloc((void **)&m->norm_seq, sizeof(unsigned), hipHostMallocCoherent));
    *m->norm_seq = 0;
    HIP_TRY(hipHostMalloc((void **)&m->iters_host, sizeof(int), hipHostMallocCoherent));
    *m->iters_host = 0;
    HIP_TRY(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    HIP_TRY(hipEventCreate(&m->ev0));
    HIP_TRY(hipEventCreate(&m->ev1));
    // the level arrays were cleared on the null stream; the handle's stream
    // does not synchronise with it
    HIP_TRY(hipDeviceSynchronize());
    *out = m.release();
    return SARAS_OK;
}

saras_status saras_mg_destroy(saras_mg *mg) {
    if (!mg) return SARAS_BAD_ARG;
    (void)hipStreamSynchronize(mg->stream);
    std::lock_guard<std::recursive_mutex> lk(saras::alloc_mutex());
    delete mg;
    return SARAS_OK;
}

int saras_mg_levels(const saras_mg *mg) { return mg ? mg->depth + 1 : -1; }

saras_status saras_mg_level_shape(const saras_mg *mg, int level, int n[3]) {
    if (!mg || !n || level < 0 || level > mg->depth) return SARAS_BAD_ARG;
    for (int a = 0; a < 3; ++a) n[a] = mg->h64.lv[level].n[a];
    return SARAS_OK;
}

static saras_status solve_fp64(saras_mg *m, hipStream_t s, saras_mg_stats *st) {
    Ops<double> ops{m, m->h64, s, true, m->p.sor};
    auto &L0 = m->h64.lv[0];
    int cycles = 0;
    double res = 0.0;
    bool conv = false;
    for (int c = 0; c < m->p.vc_count; ++c) {
        saras_status ve = run_vcycle(m, ops);
        if (ve) return ve;
        saras_status e = compute_error(m, m->p.res_type, L0.x, s, &res);
        if (e) return e;
        // compute_error read a norm launched after this cycle's coarse solve
        if (m->p.solve_flag) note_coarse_iters(m);
        cycles = c + 1;
        if (res < m->p.vc_tol) {
            conv = true;
            break;
        }
    }
    st->cycles = cycles;
    st->refinements = 0;
    st->residual = res;
    st->converged = conv;
    return SARAS_OK;
}

}  // extern "C"

template <int TYPE, int DIM, bool CX, bool CB, bool CXO = false, bool NOXW = false>
void launch_refine_split(saras_mg *m, const saras::LevelArgs<double> &a, const float *e, long esx, long esy, long ehz,
                         float *r32, const saras::FullRows &fr, hipStream_t s) {
    auto &L0 = m->h64.lv[0];
    const unsigned nb = saras::kNormBlocks, nt = saras::kNormThreads;
    if (refine_marches(m, a)) {
        if (e && !NOXW)
            launch_refine_march<TYPE, DIM, false, !NOXW, CX, CB, CXO, NOXW>(m, a, L0.x, e, esx, esy, ehz, L0.b, r32, fr, s);
        else
            launch_refine_march<TYPE, DIM, false, false, CX, CB, CXO, NOXW>(m, a, L0.x, nullptr, esx, esy, ehz, L0.b, r32, fr, s);
    } else
        hipLaunchKernelGGL((saras::k_refine_split<TYPE, DIM, false, CX, CB, CXO, NOXW>), dim3(nb), dim3(nt), 0, s, a,
                           L0.x, e, esx, esy, ehz, L0.b, m->x64b, r32, m->partial, fr);
    hipLaunchKernelGGL((saras::k_norm_final<TYPE>), dim3(1), dim3(nt), 0, s, m->partial, saras::kNormBlocks,
                       m->norm_host, m->norm_seq, ++m->norm_ticket);
}

template <int TYPE, int DIM>
void launch_refine_split(saras_mg *m, const saras::LevelArgs<double> &a, const float *e, long esx, long esy, long ehz,
                         float *r32, const saras::FullRows &fr, hipStream_t s) {
    // x_old in the caller's array with no correction: the initial residual,
    // whose iterate stays there (nothing to write but r32)
    if (fr.x && !e) launch_refine_split<TYPE, DIM, true, true, false, true>(m, a, e, esx, esy, ehz, r32, fr, s);
    else if (fr.x) launch_refine_split<TYPE, DIM, true, true>(m, a, e, esx, esy, ehz, r32, fr, s);
    else if (fr.xo) launch_refine_split<TYPE, DIM, false, true, true>(m, a, e, esx, esy, ehz, r32, fr, s);
    else if (fr.b) launch_refine_split<TYPE, DIM, false, true>(m, a, e, esx, esy, ehz, r32, fr, s);
    else launch_refine_split<TYPE, DIM, false, false>(m, a, e, esx, esy, ehz, r32, fr, s);
}

// fr: the caller's arrays when x_old and/or b are read from them instead of
// level 0, or x_new written there (fr.xo, with b from the caller and x_old
// from level 0); empty otherwise
template <int DIM>
void launch_refine(int type, saras_mg *m, const saras::LevelArgs<double> &a, const float *e, long esx, long esy,
                   long ehz, float *r32, const saras::FullRows &fr, hipStream_t s) {
    auto &L0 = m->h64.lv[0];
    if (L0.hz && ehz) {
        if (type == 0) launch_refine_split<0, DIM>(m, a, e, esx, esy, ehz, r32, fr, s);
        else if (type == 1) launch_refine_split<1, DIM>(m, a, e, esx, esy, ehz, r32, fr, s);
        else launch_refine_split<2, DIM>(m, a, e, esx, esy, ehz, r32, fr, s);
        return;
    }
    switch (type) {
        case 0:
            hipLaunchKernelGGL((saras::k_refine<0, DIM>), dim3(saras::kNormBlocks), dim3(saras::kNormThreads), 0, s, a,
                               L0.x, e, esx, esy, L0.b, m->x64b, r32, esx, esy, ehz, m->partial);
            hipLaunchKernelGGL((saras::k_norm_final<0>), dim3(1), dim3(saras::kNormThreads), 0, s, m->partial,
                               saras::kNormBlocks, m->norm_host, m->norm_seq, ++m->norm_ticket);
            break;
        case 1:
            hipLaunchKernelGGL((saras::k_refine<1, DIM>), dim3(saras::kNormBlocks), dim3(saras::kNormThreads), 0, s, a,
                               L0.x, e, esx, esy, L0.b, m->x64b, r32, esx, esy, ehz, m->partial);
            hipLaunchKernelGGL((saras::k_norm_final<1>), dim3(1), dim3(saras::kNormThreads), 0, s, m->partial,
                               saras::kNormBlocks, m->norm_host, m->norm_seq, ++m->norm_ticket);
            break;
        default:
            hipLaunchKernelGGL((saras::k_refine<2, DIM>), dim3(saras::kNormBlocks), dim3(saras::kNormThreads), 0, s, a,
                               L0.x, e, esx, esy, L0.b, m->x64b, r32, esx, esy, ehz, m->partial);
            hipLaunchKernelGGL((saras::k_norm_final<2>), dim3(1), dim3(saras::kNormThreads), 0, s, m->partial,
                               saras::kNormBlocks, m->norm_host, m->norm_seq, ++m->norm_ticket);
            break;
    }
}

// x64 <- x64 + e32 (if with_e), r32 <- b - A x64, residual norm of type res_type
static saras_status refine_step(saras_mg *m, hipStream_t s, bool with_e, const saras::FullRows &fr, double *res) {
    auto &L0 = m->h64.lv[0];
    auto &F0 = m->h32->lv[0];
    auto a = level_args(m, m->h64, 0, true);
    const float *e = with_e ? F0.x : nullptr;
    // host-side guards: the caller-layout reads and writes exist on split rows
    // only, always with b from the caller, and never read and write the
    // caller's iterate in one pass
    if ((fr.x || fr.b || fr.xo) && !(L0.hz && F0.hz && fr.b)) {
        set_error("internal error: caller-layout refinement on a level without split rows");
        return SARAS_HIP_ERROR;
    }
    if (fr.x && fr.xo) {
        set_error("internal error: refinement reading and writing the caller's iterate");
        return SARAS_HIP_ERROR;
    }
    if (m->G.dim == 3) launch_refine<3>(m->p.res_type, m, a, e, F0.sx, F0.sy, F0.hz, F0.b, fr, s);
    else launch_refine<2>(m->p.res_type, m, a, e, F0.sx, F0.sy, F0.hz, F0.b, fr, s);
    // x_new is in level 0's other buffer, or (fr.xo) in the caller's array, or
    // (x_old from the caller's array, no correction) still only there
    if (!fr.xo && !(fr.x && !with_e)) std::swap(L0.x, m->x64b);
    HIP_TRY(wait_norm(m, s));
    const double num = m->norm_host[0], den = m->norm_host[1];
    const int pointCount = L0.n[0] * L0.n[1] * L0.n[2];
    const int type = m->p.res_type;
    if (type == 0) *res = den != 0.0 ? num / den : num;
    else if (type == 1) *res = den != 0.0 ? num / den : num / pointCount;
    else *res = den != 0.0 ? std::sqrt(num / pointCount) / std::sqrt(den / pointCount) : std::sqrt(num / pointCount);
    return SARAS_OK;
}

// Mixed precision: FP64 iterate, residual and stopping test; FP32 V-cycles
// (same smoother, transfers and coarse solve as the reference, homogeneous
// walls) on the correction equation A e = r.
// full: the caller's x (initial guess) and b, read in place by the FP64
// passes when both levels 0 have split rows (empty: level 0 holds them).
// With full.xo, the refinement expected to end the solve writes its iterate
// straight into the caller's array; *x_in_caller says where the solution is.
static saras_status solve_mixed(saras_mg *m, hipStream_t s, saras_mg_stats *st,
                                const saras::FullRows &full = saras::FullRows{}, bool *x_in_caller = nullptr) {
    Ops<float> ops{m, *m->h32, s, false, (float)m->p.sor};
    auto &F0 = m->h32->lv[0];
    double res = 0.0;
    saras::FullRows first = full, later = full;
    first.xo = nullptr;
    later.x = nullptr;
    later.xo = nullptr;
    // the FP64 iterate lives in the caller's array: the initial guess until
    // the first refinement reads it from there
    bool in_caller = first.x != nullptr;
    saras_status e = refine_step(m, s, false, first, &res);
    if (e) return e;
    int cycles = 0, refs = 0;
    const int cap = m->p.vc_count > 0 ? m->p.vc_count : (1 << 30);
    // inner_cycles is the most FP32 cycles per refinement.  The first
    // refinement runs at most kProbeCycles of them, few enough that FP32
    // rounding (a correction good to about kFp32Floor of the residual) does
    // not mask the cycle's convergence factor rho, which it measures.  Each
    // later refinement runs the cycles rho needs to take the residual to half
    // the tolerance, or down to the FP32 floor when that comes first (cycles
    // past it gain nothing).  A short estimate costs one more refinement,
    // never accuracy: the FP64 residual alone decides convergence.
    constexpr int kProbeCycles = 3;
    constexpr double kFp32Floor = 1e-6;
    // level 0 is not the coarsest (whose smoothing is the coarse solve) and
    // the V-cycle opens with its pre-smoothing sweep, not the tail kernel
    const bool zero_start = !m->graphs && F0.hz && m->p.pre_smooth > 0 && m->depth > 0 &&
                            (m->tail_off || ops.tail_start() > 0);
    double rho = 1.0;
    bool measured = false;
    while (!(res < m->p.vc_tol) && refs < m->p.max_refine && cycles < cap) {
        int k = m->p.inner_cycles;
        if (!measured) {
            k = std::min(k, kProbeCycles);
        } else if (rho > 0.0 && rho < 0.9 && res > 0.0) {
            const double target = std::max(0.5 * m->p.vc_tol / res, kFp32Floor);
            const double need = std::ceil(std::log(target) / std::log(rho));
            if (need < 1.0) k = 1;
            else if (need < (double)k) k = (int)need;
        }
        // the correction starts from zero: cleared by the first red pass of
        // the round's first cycle where that pass runs on split rows (eager
        // launches; a replayed graph keeps the separate clear)
        if (zero_start) ops.zero0 = true;
        else HIP_TRY(hipMemsetAsync(F0.x, 0, F0.elems * sizeof(float), s));
        int ran = 0;
        for (int c = 0; c < k && cycles < cap; ++c) {
            e = run_vcycle(m, ops);
            if (e) return e;
            ++cycles;
            ++ran;
        }
        const double before = res;
        // where this refinement reads and writes the FP64 iterate: after a
        // refinement that wrote the caller's array, read it from there; else
        // write there when this one is expected to end the solve (the
        // measured rate predicts the tolerance, or a cap ends the loop).  A
        // wrong guess costs nothing: the next refinement reads it in place.
        saras::FullRows fr = later;
        if (in_caller) {
            fr.x = full.x;
        } else if (full.xo) {
            const bool capped = refs + 1 >= m->p.max_refine || cycles >= cap;
            const bool expect = measured && rho > 0.0 && rho < 1.0 && res * std::pow(rho, ran) < m->p.vc_tol;
            if (capped || expect) fr.xo = full.xo;
        }
        e = refine_step(m, s, true, fr, &res);
        if (e) return e;
        in_caller = fr.xo != nullptr;
        ++refs;
        if (!std::isfinite(res)) break;
        rho = (ran > 0 && before > 0.0 && res < before) ? std::pow(res / before, 1.0 / ran) : 1.0;
        measured = true;
    }
    // the last refinement's norm came after the last cycle's coarse solve
    if (m->p.solve_flag && cycles > 0) note_coarse_iters(m);
    st->cycles = cycles;
    st->refinements = refs;
    st->residual = res;
    st->converged = res < m->p.vc_tol;
    if (x_in_caller) *x_in_caller = in_caller;
    return SARAS_OK;
}

namespace saras {

void mg_level0(saras_mg *m, double **x, double **b, long *sx, long *sy, long *hz) {
    auto &L0 = m->h64.lv[0];
    *x = L0.x;
    *b = L0.b;
    *sx = L0.sx;
    *sy = L0.sy;
    if (hz) *hz = L0.hz;
}

hipStream_t mg_stream(saras_mg *m) { return m->stream; }

void set_last_error(const std::string &msg) { set_error(msg); }

std::recursive_mutex &alloc_mutex() {
    static std::recursive_mutex mu;
    return mu;
}

saras_status mg_solve_resident(saras_mg *m, hipStream_t s, saras_mg_stats *st) {
    m->coarse_iters_max = 0;
    m->coarse_capped = 0;
    saras_mg_stats r{};
    saras_status e = m->p.precision == SARAS_PREC_FP64 ? solve_fp64(m, s, &r) : solve_mixed(m, s, &r);
    if (e) return e;
    r.coarse_iters_max = m->coarse_iters_max;
    r.coarse_capped = m->coarse_capped;
    if (st) *st = r;
    return r.converged ? SARAS_OK : SARAS_NOT_CONVERGED;
}

}  // namespace saras

extern "C" {

saras_status saras_mg_solve(saras_mg *mg, double *x_full, const double *b_full, int ptr_kind, void *stream,
                            saras_mg_stats *stats) {
    if (!mg || !x_full || !b_full) {
        set_error("null argument");
        return SARAS_BAD_ARG;
    }
    if (ptr_kind != SARAS_PTR_HOST && ptr_kind != SARAS_PTR_DEVICE) return SARAS_BAD_ARG;
    saras_mg *m = mg;
    hipStream_t s = pick_stream(m, stream);
    const long fe = full_elems(m->g);
    double *dx = x_full;
    const double *db = b_full;
    if (ptr_kind == SARAS_PTR_HOST) {
        if (m->stage_elems < (size_t)fe) {
            std::lock_guard<std::recursive_mutex> lk(saras::alloc_mutex());
            (void)hipFree(m->stage_x);
            (void)hipFree(m->stage_b);
            m->stage_x = m->stage_b = nullptr;
            HIP_TRY(hipMalloc((void **)&m->stage_x, fe * sizeof(double)));
            HIP_TRY(hipMalloc((void **)&m->stage_b, fe * sizeof(double)));
            m->stage_elems = fe;
        }
        HIP_TRY(hipMemcpyAsync(m->stage_x, x_full, fe * sizeof(double), hipMemcpyHostToDevice, s));
        HIP_TRY(hipMemcpyAsync(m->stage_b, b_full, fe * sizeof(double), hipMemcpyHostToDevice, s));
        dx = m->stage_x;
        db = m->stage_b;
    }
    m->coarse_iters_max = 0;
    m->coarse_capped = 0;
    HIP_TRY(hipEventRecord(m->ev0, s));
    auto &L0 = m->h64.lv[0];
    saras_mg_stats st{};
    saras_status e = SARAS_OK;
    bool in_caller = false;   // the solution's core is in dx already
    if (m->p.precision == SARAS_PREC_FP64) {
        load_core<double>(m, db, L0, L0.b, s);
        load_core<double>(m, dx, L0, L0.x, s);
        e = solve_fp64(m, s, &st);
    } else if (L0.hz && m->h32->lv[0].hz) {
        // the FP64 passes of the mixed solve read b and the initial guess
        // from the caller's arrays; level 0 receives x from the first pass
        const long p = m->g.pad, fz = L0.n[2] + 2 * p, fy = m->g.dim == 3 ? L0.n[1] + 2 * p : 1;
        saras::FullRows fr;
        fr.x = dx;
        fr.b = db;
        fr.xo = dx;
        fr.si = m->g.dim == 3 ? fy * fz : fz;
        fr.sj = m->g.dim == 3 ? fz : 0;
        fr.off = m->g.dim == 3 ? p * fy * fz + p * fz + p : p * fz + p;
        e = solve_mixed(m, s, &st, fr, &in_caller);
    } else {
        load_core<double>(m, db, L0, L0.b, s);
        load_core<double>(m, dx, L0, L0.x, s);
        e = solve_mixed(m, s, &st);
    }
    if (e) return e;
    store_full(m, dx, in_caller ? nullptr : L0.x, s);
    HIP_TRY(hipEventRecord(m->ev1, s));
    if (ptr_kind == SARAS_PTR_HOST)
        HIP_TRY(hipMemcpyAsync(x_full, m->stage_x, fe * sizeof(double), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
    st.device_ms = ms;
    st.coarse_iters_max = m->coarse_iters_max;
    st.coarse_capped = m->coarse_capped;
    if (stats) *stats = st;
    return st.converged ? SARAS_OK : SARAS_NOT_CONVERGED;
}

saras_status saras_mg_set_graphs(saras_mg *mg, int enable) {
    if (!mg) return SARAS_BAD_ARG;
    HIP_TRY(hipStreamSynchronize(mg->stream));
    if (!enable)
        for (auto &c : mg->graph_cache) {
            for (auto &e : c) (void)hipGraphExecDestroy(e.exec);
            c.clear();
        }
    mg->graphs = enable != 0;
    return SARAS_OK;
}

size_t saras_mg_footprint(const saras_grid_desc *grid, const saras_mg_params *params) {
    if (!grid || !params) return 0;
    saras::GridLevels G;
    if (!saras::build_levels(*grid, G)) return 0;
    const int D = G.depth;
    auto level_bytes = [&](size_t word) {
        size_t tot = 0;
        for (int l = 0; l <= D; ++l) {
            int n[3];
            for (int a = 0; a < 3; ++a) n[a] = G.axes[l][a].n;
            if (grid->dim == 2) n[1] = 1;
            const long a128 = 128 / (long)word;
            const size_t sy = (size_t)((n[2] + a128 - 1) / a128 * a128);
            const size_t elems = sy * n[1] * n[0];
            tot += elems * word * (l < D ? 3 : 2);
            tot += 5 * 3 * (size_t)(n[0] + n[1] + n[2]) * word;
        }
        return tot;
    };
    size_t bytes = level_bytes(8);
    const size_t full = (size_t)full_elems(*grid);
    if (params->precision == SARAS_PREC_MIXED) {
        bytes += level_bytes(4);
        const auto &A = G.axes[0];
        const size_t sy = (size_t)((A[2].n + 15) / 16 * 16);
        bytes += sy * (grid->dim == 2 ? 1 : A[1].n) * A[0].n * 8;   // second FP64 iterate
    }
    bytes += 2 * full * 8;                      // host-pointer staging
    bytes += 2 * 1024 * 1024;                   // norms, counters, coarse workspace
    return bytes;
}

// ---- single-operation entry points ----
saras_status saras_mg_set_level(saras_mg *mg, int level, const double *lhs_pad, const double *rhs_pad) {
    if (!mg || level < 0 || level > mg->depth) return SARAS_BAD_ARG;
    auto &L = mg->h64.lv[level];
    const int nx = L.n[0], ny = L.n[1], nz = L.n[2];
    std::vector<double> core(L.elems, 0.0);
    const bool d3 = mg->g.dim == 3;
    for (int which = 0; which < 2; ++which) {
        const double *src = which == 0 ? lhs_pad : rhs_pad;
        if (!src) continue;
        for (int i = 0; i < nx; ++i)
            for (int j = 0; j < ny; ++j)
                for (int k = 0; k < nz; ++k) {
                    const long f = d3 ? ((long)(i + 1) * (ny + 2) + (j + 1)) * (nz + 2) + (k + 1)
                                      : (long)(i + 1) * (nz + 2) + (k + 1);
                    core[(size_t)i * L.sx + (size_t)j * L.sy + (L.hz ? (k & 1) * L.hz + (k >> 1) : k)] = src[f];
                }
        HIP_TRY(hipMemcpy(which == 0 ? L.x : L.b, core.data(), L.elems * sizeof(double), hipMemcpyHostToDevice));
    }
    return SARAS_OK;
}

saras_status saras_mg_get_level(saras_mg *mg, int level, double *lhs_pad, double *rhs_pad) {
    if (!mg || level < 0 || level > mg->depth) return SARAS_BAD_ARG;
    HIP_TRY(hipStreamSynchronize(mg->stream));
    auto &L = mg->h64.lv[level];
    const int nx = L.n[0], ny = L.n[1], nz = L.n[2];
    std::vector<double> core(L.elems);
    const bool d3 = mg->g.dim == 3;
    const size_t padded = d3 ? (size_t)(nx + 2) * (ny + 2) * (nz + 2) : (size_t)(nx + 2) * (nz + 2);
    for (int which = 0; which < 2; ++which) {
        double *dst = which == 0 ? lhs_pad : rhs_pad;
        if (!dst) continue;
        HIP_TRY(hipMemcpy(core.data(), which == 0 ? L.x : L.b, L.elems * sizeof(double), hipMemcpyDeviceToHost));
        std::memset(dst, 0, padded * sizeof(double));
        for (int i = 0; i < nx; ++i)
            for (int j = 0; j < ny; ++j)
                for (int k = 0; k < nz; ++k) {
                    const long f = d3 ? ((long)(i + 1) * (ny + 2) + (j + 1)) * (nz + 2) + (k + 1)
                                      : (long)(i + 1) * (nz + 2) + (k + 1);
                    dst[f] = core[(size_t)i * L.sx + (size_t)j * L.sy + (L.hz ? (k & 1) * L.hz + (k >> 1) : k)];
                }
    }
    return SARAS_OK;
}

saras_status saras_mg_smooth(saras_mg *mg, int level, int count, int zero_bc) {
    if (!mg || level < 0 || level > mg->depth || count < 0) return SARAS_BAD_ARG;
    Ops<double> ops{mg, mg->h64, mg->stream, true, mg->p.sor};
    ops.smooth(level, count, zero_bc != 0);
    if (ops.err) return ops.err;
    HIP_TRY(hipStreamSynchronize(mg->stream));
    HIP_TRY(hipGetLastError());
    return SARAS_OK;
}

saras_status saras_mg_coarse_solve(saras_mg *mg, int level, int zero_bc, int *iters) {
    if (!mg || level < 0 || level > mg->depth) return SARAS_BAD_ARG;
    if (level != mg->depth) {
        set_error("the single-workgroup solve runs on the coarsest level only");
        return SARAS_BAD_ARG;
    }
    Ops<double> ops{mg, mg->h64, mg->stream, true, mg->p.sor};
    ops.coarse(level, zero_bc != 0, 0, 0);
    if (ops.err) return ops.err;
    HIP_TRY(hipStreamSynchronize(mg->stream));
    if (iters) *iters = *mg->iters_host;
    return SARAS_OK;
}

saras_status saras_mg_residual_restrict(saras_mg *mg, int level) {
    if (!mg || level < 0 || level >= mg->depth) return SARAS_BAD_ARG;
    Ops<double> ops{mg, mg->h64, mg->stream, true, mg->p.sor};
    ops.resid_restrict(level);
    if (ops.err) return ops.err;
    HIP_TRY(hipStreamSynchronize(mg->stream));
    return SARAS_OK;
}

saras_status saras_mg_prolong_correct(saras_mg *mg, int level) {
    if (!mg || level < 0 || level >= mg->depth) return SARAS_BAD_ARG;
    Ops<double> ops{mg, mg->h64, mg->stream, true, mg->p.sor};
    ops.prolong_correct(level);
    if (ops.err) return ops.err;
    HIP_TRY(hipStreamSynchronize(mg->stream));
    return SARAS_OK;
}

saras_status saras_mg_error(saras_mg *mg, int res_type, double *value) {
    if (!mg || !value || res_type < 0 || res_type > 2) return SARAS_BAD_ARG;
    return compute_error(mg, res_type, mg->h64.lv[0].x, mg->stream, value);
}

// ---- measurement hooks ----
saras_status saras_mg_bench_cycles(saras_mg *mg, int count, double *ms) {
    if (!mg || count < 0 || !ms) return SARAS_BAD_ARG;
    hipStream_t s = mg->stream;
    HIP_TRY(hipEventRecord(mg->ev0, s));
    if (mg->p.precision == SARAS_PREC_FP64) {
        Ops<double> ops{mg, mg->h64, s, true, mg->p.sor};
        for (int c = 0; c < count; ++c) {
            saras_status e = run_vcycle(mg, ops);
            if (e) return e;
        }
    } else {
        Ops<float> ops{mg, *mg->h32, s, false, (float)mg->p.sor};
        for (int c = 0; c < count; ++c) {
            saras_status e = run_vcycle(mg, ops);
            if (e) return e;
        }
    }
    HIP_TRY(hipEventRecord(mg->ev1, s));
    HIP_TRY(hipEventSynchronize(mg->ev1));
    HIP_TRY(hipGetLastError());
    float f = 0.f;
    HIP_TRY(hipEventElapsedTime(&f, mg->ev0, mg->ev1));
    *ms = f;
    return SARAS_OK;
}

saras_status saras_mg_bench_sweeps(saras_mg *mg, int reps, double *ms) {
    if (!mg || reps < 0 || !ms) return SARAS_BAD_ARG;
    if (mg->depth == 0) {
        set_error("level 0 is the coarsest level");
        return SARAS_BAD_ARG;
    }
    hipStream_t s = mg->stream;
    HIP_TRY(hipEventRecord(mg->ev0, s));
    if (mg->p.precision == SARAS_PREC_FP64) {
        Ops<double> ops{mg, mg->h64, s, true, mg->p.sor};
        for (int c = 0; c < reps; ++c) ops.rb_sweep(0, false);
    } else {
        Ops<float> ops{mg, *mg->h32, s, false, (float)mg->p.sor};
        for (int c = 0; c < reps; ++c) ops.rb_sweep(0, true);
    }
    HIP_TRY(hipEventRecord(mg->ev1, s));
    HIP_TRY(hipEventSynchronize(mg->ev1));
    HIP_TRY(hipGetLastError());
    float f = 0.f;
    HIP_TRY(hipEventElapsedTime(&f, mg->ev0, mg->ev1));
    *ms = f;
    return SARAS_OK;
}

saras_status saras_bench_stream_copy(size_t n, int reps, double *ms) {
    if (!ms || n < 2 || reps < 1) return SARAS_BAD_ARG;
    double *a = nullptr, *b = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    const long n2 = (long)(n / 2);
    HIP_TRY(hipMalloc((void **)&a, n2 * 2 * sizeof(double)));
    HIP_TRY(hipMalloc((void **)&b, n2 * 2 * sizeof(double)));
    HIP_TRY(hipMemset(a, 0, n2 * 2 * sizeof(double)));
    HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    const unsigned blocks = (unsigned)((n2 + 255) / 256);
    hipLaunchKernelGGL(saras::k_stream_copy, dim3(blocks), dim3(256), 0, s, (const double2 *)a, (double2 *)b, n2);
    HIP_TRY(hipEventRecord(e0, s));
    for (int r = 0; r < reps; ++r)
        hipLaunchKernelGGL(saras::k_stream_copy, dim3(blocks), dim3(256), 0, s, (const double2 *)a, (double2 *)b, n2);
    HIP_TRY(hipEventRecord(e1, s));
    HIP_TRY(hipEventSynchronize(e1));
    float f = 0.f;
    HIP_TRY(hipEventElapsedTime(&f, e0, e1));
    *ms = f;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(s);
    (void)hipFree(a);
    (void)hipFree(b);
    return SARAS_OK;
}

// ---- device memory helpers ----
saras_status saras_device_alloc(void **ptr, size_t bytes) {
    if (!ptr) return SARAS_BAD_ARG;
    HIP_TRY(hipMalloc(ptr, bytes));
    return SARAS_OK;
}
saras_status saras_device_free(void *ptr) {
    HIP_TRY(hipFree(ptr));
    return SARAS_OK;
}
saras_status saras_memcpy_h2d(void *dst, const void *src, size_t bytes) {
    HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return SARAS_OK;
}
saras_status saras_memcpy_d2h(void *dst, const void *src, size_t bytes) {
    HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return SARAS_OK;
}
saras_status saras_device_sync(void) {
    HIP_TRY(hipDeviceSynchronize());
    return SARAS_OK;
}
saras_status saras_device_zero(void *ptr, size_t bytes) {
    if (!ptr) return SARAS_BAD_ARG;
    HIP_TRY(hipMemset(ptr, 0, bytes));
    // hipMemset on device memory may return before the fill has run; the
    // solver handles' streams do not wait for the null stream
    HIP_TRY(hipDeviceSynchronize());
    return SARAS_OK;
}

}  // extern "C"
