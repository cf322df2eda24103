// mg_tail.hpp -- the small bottom of the V-cycle in one workgroup.
//
// Below a few thousand cells per level a V-cycle is all launch latency: the
// levels S..D of the reference V-cycle (poisson.cc:227-277 restricted to
// those levels) run here inside one workgroup, every level held in LDS.
// Arithmetic follows the same expressions as the multi-block kernels, so the
// FP64 path stays bit-identical to the reference ordering.
//
// One compute unit runs the kernel, and most of its levels have fewer cells
// than the workgroup has threads: what bounds it is the number of
// instructions a wave issues from one barrier to the next.  So
//  * a level is stored by colour (all red cells, then all black, each in
//    (i, j, k / 2) order): the lanes of a pass read and write consecutive
//    words;
//  * there are no ghost cells to refresh: a wall neighbour is a function of
//    the cell's own value (its address is the cell's own, its sign flipped
//    for Dirichlet), a periodic one is the opposite core cell (as in the
//    multi-block kernels; see mg_kernels.hpp), so a sweep is two phases;
//  * the neighbour addresses of every cell are tabulated on the host (TailCell)
//    and kept in registers through a smoothing call, with the coefficients,
//    the divisor's reciprocal (FP32), the right-hand side and the value;
//  * the residual before a restriction is taken by all fine cells at once;
//  * the coarsest solve tests max|r| < tol by a ballot instead of a
//    reduction, and a level of at most 64 cells of a colour runs on one wave
//    without barriers.
// Measured against literal ghost layers with colour lists, per V(2,2) cycle:
// 16^3..2^3 FP32 47 -> 35 us, FP64 55 -> 43 us; 64^2..4^2 FP64 53 -> 38 us; V(3,6)
// 16^3..2^3 FP32 70 -> 47 us; three sweeps of an 18 x 14 x 25 coarsest level FP64
// 49 -> 24 us.  A pass of 16^3 takes about 0.7 us, the vector issue of its 32
// wave iterations; a pass of 8^3 and below 0.2-0.3 us.
#pragma once
#include <type_traits>

#include "mg_kernels.hpp"
#include "mg_plan.hpp"

namespace saras {

// One cell of a level stored by colour.  Directions: x+, x-, y+, y-, z+, z-.
struct TailCell {
    unsigned a[3];   // LDS offsets of the neighbours, two per word (a wall: the cell itself)
    unsigned cxy;    // LDS offsets of the x and y coefficient pairs (c2, c1)
    unsigned czf;    // of the z pair, | flags << 16
};
// flags: bit d, direction d is a Dirichlet wall; bit 6 + d, the coarsest
// residual sees an old value there (see tail_smooth); kNoCell: a row of odd
// length has no such cell
constexpr unsigned kTailNoCell = 1u << 15;

// One tail level; every array is an LDS offset in elements.
struct TailLevel {
    int n[3];
    int hz, half;              // cells of one colour per row (rounded up) and per level
    int x, b, old;             // iterate, right-hand side (-1: at TailArgs::bcol), old values of a coarsest solve
    int lo[3], hi[3], wd[3];   // restriction factors of this (coarse) level, 3-D
    int neg;                   // some wall is Dirichlet
    int odd;                   // an odd periodic extent (the coarsest level alone can have one)
    int cell4;                 // the level's TailCell table, by words: LDS offset of the first four
    int cell1;                 // ... and of the fifth; -1: the table is in global memory, from entry cell4
};

template <typename T>
struct TailArgs {
    int first, last;                     // levels S and D
    TailLevel L[kTailMaxLevels];         // levels S..D (index l - S)
    long sx, sy, hz;                     // level S's layout in global memory
    int res;                             // LDS offset of the residual of a level (by colour, as its iterate)
    int coff, ncoef;                     // the coefficients' place in LDS and their number
    int cellw, ncellw;                   // the cell tables' place in LDS and size, in 32-bit words
    const T *coef;                       // their packed image in global memory (the LDS region's order)
    const unsigned *cellimg;             // the same of the cell tables
    const uint4 *cells4;                 // the tables that are not in LDS
    const unsigned *cells1;
    T *x;                                // global core array of level S (in/out)
    const T *b;                          // global core array of level S
    T *bcol;                             // the right-hand side of a level without room for it in LDS, by colour
    int pre, post, solve_flag, max_count;
    T w;
    double tol;
    double rel_floor;                    // as CoarseCtl::rel_floor
    int *iters_out;
};

// position of core cell (i, j, k) in a level stored by colour
template <int DIM>
__host__ __device__ __forceinline__ int tail_at(const TailLevel &V, int i, int j, int k) {
    const int row = DIM == 3 ? i * V.n[1] + j : i;
    return ((i + j + k) & 1) * V.half + row * V.hz + (k >> 1);
}

// (i, j, k) of core index t of a small level (32-bit unsigned arithmetic)
__device__ __forceinline__ void tcoords(int t, int ny, int nz, int &i, int &j, int &k) {
    const unsigned r = (unsigned)t / (unsigned)nz;
    k = t - (int)(r * (unsigned)nz);
    const unsigned q = r / (unsigned)ny;
    j = (int)(r - q * (unsigned)ny);
    i = (int)q;
}

// the TailCell of every cell of a level: col * half + u
template <int DIM>
inline void tail_cells(const TailLevel &V, const int (&c)[3], const int (&bc_lo)[3], const int (&bc_hi)[3],
                       TailCell *out) {
    for (int q = 0; q < 2 * V.half; ++q) out[q].czf = kTailNoCell << 16;
    const int ny = DIM == 3 ? V.n[1] : 1;
    for (int i = 0; i < V.n[0]; ++i)
        for (int j = 0; j < ny; ++j)
            for (int k = 0; k < V.n[2]; ++k) {
                const int own = tail_at<DIM>(V, i, j, k);
                TailCell &t = out[own];
                unsigned flags = 0, a[6] = {0, 0, 0, 0, 0, 0};
                for (int d = 0; d < 6; ++d) {
                    const int ax = d / 2;
                    if (DIM == 2 && ax == 1) continue;
                    int p[3] = {i, j, k};
                    const int n = V.n[ax], bc = d & 1 ? bc_lo[ax] : bc_hi[ax];
                    p[ax] += d & 1 ? -1 : 1;
                    if (p[ax] < 0 || p[ax] >= n) {
                        if (bc != BC_PER) {
                            a[d] = (unsigned)(V.x + own);
                            flags |= 64u << d;
                            if (bc == BC_DIR) flags |= 1u << d;
                            continue;
                        }
                        p[ax] = p[ax] < 0 ? n - 1 : 0;
                        if ((p[0] + p[1] + p[2]) & 1) flags |= 64u << d;   // a black cell
                    }
                    a[d] = (unsigned)(V.x + tail_at<DIM>(V, p[0], p[1], p[2]));
                }
                for (int ax = 0; ax < 3; ++ax) t.a[ax] = a[2 * ax] | a[2 * ax + 1] << 16;
                t.cxy = (unsigned)(c[0] + 2 * i) | (unsigned)(c[1] + 2 * j) << 16;
                t.czf = (unsigned)(c[2] + 2 * k) | flags << 16;
            }
}

// the coefficient pair (c2, c1) at an LDS offset
template <typename T>
__device__ __forceinline__ void tail_coef(const T *lds, unsigned at, T &c2, T &c1) {
    using P = std::conditional_t<sizeof(T) == 4, float2, double2>;
    const P p = *reinterpret_cast<const P *>(lds + at);
    c2 = p.x;
    c1 = p.y;
}

template <typename T>
struct TailCoef {
    T c2x, c1x, c2y, c1y, c2z, c1z;
};
template <typename T, int DIM>
__device__ __forceinline__ TailCoef<T> tail_coefs(const T *lds, const TailCell &t) {
    TailCoef<T> m;
    m.c2y = m.c1y = T(0);
    tail_coef(lds, t.cxy & 0xffffu, m.c2x, m.c1x);
    if (DIM == 3) tail_coef(lds, t.cxy >> 16, m.c2y, m.c1y);
    tail_coef(lds, t.czf & 0xffffu, m.c2z, m.c1z);
    return m;
}

// A thread's cell: right-hand side, sor_inv of the divisor, value; KEEP: the
// coefficients too.
template <typename T, bool KEEP>
struct TailOwn {
    TailCell t;
    T b, d, x;
};
template <typename T>
struct TailOwn<T, true> {
    TailCell t;
    T b, d, x;
    TailCoef<T> m;
};

// The six neighbour values of a cell; STALE: as the coarsest residual sees
// them, `delta` from the iterate to its old values.
template <typename T, int DIM, bool STALE>
__device__ __forceinline__ Stencil<T, DIM> tail_gather(const T *lds, const TailCell &t, T c, bool neg, int delta) {
    T v[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) {
        if (DIM == 2 && (d == 2 || d == 3)) continue;
        int a = (int)(d & 1 ? t.a[d >> 1] >> 16 : t.a[d >> 1] & 0xffffu);
        if (STALE && (t.czf & (64u << 16 << d))) a += delta;
        v[d] = lds[a];
    }
    if (neg) {
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            if (DIM == 2 && (d == 2 || d == 3)) continue;
            if (t.czf & (1u << 16 << d)) v[d] = -v[d];
        }
    }
    Stencil<T, DIM> s;
    s.c = c;
    s.xE = v[0];
    s.xW = v[1];
    if (DIM == 3) {
        s.yN = v[2];
        s.yS = v[3];
    }
    s.zT = v[4];
    s.zB = v[5];
    return s;
}

// The smoothing sweeps of a level, or its coarsest solve: with `pro`, first
// the correction of coarse level C is added (injection plus the saved
// iterate, poisson_d3.cc:548-558, poisson.cc:266); then `count` RB-SOR
// sweeps, or with `solve` sweeps until max|r| < tol or the iteration cap
// (poisson_d3.cc:249-432), returning the iteration count; with `emit`, last
// the residual of every cell into A.res.
//
// The reference takes the coarsest residual with its ghosts as they stand
// after a sweep (poisson_d3.cc:398-415): a wall ghost is the rule applied to
// the cell's value before the sweep, and a periodic ghost was refreshed
// between the colours, so it holds a wrapped black cell's value from before
// the black pass.  A pass of the solve leaves each cell's old value at
// V.old, and the residual reads those neighbours there.
//
// Where a periodic extent is odd, a wrapped neighbour has the cell's own
// colour, and its ghost its value from before the pass: all cells are read
// before the first is written.
//
// CPT cells of a colour per thread are kept in registers; the cells of a
// larger level beyond them (a coarsest one: the others are limited to
// kTailColourCells) are loaded anew in each pass (and with an odd periodic
// extent wait at V.old for the others' reads).
//
// BG: the right-hand side of the level (a coarsest one by itself) is at A.bcol.
template <typename T, int DIM, int CPT, bool BG>
__device__ __forceinline__ int tail_smooth(T *lds, const TailArgs<T> &A, const TailLevel &V, const TailLevel &C,
                                           bool pro, bool solve, int count, bool emit, double *red, int *wflag) {
    // FP64 with several cells per thread: the coefficients do not fit beside them
    constexpr bool KEEP = CPT == 1 || sizeof(T) == 4;
    using Own = TailOwn<T, KEEP>;
    const int tid = threadIdx.x;
    constexpr int nthr = kTailThreads, nwave = kTailThreads / 64;
    constexpr int PAIR = CPT > 1 ? 2 : 1;   // cells whose neighbours are read together
    const int lane = tid & 63, wv = tid >> 6;
    const int half = V.half;
    // at most one cell of a colour per lane of wave 0: the other waves wait
    // at the closing barrier and the phases need none
    const bool wave = CPT == 1 && half <= 64;
    const bool neg = V.neg != 0, odd = V.odd != 0;
    const bool rest = CPT > 1 && half > CPT * nthr;
    const int delta = V.old - V.x;
    const T w = A.w;
    auto sync = [&]() __attribute__((always_inline)) {
        if (wave) wave_lds_sync();
        else __syncthreads();
    };
    auto cell = [&](int q) __attribute__((always_inline)) {
        TailCell t;
        uint4 v;
        if (CPT == 1) {
            const unsigned *lw = reinterpret_cast<const unsigned *>(lds);
            v = *reinterpret_cast<const uint4 *>(lw + V.cell4 + 4 * q);
            t.czf = lw[V.cell1 + q];
        } else {
            v = A.cells4[V.cell4 + q];
            t.czf = A.cells1[V.cell4 + q];
        }
        t.a[0] = v.x;
        t.a[1] = v.y;
        t.a[2] = v.z;
        t.cxy = v.w;
        return t;
    };
    // cell q of the level (col * half + u) with its value; false: none there
    // (the addresses are valid all the same, so a caller may go on with it)
    auto load = [&](int q, Own &o) __attribute__((always_inline)) {
        o.t = cell(q);
        o.b = BG ? A.bcol[q] : lds[V.b + q];
        o.x = lds[V.x + q];
        const TailCoef<T> m = tail_coefs<T, DIM>(lds, o.t);
        if constexpr (KEEP) o.m = m;
        o.d = sor_inv(sor_den<T, DIM>(m.c2x, m.c2y, m.c2z));
        return !(o.t.czf & (kTailNoCell << 16));
    };
    auto coefs = [&](const Own &o) __attribute__((always_inline)) {
        if constexpr (KEEP) return o.m;
        else return tail_coefs<T, DIM>(lds, o.t);
    };
    auto update = [&](const Own &o) __attribute__((always_inline)) {
        const Stencil<T, DIM> s = tail_gather<T, DIM, false>(lds, o.t, o.x, neg, 0);
        const TailCoef<T> m = coefs(o);
        const T num = sor_num<T, DIM>(s, m.c2x, m.c1x, m.c2y, m.c1y, m.c2z, m.c1z, o.b, w);
        return (T(1.0) - w) * o.x + sor_quot_inv(num, o.d);
    };
    auto resid = [&](const Own &o, auto stale) __attribute__((always_inline)) {
        constexpr bool STALE = decltype(stale)::value;
        const Stencil<T, DIM> s = tail_gather<T, DIM, STALE>(lds, o.t, o.x, neg, delta);
        const TailCoef<T> m = coefs(o);
        return residual<T, DIM>(s, m.c2x, m.c1x, m.c2y, m.c1y, m.c2z, m.c1z, o.b);
    };
    int iter = 0;
    if (!wave || wv == 0) {
        Own o[2][CPT];
        bool act[2][CPT];
        if (pro) {
            for (int q = tid; q < 2 * half; q += wave ? 64 : nthr) {
                const int col = q >= half, u = q - col * half;
                const unsigned row = (unsigned)u / (unsigned)V.hz;
                const int m = u - (int)(row * (unsigned)V.hz);
                // rows (i, j) -> coarse (i / 2, j / 2); both cells m of a row have K = m
                const int i = DIM == 3 ? (int)(row / (unsigned)V.n[1]) : (int)row;
                const int j = DIM == 3 ? (int)(row - (unsigned)i * (unsigned)V.n[1]) : 0;
                lds[V.x + q] = lds[C.x + tail_at<DIM>(C, i >> 1, j >> 1, m)] + lds[V.x + q];
            }
            sync();
        }
        // a thread beyond the level's last cell takes that cell too, without
        // writing it: no load waits behind a branch
#pragma unroll
        for (int col = 0; col < 2; ++col)
#pragma unroll
            for (int e = 0; e < CPT; ++e) {
                const int u = tid + e * nthr;
                act[col][e] = load(col * half + min(u, half - 1), o[col][e]) && u < half;
            }
        auto pass = [&](auto colc) __attribute__((always_inline)) {
            constexpr int col = decltype(colc)::value;
            const int base = V.x + col * half;
#pragma unroll
            for (int p = 0; p < CPT; p += PAIR) {
                if (p > 0 && p * nthr >= half) continue;
                T v[PAIR];
#pragma unroll
                for (int e = 0; e < PAIR; ++e) v[e] = update(o[col][p + e]);
#pragma unroll
                for (int e = 0; e < PAIR; ++e) {
                    const int at = base + tid + (p + e) * nthr;
                    if (act[col][p + e]) {
                        if (solve) lds[at + delta] = o[col][p + e].x;
                        if (!odd) lds[at] = v[e];
                    }
                    o[col][p + e].x = v[e];
                }
            }
            if (rest)
                for (int u = tid + CPT * nthr; u < half; u += nthr) {
                    Own q;
                    if (!load(col * half + u, q)) continue;
                    const T v = update(q);
                    lds[base + u] = odd ? q.x : v;
                    if (solve || odd) lds[base + u + delta] = odd ? v : q.x;
                }
            if (odd) {
                sync();
#pragma unroll
                for (int e = 0; e < CPT; ++e)
                    if (act[col][e]) lds[base + tid + e * nthr] = o[col][e].x;
                if (rest)
                    for (int u = tid + CPT * nthr; u < half; u += nthr) {
                        const T v = lds[base + u + delta];
                        lds[base + u + delta] = lds[base + u];
                        lds[base + u] = v;
                    }
            }
            sync();
        };
        double tol = A.tol;
        if (solve && A.rel_floor > 0.0) {
            // the FP32 floor of the correction equation (CoarseCtl::rel_floor)
            double bm = 0.0;
#pragma unroll
            for (int col = 0; col < 2; ++col) {
#pragma unroll
                for (int e = 0; e < CPT; ++e)
                    if (act[col][e]) bm = fmax(bm, fabs((double)o[col][e].b));
                if (rest)
                    for (int u = tid + CPT * nthr; u < half; u += nthr) {
                        Own q;
                        if (load(col * half + u, q)) bm = fmax(bm, fabs((double)q.b));
                    }
            }
            tol = fmax(tol, A.rel_floor * (wave ? group_max<true>(bm, red) : group_max<false>(bm, red)));
        }
        for (int n = 0; solve || n < count; ++n) {
            pass(std::integral_constant<int, 0>{});
            pass(std::integral_constant<int, 1>{});
            if (!solve) continue;
            bool any = false;
            // |r| >= tol of some cell; the reference's maximum starts at
            // -1e-10 and passes over NaN
#pragma unroll
            for (int col = 0; col < 2; ++col) {
#pragma unroll
                for (int e = 0; e < CPT; ++e) {
                    if (e > 0 && e * nthr >= half) continue;
                    any = (fabs((double)resid(o[col][e], std::true_type{})) >= tol && act[col][e]) || any;
                }
                if (rest)
                    for (int u = tid + CPT * nthr; u < half; u += nthr) {
                        Own q;
                        if (load(col * half + u, q)) any = fabs((double)resid(q, std::true_type{})) >= tol || any;
                    }
            }
            any = __ballot(any) != 0;
            if (!wave) {
                if (lane == 0) wflag[wv] = any ? 1 : 0;
                __syncthreads();
                any = __ballot(lane < nwave && wflag[lane < nwave ? lane : 0] != 0) != 0;
            }
            if (!any && -1.0e-10 < tol) break;
            iter += 1;
            if (iter > A.max_count) break;
        }
        if (emit) {
#pragma unroll
            for (int col = 0; col < 2; ++col)
#pragma unroll
                for (int e = 0; e < CPT; ++e) {
                    if (e > 0 && e * nthr >= half) continue;
                    const T r = resid(o[col][e], std::false_type{});
                    if (act[col][e]) lds[A.res + col * half + tid + e * nthr] = r;
                }
        }
    }
    // a one-wave level is read by the whole workgroup next
    __syncthreads();
    return iter;
}

// BG: the coarsest level alone, its right-hand side in global memory (see
// plan_tail; a kernel of its own, since a pointer to either memory would make
// each access a flat one)
template <typename T, int DIM, bool BG>
__global__ void __launch_bounds__(kTailThreads) k_tail(TailArgs<T> A) {
    extern __shared__ __align__(16) unsigned char tail_raw[];
    T *lds = reinterpret_cast<T *>(tail_raw);
    __shared__ double red[16];
    __shared__ int wflag[kTailThreads / 64];
    const int S = A.first, D = A.last;

    // Staging, with every global load issued before the first barrier: the
    // metric coefficients and restriction factors and the cell tables as flat
    // coalesced copies of their packed images, level S's iterate and
    // right-hand side beside them.
    {
        unsigned *lw = reinterpret_cast<unsigned *>(lds);
        for (int e = threadIdx.x; e < A.ncoef; e += kTailThreads) lds[A.coff + e] = A.coef[e];
        for (int e = threadIdx.x; e < A.ncellw / 4; e += kTailThreads)
            *reinterpret_cast<uint4 *>(lw + A.cellw + 4 * e) = reinterpret_cast<const uint4 *>(A.cellimg)[e];
        const TailLevel &V = A.L[0];
        const int total = V.n[0] * V.n[1] * V.n[2];
        for (int t = threadIdx.x; t < total; t += kTailThreads) {
            int i, j, k;
            tcoords(t, V.n[1], V.n[2], i, j, k);
            const long g = (long)i * A.sx + (long)j * A.sy + (A.hz ? (long)(k & 1) * A.hz + (k >> 1) : (long)k);
            const int at = tail_at<DIM>(V, i, j, k);
            lds[V.x + at] = A.x[g];
            if constexpr (BG) A.bcol[at] = A.b[g];
            else lds[V.b + at] = A.b[g];
        }
        __syncthreads();
    }

    // The V-cycle over levels S..D as one loop of steps, so that each phase's
    // code appears once in the kernel (a single CU runs this kernel, and its
    // instruction cache holds far less than one copy per call site):
    //   down-leg, l = S..D: pre-smoothing (the coarsest treatment at D > 0;
    //     l = S = D = 0 is the whole V-cycle of a single-level hierarchy,
    //     poisson.cc:228), then the residual of l restricted into the
    //     right-hand side of l + 1, whose iterate starts at zero;
    //   up-leg, l = D-1..S: injection plus the saved iterate, then
    //     post-smoothing of l.
    int iters = 0;  // meaningful in thread 0
    const int nsteps = 2 * (D - S) + 1;
    for (int st = 0; st < nsteps; ++st) {
        const bool up = st > D - S;
        const int l = up ? D - (st - (D - S)) : S + st;
        const bool solve = l == D && D > 0 && A.solve_flag;
        const bool emit = !up && l < D;
        const int count = up ? A.post : A.pre;
        const TailLevel &V = A.L[l - S], &C = A.L[l < D ? l + 1 - S : l - S];
        int it;
        if (!BG && V.cell1 >= 0) it = tail_smooth<T, DIM, 1, false>(lds, A, V, C, up, solve, count, emit, red, wflag);
        else it = tail_smooth<T, DIM, kTailColourCells, BG>(lds, A, V, C, up, solve, count, emit, red, wflag);
        if (solve) iters = it;
        if (BG || !emit) continue;
        // computeResidual + coarsen (poisson_d3.cc:71-93, 484-511; poisson_d2.cc:288-297)
        const int ctotal = C.n[0] * C.n[1] * C.n[2];
        const T *R = lds + A.res;
        for (int q = threadIdx.x; q < 2 * C.half; q += kTailThreads) lds[C.x + q] = T(0);
        for (int t = threadIdx.x; t < ctotal; t += kTailThreads) {
            int I, J, K;
            tcoords(t, C.n[1], C.n[2], I, J, K);
            // child (di, dj, dk): row (2I + di, 2J + dj), position K of the colour of its k parity
            auto r = [&](int di, int dj, int dk) {
                return R[((di + dj + dk) & 1) * V.half + (DIM == 3 ? (2 * I + di) * V.n[1] + 2 * J + dj : 2 * I + di) * V.hz + K];
            };
            T out;
            if (DIM == 3) {
                const T lx = lds[C.lo[0] + I], hx = lds[C.hi[0] + I], ly = lds[C.lo[1] + J], hy = lds[C.hi[1] + J],
                        lz = lds[C.lo[2] + K], hz = lds[C.hi[2] + K];
                const T v000 = lx * ly * lz, v100 = hx * ly * lz, v010 = lx * hy * lz, v001 = lx * ly * hz;
                const T v011 = lx * hy * hz, v101 = hx * ly * hz, v110 = hx * hy * lz, v111 = hx * hy * hz;
                const T vtot = lds[C.wd[0] + I] * lds[C.wd[1] + J] * lds[C.wd[2] + K];
                out = (v111 * r(1, 1, 1) + v000 * r(0, 0, 0) + v110 * r(1, 1, 0) + v001 * r(0, 0, 1) +
                       v101 * r(1, 0, 1) + v010 * r(0, 1, 0) + v011 * r(0, 1, 1) + v100 * r(1, 0, 0)) / vtot;
            } else {
                out = (r(1, 0, 1) + r(0, 0, 0) + r(1, 0, 0) + r(0, 0, 1)) / T(4);
            }
            lds[C.b + tail_at<DIM>(C, I, J, K)] = out;
        }
        __syncthreads();
    }
    // level S back to global memory
    {
        const TailLevel &V = A.L[0];
        const int total = V.n[0] * V.n[1] * V.n[2];
        for (int t = threadIdx.x; t < total; t += kTailThreads) {
            int i, j, k;
            tcoords(t, V.n[1], V.n[2], i, j, k);
            A.x[(long)i * A.sx + (long)j * A.sy + (A.hz ? (long)(k & 1) * A.hz + (k >> 1) : (long)k)] =
                lds[V.x + tail_at<DIM>(V, i, j, k)];
        }
    }
    if (threadIdx.x == 0 && A.iters_out && A.solve_flag) *A.iters_out = iters;
}

}  // namespace saras
