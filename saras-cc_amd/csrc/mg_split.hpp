// mg_split.hpp -- red-black SOR colour pass on colour-split rows.
//
// In a split row the cells of one colour are one contiguous half-row (even k
// in [0, nz/2), odd k at hz + [0, nz/2)), so one colour pass (poisson_d3.cc:
// 105-170 for red, 177-242 for black) reads and writes whole 16-byte vectors:
// each lane updates W = 16 / sizeof(T) consecutive cells of its row's
// colour.  Per cell it loads the same-half vectors of the four x/y
// neighbour rows, the other half of its own row (the two z neighbours of
// each cell; the one that lies in the adjacent vector comes from the
// neighbouring lane), the right-hand side and the reordered z metric
// coefficients.  The update is the same sor_update expression as the
// z-contiguous pass, so both layouts give identical values.
//
// Blocks are remapped so that each XCD works through one contiguous range of
// rows: the neighbour rows of a row were fetched by the same XCD a moment
// earlier and are read from its L2.
#pragma once
#include <type_traits>

#include "mg_kernels.hpp"

namespace saras {

template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
    using V = float4;
    static constexpr int W = 4;
    __device__ static float get(const float4 &v, int e) { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; }
    __device__ static float4 make(const float *a) { return make_float4(a[0], a[1], a[2], a[3]); }
};
template <>
struct Vec16<double> {
    using V = double2;
    static constexpr int W = 2;
    __device__ static double get(const double2 &v, int e) { return e == 0 ? v.x : v.y; }
    __device__ static double2 make(const double *a) { return make_double2(a[0], a[1]); }
};

constexpr int kSplitThreads = 256;

// W consecutive coarse cells K0..K0+W-1 of coarse row (I, J) in the coarse
// level's own layout (split or z-contiguous), as one vector
template <typename T>
__device__ __forceinline__ void coarse_vec(const T *__restrict__ e, long base, long chz, int K0, T (&out)[Vec16<T>::W]) {
    using VT = Vec16<T>;
    constexpr int W = VT::W;
    if (chz == 0) {
        const typename VT::V v = *reinterpret_cast<const typename VT::V *>(e + base + K0);
#pragma unroll
        for (int q = 0; q < W; ++q) out[q] = VT::get(v, q);
    } else {
        if constexpr (W == 4) {
            // even K at K/2, odd K at chz + K/2 (K0 is a multiple of 4): two pairs
            const float2 ev = *reinterpret_cast<const float2 *>(e + base + (K0 >> 1));
            const float2 od = *reinterpret_cast<const float2 *>(e + base + chz + (K0 >> 1));
            out[0] = ev.x;
            out[1] = od.x;
            out[2] = ev.y;
            out[3] = od.y;
        } else {
#pragma unroll
            for (int q = 0; q < W; ++q) out[q] = e[base + (q & 1) * chz + ((K0 + q) >> 1)];
        }
    }
}

template <typename T>
__device__ __forceinline__ void coarse_store(T *__restrict__ dst, long base, long chz, int K0,
                                             const T (&in)[Vec16<T>::W]) {
    using VT = Vec16<T>;
    constexpr int W = VT::W;
    if (chz == 0) {
        *reinterpret_cast<typename VT::V *>(dst + base + K0) = VT::make(in);
    } else {
#pragma unroll
        for (int q = 0; q < W; ++q) dst[base + (q & 1) * chz + ((K0 + q) >> 1)] = in[q];
    }
}


// N consecutive values of a row at p: one vector load where N fills 16 bytes
template <typename T, int N>
__device__ __forceinline__ void load_n(const T *__restrict__ p, T (&out)[N]) {
    if constexpr (N == Vec16<T>::W) {
        const typename Vec16<T>::V v = *reinterpret_cast<const typename Vec16<T>::V *>(p);
#pragma unroll
        for (int q = 0; q < N; ++q) out[q] = Vec16<T>::get(v, q);
    } else if constexpr (N == 2 && sizeof(T) == 4) {
        const float2 v = *reinterpret_cast<const float2 *>(p);
        out[0] = v.x;
        out[1] = v.y;
    } else {
#pragma unroll
        for (int q = 0; q < N; ++q) out[q] = p[q];
    }
}

// N consecutive coarse cells K0.. of a coarse row in the coarse level's layout
template <typename T, int N>
__device__ __forceinline__ void coarse_store_n(T *__restrict__ dst, long base, long chz, int K0, const T (&in)[N]) {
    if (chz == 0 && N == Vec16<T>::W) {
        *reinterpret_cast<typename Vec16<T>::V *>(dst + base + K0) = Vec16<T>::make(in);
    } else {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int K = K0 + q;
            dst[base + (chz ? (long)(K & 1) * chz + (K >> 1) : (long)K)] = in[q];
        }
    }
}

// one coarse cell (I, J, K) of a level in its own layout
template <typename T>
__device__ __forceinline__ T coarse_at(const T *__restrict__ e, long base, long chz, int K) {
    return e[base + (chz ? (long)(K & 1) * chz + (K >> 1) : (long)K)];
}

// n / d for n < 2^31 by a multiplication (Granlund and Montgomery, "Division
// by invariant integers using multiplication", 1994): m = ceil(2^(31 + l) / d),
// l = ceil(log2 d), and the quotient is the high word of m n shifted by l - 1.
struct FastDiv {
    unsigned m = 0, s = 0, d = 1;   // m = 0: d = 1
    __host__ static FastDiv of(unsigned d) {
        FastDiv f;
        f.d = d;
        if (d <= 1) return f;
        unsigned l = 0;
        while ((1ull << l) < d) ++l;
        f.m = (unsigned)(((1ull << (31 + l)) + d - 1) / d);
        f.s = l - 1;
        return f;
    }
    __device__ __forceinline__ unsigned div(unsigned n) const { return m ? __umulhi(n, m) >> s : n; }
};

// How the vectors of a colour pass are numbered: vector v of row group g, the
// R rows (i, R jp ..) of a 3-D level or (R g ..) of a planar one.  Groups run
// over the rows of a tile of wj groups, i by i, then the next tile (wj covers
// the whole y axis where rows need no tiles, see LevelArgs::rtile).
struct RowMap {
    FastDiv q, tile, wj;   // vectors of a half-row; groups of a tile; groups of a tile's i-row
    unsigned total;        // vectors of the level
    bool div64 = false;    // their numbers take no FastDiv (2^31 and more; not in RB_PAIR, see plan_pass)
};

// What the iterate is when a colour pass reads it.
//   RB_PLAIN  the level's iterate.
//   RB_ZERO   zero (a red pass): x is not read, +0 stands wherever a cell would
//             have been, and the black half is written as +0, the same values
//             as clearing x and running the ordinary pass.
//   RB_RED, RB_BLACK  the first sweep after the prolongation, whose input is
//             x + P e with P the injection from the coarse iterate e
//             (poisson_d3.cc:548-558, poisson.cc:266): the red pass reads every
//             cell as e(coarse) + x, the black pass its own cells (its
//             neighbours are the red values just written), so the separate
//             prolongation pass is not needed.
enum RbMode { RB_PLAIN, RB_ZERO, RB_RED, RB_BLACK };
enum RbForm { RB_PAIR, RB_PAIR64, RB_GENERAL };

// One colour pass over a split level; the grid is a multiple of kXcds blocks.
// A lane updates one vector of each of R rows that follow one another along y
// (x in a planar level).  With R = 2 each row's vector of the other colour is
// also the neighbour row of the other, so the pair loads 10 vectors of the
// iterate and right-hand side where two single rows load 14.
//
// W1: w == 1 (the "SOR Parameter" of every reference deck).  The update
// (1 - w) x + q then equals q whenever q != 0 and x is finite (0 x is a
// signed zero), so the cells' own values are read only where q is a zero
// (to give the sign the reference's sum has).
// UNI: every axis is uniform, so the coefficients are one value per axis and
// the divisor (FP32: its reciprocal) is formed once.
// FORM: RB_PAIR; RB_PAIR64, the same with 64-bit offsets (arrays of 4 GB and
// more); RB_GENERAL (R = 1, any w, 64-bit offsets, inhomogeneous walls).
//
// No load waits behind a lane-dependent branch: a neighbour beyond a wall is
// read at the cell's own place (which is the Neumann rule) and its sign
// flipped for a Dirichlet wall, and a row's parity selects between loaded
// values; byte offsets are 32 bits wide on scalar bases, divisions by the row
// length are multiplications.  Issuing that arithmetic and waiting for one
// load after another took as long as the traffic before: see the measured
// times at Ops::rb_pass (mg_solver.hip).
template <typename T, int DIM, int MODE, bool W1, bool UNI, int FORM>
__global__ void __launch_bounds__(kSplitThreads) k_rb_split(LevelArgs<T> L, RowMap M, T *__restrict__ x,
                                                            const T *__restrict__ b, int colour, T w,
                                                            const T *__restrict__ e, long esx, long esy, long ehz) {
    constexpr bool GEN = FORM == RB_GENERAL;
    static_assert(!GEN || (!W1 && !UNI), "the general form takes any w and any metric");
    using VT = Vec16<T>;
    using V = typename VT::V;
    using OFF = std::conditional_t<FORM != RB_PAIR, unsigned long, unsigned>;   // byte offset
    constexpr int W = VT::W, R = GEN ? 1 : 2;
    constexpr bool RED = MODE == RB_RED, BLACK = MODE == RB_BLACK, ZERO = MODE == RB_ZERO;
    const unsigned per = gridDim.x / kXcds;
    const unsigned logical = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    const unsigned t = logical * kSplitThreads + threadIdx.x;
    if (t >= M.total) return;
    const int nx = L.n[0], ny = L.n[1], half = L.n[2] >> 1;
    const unsigned g = FORM != RB_PAIR && M.div64 ? t / M.q.d : M.q.div(t);
    const int m0 = (int)(t - g * M.q.d) * W;
    int i, j;
    if (DIM == 3) {
        const unsigned tile = M.tile.div(g), rem = g - tile * M.tile.d, gi = M.wj.div(rem);
        i = (int)gi;
        j = R * (int)(tile * M.wj.d + rem - gi * M.wj.d);
    } else {
        i = R * (int)g;
        j = 0;
    }
    const OFF sx = (OFF)L.sx * sizeof(T), sy = (OFF)L.sy * sizeof(T), hz = (OFF)L.hz * sizeof(T);
    const OFF vo = (OFF)m0 * sizeof(T);
    auto xv = [&](OFF o) __attribute__((always_inline)) {
        return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(x) + o);
    };
    auto ld = [](const T *p, OFF o) __attribute__((always_inline)) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + o);
    };
    // the axis along which the R rows follow one another (P), and x in 3-D (Q)
    constexpr int AP = DIM == 3 ? 1 : 0;
    const OFF sp = DIM == 3 ? sy : sx;
    const int p0 = DIM == 3 ? j : i, np = DIM == 3 ? ny : nx;
    const int h0 = (i + j + colour) & 1;
    OFF row[R], own[R], oth[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int h = h0 ^ (r & 1);
        row[r] = (OFF)i * sx + (OFF)j * sy + (OFF)r * sp;
        own[r] = row[r] + (h ? hz : 0) + vo;
        oth[r] = row[r] + (h ? 0 : hz) + vo;
    }
    // neighbour rows: wrapped, or beyond a wall the row itself
    const bool inl = p0 > 0, inr = p0 + R < np, perp = L.bc_lo[AP] == BC_PER;
    const OFF pl = own[0] + (inl ? (OFF)0 - sp : (perp ? (OFF)(np - 1) * sp : (OFF)0));
    const OFF pr = own[R - 1] + (inr ? sp : (perp ? (OFF)0 - (OFF)(np - 1) * sp : (OFF)0));
    const bool ine = i + 1 < nx, inw = i > 0, perx = L.bc_lo[0] == BC_PER;
    const OFF de = ine ? sx : (perx ? (OFF)0 - (OFF)(nx - 1) * sx : (OFF)0);
    const OFF dw = inw ? (OFF)0 - sx : (perx ? (OFF)(nx - 1) * sx : (OFF)0);
    const bool perz = L.bc_lo[2] == BC_PER;
    const int lane = threadIdx.x & 63;

    // ---- loads ----
    V ov[R], bv[R], plv{}, prv{}, ev[R], wv[R], cv[R];
    T zx[R];
    bool zend[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ov[r] = ev[r] = wv[r] = cv[r] = V{};
        if (!ZERO) {
            ov[r] = xv(oth[r]);
            if (DIM == 3) {
                ev[r] = xv(own[r] + de);
                wv[r] = xv(own[r] + dw);
            }
            if (!W1) cv[r] = xv(own[r]);
        }
        bv[r] = *reinterpret_cast<const V *>(reinterpret_cast<const char *>(b) + own[r]);
    }
    if (!ZERO) {
        plv = xv(pl);
        prv = xv(pr);
    }
    // The z neighbour beyond a lane's vector, below its first even cell or
    // above its last odd one, where no adjacent lane of the wave holds it: the
    // row's end (wrapped, or the cell itself at a wall) or the next vector in
    // another wave.
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int h = h0 ^ (r & 1);
        zend[r] = h ? m0 + W == half : m0 == 0;
        const OFF zw = h ? row[r] : row[r] + hz + (OFF)(half - 1) * sizeof(T);
        const OFF zs = h ? own[r] + (W - 1) * sizeof(T) : own[r];
        const OFF zn = h ? oth[r] + W * sizeof(T) : oth[r] - sizeof(T);
        zx[r] = T(0);
        if (!ZERO && (zend[r] || lane == (h ? 63 : 0))) zx[r] = ld(x, zend[r] ? (perz ? zw : zs) : zn);
    }
    T c2x, c1x, c2y[R], c1y[R], c2z[R][W], c1z[R][W];
    if constexpr (UNI) {
        c2x = L.c2[0][0];
        c1x = L.c1[0][0];
    } else {
        c2x = DIM == 3 ? L.c2[0][i] : T(0);
        c1x = DIM == 3 ? L.c1[0][i] : T(0);
    }
    T c2r[R], c1r[R];   // planar: the x coefficients of each row
#pragma unroll
    for (int r = 0; r < R; ++r) {
        c2r[r] = DIM == 3 || UNI ? c2x : L.c2[0][i + r];
        c1r[r] = DIM == 3 || UNI ? c1x : L.c1[0][i + r];
        c2y[r] = DIM == 3 ? (UNI ? L.c2[1][0] : L.c2[1][j + r]) : T(0);
        c1y[r] = DIM == 3 ? (UNI ? L.c1[1][0] : L.c1[1][j + r]) : T(0);
        if constexpr (UNI) {
#pragma unroll
            for (int q = 0; q < W; ++q) {
                c2z[r][q] = L.c2[2][0];
                c1z[r][q] = L.c1[2][0];
            }
        } else {
            const int at = (h0 ^ (r & 1)) * half + m0;
            const V a = *reinterpret_cast<const V *>(L.c2zs + at), c = *reinterpret_cast<const V *>(L.c1zs + at);
#pragma unroll
            for (int q = 0; q < W; ++q) {
                c2z[r][q] = VT::get(a, q);
                c1z[r][q] = VT::get(c, q);
            }
        }
    }
    // ---- the prolongation: the coarse vector over cells m0.. of a row ----
    auto coarse = [&](int ci, int cj, T(&out)[W]) __attribute__((always_inline)) {
        coarse_vec(e, (long)ci * esx + (long)cj * esy, ehz, m0, out);
    };
    // the rows of a pair lie in one coarse row (j, or i in a planar level, is even)
    T eo[W];
#pragma unroll
    for (int q = 0; q < W; ++q) eo[q] = T(0);
    const bool walls = !perz || !perp || (DIM == 3 && !perx);
    if (RED || (BLACK && (walls || !W1))) coarse(i >> 1, j >> 1, eo);
    T o[R][W], xe[R][W], xw[R][W], yl[W], yr[W], c[R][W], z[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < W; ++q) {
            o[r][q] = VT::get(ov[r], q);
            xe[r][q] = VT::get(ev[r], q);
            xw[r][q] = VT::get(wv[r], q);
            c[r][q] = VT::get(cv[r], q);
        }
#pragma unroll
    for (int q = 0; q < W; ++q) {
        yl[q] = VT::get(plv, q);
        yr[q] = VT::get(prv, q);
    }
    if (RED) {
        // every cell read is e + x; one of the x rows, and in a row pair both y
        // rows, lie in another coarse row
        T el[W], er[W], eq[W];
        const int lp = inl ? p0 - 1 : (perp ? np - 1 : p0), rp = inr ? p0 + R : (perp ? 0 : p0 + R - 1);
        coarse(DIM == 3 ? i >> 1 : lp >> 1, DIM == 3 ? lp >> 1 : 0, el);
        coarse(DIM == 3 ? i >> 1 : rp >> 1, DIM == 3 ? rp >> 1 : 0, er);
        const int ie = ine ? i + 1 : (perx ? 0 : i), iw = inw ? i - 1 : (perx ? nx - 1 : i);
        // i even: x+ lies in the cell's coarse row; i odd: x- does (an even extent's wrap: i = n - 1 and 0)
        const bool eshare = (ie >> 1) == (i >> 1), wshare = (iw >> 1) == (i >> 1);
        if (DIM == 3) coarse(eshare ? iw >> 1 : ie >> 1, j >> 1, eq);
#pragma unroll
        for (int q = 0; q < W; ++q) {
            yl[q] = el[q] + yl[q];
            yr[q] = er[q] + yr[q];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                o[r][q] = eo[q] + o[r][q];
                c[r][q] = eo[q] + c[r][q];
                if (DIM == 3) {
                    xe[r][q] = (eshare ? eo[q] : eq[q]) + xe[r][q];
                    xw[r][q] = (wshare ? eo[q] : eq[q]) + xw[r][q];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int h = h0 ^ (r & 1);
            const int kz = zend[r] ? (perz ? (h ? 0 : half - 1) : (h ? m0 + W - 1 : m0)) : (h ? m0 + W : m0 - 1);
            if (zend[r] || lane == (h ? 63 : 0)) zx[r] = coarse_at(e, (long)(i >> 1) * esx + (long)(j >> 1) * esy, ehz, kz) + zx[r];
        }
    }
    if (BLACK && (walls || !W1)) {
        // the cells' own values, which walls and (1 - w) x read
#pragma unroll
        for (int q = 0; q < W; ++q) {
            if (!inl && !perp) yl[q] = eo[q] + yl[q];
            if (!inr && !perp) yr[q] = eo[q] + yr[q];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                c[r][q] = eo[q] + c[r][q];
                if (DIM == 3 && !ine && !perx) xe[r][q] = eo[q] + xe[r][q];
                if (DIM == 3 && !inw && !perx) xw[r][q] = eo[q] + xw[r][q];
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (zend[r] && !perz) zx[r] = ((h0 ^ (r & 1)) ? eo[W - 1] : eo[0]) + zx[r];
    }
    // ---- wall rules ----
    auto flip = [&](bool wall, int bc, T v) __attribute__((always_inline)) { return wall && bc == BC_DIR ? -v : v; };
#pragma unroll
    for (int q = 0; q < W; ++q) {
        yl[q] = flip(!inl, L.bc_lo[AP], yl[q]);
        yr[q] = flip(!inr, L.bc_hi[AP], yr[q]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (DIM == 3) {
                xe[r][q] = flip(!ine, L.bc_hi[0], xe[r][q]);
                xw[r][q] = flip(!inw, L.bc_lo[0], xw[r][q]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int h = h0 ^ (r & 1);
        const T edge = flip(zend[r], h ? L.bc_hi[2] : L.bc_lo[2], zx[r]);
        // the adjacent lane's value where it holds the same row
        const T prev = __shfl_up(o[r][W - 1], 1, 64), next = __shfl_down(o[r][0], 1, 64);
        z[r] = zend[r] || lane == (h ? 63 : 0) ? edge : (h ? next : prev);
    }
    if (GEN) {
        // inhomogeneous walls: 2 w - x (bc_value)
        const int nz = L.n[2];
#pragma unroll
        for (int q = 0; q < W; ++q) {
            const int k = 2 * (m0 + q) + h0;
            const T own_c = c[0][q];
            if (DIM == 3) {
                if (!ine && L.bc_hi[0] == BC_DIRV) xe[0][q] = bc_value(BC_DIRV, own_c, T(0), L.wall[0][(j + 1) * (nz + 2) + k + 1]);
                if (!inw && L.bc_lo[0] == BC_DIRV) xw[0][q] = bc_value(BC_DIRV, own_c, T(0), L.wall[0][(j + 1) * (nz + 2) + k + 1]);
                if (!inr && L.bc_hi[1] == BC_DIRV) yr[q] = bc_value(BC_DIRV, own_c, T(0), L.wall[1][(i + 1) * (nz + 2) + k + 1]);
                if (!inl && L.bc_lo[1] == BC_DIRV) yl[q] = bc_value(BC_DIRV, own_c, T(0), L.wall[1][(i + 1) * (nz + 2) + k + 1]);
            } else {
                if (!inr && L.bc_hi[0] == BC_DIRV) yr[q] = bc_value(BC_DIRV, own_c, T(0), L.wall[0][k + 1]);
                if (!inl && L.bc_lo[0] == BC_DIRV) yl[q] = bc_value(BC_DIRV, own_c, T(0), L.wall[0][k + 1]);
            }
        }
        const T zw = (zend[0] && (h0 ? L.bc_hi[2] : L.bc_lo[2]) == BC_DIRV)
                         ? (DIM == 3 ? L.wall[2][(i + 1) * (ny + 2) + j + 1] : L.wall[2][i + 1])
                         : T(0);
        if (zend[0] && (h0 ? L.bc_hi[2] : L.bc_lo[2]) == BC_DIRV) z[0] = bc_value(BC_DIRV, h0 ? c[0][W - 1] : c[0][0], T(0), zw);
    }
    // ---- the updates ----
    const T dinv = UNI ? sor_inv(sor_den<T, DIM>(c2x, c2y[0], c2z[0][0])) : T(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int h = h0 ^ (r & 1);
        T out[W];
        bool zero = false;
#pragma unroll
        for (int q = 0; q < W; ++q) {
            Stencil<T, DIM> s;
            // along P: the neighbour rows, within the pair the other row's other-colour vector
            const T lo = r > 0 ? o[r > 0 ? r - 1 : 0][q] : yl[q], hi = r < R - 1 ? o[r < R - 1 ? r + 1 : r][q] : yr[q];
            s.c = c[r][q];
            if (DIM == 3) {
                s.xE = xe[r][q];
                s.xW = xw[r][q];
                s.yN = hi;
                s.yS = lo;
            } else {
                s.xE = hi;
                s.xW = lo;
            }
            s.zB = h ? o[r][q] : (q > 0 ? o[r][q > 0 ? q - 1 : 0] : z[r]);
            s.zT = h ? (q < W - 1 ? o[r][q < W - 1 ? q + 1 : q] : z[r]) : o[r][q];
            const T num = sor_num<T, DIM>(s, c2r[r], c1r[r], c2y[r], c1y[r], c2z[r][q], c1z[r][q], VT::get(bv[r], q), w);
            out[q] = UNI ? sor_quot_inv(num, dinv) : sor_div(num, sor_den<T, DIM>(c2r[r], c2y[r], c2z[r][q]));
            zero = zero || out[q] == T(0);
        }
        if (W1 && zero) {
            // a zero quotient takes the sign of (1 - w) x + q: read the cells now
            V lv{};
            if (!ZERO) lv = xv(own[r]);
            if (BLACK && !walls) coarse(i >> 1, j >> 1, eo);
#pragma unroll
            for (int q = 0; q < W; ++q) c[r][q] = RED || BLACK ? eo[q] + VT::get(lv, q) : VT::get(lv, q);
        }
#pragma unroll
        for (int q = 0; q < W; ++q)
            if (!W1 || out[q] == T(0)) out[q] = (T(1.0) - w) * c[r][q] + out[q];
        *reinterpret_cast<V *>(reinterpret_cast<char *>(x) + own[r]) = VT::make(out);
        if (ZERO) *reinterpret_cast<V *>(reinterpret_cast<char *>(x) + oth[r]) = V{};
    }
}

// ---------------------------------------------------------------------------
// residual of a split level restricted to the next level (the same
// computeResidual + coarsen expressions as k_resid_restrict,
// poisson_d3.cc:71-93, 484-511; poisson_d2.cc:288-297), and x(l+1) = 0.  A
// lane owns W consecutive coarse cells K0.. of coarse row (I, J): their fine
// children are the even and odd half-rows at K0.. of the 2 x 2 child rows.
// RED: the coarse level's first pre-smoothing red pass is applied as well.
// Its input iterate is the zero just written, so each red cell's update reads
// only zeros (wall rules of zero give zero) and its own new right-hand side:
// the same sor_update expression, evaluated here instead of in a launch of
// its own.
// ---------------------------------------------------------------------------
// Coarse cells per lane: 2 in FP32 (4 measured slower); 1 in FP64, where two per lane need
// more than 256 registers.
template <typename T>
constexpr int rr_width() {
    return sizeof(T) == 4 ? 2 : 1;
}

template <typename T, int DIM, bool RED = false>
__global__ void __launch_bounds__(kSplitThreads) k_rr_split(LevelArgs<T> F, const T *__restrict__ x,
                                                            const T *__restrict__ b, LevelArgs<T> C,
                                                            T *__restrict__ bc, T *__restrict__ xc, RestrictArgs<T> R,
                                                            int nblocks, T w) {
    constexpr int W = rr_width<T>();
    const int per = gridDim.x / kXcds;
    const int logical = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (logical >= nblocks) return;
    const int nx = F.n[0], ny = F.n[1], nz = F.n[2];
    const int half = nz >> 1, q = half / W;
    const int cy = C.n[1];
    const long total = (long)C.n[0] * cy * q;
    const long t = (long)logical * kSplitThreads + threadIdx.x;
    if (t >= total) return;
    const int crow = (int)(t / q);
    const int v = (int)(t - (long)crow * q);
    const int I = crow / cy, J = crow - (crow / cy) * cy;
    const int K0 = v * W;
    const long hz = F.hz;
    const int lane = threadIdx.x & 63;
    auto ldv = [&](const T *p, T (&out)[W]) { load_n<T, W>(p, out); };
    // residuals of the children: [di][dj][dk][e], dk = 0 the even cell 2K, 1 the odd cell 2K+1
    T res[2][DIM == 3 ? 2 : 1][2][W];
    const T c2e0 = T(0);
    (void)c2e0;
    T cz2e[W], cz1e[W], cz2o[W], cz1o[W];
    ldv(F.c2zs + K0, cz2e);
    ldv(F.c1zs + K0, cz1e);
    ldv(F.c2zs + half + K0, cz2o);
    ldv(F.c1zs + half + K0, cz1o);
#pragma unroll
    for (int di = 0; di < 2; ++di) {
#pragma unroll
        for (int dj = 0; dj < (DIM == 3 ? 2 : 1); ++dj) {
            const int i = 2 * I + di, j = DIM == 3 ? 2 * J + dj : 0;
            const long rb = (long)i * F.sx + (long)j * F.sy;
            T xe[W], xo[W], be[W], bo[W];
            ldv(x + rb + K0, xe);
            ldv(x + rb + hz + K0, xo);
            ldv(b + rb + K0, be);
            ldv(b + rb + hz + K0, bo);
            // neighbour rows: [0] E, [1] W, [2] N, [3] S; even and odd halves
            T ne[4][W], no[4][W];
            auto nbr = [&](int slot, bool inside, long off, int bc, int axis) {
                if (inside || bc == BC_PER) {
                    ldv(x + rb + off + K0, ne[slot]);
                    ldv(x + rb + off + hz + K0, no[slot]);
                } else {
#pragma unroll
                    for (int e = 0; e < W; ++e) {
                        T wve = T(0), wvo = T(0);
                        if (bc == BC_DIRV) {
                            const int ke = 2 * (K0 + e), ko = ke + 1;
                            if (axis == 0) {
                                wve = DIM == 3 ? F.wall[0][(j + 1) * (nz + 2) + ke + 1] : F.wall[0][ke + 1];
                                wvo = DIM == 3 ? F.wall[0][(j + 1) * (nz + 2) + ko + 1] : F.wall[0][ko + 1];
                            } else {
                                wve = F.wall[1][(i + 1) * (nz + 2) + ke + 1];
                                wvo = F.wall[1][(i + 1) * (nz + 2) + ko + 1];
                            }
                        }
                        ne[slot][e] = bc_value(bc, xe[e], T(0), wve);
                        no[slot][e] = bc_value(bc, xo[e], T(0), wvo);
                    }
                }
            };
            nbr(0, i + 1 < nx, i + 1 < nx ? F.sx : -(long)(nx - 1) * F.sx, F.bc_hi[0], 0);
            nbr(1, i > 0, i > 0 ? -F.sx : (long)(nx - 1) * F.sx, F.bc_lo[0], 0);
            if (DIM == 3) {
                nbr(2, j + 1 < ny, j + 1 < ny ? F.sy : -(long)(ny - 1) * F.sy, F.bc_hi[1], 1);
                nbr(3, j > 0, j > 0 ? -F.sy : (long)(ny - 1) * F.sy, F.bc_lo[1], 1);
            }
            // z: even cell 2K has zB = odd[K-1], zT = odd[K]; odd cell has zB = even[K], zT = even[K+1]
            const T from_prev = __shfl_up(xo[W - 1], 1, 64);
            const T from_next = __shfl_down(xe[0], 1, 64);
            T zlo0, zhi_last;
            if (K0 == 0) {
                if (F.bc_lo[2] == BC_PER) zlo0 = x[rb + hz + (half - 1)];
                else {
                    const T wv = F.bc_lo[2] == BC_DIRV ? (DIM == 3 ? F.wall[2][(i + 1) * (ny + 2) + j + 1] : F.wall[2][i + 1])
                                                       : T(0);
                    zlo0 = bc_value(F.bc_lo[2], xe[0], T(0), wv);
                }
            } else {
                zlo0 = lane > 0 ? from_prev : x[rb + hz + K0 - 1];
            }
            if (K0 + W == half) {
                if (F.bc_hi[2] == BC_PER) zhi_last = x[rb];
                else {
                    const T wv = F.bc_hi[2] == BC_DIRV ? (DIM == 3 ? F.wall[2][(i + 1) * (ny + 2) + j + 1] : F.wall[2][i + 1])
                                                       : T(0);
                    zhi_last = bc_value(F.bc_hi[2], xo[W - 1], T(0), wv);
                }
            } else {
                zhi_last = lane < 63 ? from_next : x[rb + K0 + W];
            }
            const T c2x = F.c2[0][i], c1x = F.c1[0][i];
            const T c2y = DIM == 3 ? F.c2[1][j] : T(0), c1y = DIM == 3 ? F.c1[1][j] : T(0);
#pragma unroll
            for (int e = 0; e < W; ++e) {
                Stencil<T, DIM> s;
                s.c = xe[e];
                s.xE = ne[0][e];
                s.xW = ne[1][e];
                if (DIM == 3) {
                    s.yN = ne[2][e];
                    s.yS = ne[3][e];
                }
                s.zB = e > 0 ? xo[e - 1] : zlo0;
                s.zT = xo[e];
                res[di][dj][0][e] = residual<T, DIM>(s, c2x, c1x, c2y, c1y, cz2e[e], cz1e[e], be[e]);
                s.c = xo[e];
                s.xE = no[0][e];
                s.xW = no[1][e];
                if (DIM == 3) {
                    s.yN = no[2][e];
                    s.yS = no[3][e];
                }
                s.zB = xe[e];
                s.zT = e < W - 1 ? xe[e + 1] : zhi_last;
                res[di][dj][1][e] = residual<T, DIM>(s, c2x, c1x, c2y, c1y, cz2o[e], cz1o[e], bo[e]);
            }
        }
    }
    T out[W], zero[W];
#pragma unroll
    for (int e = 0; e < W; ++e) {
        zero[e] = T(0);
        if (DIM == 3) {
            const T lx = R.lo[0][I], hx = R.hi[0][I], ly = R.lo[1][J], hy = R.hi[1][J];
            const T lz = R.lo[2][K0 + e], hz2 = R.hi[2][K0 + e];
            const T v000 = lx * ly * lz, v100 = hx * ly * lz, v010 = lx * hy * lz, v001 = lx * ly * hz2;
            const T v011 = lx * hy * hz2, v101 = hx * ly * hz2, v110 = hx * hy * lz, v111 = hx * hy * hz2;
            const T vtot = R.wd[0][I] * R.wd[1][J] * R.wd[2][K0 + e];
            out[e] = (v111 * res[1][DIM == 3 ? 1 : 0][1][e] + v000 * res[0][0][0][e] +
                      v110 * res[1][DIM == 3 ? 1 : 0][0][e] + v001 * res[0][0][1][e] + v101 * res[1][0][1][e] +
                      v010 * res[0][DIM == 3 ? 1 : 0][0][e] + v011 * res[0][DIM == 3 ? 1 : 0][1][e] +
                      v100 * res[1][0][0][e]) /
                     vtot;
        } else {
            out[e] = (res[1][0][1][e] + res[0][0][0][e] + res[1][0][0][e] + res[0][0][1][e]) / T(4);
        }
    }
    const long cb = (long)I * C.sx + (long)J * C.sy;
    coarse_store_n<T, W>(bc, cb, C.hz, K0, out);
    if (RED) {
        T xr[W];
        const T c2x = C.c2[0][I], c1x = C.c1[0][I];
        const T c2y = DIM == 3 ? C.c2[1][J] : T(0), c1y = DIM == 3 ? C.c1[1][J] : T(0);
#pragma unroll
        for (int e = 0; e < W; ++e) {
            const int K = K0 + e;
            if (((I + J + K) & 1) == 0) {
                Stencil<T, DIM> s;
                s.c = T(0);
                s.xE = bc_value(C.bc_hi[0], T(0), T(0), T(0));
                s.xW = bc_value(C.bc_lo[0], T(0), T(0), T(0));
                if (DIM == 3) {
                    s.yN = bc_value(C.bc_hi[1], T(0), T(0), T(0));
                    s.yS = bc_value(C.bc_lo[1], T(0), T(0), T(0));
                }
                s.zT = bc_value(C.bc_hi[2], T(0), T(0), T(0));
                s.zB = bc_value(C.bc_lo[2], T(0), T(0), T(0));
                xr[e] = sor_update<T, DIM>(s, c2x, c1x, c2y, c1y, C.c2[2][K], C.c1[2][K], out[e], w);
            } else {
                xr[e] = T(0);
            }
        }
        coarse_store_n<T, W>(xc, cb, C.hz, K0, xr);
    } else {
        coarse_store_n<T, W>(xc, cb, C.hz, K0, zero);
    }
}

// ---------------------------------------------------------------------------
// Residual + restriction of a split 3-D level.  A task is one vector of W
// coarse cells of a coarse row; a block owns kRrTasks of them.  A lane takes
// the fine rows (2I + di, 2J) and (2I + di, 2J + 1) under a task -- di by wave --
// both halves of each at the task's W fine positions, as whole 16-byte vectors
// (each row is the other's y neighbour: 20 vectors for the pair where single
// rows load 32), and leaves the products v_{di dj dk} r in LDS.  After one
// barrier each thread adds the eight products of one coarse cell in the
// reference's order and divides by the volume (poisson_d3.cc:494-511).  Every
// product and partial sum is the same rounding as in the one-lane form, so the
// values are identical.  RED as in k_rr_split; UNI, FORM and the form of the
// loads as in k_rb_split.
// Measured per launch, one row per lane with branches around each load / now:
// see Ops::resid_restrict (mg_solver.hip).
// ---------------------------------------------------------------------------
constexpr int kRrTasks = 128;

// position of v_{di dj dk} r_{di dj dk} in the reference's sum
// v111 r111 + v000 r000 + v110 r110 + v001 r001 + v101 r101 + v010 r010 + v011 r011 + v100 r100
__device__ __forceinline__ int rr_slot(int di, int dj, int dk) {
    switch (di * 4 + dj * 2 + dk) {   // codes 7, 0, 6, 1, 5, 2, 3, 4 in sum order
        case 7: return 0;
        case 0: return 1;
        case 6: return 2;
        case 1: return 3;
        case 5: return 4;
        case 2: return 5;
        case 3: return 6;
        default: return 7;
    }
}

template <typename T, bool RED, bool UNI, int FORM>
__global__ void __launch_bounds__(kSplitThreads) k_rr_pair(LevelArgs<T> F, const T *__restrict__ x,
                                                           const T *__restrict__ b, LevelArgs<T> C,
                                                           T *__restrict__ bc, T *__restrict__ xc, RestrictArgs<T> R,
                                                           RowMap M, T w) {
    using VT = Vec16<T>;
    using V = typename VT::V;
    using OFF = std::conditional_t<FORM != RB_PAIR, unsigned long, unsigned>;   // byte offset
    constexpr int W = VT::W;
    __shared__ __align__(16) T prod[8][kRrTasks * W];
    const unsigned per = gridDim.x / kXcds;
    const unsigned logical = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    const unsigned ntask = M.total;
    if (logical * kRrTasks >= ntask) return;
    // coarse row and first coarse cell of a task
    auto place = [&](unsigned tk, int &I, int &J, int &K) __attribute__((always_inline)) {
        const unsigned g = M.q.div(tk), tile = M.tile.div(g), rem = g - tile * M.tile.d, gi = M.wj.div(rem);
        I = (int)gi;
        J = (int)(tile * M.wj.d + rem - gi * M.wj.d);
        K = (int)(tk - g * M.q.d) * W;
    };
    const int nx = F.n[0], ny = F.n[1], nz = F.n[2], half = nz >> 1;
    const int lane = threadIdx.x & 63, di = threadIdx.x >> 7, slot = threadIdx.x & 127;
    const unsigned task = logical * kRrTasks + slot;
    const bool live = task < ntask;
    const unsigned tt = live ? task : ntask - 1;   // a lane without a task repeats the last one, unread
    int I, J, K0;
    place(tt, I, J, K0);
    const int i = 2 * I + di, j = 2 * J;
    const OFF sx = (OFF)F.sx * sizeof(T), sy = (OFF)F.sy * sizeof(T), hz = (OFF)F.hz * sizeof(T);
    const OFF r0 = (OFF)i * sx + (OFF)j * sy, ko = (OFF)K0 * sizeof(T);
    const bool perx = F.bc_lo[0] == BC_PER, pery = F.bc_lo[1] == BC_PER, perz = F.bc_lo[2] == BC_PER;
    const bool ine = i + 1 < nx, inw = i > 0, inn = j + 2 < ny, ins = j > 0;
    const OFF de = ine ? sx : (perx ? (OFF)0 - (OFF)(nx - 1) * sx : (OFF)0);
    const OFF dw = inw ? (OFF)0 - sx : (perx ? (OFF)(nx - 1) * sx : (OFF)0);
    // the rows beyond the pair: row j - 1 of row j, row j + 2 of row j + 1
    const OFF ps = ins ? (OFF)0 - sy : (pery ? (OFF)(ny - 1) * sy : (OFF)0);
    const OFF pn = (inn ? sy : (pery ? (OFF)0 - (OFF)(ny - 1) * sy : (OFF)0)) + sy;
    auto ldv = [](const T *p, OFF o) __attribute__((always_inline)) {
        return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(p) + o);
    };
    auto ld = [](const T *p, OFF o) __attribute__((always_inline)) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + o);
    };
    // ---- loads: [row of the pair][half] ----
    V xv[2][2], bv[2][2], ev[2][2], wv[2][2], sv[2], nv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const OFF o = r0 + ko + (h ? hz : 0);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            xv[r][h] = ldv(x, o + (r ? sy : 0));
            ev[r][h] = ldv(x, o + (r ? sy : 0) + de);
            wv[r][h] = ldv(x, o + (r ? sy : 0) + dw);
            bv[r][h] = ldv(b, o + (r ? sy : 0));
        }
        sv[h] = ldv(x, o + ps);
        nv[h] = ldv(x, o + pn);
    }
    // z neighbours no adjacent lane holds: below the first even cell and above the last odd one
    const bool zlo = K0 == 0, zhi = K0 + W == half;
    T zl[2], zh[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const OFF row = r0 + (r ? sy : 0);
        zl[r] = zh[r] = T(0);
        if (zlo || lane == 0)
            zl[r] = ld(x, zlo ? (perz ? row + hz + (OFF)(half - 1) * sizeof(T) : row + ko) : row + hz + ko - sizeof(T));
        if (zhi || lane == 63)
            zh[r] = ld(x, zhi ? (perz ? row : row + hz + ko + (W - 1) * sizeof(T)) : row + ko + W * sizeof(T));
    }
    T c2z[2][W], c1z[2][W], c2y[2], c1y[2];
    const T c2x = F.c2[0][UNI ? 0 : i], c1x = F.c1[0][UNI ? 0 : i];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        c2y[r] = F.c2[1][UNI ? 0 : j + r];
        c1y[r] = F.c1[1][UNI ? 0 : j + r];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if constexpr (UNI) {
#pragma unroll
            for (int q = 0; q < W; ++q) {
                c2z[h][q] = F.c2[2][0];
                c1z[h][q] = F.c1[2][0];
            }
        } else {
            load_n<T, W>(F.c2zs + h * half + K0, c2z[h]);
            load_n<T, W>(F.c1zs + h * half + K0, c1z[h]);
        }
    }
    const T ax = di ? R.hi[0][I] : R.lo[0][I], ay[2] = {R.lo[1][J], R.hi[1][J]};
    T fz[2][W];
    load_n<T, W>(R.lo[2] + K0, fz[0]);
    load_n<T, W>(R.hi[2] + K0, fz[1]);
    // ---- residuals ----
    auto flip = [](bool wall, int code, T v) __attribute__((always_inline)) { return wall && code == BC_DIR ? -v : v; };
    T xs[2][2][W];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < W; ++q) xs[r][h][q] = VT::get(xv[r][h], q);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        // cross-vector z neighbours: the adjacent lanes', or the loaded ones
        const T prev = __shfl_up(xs[r][1][W - 1], 1, 64), next = __shfl_down(xs[r][0][0], 1, 64);
        T zb = zlo || lane == 0 ? flip(zlo, F.bc_lo[2], zl[r]) : prev;
        T zt = zhi || lane == 63 ? flip(zhi, F.bc_hi[2], zh[r]) : next;
        if (FORM == RB_GENERAL) {
            const T wz = F.bc_lo[2] == BC_DIRV ? F.wall[2][(i + 1) * (ny + 2) + j + r + 1] : T(0);
            if (zlo && F.bc_lo[2] == BC_DIRV) zb = bc_value(BC_DIRV, xs[r][0][0], T(0), wz);
            if (zhi && F.bc_hi[2] == BC_DIRV) zt = bc_value(BC_DIRV, xs[r][1][W - 1], T(0), wz);
        }
        const T axy = ax * ay[r];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            T p[W];
#pragma unroll
            for (int q = 0; q < W; ++q) {
                Stencil<T, 3> s;
                s.c = xs[r][h][q];
                s.xE = flip(!ine, F.bc_hi[0], VT::get(ev[r][h], q));
                s.xW = flip(!inw, F.bc_lo[0], VT::get(wv[r][h], q));
                s.yN = r == 0 ? xs[1][h][q] : flip(!inn, F.bc_hi[1], VT::get(nv[h], q));
                s.yS = r == 1 ? xs[0][h][q] : flip(!ins, F.bc_lo[1], VT::get(sv[h], q));
                s.zB = h ? xs[r][0][q] : (q > 0 ? xs[r][1][q > 0 ? q - 1 : 0] : zb);
                s.zT = h ? (q < W - 1 ? xs[r][0][q < W - 1 ? q + 1 : q] : zt) : xs[r][1][q];
                if (FORM == RB_GENERAL) {
                    const int k = 2 * (K0 + q) + h;
                    if (!ine && F.bc_hi[0] == BC_DIRV) s.xE = bc_value(BC_DIRV, s.c, T(0), F.wall[0][(j + r + 1) * (nz + 2) + k + 1]);
                    if (!inw && F.bc_lo[0] == BC_DIRV) s.xW = bc_value(BC_DIRV, s.c, T(0), F.wall[0][(j + r + 1) * (nz + 2) + k + 1]);
                    if (r == 1 && !inn && F.bc_hi[1] == BC_DIRV) s.yN = bc_value(BC_DIRV, s.c, T(0), F.wall[1][(i + 1) * (nz + 2) + k + 1]);
                    if (r == 0 && !ins && F.bc_lo[1] == BC_DIRV) s.yS = bc_value(BC_DIRV, s.c, T(0), F.wall[1][(i + 1) * (nz + 2) + k + 1]);
                }
                const T d = residual<T, 3>(s, c2x, c1x, c2y[r], c1y[r], c2z[h][q], c1z[h][q], VT::get(bv[r][h], q));
                p[q] = (axy * fz[h][q]) * d;
            }
            *reinterpret_cast<V *>(&prod[rr_slot(di, r, h)][slot * W]) = VT::make(p);
        }
    }
    __syncthreads();
    // ---- sums: coarse cell c of the block's tasks ----
#pragma unroll
    for (int u = 0; u < kRrTasks * W / kSplitThreads; ++u) {
        const int c = threadIdx.x + u * kSplitThreads;
        const unsigned tk = logical * kRrTasks + c / W;
        if (tk >= ntask) continue;
        int CI, CJ, K;
        place(tk, CI, CJ, K);
        K += c % W;
        T sum = prod[0][c] + prod[1][c];
        sum = sum + prod[2][c];
        sum = sum + prod[3][c];
        sum = sum + prod[4][c];
        sum = sum + prod[5][c];
        sum = sum + prod[6][c];
        sum = sum + prod[7][c];
        const T vtot = R.wd[0][CI] * R.wd[1][CJ] * R.wd[2][K];
        const T out = sum / vtot;
        const long cidx = (long)CI * C.sx + (long)CJ * C.sy + kof(C, K);
        bc[cidx] = out;
        T xr = T(0);
        if (RED && ((CI + CJ + K) & 1) == 0) {
            Stencil<T, 3> s;
            s.c = T(0);
            s.xE = bc_value(C.bc_hi[0], T(0), T(0), T(0));
            s.xW = bc_value(C.bc_lo[0], T(0), T(0), T(0));
            s.yN = bc_value(C.bc_hi[1], T(0), T(0), T(0));
            s.yS = bc_value(C.bc_lo[1], T(0), T(0), T(0));
            s.zT = bc_value(C.bc_hi[2], T(0), T(0), T(0));
            s.zB = bc_value(C.bc_lo[2], T(0), T(0), T(0));
            xr = sor_update<T, 3>(s, C.c2[0][CI], C.c1[0][CI], C.c2[1][CJ], C.c1[1][CJ], C.c2[2][K], C.c1[2][K], out, w);
        }
        xc[cidx] = xr;
    }
}

// ---------------------------------------------------------------------------
// prolongation by injection plus the saved iterate on a split level
// (poisson_d3.cc:548-558, poisson.cc:266): both halves of W fine positions
// m0.. of row (i, j) take the correction of coarse cells K = m0.. of coarse
// row (i/2, j/2).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(kSplitThreads) k_prolong_split(int nx, int ny, int nz, long sx, long sy, long hz,
                                                                 T *__restrict__ x, const T *__restrict__ e,
                                                                 long csx, long csy, long chz, int nblocks) {
    using VT = Vec16<T>;
    using V = typename VT::V;
    constexpr int W = VT::W;
    const int per = gridDim.x / kXcds;
    const int logical = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (logical >= nblocks) return;
    const int half = nz >> 1, q = half / W;
    const long total = (long)nx * ny * q;
    const long t = (long)logical * kSplitThreads + threadIdx.x;
    if (t >= total) return;
    const int row = (int)(t / q);
    const int v = (int)(t - (long)row * q);
    const int i = row / ny, j = row - (row / ny) * ny;
    const int m0 = v * W;
    T ev[W];
    coarse_vec(e, (long)(i >> 1) * csx + (long)(j >> 1) * csy, chz, m0, ev);
    const long rb = (long)i * sx + (long)j * sy;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
        V *p = reinterpret_cast<V *>(x + rb + hh * hz + m0);
        const V xv = *p;
        T r[W];
#pragma unroll
        for (int q2 = 0; q2 < W; ++q2) r[q2] = ev[q2] + VT::get(xv, q2);
        *p = VT::make(r);
    }
}

// ---------------------------------------------------------------------------
// FP64 refinement step of the mixed-precision solve on split rows (the same
// expressions as k_refine): x_new = x_old + e, r = b - A x_new with the wall
// rules applied to x_new, r32 = (float) r, per-block norm partials of r and
// b.  A lane owns W = 2 positions m0.. of both halves of one row, i.e. the
// four cells k = 2 m0 .. 2 m0 + 3; FP64 arrays use the FP64 level's split
// rows (hz), the FP32 correction and residual the FP32 level's (ehz).
// ---------------------------------------------------------------------------
// NORM_ONLY: the residual norm partials of computeError alone
// (poisson_d3.cc:563-663): no correction, nothing written but the partials.
// CX / CB: x_old / b are read from the caller's padded array (FullRows: the
// core cell (i, j, k) at off + i si + j sj + k) instead of the level's split
// rows, so the solve needs no separate layout conversion of its inputs; the
// values, and so the results, are the same.  CXO: x_new is written into the
// caller's array (xo) instead of the split rows -- the refinement expected
// to be the last, which then needs no layout conversion of its output either
// (never together with CX: x_old and x_new are then the same array).
struct FullRows {
    const double *x = nullptr, *b = nullptr;
    double *xo = nullptr;
    long si = 0, sj = 0, off = 0;
};

// Four consecutive doubles of a caller's row, whose start need not be
// 16-byte aligned (an odd pad puts the core at an odd element): two 16-byte
// accesses when it is, else 8 + 16 + 8 bytes.  The parity is the same along
// a row, so the lanes of a wave take one branch.
__device__ __forceinline__ void load4(const double *__restrict__ p, double (&v)[4]) {
    if ((reinterpret_cast<unsigned long>(p) & 15) == 0) {
        const double2 a = *reinterpret_cast<const double2 *>(p), c = *reinterpret_cast<const double2 *>(p + 2);
        v[0] = a.x;
        v[1] = a.y;
        v[2] = c.x;
        v[3] = c.y;
    } else {
        const double2 m = *reinterpret_cast<const double2 *>(p + 1);
        v[0] = p[0];
        v[1] = m.x;
        v[2] = m.y;
        v[3] = p[3];
    }
}
__device__ __forceinline__ void store4(double *__restrict__ p, double v0, double v1, double v2, double v3) {
    if ((reinterpret_cast<unsigned long>(p) & 15) == 0) {
        *reinterpret_cast<double2 *>(p) = make_double2(v0, v1);
        *reinterpret_cast<double2 *>(p + 2) = make_double2(v2, v3);
    } else {
        p[0] = v0;
        *reinterpret_cast<double2 *>(p + 1) = make_double2(v1, v2);
        p[3] = v3;
    }
}

// NOXW: r32 and the norm only, x_new not written (the initial residual of a
// solve whose iterate stays in the caller's array until the first refinement).
template <int TYPE, int DIM, bool NORM_ONLY = false, bool CX = false, bool CB = false, bool CXO = false,
          bool NOXW = false>
__global__ void __launch_bounds__(kNormThreads) k_refine_split(LevelArgs<double> L, const double *__restrict__ xold,
                                                               const float *__restrict__ e, long esx, long esy,
                                                               long ehz, const double *__restrict__ b,
                                                               double *__restrict__ xnew, float *__restrict__ r32,
                                                               double *__restrict__ partial, FullRows F) {
    static_assert(!(CX && CXO), "x_old and x_new cannot both be the caller's array");
    constexpr int W = 2;
    const int nx = L.n[0], ny = L.n[1], nz = L.n[2];
    const int half = nz >> 1, q = half / W;
    const long total = (long)nx * ny * q;
    const long hz = L.hz;
    const int lane = threadIdx.x & 63;
    double ar = 0.0, ab = 0.0;
    // rows of the x_old + e iterate: even and odd halves at m0
    auto row_vals = [&](int ii, int jj, int m0, double (&ve)[W], double (&vo)[W]) {
        if (CX) {
            double xr[4];
            load4(F.x + F.off + (long)ii * F.si + (long)jj * F.sj + 2 * m0, xr);
            ve[0] = xr[0];
            vo[0] = xr[1];
            ve[1] = xr[2];
            vo[1] = xr[3];
            if (e) {
                const long eb = (long)ii * esx + (long)jj * esy;
                const float2 fe = *reinterpret_cast<const float2 *>(e + eb + m0);
                const float2 fo = *reinterpret_cast<const float2 *>(e + eb + ehz + m0);
                ve[0] = ve[0] + (double)fe.x;
                ve[1] = ve[1] + (double)fe.y;
                vo[0] = vo[0] + (double)fo.x;
                vo[1] = vo[1] + (double)fo.y;
            }
            return;
        }
        const long rb = (long)ii * L.sx + (long)jj * L.sy;
        const double2 xe = *reinterpret_cast<const double2 *>(xold + rb + m0);
        const double2 xo = *reinterpret_cast<const double2 *>(xold + rb + hz + m0);
        ve[0] = xe.x;
        ve[1] = xe.y;
        vo[0] = xo.x;
        vo[1] = xo.y;
        if (e) {
            const long eb = (long)ii * esx + (long)jj * esy;
            const float2 fe = *reinterpret_cast<const float2 *>(e + eb + m0);
            const float2 fo = *reinterpret_cast<const float2 *>(e + eb + ehz + m0);
            ve[0] = ve[0] + (double)fe.x;
            ve[1] = ve[1] + (double)fe.y;
            vo[0] = vo[0] + (double)fo.x;
            vo[1] = vo[1] + (double)fo.y;
        }
    };
    // Rows are walked in one of two orders.  Where a level's neighbour
    // planes exceed half an XCD's L2 (L.rtile, set for the colour passes too),
    // each XCD walks one contiguous range of j-tiled rows, its blocks striding
    // through it together, so a row's x and y neighbours were fetched into
    // the same L2 a few rows before; otherwise the grid strides over all rows
    // in order (the level's x and b are then served from the Infinity Cache
    // and this order measured faster).  The grid is a multiple of kXcds.
    const bool xwalk = L.rtile != 0;
    const int per = xwalk ? gridDim.x / kXcds : gridDim.x;
    const int xcd = xwalk ? blockIdx.x % kXcds : 0, kb = xwalk ? blockIdx.x / kXcds : blockIdx.x;
    const long rows = (long)nx * ny;
    const long xrows = xwalk ? (rows + kXcds - 1) / kXcds : rows;
    const long lo = (long)xcd * xrows * q, hi = min(total, lo + xrows * q);
    for (long t = lo + (long)kb * blockDim.x + threadIdx.x; t < hi; t += (long)per * blockDim.x) {
        const int row = (int)(t / q);
        const int v = (int)(t - (long)row * q);
        int i, j;
        if (xwalk) {
            const int jt = L.rtile, tile = row / (nx * jt), rem = row - tile * (nx * jt);
            i = rem >> __builtin_ctz(jt);
            j = tile * jt + (rem & (jt - 1));
        } else {
            i = row / ny;
            j = row - i * ny;
        }
        const int m0 = v * W;
        const long rb = (long)i * L.sx + (long)j * L.sy;
        const long eb = (long)i * esx + (long)j * esy;
        // the iterate at cell k of this row
        auto cell = [&](int k) {
            const long h = k & 1, m = k >> 1;
            double x = CX ? F.x[F.off + (long)i * F.si + (long)j * F.sj + k] : xold[rb + h * hz + m];
            if (e) x = x + (double)e[eb + h * ehz + m];
            return x;
        };
        // the z neighbours beyond this lane's vectors that no adjacent lane
        // holds (periodic wrap, or the row's vector in another wave), loaded
        // first so that their latency overlaps the row loads
        const bool need_lo = m0 == 0 ? L.bc_lo[2] == BC_PER : lane == 0;
        const bool need_hi = m0 + W == half ? L.bc_hi[2] == BC_PER : lane == 63;
        double zl = 0.0, zh = 0.0;
        if (need_lo) zl = cell(m0 == 0 ? nz - 1 : 2 * m0 - 1);
        if (need_hi) zh = cell(m0 + W == half ? 0 : 2 * (m0 + W));
        double ce[W], co[W];
        row_vals(i, j, m0, ce, co);
        // x/y neighbours: [0] E, [1] W, [2] N, [3] S
        double ne[4][W], no[4][W];
        auto nbr = [&](int slot, bool inside, int ii, int jj, int bc, int axis) {
            if (inside || bc == BC_PER) {
                row_vals(ii, jj, m0, ne[slot], no[slot]);
            } else {
#pragma unroll
                for (int p = 0; p < W; ++p) {
                    double wve = 0.0, wvo = 0.0;
                    if (bc == BC_DIRV) {
                        const int ke = 2 * (m0 + p), ko = ke + 1;
                        if (axis == 0) {
                            wve = DIM == 3 ? L.wall[0][(j + 1) * (nz + 2) + ke + 1] : L.wall[0][ke + 1];
                            wvo = DIM == 3 ? L.wall[0][(j + 1) * (nz + 2) + ko + 1] : L.wall[0][ko + 1];
                        } else {
                            wve = L.wall[1][(i + 1) * (nz + 2) + ke + 1];
                            wvo = L.wall[1][(i + 1) * (nz + 2) + ko + 1];
                        }
                    }
                    ne[slot][p] = bc_value<double>(bc, ce[p], 0.0, wve);
                    no[slot][p] = bc_value<double>(bc, co[p], 0.0, wvo);
                }
            }
        };
        nbr(0, i + 1 < nx, i + 1 < nx ? i + 1 : 0, j, L.bc_hi[0], 0);
        nbr(1, i > 0, i > 0 ? i - 1 : nx - 1, j, L.bc_lo[0], 0);
        if (DIM == 3) {
            nbr(2, j + 1 < ny, i, j + 1 < ny ? j + 1 : 0, L.bc_hi[1], 1);
            nbr(3, j > 0, i, j > 0 ? j - 1 : ny - 1, L.bc_lo[1], 1);
        }
        // z: even cell 2m: zB = odd[m-1], zT = odd[m]; odd cell 2m+1: zB = even[m], zT = even[m+1]
        const double from_prev = __shfl_up(co[W - 1], 1, 64);
        const double from_next = __shfl_down(ce[0], 1, 64);
        double zlo0, zhi_last;
        if (m0 == 0) {
            if (L.bc_lo[2] == BC_PER) zlo0 = zl;
            else {
                const double wv = L.bc_lo[2] == BC_DIRV ? (DIM == 3 ? L.wall[2][(i + 1) * (ny + 2) + j + 1] : L.wall[2][i + 1])
                                                        : 0.0;
                zlo0 = bc_value<double>(L.bc_lo[2], ce[0], 0.0, wv);
            }
        } else {
            zlo0 = lane > 0 ? from_prev : zl;
        }
        if (m0 + W == half) {
            if (L.bc_hi[2] == BC_PER) zhi_last = zh;
            else {
                const double wv = L.bc_hi[2] == BC_DIRV ? (DIM == 3 ? L.wall[2][(i + 1) * (ny + 2) + j + 1] : L.wall[2][i + 1])
                                                        : 0.0;
                zhi_last = bc_value<double>(L.bc_hi[2], co[W - 1], 0.0, wv);
            }
        } else {
            zhi_last = lane < 63 ? from_next : zh;
        }
        const double c2x = L.c2[0][i], c1x = L.c1[0][i];
        const double c2y = DIM == 3 ? L.c2[1][j] : 0.0, c1y = DIM == 3 ? L.c1[1][j] : 0.0;
        double bev[W], bov[W];
        if (CB) {
            double br[4];
            load4(F.b + F.off + (long)i * F.si + (long)j * F.sj + 2 * m0, br);
            bev[0] = br[0];
            bov[0] = br[1];
            bev[1] = br[2];
            bov[1] = br[3];
        } else {
            const double2 be = *reinterpret_cast<const double2 *>(b + rb + m0);
            const double2 bo = *reinterpret_cast<const double2 *>(b + rb + hz + m0);
            bev[0] = be.x;
            bev[1] = be.y;
            bov[0] = bo.x;
            bov[1] = bo.y;
        }
        double re[W], ro[W];
#pragma unroll
        for (int p = 0; p < W; ++p) {
            Stencil<double, DIM> s;
            s.c = ce[p];
            s.xE = ne[0][p];
            s.xW = ne[1][p];
            if (DIM == 3) {
                s.yN = ne[2][p];
                s.yS = ne[3][p];
            }
            s.zB = p > 0 ? co[p - 1] : zlo0;
            s.zT = co[p];
            re[p] = residual<double, DIM>(s, c2x, c1x, c2y, c1y, L.c2zs[m0 + p], L.c1zs[m0 + p], bev[p]);
            s.c = co[p];
            s.xE = no[0][p];
            s.xW = no[1][p];
            if (DIM == 3) {
                s.yN = no[2][p];
                s.yS = no[3][p];
            }
            s.zB = ce[p];
            s.zT = p < W - 1 ? ce[p + 1] : zhi_last;
            ro[p] = residual<double, DIM>(s, c2x, c1x, c2y, c1y, L.c2zs[half + m0 + p], L.c1zs[half + m0 + p], bov[p]);
        }
        if (!NORM_ONLY) {
            if (NOXW) {
            } else if (CXO) {
                store4(F.xo + F.off + (long)i * F.si + (long)j * F.sj + 2 * m0, ce[0], co[0], ce[1], co[1]);
            } else {
                *reinterpret_cast<double2 *>(xnew + rb + m0) = make_double2(ce[0], ce[1]);
                *reinterpret_cast<double2 *>(xnew + rb + hz + m0) = make_double2(co[0], co[1]);
            }
            *reinterpret_cast<float2 *>(r32 + eb + m0) = make_float2((float)re[0], (float)re[1]);
            *reinterpret_cast<float2 *>(r32 + eb + ehz + m0) = make_float2((float)ro[0], (float)ro[1]);
        }
#pragma unroll
        for (int p = 0; p < W; ++p) {
            ar = norm_acc<TYPE>(ar, re[p]);
            ab = norm_acc<TYPE>(ab, bev[p]);
            ar = norm_acc<TYPE>(ar, ro[p]);
            ab = norm_acc<TYPE>(ab, bov[p]);
        }
    }
    block_reduce2<TYPE>(ar, ab);
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = ar;
        partial[2 * blockIdx.x + 1] = ab;
    }
}

// ---------------------------------------------------------------------------
// k_refine_split for the levels it mostly meets: homogeneous walls and arrays
// below 4 GB.  The same values and the same norms.  Bound by memory: walking
// the rows in order, each plane was read again for its x neighbours from
// beyond L2 (1.3 to 2 times the words a pass cannot do without).  Here a lane
// keeps its place in the (y, z) plane -- W positions of both halves of a row --
// and marches along x through one chunk of planes, with the plane behind and
// its own in registers, so a plane is read once; its y neighbours are read by
// the blocks beside it at about the same time, on the same XCD.  E: with a
// correction; UNI: every axis uniform, so the coefficients are one value per
// axis; loads do not wait behind a lane-dependent branch, byte offsets have 32
// bits.  Measured: see launch_refine_march (mg_solver.hip).
// ---------------------------------------------------------------------------
// two doubles of a caller's row, whose start need not be 16-byte aligned (a
// 16-byte global access needs 4-byte alignment only)
typedef double double2u __attribute__((ext_vector_type(2), aligned(8)));

// The items of a march: block vectors of the (y, z) plane times chunks of
// planes, chunk by chunk.
struct MarchMap {
    FastDiv q, pb;            // vectors of a half-row; items of a chunk
    unsigned plane;           // vectors of a plane
    unsigned items;
    int len;                  // planes of a chunk
};

template <int TYPE, int DIM, bool NORM_ONLY, bool E, bool CX, bool CB, bool CXO, bool NOXW, bool UNI>
__global__ void __launch_bounds__(kNormThreads) k_refine_march(LevelArgs<double> L, MarchMap M,
                                                               const double *__restrict__ xold,
                                                               const float *__restrict__ e, long esx_, long esy_,
                                                               long ehz_, const double *__restrict__ b,
                                                               double *__restrict__ xnew, float *__restrict__ r32,
                                                               double *__restrict__ partial, FullRows F) {
    static_assert(!(CX && CXO), "x_old and x_new cannot both be the caller's array");
    constexpr int W = 2;
    using u32 = unsigned;
    const int nx = L.n[0], ny = DIM == 3 ? L.n[1] : 1, nz = L.n[2], half = nz >> 1;
    const int lane = threadIdx.x & 63;
    const u32 sx = (u32)L.sx * 8u, sy = (u32)L.sy * 8u, hz = (u32)L.hz * 8u;
    const u32 esx = (u32)esx_ * 4u, esy = (u32)esy_ * 4u, ehz = (u32)ehz_ * 4u;
    const u32 fi = (u32)F.si * 8u, fj = (u32)F.sj * 8u, f0 = (u32)F.off * 8u;
    const bool perx = L.bc_lo[0] == BC_PER, pery = DIM == 3 && L.bc_lo[1] == BC_PER, perz = L.bc_lo[2] == BC_PER;
    auto at = [](const void *p, u32 o) __attribute__((always_inline)) { return reinterpret_cast<const char *>(p) + o; };
    const char *X = reinterpret_cast<const char *>(CX ? F.x : xold);
    double ar = 0.0, ab = 0.0;
    // each XCD takes one contiguous range of items
    const u32 per = gridDim.x / kXcds;
    for (u32 it = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds; it < M.items; it += gridDim.x) {
        const u32 chunk = M.pb.div(it), s0 = (it - chunk * M.pb.d) * kNormThreads + threadIdx.x;
        const bool live = s0 < M.plane;
        const u32 sv = live ? s0 : M.plane - 1;   // a lane beyond the plane repeats its last vector, unwritten
        const int j = (int)M.q.div(sv), m0 = (int)(sv - (u32)j * M.q.d) * W;
        const int i0 = (int)chunk * M.len, i1 = min(nx, i0 + M.len);
        const u32 mo = (u32)m0 * 8u, me = (u32)m0 * 4u;
        const u32 row = (u32)j * sy, erow = (u32)j * esy, frow = f0 + (u32)j * fj;
        const bool inn = j + 1 < ny, ins = j > 0;
        const u32 jn = (u32)(inn ? 1 : (pery ? 1 - ny : 0)), js = (u32)(ins ? -1 : (pery ? ny - 1 : 0));
        struct Raw {
            double2 a, b;   // split rows: even, odd; caller rows: cells 2 m0.., 2 m0 + 2..
            float2 ea, eb;
        };
        // the lane's four cells of row (i, j + dj)
        auto load = [&](int i, u32 dj) __attribute__((always_inline)) {
            Raw r;
            if (CX) {
                const u32 o = frow + (u32)i * fi + dj * fj + 2u * mo;
                const double2u p = *reinterpret_cast<const double2u *>(X + o), t = *reinterpret_cast<const double2u *>(X + o + 16u);
                r.a = make_double2(p.x, t.x);
                r.b = make_double2(p.y, t.y);
            } else {
                const u32 o = row + (u32)i * sx + dj * sy + mo;
                r.a = *reinterpret_cast<const double2 *>(X + o);
                r.b = *reinterpret_cast<const double2 *>(X + o + hz);
            }
            if (E) {
                const u32 o = erow + (u32)i * esx + dj * esy + me;
                r.ea = *reinterpret_cast<const float2 *>(at(e, o));
                r.eb = *reinterpret_cast<const float2 *>(at(e, o + ehz));
            }
            return r;
        };
        struct Cells {
            double v[2][W];   // [half][position]
        };
        auto value = [&](const Raw &r) __attribute__((always_inline)) {
            Cells c{{{r.a.x, r.a.y}, {r.b.x, r.b.y}}};
            if (E) {
                c.v[0][0] = c.v[0][0] + (double)r.ea.x;
                c.v[0][1] = c.v[0][1] + (double)r.ea.y;
                c.v[1][0] = c.v[1][0] + (double)r.eb.x;
                c.v[1][1] = c.v[1][1] + (double)r.eb.y;
            }
            return c;
        };
        auto flip = [](bool wall, int code, Cells c) __attribute__((always_inline)) {
            if (code == BC_DIR && wall) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int p = 0; p < W; ++p) c.v[h][p] = -c.v[h][p];
            }
            return c;
        };
        const double c2y = DIM == 3 ? L.c2[1][UNI ? 0 : j] : 0.0, c1y = DIM == 3 ? L.c1[1][UNI ? 0 : j] : 0.0;
        double c2z[2][W], c1z[2][W];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (UNI) {
#pragma unroll
                for (int p = 0; p < W; ++p) {
                    c2z[h][p] = L.c2[2][0];
                    c1z[h][p] = L.c1[2][0];
                }
            } else {
                load_n<double, W>(L.c2zs + h * half + m0, c2z[h]);
                load_n<double, W>(L.c1zs + h * half + m0, c1z[h]);
            }
        }
        // z neighbours no adjacent lane holds: below the first even cell, above the last odd one
        const bool zlo = m0 == 0, zhi = m0 + W == half;
        const bool zll = zlo || lane == 0, zhl = zhi || lane == 63;
        const int kl = zlo ? (perz ? nz - 1 : 0) : 2 * m0 - 1, kh = zhi ? (perz ? 0 : nz - 1) : 2 * (m0 + W);
        auto cell = [&](int i, int k) __attribute__((always_inline)) {
            double v = CX ? *reinterpret_cast<const double *>(X + frow + (u32)i * fi + (u32)k * 8u)
                          : *reinterpret_cast<const double *>(X + row + (u32)i * sx + (k & 1 ? hz : 0u) + (u32)(k >> 1) * 8u);
            if (E)
                v = v + (double)*reinterpret_cast<const float *>(
                            at(e, erow + (u32)i * esx + (k & 1 ? ehz : 0u) + (u32)(k >> 1) * 4u));
            return v;
        };
        // the plane behind, and the first one
        Cells west, cur;
        {
            const Raw w = load(i0 > 0 ? i0 - 1 : (perx ? nx - 1 : 0), 0u), c = load(i0, 0u);
            cur = value(c);
            west = flip(i0 == 0 && !perx, L.bc_lo[0], value(w));
        }
        for (int i = i0; i < i1; ++i) {
            const bool ine = i + 1 < nx;
            const Raw re = load(ine ? i + 1 : (perx ? 0 : i), 0u);
            Raw rn{}, rs{};
            if (DIM == 3) {
                rn = load(i, jn);
                rs = load(i, js);
            }
            double2 ba, bb;
            if (CB) {
                const char *p = at(F.b, frow + (u32)i * fi + 2u * mo);
                const double2u u = *reinterpret_cast<const double2u *>(p), t = *reinterpret_cast<const double2u *>(p + 16);
                ba = make_double2(u.x, t.x);
                bb = make_double2(u.y, t.y);
            } else {
                ba = *reinterpret_cast<const double2 *>(at(b, row + (u32)i * sx + mo));
                bb = *reinterpret_cast<const double2 *>(at(b, row + (u32)i * sx + mo + hz));
            }
            double zl = 0.0, zh = 0.0;
            if (zll) zl = cell(i, kl);
            if (zhl) zh = cell(i, kh);
            const double c2x = L.c2[0][UNI ? 0 : i], c1x = L.c1[0][UNI ? 0 : i];
            const Cells next = value(re);
            const Cells east = flip(!ine && !perx, L.bc_hi[0], next);
            Cells north{}, south{};
            if (DIM == 3) {
                north = flip(!inn, L.bc_hi[1], value(rn));
                south = flip(!ins, L.bc_lo[1], value(rs));
            }
            const double prev = __shfl_up(cur.v[1][W - 1], 1, 64), foll = __shfl_down(cur.v[0][0], 1, 64);
            const double zb = zll ? (zlo && L.bc_lo[2] == BC_DIR ? -zl : zl) : prev;
            const double zt = zhl ? (zhi && L.bc_hi[2] == BC_DIR ? -zh : zh) : foll;
            const double bv[2][W] = {{ba.x, ba.y}, {bb.x, bb.y}};
            double r[2][W];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < W; ++p) {
                    Stencil<double, DIM> s;
                    s.c = cur.v[h][p];
                    s.xE = east.v[h][p];
                    s.xW = west.v[h][p];
                    if (DIM == 3) {
                        s.yN = north.v[h][p];
                        s.yS = south.v[h][p];
                    }
                    s.zB = h ? cur.v[0][p] : (p > 0 ? cur.v[1][p > 0 ? p - 1 : 0] : zb);
                    s.zT = h ? (p < W - 1 ? cur.v[0][p < W - 1 ? p + 1 : p] : zt) : cur.v[1][p];
                    r[h][p] = residual<double, DIM>(s, c2x, c1x, c2y, c1y, c2z[h][p], c1z[h][p], bv[h][p]);
                }
            if (live) {
                if (!NORM_ONLY) {
                    if (NOXW) {
                    } else if (CXO) {
                        char *p = reinterpret_cast<char *>(F.xo) + frow + (u32)i * fi + 2u * mo;
                        *reinterpret_cast<double2u *>(p) = double2u{cur.v[0][0], cur.v[1][0]};
                        *reinterpret_cast<double2u *>(p + 16) = double2u{cur.v[0][1], cur.v[1][1]};
                    } else {
                        char *p = reinterpret_cast<char *>(xnew) + row + (u32)i * sx + mo;
                        *reinterpret_cast<double2 *>(p) = make_double2(cur.v[0][0], cur.v[0][1]);
                        *reinterpret_cast<double2 *>(p + hz) = make_double2(cur.v[1][0], cur.v[1][1]);
                    }
                    char *p = reinterpret_cast<char *>(r32) + erow + (u32)i * esx + me;
                    *reinterpret_cast<float2 *>(p) = make_float2((float)r[0][0], (float)r[0][1]);
                    *reinterpret_cast<float2 *>(p + ehz) = make_float2((float)r[1][0], (float)r[1][1]);
                }
#pragma unroll
                for (int p = 0; p < W; ++p) {
                    ar = norm_acc<TYPE>(ar, r[0][p]);
                    ab = norm_acc<TYPE>(ab, bv[0][p]);
                    ar = norm_acc<TYPE>(ar, r[1][p]);
                    ab = norm_acc<TYPE>(ab, bv[1][p]);
                }
            }
            west = cur;
            cur = next;
        }
    }
    block_reduce2<TYPE>(ar, ab);
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = ar;
        partial[2 * blockIdx.x + 1] = ab;
    }
}

}  // namespace saras
