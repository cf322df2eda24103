// mg_tile.hpp -- several colour passes of a small level in one launch.
//
// On a level between the tail's few thousand cells and about 64^3 a colour
// pass is all launch: every kernel takes about 4 us there however little it
// does, and a V(2,2) cycle visits such a level with nine of them.  Here a
// workgroup keeps a tile of rows (all of z) and a halo of H rows around it in
// LDS and runs all passes of a visit on it, each pass on one ring of rows less
// than the one before: the cells of the halo are computed by every tile that
// needs them, with the same expressions from the same inputs, so every value is
// the one the separate passes give.  The result goes to the level's other
// iterate buffer, since neighbouring tiles still read the old one.
//
//   zero   the iterate is zero (a coarse level after the restriction, or a
//          correction just started): x is not read;
//   pro    the coarse level's correction is added first (poisson_d3.cc:548-558,
//          poisson.cc:266);
//   restr  the residual of the result is restricted into the coarse level's
//          right-hand side, whose iterate becomes zero (poisson_d3.cc:71-93,
//          484-511; poisson_d2.cc:288-297).
//
// What bounds it is the vector issue of the halo's extra cells, so a row's
// cells are handled as 16-byte vectors of one colour, as in the split passes.
// Four passes with the restriction or the prolongation take 9-11 us at
// 32^3-64^3 FP32 (36-38 us for the visit's nine launches before, two launches
// now); V(2,2) cycles: 64^3 FP32 102 -> 73 us, FP64 104 -> 88, 128 x 128 FP64
// 75 -> 54, 1024 x 1024 FP32 160 -> 100, 256^3 FP32 345 -> 327; V(3,6) at 256^3 FP32
// 667 -> 620 us.
#pragma once
#include <type_traits>

#include "mg_plan.hpp"
#include "mg_split.hpp"

namespace saras {

template <typename T>
struct TileArgs {
    LevelArgs<T> L;          // the level
    const T *x;              // iterate in (not read with `zero`)
    T *y;                    // iterate out
    const T *b;
    int ti, tj;              // rows of a tile along x and y (tj = 1 in 2-D)
    int nti, ntj;            // tiles along x and y
    int halo;                // rows around a tile (x; also y in 3-D): tile_halo
    int sweeps, zero, pro, restr;
    T w;
    const T *e;              // pro: the coarse iterate and its layout
    long esx, esy, ehz;
    LevelArgs<T> C;          // restr: the coarse level
    T *cb, *cx;
    RestrictArgs<T> R;
};

// What the iterate is at the first pass.
enum TileMode { TILE_PLAIN, TILE_ZERO, TILE_PRO };

// HZ: the level's rows are colour-split (see mg_kernels.hpp).  Loads never
// wait behind a lane-dependent branch: a neighbour beyond a wall is read at
// the cell's own address (which is the Neumann rule) and its sign flipped for
// a Dirichlet one, and a row's parity selects between loaded values.
template <typename T, int DIM, bool HZ, int MODE>
__global__ void __launch_bounds__(kTileThreads) k_tile(TileArgs<T> A) {
    using VT = Vec16<T>;
    using V = typename VT::V;
    constexpr int W = VT::W;
    extern __shared__ __align__(16) unsigned char tile_raw[];
    const LevelArgs<T> &L = A.L;
    const int nx = L.n[0], ny = DIM == 3 ? L.n[1] : 1, nz = L.n[2];
    const int half = nz >> 1, nv = (half + W - 1) / W, hp = nv * W;
    const int H = A.halo, HJ = DIM == 3 ? H : 0;
    const int RI = A.ti + 2 * H, RJ = DIM == 3 ? A.tj + 2 * H : 1;
    const int rs = 2 * hp;   // LDS elements of a row: its even cells, then its odd cells
    T *X = reinterpret_cast<T *>(tile_raw);
    T *B = X + RI * RJ * rs;
    T *cz2 = B + RI * RJ * rs, *cz1 = cz2 + rs;   // z coefficients by colour half
    T *cx = cz1 + rs, *cy = cx + 2 * RI;          // (c2, c1) of the tile's rows
    // tiles of one XCD are neighbours: they share halo rows in its L2
    const int ntile = A.nti * A.ntj, per = gridDim.x / kXcds;
    const int tile = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (tile >= ntile) return;
    const int i0 = (tile / A.ntj) * A.ti, j0 = (tile % A.ntj) * A.tj;
    const bool perx = L.bc_lo[0] == BC_PER, pery = DIM == 3 && L.bc_lo[1] == BC_PER, perz = L.bc_lo[2] == BC_PER;
    const int tid = threadIdx.x;
    const int v = tid % nv, slot = tid / nv, nslot = kTileThreads / nv;
    const int m0 = v * W;
    const bool on = slot < nslot;
    const bool ragged = !HZ && half % W != 0;   // the last vector of a row is not full

    // the rows there are to work on (see TileAxis), by their unwrapped numbers
    const TileAxis AX = TileAxis::of(nx, H, perx), AY = TileAxis::of(ny, HJ, pery);
    auto inside = [&](int i, int j) __attribute__((always_inline)) { return AX.has(i) && (DIM == 2 || AY.has(j)); };
    // rows of radius r around the tile, dealt to the thread's slot
    auto rows = [&](int r, auto &&f) __attribute__((always_inline)) {
        const int wi = A.ti + 2 * r, wj = DIM == 3 ? A.tj + 2 * r : 1;
        const unsigned magic = 65536u / (unsigned)wj + 1;   // exact below 65536 / wj rows
        if (!on) return;
        for (int q = slot; q < wi * wj; q += nslot) {
            const int di = (int)(((unsigned)q * magic) >> 16);
            const int ti = di + H - r, tj = q - di * wj + HJ - (DIM == 3 ? r : 0);
            const int i = i0 - H + ti, j = j0 - HJ + tj;
            if (inside(i, j)) f(ti, tj, i, j);
        }
    };
    auto vec = [&](T *p) __attribute__((always_inline)) { return reinterpret_cast<V *>(p); };
    // W pairs (even, odd cell) m0.. of a row in the level's own layout
    auto load_pairs = [&](const T *p, T(&ev)[W], T(&od)[W]) __attribute__((always_inline)) {
        if constexpr (HZ) {
            load_n<T, W>(p + m0, ev);
            load_n<T, W>(p + L.hz + m0, od);
        } else {
#pragma unroll
            for (int q = 0; q < W; ++q) {
                const int m = min(m0 + q, half - 1);
                ev[q] = p[2 * m];
                od[q] = p[2 * m + 1];
            }
        }
    };

    // ---- load the tile and its halo ----
    // All loads are issued before the first is waited for: kBatch rows of a
    // thread at a time, then the coefficients.
    constexpr int kBatch = MODE == TILE_ZERO ? 4 : 2;
    {
        const int nrow = RI * RJ;
        const unsigned magic = 65536u / (unsigned)RJ + 1;
        // at least one turn for every thread: the first also loads the coefficients
        for (int q0 = slot, turn = 0; turn == 0 || q0 < nrow; q0 += kBatch * nslot, ++turn) {
            T be[kBatch][W], bo[kBatch][W], xe[kBatch][W], xo[kBatch][W], ev[kBatch][W];
            int at[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const int q = q0 + u * nslot;
                const int ti = (int)(((unsigned)q * magic) >> 16), tj = q - ti * RJ;
                const int i = i0 - H + ti, j = j0 - HJ + tj;
                const bool in = on && q < nrow && inside(i, j);
                at[u] = in ? q * rs : -1;
                // a row that does not exist: the tile's first one, not stored
                const int gi = in ? AX.row(i) : i0, gj = in && DIM == 3 ? AY.row(j) : j0;
                const long g = (long)gi * L.sx + (long)gj * L.sy;
                load_pairs(A.b + g, be[u], bo[u]);
                if constexpr (MODE != TILE_ZERO) load_pairs(A.x + g, xe[u], xo[u]);
                if constexpr (MODE == TILE_PRO) {
                    // both cells m of a row lie under coarse cell K = m
                    const T *ep = A.e + (long)(gi >> 1) * A.esx + (long)(gj >> 1) * A.esy;
                    if constexpr (HZ) {
                        coarse_vec(ep, 0, A.ehz, m0, ev[u]);
                    } else {
#pragma unroll
                        for (int c = 0; c < W; ++c) ev[u][c] = coarse_at(ep, 0, A.ehz, min(m0 + c, half - 1));
                    }
                }
            }
            if (turn == 0) {
                for (int k = tid; k < nz; k += kTileThreads) {
                    cz2[(k & 1) * hp + (k >> 1)] = L.c2[2][k];
                    cz1[(k & 1) * hp + (k >> 1)] = L.c1[2][k];
                }
                for (int t = tid; t < RI + (DIM == 3 ? RJ : 0); t += kTileThreads) {
                    const int ax = t < RI ? 0 : 1, n = ax ? ny : nx;
                    const int q = ax ? j0 - HJ + t - RI : i0 - H + t;
                    const int g = min(max(ax ? AY.row(q) : AX.row(q), 0), n - 1);
                    cx[2 * t] = ax ? L.c2[1][g] : L.c2[0][g];
                    cx[2 * t + 1] = ax ? L.c1[1][g] : L.c1[0][g];
                }
            }
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                if (at[u] < 0) continue;
#pragma unroll
                for (int c = 0; c < W; ++c) {
                    if (MODE == TILE_ZERO) xe[u][c] = xo[u][c] = T(0);
                    if (MODE == TILE_PRO) {
                        xe[u][c] = ev[u][c] + xe[u][c];
                        xo[u][c] = ev[u][c] + xo[u][c];
                    }
                }
                *vec(B + at[u] + m0) = VT::make(be[u]);
                *vec(B + at[u] + hp + m0) = VT::make(bo[u]);
                *vec(X + at[u] + m0) = VT::make(xe[u]);
                *vec(X + at[u] + hp + m0) = VT::make(xo[u]);
            }
        }
    }
    // the coarse cells' restriction factors, needed last: kept in registers
    // (one coarse cell per thread; further ones load theirs)
    const int cti = A.ti / 2, ctj = DIM == 3 ? A.tj / 2 : 1;
    struct Factors {
        T lx, hx, ly, hy, lz, hz, wx, wy, wz;
    };
    auto factors = [&](int q) __attribute__((always_inline)) {
        Factors f{};
        const int row = q / half, K = q - row * half, ci = row / ctj, cj = row - ci * ctj;
        const int I = i0 / 2 + ci, J = j0 / 2 + cj;
        if (DIM == 3 && A.restr && q < cti * ctj * half && I < A.C.n[0] && J < A.C.n[1])
            f = Factors{A.R.lo[0][I], A.R.hi[0][I], A.R.lo[1][J], A.R.hi[1][J], A.R.lo[2][K],
                        A.R.hi[2][K], A.R.wd[0][I], A.R.wd[1][J], A.R.wd[2][K]};
        return f;
    };
    const Factors f0 = factors(tid);
    __syncthreads();

    const bool dir[6] = {L.bc_hi[0] == BC_DIR, L.bc_lo[0] == BC_DIR, L.bc_hi[1] == BC_DIR,
                         L.bc_lo[1] == BC_DIR, L.bc_hi[2] == BC_DIR, L.bc_lo[2] == BC_DIR};
    // The stencils of W cells m0.. of half h of tile row (ti, tj).  ZERO: of a
    // zero iterate (no row beyond the halo's last ring is read).
    auto stencils = [&](int ti, int tj, int i, int j, int h, Stencil<T, DIM>(&s)[W], auto zeroc)
        __attribute__((always_inline)) {
        constexpr bool ZERO = decltype(zeroc)::value;
        const int r = (ti * RJ + tj) * rs, own = r + h * hp + m0, oth = r + (1 - h) * hp + m0;
        const bool in[4] = {perx || i + 1 < nx, perx || i > 0, pery || j + 1 < ny, pery || j > 0};
        const int off[4] = {RJ * rs, -RJ * rs, rs, -rs};
        // the z neighbour beyond the vector, below an even cell or above an odd one
        const bool end = h ? m0 + W >= half : m0 == 0;
        const int zw = h ? r : r + hp + half - 1, ze = h ? own + W - 1 : own;   // wrapped; the cell itself
        const int za = end ? (perz ? zw : ze) : (h ? oth + W : oth - 1);
        V cv{}, ov{}, nv_[4] = {V{}, V{}, V{}, V{}};
        T z = T(0);
        if (!ZERO) {
            cv = *vec(X + own);
            ov = *vec(X + oth);
#pragma unroll
            for (int d = 0; d < (DIM == 3 ? 4 : 2); ++d) nv_[d] = *vec(X + own + (in[d] ? off[d] : 0));
            z = X[za];
        }
        if (end && !perz && (h ? dir[4] : dir[5])) z = -z;
        T c[W], o[W], n[4][W];
#pragma unroll
        for (int q = 0; q < W; ++q) {
            c[q] = VT::get(cv, q);
            o[q] = VT::get(ov, q);
#pragma unroll
            for (int d = 0; d < (DIM == 3 ? 4 : 2); ++d) {
                n[d][q] = VT::get(nv_[d], q);
                if (dir[d] && !in[d]) n[d][q] = -n[d][q];
            }
            s[q].c = c[q];
            s[q].xE = n[0][q];
            s[q].xW = n[1][q];
            if (DIM == 3) {
                s[q].yN = n[2][q];
                s[q].yS = n[3][q];
            }
        }
        // even cell m: other[m - 1], other[m]; odd cell: other[m], other[m + 1]
#pragma unroll
        for (int q = 0; q < W; ++q) {
            s[q].zB = h ? o[q] : (q > 0 ? o[q - 1] : z);
            s[q].zT = h ? (q < W - 1 ? o[q + 1] : z) : o[q];
        }
        if (ragged && h && m0 + W >= half) {
            // the row's last odd cell lies inside the vector
            const T first = ZERO ? T(0) : X[r];
#pragma unroll
            for (int q = 0; q < W; ++q)
                if (m0 + q == half - 1) s[q].zT = perz ? first : (dir[4] ? -c[q] : c[q]);
        }
    };
    // one colour pass on the rows of radius r
    auto pass = [&](int r, int colour, auto zeroc) __attribute__((always_inline)) {
        rows(r, [&](int ti, int tj, int i, int j) __attribute__((always_inline)) {
            const int h = (i + j + colour) & 1;
            Stencil<T, DIM> s[W];
            stencils(ti, tj, i, j, h, s, zeroc);
            const int own = (ti * RJ + tj) * rs + h * hp + m0;
            const V bv = *vec(B + own), c2v = *vec(cz2 + h * hp + m0), c1v = *vec(cz1 + h * hp + m0);
            const T c2x = cx[2 * ti], c1x = cx[2 * ti + 1];
            const T c2y = DIM == 3 ? cy[2 * tj] : T(0), c1y = DIM == 3 ? cy[2 * tj + 1] : T(0);
            T x[W];
#pragma unroll
            for (int q = 0; q < W; ++q)
                x[q] = sor_update<T, DIM>(s[q], c2x, c1x, c2y, c1y, VT::get(c2v, q), VT::get(c1v, q), VT::get(bv, q), A.w);
            *vec(X + own) = VT::make(x);
        });
        __syncthreads();
    };

    // ---- the sweeps: pass p on the rows that later passes still need ----
    const int npass = 2 * A.sweeps, last = npass - 1 + (A.restr ? 1 : 0);
    if constexpr (MODE == TILE_ZERO) pass(last, 0, std::true_type{});
    for (int p = MODE == TILE_ZERO ? 1 : 0; p < npass; ++p) pass(last - p, p & 1, std::false_type{});

    // ---- the tile's rows out, and their residuals in place of b ----
    rows(0, [&](int ti, int tj, int i, int j) __attribute__((always_inline)) {
        if (i >= nx || j >= ny) return;   // beyond the level in its last tile
        const long g = (long)i * L.sx + (long)j * L.sy;
        const int r = (ti * RJ + tj) * rs;
        if constexpr (HZ) {
            *vec(A.y + g + m0) = *vec(X + r + m0);
            *vec(A.y + g + L.hz + m0) = *vec(X + r + hp + m0);
        } else {
#pragma unroll
            for (int q = 0; q < W; ++q)
                if (m0 + q < half) {
                    A.y[g + 2 * (m0 + q)] = X[r + m0 + q];
                    A.y[g + 2 * (m0 + q) + 1] = X[r + hp + m0 + q];
                }
        }
        if (!A.restr) return;
        const T c2x = cx[2 * ti], c1x = cx[2 * ti + 1];
        const T c2y = DIM == 3 ? cy[2 * tj] : T(0), c1y = DIM == 3 ? cy[2 * tj + 1] : T(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            Stencil<T, DIM> s[W];
            stencils(ti, tj, i, j, h, s, std::false_type{});
            const int own = r + h * hp + m0;
            const V bv = *vec(B + own), c2v = *vec(cz2 + h * hp + m0), c1v = *vec(cz1 + h * hp + m0);
            T d[W];
#pragma unroll
            for (int q = 0; q < W; ++q)
                d[q] = residual<T, DIM>(s[q], c2x, c1x, c2y, c1y, VT::get(c2v, q), VT::get(c1v, q), VT::get(bv, q));
            *vec(B + own) = VT::make(d);
        }
    });
    if (!A.restr) return;
    __syncthreads();
    // ---- restriction: one coarse cell per thread and turn ----
    const LevelArgs<T> &C = A.C;
    for (int q = tid; q < cti * ctj * half; q += kTileThreads) {
        const int row = q / half, K = q - row * half;
        const int ci = row / ctj, cj = row - ci * ctj;
        const int I = i0 / 2 + ci, J = j0 / 2 + cj;
        if (I >= C.n[0] || (DIM == 3 && J >= C.n[1])) continue;
        auto r = [&](int di, int dj, int dk) __attribute__((always_inline)) {
            return B[((2 * ci + di + H) * RJ + (DIM == 3 ? 2 * cj + dj + HJ : 0)) * rs + dk * hp + K];
        };
        T out;
        if (DIM == 3) {
            const Factors f = q == tid ? f0 : factors(q);
            const T lx = f.lx, hx = f.hx, ly = f.ly, hy = f.hy, lz = f.lz, hz = f.hz;
            const T v000 = lx * ly * lz, v100 = hx * ly * lz, v010 = lx * hy * lz, v001 = lx * ly * hz;
            const T v011 = lx * hy * hz, v101 = hx * ly * hz, v110 = hx * hy * lz, v111 = hx * hy * hz;
            const T vtot = f.wx * f.wy * f.wz;
            out = (v111 * r(1, 1, 1) + v000 * r(0, 0, 0) + v110 * r(1, 1, 0) + v001 * r(0, 0, 1) + v101 * r(1, 0, 1) +
                   v010 * r(0, 1, 0) + v011 * r(0, 1, 1) + v100 * r(1, 0, 0)) / vtot;
        } else {
            out = (r(1, 0, 1) + r(0, 0, 0) + r(1, 0, 0) + r(0, 0, 1)) / T(4);
        }
        const long c = (long)I * C.sx + (long)J * C.sy + kof(C, K);
        A.cb[c] = out;
        A.cx[c] = T(0);
    }
}

}  // namespace saras
