// mg_plan.hpp -- how a level's work is cut: the tiles of k_tile (mg_tile.hpp), the
// rows of a level each of them touches and the plan of a V-cycle's visit; the
// form of a colour pass (k_rb_split, mg_split.hpp) and its vectors; the LDS of
// the tail (k_tail, mg_tail.hpp).
// Plain arithmetic shared by the host code, the kernel and the CPU tests.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace saras {

constexpr int kTileThreads = 512;
// LDS of a tile (k_tile has no static LDS), of the 160 KB a workgroup may hold
constexpr size_t kTileLds = 156 * 1024;

// 16-byte vectors of one colour in a row of nz cells of `word` bytes
constexpr int tile_vecs(size_t word, int nz) { return (nz / 2 + 16 / (int)word - 1) / (16 / (int)word); }

// Rows around a tile that `sweeps` sweeps need: pass p runs on the rows of
// radius 2 sweeps - 1 - p (one more before a residual) and reads one row
// further, except that the first pass of a zero iterate reads none.
constexpr int tile_halo(int sweeps, bool zero, bool restr) { return 2 * sweeps + (restr ? 1 : 0) - (zero ? 1 : 0); }

// LDS bytes of a tile: iterate, right-hand side and the coefficients of its rows
constexpr size_t tile_bytes(size_t word, int dim, int nz, int ti, int tj, int halo) {
    const size_t ri = ti + 2 * halo, rj = dim == 3 ? tj + 2 * halo : 1;
    const size_t row = 2 * (size_t)tile_vecs(word, nz) * 16;
    return 2 * ri * rj * row + 2 * row + 2 * (ri + rj) * word;
}

// The rows along one axis (x, or y in 3-D) that tiles work on, numbered without
// wrapping: the level's n and, on a periodic axis, the `halo` images before and
// after them.  The last tile of an axis covers rows beyond those where its
// extent does not divide n; no row of the level needs them, and with
// halo <= n every row named here is an image at most one extent away.
struct TileAxis {
    int n, lo, hi;
    static constexpr TileAxis of(int n, int halo, bool periodic) {
        return TileAxis{n, periodic ? -halo : 0, periodic ? n + halo : n};
    }
    constexpr bool has(int q) const { return q >= lo && q < hi; }
    constexpr int row(int q) const { return q < 0 ? q + n : (q >= n ? q - n : q); }   // of a row it has
};

// The visits of a level by tiles: rows of a tile and sweeps of a launch; none
// (sweeps 0) where separate passes are faster.
struct TilePlan {
    int ti = 0, tj = 0, sweeps = 0;
};

// The plan of one visit of a level of n cells of `word` bytes, or none where
// separate passes are faster by this estimate (us).  A kernel takes about 4 us
// however little it does; a pass beyond that is bound by its 1.5 words per cell
// at about 7 TB/s (levels of this size sit in the Infinity Cache).  A tile launch
// adds, per workgroup of a compute unit, its rows' vectors: about kVec cycles of
// vector issue for 64 of them, and about 350 cycles a pass for the barrier and
// the LDS latency.  Measured over tiles of 2 to 16 by 1 to 8 rows, 1 to 6 sweeps
// a launch, 32^3..128^3 and 128^2..2048^2 in both precisions: the estimate's
// choice is within 3 % of the fastest V-cycle, and turns to separate passes where
// those are (64^3 with six sweeps FP64, 128^3, 2048^2).
// split: the level's rows are colour-split.
inline TilePlan plan_tile(size_t word, int dim, const int (&n)[3], bool split, int count, bool zero, bool pro,
                          bool restr) {
    TilePlan best;
    const int nv = tile_vecs(word, n[2]);
    if (count < 1 || (n[2] & 1) || nv > kTileThreads) return best;
    constexpr double kLaunch = 4.0, kVec = 125.0, kClock = 2400.0, kCus = 256.0;
    const double cells = (double)n[0] * n[1] * n[2];
    const double pass = std::max(kLaunch + 0.2, 2.8 + 1.5 * cells * word / 7e6);
    double cost = 2 * count * pass + (restr ? 1.4 * pass : 0.0) + (pro ? 0.4 * pass : 0.0);
    if (!split && pro) cost += pass;   // a prolongation pass of its own
    cost *= 0.95;
    const int jmax = dim == 3 ? 8 : 1;
    for (int ti = 2; ti <= 32; ti *= 2)
        for (int tj = dim == 3 ? 2 : 1; tj <= jmax; tj *= 2)
            for (int s = 1; s <= count; ++s) {
                double c = 0.0;
                bool ok = true;
                for (int done = 0; done < count && ok; done += s) {
                    const bool z = zero && done == 0, r = restr && done + s >= count;
                    const int sw = std::min(s, count - done), halo = tile_halo(sw, z, r);
                    ok = tile_bytes(word, dim, n[2], ti, tj, halo) <= kTileLds && halo <= n[0] &&
                         (dim == 2 || halo <= n[1]);
                    auto rows = [&](int q) { return (double)(ti + 2 * q) * (dim == 3 ? tj + 2 * q : 1); };
                    double vecs = (z ? 1.0 : 1.5) * rows(halo) + (r ? 3.0 * rows(0) : 0.0);
                    for (int p = 0; p < 2 * sw; ++p) vecs += rows(2 * sw - 1 - p + (r ? 1 : 0));
                    const double tiles = std::ceil((double)n[0] / ti) * (dim == 3 ? std::ceil((double)n[1] / tj) : 1.0);
                    const double per_cu = std::max(1.0, tiles / kCus);
                    c += kLaunch + 1.0 + (std::ceil(per_cu) * vecs * nv / 64.0 * kVec + 350.0 * 2 * sw) / kClock;
                }
                if (ok && c < cost) {
                    cost = c;
                    best.ti = ti;
                    best.tj = tj;
                    best.sweeps = s;
                }
            }
    return best;
}

constexpr int kTailMaxLevels = 8;
constexpr int kTailThreads = 512;
// cells of one colour that a thread of the tail keeps in registers
constexpr int kTailColourCells = 4;
// LDS that the tail takes by default, of the 160 KB a workgroup may hold (its
// static LDS is under 1 KB).  Taking 156 KB lets in 2-D levels of 4096 cells in
// long boxes, which are faster by tiles (1024 x 64 FP64, four V(2,2) cycles: 1.01
// against 1.09 ms).
constexpr size_t kTailLds = 150 * 1024;

// The LDS of the tail (k_tail) for levels S..D, offsets in elements (the
// tables' in 32-bit words).
struct TailPlan {
    size_t bytes = 0;          // 0: the tail does not take these levels
    bool b_global = false;     // the right-hand side of the single level stays in global memory
    struct Level {
        int n[3];
        int hz, half;          // cells of one colour per row (rounded up) and per level
        bool odd;              // an odd periodic extent
        int x, b, old;         // iterate, right-hand side, old values
        int cell4, cell1;      // tables (see TailLevel); cell1 -1: not in LDS
    } L[kTailMaxLevels];
    int res = 0, coff = 0, ncoef = 0, cellw = 0, ncellw = 0;
};

// n: extents of the levels S..D (`count` of them, 1 along y in 2-D); periodic:
// per axis; solve: the coarsest level is solved; limit: bytes of LDS.
//
// A solved coarsest level holds three arrays, the third the old values that its
// stopping residual reads; one that fits only without its right-hand side keeps
// that in global memory, from where each thread reads it into registers once a
// solve, and in each pass for the cells beyond those.  Four cycles with the
// coarsest level solved by k_coarse in global memory / here: FP64 82 x 86, 2256
// iterations a solve at most, 62 / 23 ms; 18 x 18 x 22, 119 iterations, 5.8 / 2.5 ms;
// 19 x 18 x 19, 125 iterations, 5.7 / 2.4 ms; FP32 115 x 123 189 / 151 ms, 24 x 23 x 25
// 56 / 28 ms.
inline TailPlan plan_tail(size_t word, int dim, const int (*n)[3], int count, const int (&periodic)[3], bool solve,
                          size_t limit) {
    TailPlan P;
    if (count < 1 || count > kTailMaxLevels) return P;
    const size_t reg = (size_t)kTailColourCells * kTailThreads;
    auto up4 = [](size_t v) { return (v + 3) / 4 * 4; };
    auto place = [&](bool b_global) -> size_t {
        size_t off = 0, ncoef = 0, ncell = 0;
        for (int l = 0; l < count; ++l) {
            TailPlan::Level &V = P.L[l];
            const bool last = l == count - 1;
            for (int a = 0; a < 3; ++a) V.n[a] = n[l][a];
            const int ny = dim == 3 ? n[l][1] : 1;
            V.hz = (n[l][2] + 1) / 2;
            const size_t half = (size_t)n[l][0] * ny * V.hz;
            if (2 * half > 65535) return 0;   // a cell's LDS offset takes 16 bits
            V.half = (int)half;
            V.odd = false;
            for (int a = 0; a < 3; ++a)
                if (dim == 3 || a != 1) V.odd = V.odd || (periodic[a] && (n[l][a] & 1));
            // levels above the coarsest: the cells that the threads keep in
            // registers; larger ones run faster as multi-workgroup passes
            if (!last && (half > reg || V.odd)) return 0;
            V.x = (int)off;
            off += up4(2 * half);
            V.b = b_global ? -1 : (int)off;
            if (!b_global) off += up4(2 * half);
            V.old = (int)off;
            if (last && (solve || (V.odd && half > reg))) off += up4(2 * half);
            ncoef += 2 * ((size_t)n[l][0] + ny + n[l][2]);
            if (dim == 3 && l > 0) ncoef += 3 * ((size_t)n[l][0] + ny + n[l][2]);
            // cell tables of levels with at most one cell of a colour per thread
            V.cell1 = half <= (size_t)kTailThreads ? 0 : -1;
            V.cell4 = 0;
            if (V.cell1 >= 0) ncell += 2 * up4(2 * half) * 5 / 2;
        }
        P.res = (int)off;
        if (count > 1) off += up4(2 * (size_t)P.L[0].half);
        P.coff = (int)off;
        P.ncoef = (int)ncoef;
        off += up4(ncoef);
        const size_t words = word / 4;
        size_t w = off * words;
        P.cellw = (int)w;
        P.ncellw = (int)ncell;
        for (int l = 0; l < count; ++l) {
            TailPlan::Level &V = P.L[l];
            if (V.cell1 < 0) continue;
            const size_t cells = up4(2 * (size_t)V.half);
            V.cell4 = (int)w;
            V.cell1 = (int)(w + 4 * cells);
            w += 5 * cells;
        }
        return w * 4 <= limit && w / words < 65536 ? w * 4 : 0;
    };
    P.bytes = place(false);
    if (!P.bytes && count == 1 && solve) {
        P.b_global = true;
        P.bytes = place(true);
    }
    return P;
}

// One colour pass of a split level (see k_rb_split): rows a lane takes, byte
// offsets and vector numbers beyond 32 and 31 bits, and the number of vectors.
struct PassPlan {
    int rows = 1;
    bool off64 = false, div64 = false, ok = false;
    unsigned total = 0;
};

// Pairs of rows along y (x in a planar level) where the rows pair up and the
// walls are homogeneous; the general form (one row a lane, any SOR parameter,
// 64-bit offsets) elsewhere, and for other parameters than 1 in arrays of 4 GB
// and more, which no deck has.  A launch numbers its lanes with 32 bits (ok);
// numbers of 2^31 and more, which the division by multiplication does not take,
// are divided as they are (div64): general-form levels of 69 GB an array reach
// them, pairs those of twice that.
// dirv: stored wall values; w1: SOR parameter 1; general, wide: forced forms.
inline PassPlan plan_pass(size_t word, int dim, const int (&n)[3], size_t elems, int rtile, bool dirv, bool w1,
                          bool general, bool wide) {
    PassPlan P;
    P.off64 = elems * word > 0xffffffffull || wide;
    const bool one = ((dim == 3 ? n[1] : n[0]) & 1) || dirv || general || (P.off64 && !w1);
    P.rows = one ? 1 : 2;
    const size_t total = (size_t)n[0] * n[1] / P.rows * (n[2] / 2 / (16 / word));
    // (a launch rounds up to whole blocks on every XCD)
    P.ok = total + 4096 <= 0xffffffffull && !(rtile && rtile % P.rows);
    P.total = P.ok ? (unsigned)total : 0;
    P.div64 = total > 0x7fffffffull || wide;
    return P;
}

}  // namespace saras
