// Every row that the tiles of a planned visit load or need, over axes from a few
// rows (thin periodic ones among them) to many: a loaded row lies inside the
// level, and every row that a stored row's passes read is one of those.
// Arguments: bytes of a word, dimension.  Prints the plans checked and how many
// of them leave rows of their last tile out.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <tuple>

#include "mg_plan.hpp"

using namespace saras;

namespace {

int failures = 0;

// the tiles of `t` rows along an axis of n rows
void axis(const char *what, int n, int t, int halo, bool periodic) {
    static std::set<std::tuple<int, int, int, bool>> seen;
    if (!seen.insert({n, t, halo, periodic}).second) return;
    const TileAxis A = TileAxis::of(n, halo, periodic);
    for (int i0 = 0; i0 < n; i0 += t) {
        for (int q = i0 - halo; q < i0 + t + halo; ++q)
            if (A.has(q) && (A.row(q) < 0 || A.row(q) >= n || (A.row(q) - q) % n)) {
                std::printf("%s: n %d tile %d halo %d %s: row %d -> %d\n", what, n, t, halo, periodic ? "periodic" : "walls", q,
                            A.row(q));
                ++failures;
            }
        for (int i = i0; i < std::min(i0 + t, n); ++i)
            for (int q = i - halo; q <= i + halo; ++q)
                if (!A.has(q) && (periodic || (q >= 0 && q < n))) {
                    std::printf("%s: n %d tile %d halo %d: row %d, which row %d needs, is left out\n", what, n, t, halo, q, i);
                    ++failures;
                }
    }
}

}  // namespace

int main(int argc, char **argv) {
    if (argc != 3) return 2;
    const size_t word = (size_t)std::atoi(argv[1]);
    const int dim = std::atoi(argv[2]);
    long plans = 0, cut = 0;
    const int xs[] = {4, 6, 8, 10, 12, 14, 18, 20, 22, 28, 36, 44, 50, 64, 72, 100, 160, 192, 256, 512};
    const int zs[] = {8, 16, 20, 32, 44, 64, 100, 128, 256};
    for (int nx : xs)
        for (int ny : xs)
            for (int nz : zs) {
                if (dim == 2 && ny != xs[0]) continue;
                const int n[3] = {nx, dim == 3 ? ny : 1, nz};
                for (int split = 0; split < 2; ++split)
                    for (int count = 1; count <= 8; ++count)
                        for (int visit = 0; visit < 3; ++visit) {   // down from zero, down, up
                            const bool zero = visit == 0, pro = visit == 2, restr = visit < 2;
                            const TilePlan t = plan_tile(word, dim, n, split != 0, count, zero, pro, restr);
                            if (!t.sweeps) continue;
                            ++plans;
                            bool over = false;
                            for (int done = 0; done < count; done += t.sweeps) {
                                const int halo = tile_halo(std::min(t.sweeps, count - done), zero && done == 0,
                                                           restr && done + t.sweeps >= count);
                                for (int periodic = 0; periodic < 2; ++periodic) {
                                    axis("x", nx, t.ti, halo, periodic != 0);
                                    if (dim == 3) axis("y", ny, t.tj, halo, periodic != 0);
                                }
                                over = over || (nx + t.ti - 1) / t.ti * t.ti + halo > 2 * nx ||
                                       (dim == 3 && (ny + t.tj - 1) / t.tj * t.tj + halo > 2 * ny);
                            }
                            cut += over;
                        }
            }
    std::printf("plans %ld cut %ld failures %d\n", plans, cut, failures);
    return failures ? 1 : 0;
}
