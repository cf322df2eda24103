// The tail's LDS (plan_tail): which solved coarsest levels it takes and how.
// Prints the levels checked.
#include <cstdio>

#include "mg_plan.hpp"

using namespace saras;

int main() {
    int failures = 0;
    long checked = 0, global = 0;
    for (size_t word = 4; word <= 8; word += 4)
        for (int dim = 2; dim <= 3; ++dim)
            for (int nx = 2; nx <= 130; ++nx)
                for (int ny = dim == 3 ? 2 : 1; ny <= (dim == 3 ? 40 : 1); ++ny)
                    for (int nz = 2; nz <= 130; ++nz) {
                        const size_t cells = (size_t)nx * ny * nz;
                        const size_t shell = dim == 3 ? (size_t)(nx + 2) * (ny + 2) * (nz + 2) : (size_t)(nx + 2) * (nz + 2);
                        // two arrays, one with ghost layers, and the coefficients in
                        // 128 KB: what a tail without tables and old values takes
                        if ((shell + cells + 5 * (nx + ny + nz)) * word > 128 * 1024) continue;
                        const int n[1][3] = {{nx, ny, nz}}, per[3] = {1, 1, 1};
                        const TailPlan P = plan_tail(word, dim, n, 1, per, true, kTailLds);
                        ++checked;
                        const TailPlan::Level &V = P.L[0];
                        const int len = 2 * V.half;
                        bool ok = P.bytes > 0 && P.bytes <= kTailLds && len >= (int)cells && V.x == 0 && V.old >= V.x + len &&
                                  P.coff >= V.old + len && P.coff + P.ncoef <= (int)(P.bytes / word) && P.coff < 65536;
                        if (P.b_global) {
                            ++global;
                            ok = ok && V.b == -1 && V.cell1 == -1;
                        } else {
                            ok = ok && V.b >= V.x + len && V.old >= V.b + len;
                        }
                        if (!ok && ++failures < 20) std::printf("word %zu: %d x %d x %d: %zu bytes\n", word, nx, ny, nz, P.bytes);
                    }
    // by colour passes where nothing is solved and a third array does not fit
    const int n[1][3] = {{85, 1, 78}}, per[3] = {1, 0, 0};
    failures += plan_tail(8, 2, n, 1, per, false, kTailLds).bytes != 0;
    std::printf("levels %ld, %ld of them without the right-hand side; failures %d\n", checked, global, failures);
    return failures ? 1 : 0;
}
