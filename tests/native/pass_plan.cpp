// The form of a colour pass (plan_pass) at the sizes where it changes.
#include <cstdio>

#include "mg_plan.hpp"

using namespace saras;

static int failures = 0;
#define CHECK(c) \
    do { \
        if (!(c)) { \
            std::printf("line %d: %s\n", __LINE__, #c); \
            ++failures; \
        } \
    } while (0)

static PassPlan plan(size_t word, int dim, int nx, int ny, int nz, bool dirv, bool w1, bool general = false,
                     bool wide = false) {
    const int n[3] = {nx, ny, nz};
    return plan_pass(word, dim, n, (size_t)nx * ny * nz, 0, dirv, w1, general, wide);
}

int main() {
    // pairs of rows, 32-bit offsets
    PassPlan p = plan(8, 3, 256, 256, 256, false, true);
    CHECK(p.ok && p.rows == 2 && !p.off64 && !p.div64 && p.total == 256u * 256 / 2 * 64);
    p = plan(4, 2, 1024, 1, 1024, false, false);
    CHECK(p.ok && p.rows == 2 && !p.off64 && p.total == 512u * 128);
    // one row: odd rows, stored walls, forced
    CHECK(plan(8, 3, 8, 9, 16, false, true).rows == 1);
    CHECK(plan(8, 2, 9, 1, 16, false, true).rows == 1);
    CHECK(plan(8, 3, 8, 8, 16, true, true).rows == 1);
    CHECK(plan(8, 3, 8, 8, 16, false, true, true).rows == 1);
    // 4 GB: the last array of 32-bit offsets and the first beyond
    CHECK(!plan(4, 3, 1024, 1023, 1024, false, true).off64);
    p = plan(4, 3, 1024, 1024, 1024, false, true);
    CHECK(p.ok && p.off64 && p.rows == 2 && !p.div64);
    CHECK(plan(4, 3, 1024, 1024, 1024, false, false).rows == 1);
    // 69 GB: 2^31 vectors of single rows
    p = plan(8, 3, 2048, 2048, 2048, false, false);
    CHECK(p.ok && p.rows == 1 && p.off64 && p.div64 && p.total == 1u << 31);
    p = plan(8, 3, 2048, 2048, 2044, false, false);
    CHECK(p.ok && !p.div64);
    p = plan(8, 2, 65536, 1, 131072, true, true);
    CHECK(p.ok && p.rows == 1 && p.div64);
    p = plan(8, 3, 2048, 2048, 2048, false, true);
    CHECK(p.ok && p.rows == 2 && p.off64 && !p.div64);
    // beyond the lanes of a launch
    CHECK(!plan(8, 3, 2048, 4096, 2048, false, false).ok);
    // forced
    p = plan(8, 3, 16, 16, 16, false, true, false, true);
    CHECK(p.ok && p.rows == 2 && p.off64 && p.div64);
    std::printf("failures %d\n", failures);
    return failures ? 1 : 0;
}
