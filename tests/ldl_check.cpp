// Checks of the LDL preconditioner's host side (csrc/ldl_host.cpp), built and
// run by test_ldl_host.py.
//   ldl_check alloc nx ny   every allocation of ldl_blocks fails in turn, in
//                           whichever thread makes it: the caller gets a
//                           std::bad_alloc, or (a helper thread that cannot
//                           start) the blocks
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "fvh_internal.h"
#include "ldl_host.h"

namespace fvh {
int set_error(int code, const char *fmt, ...) {
    va_list a;
    va_start(a, fmt);
    std::vprintf(fmt, a);
    va_end(a);
    return code;
}
}  // namespace fvh

using namespace fvh;

static std::atomic<long> g_left{-1};  // allocations until one fails (-1: none does)
static std::atomic<bool> g_failed{false};

void *operator new(std::size_t n) {
    if (g_left.load() >= 0 && g_left.fetch_sub(1) == 0) {
        g_failed = true;
        throw std::bad_alloc();
    }
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

// A on an nx x ny grid of five-point rows: off(a, b) for neighbours a < b, diag(r, sum of the row's |off|).
struct Grid {
    int n = 0;
    std::vector<int> rp{0}, col;
    std::vector<double> val, x, y;
    template <class Off, class Diag>
    Grid(int nx, int ny, Off off, Diag diag) : n(nx * ny), x(n), y(n) {
        for (int r = 0; r < n; ++r) {
            const int i = r % nx, j = r / nx;
            x[r] = i;
            y[r] = j;
            const int nb[5] = {j ? r - nx : -1, i ? r - 1 : -1, r, i < nx - 1 ? r + 1 : -1, j < ny - 1 ? r + nx : -1};
            double sum = 0.0;
            size_t at = 0;
            for (int c : nb) {
                if (c < 0) continue;
                if (c == r) at = val.size();
                col.push_back(c);
                val.push_back(c == r ? 0.0 : off(std::min(r, c), std::max(r, c)));
                sum += std::fabs(val.back());
            }
            val[at] = diag(r, sum);
            rp.push_back((int)col.size());
        }
    }
};

static int factor(const Grid &g, LdlHost &F, std::vector<int> &bounds) {
    std::vector<int> perm;
    ldl_order(g.n, g.rp.data(), g.col.data(), g.x.data(), g.y.data(), perm, &bounds);
    return ldl_factor(g.n, g.rp.data(), g.col.data(), g.val.data(), perm, F);
}

static int check_alloc(int nx, int ny) {
    const Grid g(nx, ny, [](int, int) { return -1.0; }, [](int, double s) { return s + 0.01; });
    LdlHost F;
    std::vector<int> bounds;
    if (factor(g, F, bounds)) return 1;
    int thrown = 0, served = 0;
    for (long k = 0;; ++k) {
        g_failed = false;
        g_left = k;
        try {
            LdlBlocks B;
            ldl_blocks(F, bounds, B);
            g_left = -1;
            if (B.f.blocks.empty() || B.b.blocks.empty()) return 2;
            if (!g_failed) break;
            ++served;
        } catch (const std::bad_alloc &) {
            g_left = -1;
            ++thrown;
        }
    }
    std::printf("%d failures reported, %d served by fewer threads\n", thrown, served);
    return thrown > 0 ? 0 : 3;
}

int main(int argc, char **argv) {
    if (argc >= 4 && !std::strcmp(argv[1], "alloc")) return check_alloc(std::atoi(argv[2]), std::atoi(argv[3]));
    return 64;
}
