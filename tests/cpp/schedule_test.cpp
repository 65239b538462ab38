// Chunks of a batch solve (csrc/schedule.h) on the host: simulated solves whose
// residual falls at a steady rate, and states at the limits of their ranges.
#define __host__
#define __device__
#include "schedule.h"

#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <limits>

using namespace cpmgpu;

#define CHECK(c) \
    if (!(c)) { std::fprintf(stderr, "line %d: %s\n", __LINE__, #c); std::exit(1); }

static KState lane(int iters, int max_it, double rr, double bsq, double tol2) {
    KState s{};
    s.status = ST_RUN;
    s.iters = iters;
    s.max_it = max_it;
    s.rr = rr;
    s.bsq = bsq;
    s.tol2 = tol2;
    return s;
}

// Iterations that the solve's loop launches for a system that ends after `need`.
static int launched(int need, int max_it, double tol2) {
    const int end = std::min(need, max_it);
    int total = 0, flight[2] = {0, 0}, pending = 0;
    auto queue = [&](int n) {
        total += n;
        flight[pending++] = n;
    };
    queue(4);
    for (;;) {
        const int seen = total - (pending == 2 ? flight[1] : 0);   // iterations behind the oldest states
        const int fly = total - seen;
        flight[0] = flight[1];
        --pending;
        if (seen >= end) return total;
        const double left = iterations_left(lane(seen, max_it, std::pow(tol2, (double)seen / need), 1.0, tol2), false);
        for (int f = fly; pending < 2;) {
            const int n = next_chunk(left, f);
            if (n == 0) break;
            queue(n);
            f += n;
        }
        CHECK(pending > 0);
    }
}

int main() {
    // at most a chunk of four more than the system takes, when its residual falls steadily
    for (int need : {1, 2, 4, 5, 8, 9, 12, 13, 60, 61, 129, 130, 448, 1000})
        CHECK(launched(need, 100000, 1e-20) <= (need + 3) / 4 * 4 + 4);
    // and none past the limit's last four
    for (int max_it : {1, 2, 4, 5, 8, 12, 13, 60, 61, 130})
        CHECK(launched(5000, max_it, 1e-20) == (max_it + 3) / 4 * 4);
    // residuals that say nothing
    const double eps = std::numeric_limits<double>::epsilon(), inf = std::numeric_limits<double>::infinity();
    for (double rr : {1.0 - eps / 2, 1.0, 2.0, 0.0, inf, std::nan(""), std::numeric_limits<double>::denorm_min()})
        for (double tol2 : {1e-20, 0.0, std::numeric_limits<double>::denorm_min()})
            for (int it : {0, 1, 99999}) {
                const double left = iterations_left(lane(it, 100000, rr, 1.0, tol2), false);
                CHECK(left >= 1.0 && left <= 1e6);
                for (int f : {0, 4, 64}) {
                    const int n = next_chunk(left, f);
                    CHECK(n >= 0 && n <= 32 && n % 4 == 0 && (n > 0 || f > 0));
                }
            }
    CHECK(next_chunk(iterations_left(lane(99999, 100000, 1.0 - eps / 2, 1.0, 1e-20), false), 0) == 4);
    std::puts("schedule ok");
    return 0;
}
