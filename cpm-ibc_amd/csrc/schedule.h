// How many iterations a batch solve queues between two looks at its states.
// Plain C++, tested on the host (tests/cpp/schedule_test.cpp).
#pragma once
#include <algorithm>
#include <cmath>

#include "refine.h"

namespace cpmgpu {

inline bool lane_running(const KState& s) { return s.status == ST_RUN || (s.status >= ST_UPDATE && s.status <= ST_READY); }

// Iterations a running lane is expected to need until its residual meets the
// tolerance, at its mean rate so far, or kUnknownLeft while that says nothing
// (no iteration yet, or a residual that has not fallen); never more than its
// iteration limit leaves, nor fewer than one.
constexpr double kUnknownLeft = 8.0;
inline double iterations_left(const KState& s, bool refine) {
    double rr = s.rr;
    if (refine) {
        rr = s.scale > 0 ? s.rr / (s.scale * s.scale) : s.rr_true;
        if (!(rr < s.rr_true)) rr = s.rr_true;
    }
    double left = kUnknownLeft;
    if (s.iters > 0 && s.bsq > 0 && rr > 0 && rr < s.bsq && s.tol2 > 0) {
        const double est = s.iters * (std::log(s.tol2 / rr) / std::log(rr / s.bsq));
        if (est < 1e6) left = est;   // a residual that has hardly fallen says no more than none
    }
    // a mixed lane takes an iteration more for each refinement step, the last one after its limit
    const double most = (double)s.max_it - s.iters + (refine ? 1 : 0);
    return std::max(1.0, std::min(left, most));
}

// Iterations to queue next, a multiple of 4 up to 32, with `left` expected
// from the states just seen and `flight` of those queued already; 0: what is
// in flight is expected to finish.
inline int next_chunk(double left, int flight) {
    if (!(left > flight)) return 0;
    return std::max(4, std::min(32, (int)((left - flight) / 3.0) & ~3));
}

}  // namespace cpmgpu
