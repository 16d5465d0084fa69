// How a Krylov solve hands its iterations to the device: how many to launch
// before the host looks at the scalars, and whether as graphs of several.
// Host arithmetic only.
#ifndef SOLVE_PLAN_H
#define SOLVE_PLAN_H

#include <algorithm>
#include <cmath>

namespace sph {

constexpr int KR_RUN = 4;   // iterations of the larger graph

struct SolvePlan {
    int pred;    // iterations of the last such solve, 0: none yet
    int maxit;

    bool brief() const { return pred > 0 && pred <= 8; }

    // Iterations to launch after `launched` before the next look.  A look costs a
    // stop of the device of about 25 us, an iteration past the end about as much
    // in launches that return at once: with a prediction the solve runs straight
    // to it (a long one to just before it) and then looks often, less so the
    // further it is past it (with the root, looks and launches past the end stay
    // equally dear); without one the batches grow geometrically.  Looked at one by
    // one past a prediction of at most eight, a solve after one at rest took 3.72
    // ms (16^3 box, 44 iterations), 3.90 (20 k canyon, 44), 8.42 (150 k, 64) and
    // 6.80 (32^3 box, 79); so 3.31, 3.55, 7.72 and 6.38.
    int batch(int launched) const {
        const int past = (int)std::sqrt(2.0 * std::max(0, launched - pred));
        int n;
        if (pred == 0) n = std::max(4, launched / 2);
        else if (brief()) n = launched == 0 ? pred : std::max(1, past);
        else if (launched + 4 < pred * 9 / 10) n = pred * 9 / 10 - launched;
        else n = std::max(2, past);
        return std::min(n, maxit - launched);
    }

    // Whether the next KR_RUN of `left` iterations go as one graph, which saves
    // some 7 us an iteration: in solves that are long, or were expected to be.  Its
    // capture takes 0.3 ms; in a solve that was expected to end by now the device
    // waits for it.
    bool run_graph(int launched, int left) const {
        return left >= KR_RUN && (pred == 0 ? launched >= 16 : !brief() || launched >= 64);
    }
};

}  // namespace sph

#endif
