// time_loop.hpp -- the host side of the device time loop: queue a chunk of steps,
// wait once, read the steps' log.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace trixi_hip {

// Steps from *t to t_end, at most max_steps, in chunks of at most max_chunk.
// queue(i) queues step i of the chunk and wait() waits for everything queued; both
// return 0 or an error.  Step i leaves {t after it, h} in log[2 i], log[2 i + 1],
// h < 0 for a step that was not taken because t_end had been reached.  h: the size
// of the next step if known, else 0 (a guess of how many steps are left).
// *t and *nsteps follow the steps that were taken.  If a step cannot be queued,
// those queued before it in its chunk are waited for and counted before the error
// is returned, so that nothing is still running then and *t and *nsteps are those
// of the state.
template <class Queue, class Wait>
int run_steps(double* t, double t_end, double h, int64_t max_steps, int64_t max_chunk, const double* log,
              int64_t* nsteps, Queue queue, Wait wait) {
    *nsteps = 0;
    while (*t < t_end && *nsteps < max_steps) {
        // by the last step size, two where there is none yet
        const double left = h > 0.0 ? std::ceil((t_end - *t) / h) : 2.0;
        int64_t chunk = std::min<int64_t>(max_chunk, max_steps - *nsteps);
        if (left < (double)chunk) chunk = left > 1.0 ? (int64_t)left : 1;
        int64_t queued = 0;
        int rc = 0;
        while (queued < chunk && (rc = queue(queued)) == 0) ++queued;
        const int waited = wait();
        if (waited) return rc ? rc : waited;
        for (int64_t i = 0; i < queued; ++i) {
            if (log[2 * i + 1] < 0.0) break;
            *t = log[2 * i];
            h = log[2 * i + 1];
            ++*nsteps;
        }
        if (rc) return rc;
    }
    return 0;
}

}  // namespace trixi_hip
