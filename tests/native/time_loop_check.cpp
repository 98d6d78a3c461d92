// The host side of the device time loop (csrc/time_loop.hpp) against a device that
// is played on the host: steps queued run when they are waited for, each logging
// its time.  Checked: the steps and times of a run that ends well (fixed and
// shrinking steps, limits on the steps), and of runs whose queueing or waiting
// fails at any step: then the time and the count are those of the steps that ran,
// everything queued has been waited for, and nothing is queued afterwards.
// Prints "runs <n>" and "ok" or "FAIL ...".
#include <cstdio>
#include <vector>

#include "time_loop.hpp"

static const int64_t kChunk = 8;

struct Device {  // the device's time, and the log of a chunk
    double t, t_end, dt, shrink;
    std::vector<double> log = std::vector<double>(2 * kChunk);
    std::vector<int64_t> pending;
    int64_t steps = 0, queued = 0, waits = 0;
    int64_t fail_queue = -1, fail_wait = -1;
    bool after_error = false, failed = false;
    int queue(int64_t i) {
        after_error = after_error || failed;
        if (queued++ == fail_queue) {
            failed = true;
            return 7;
        }
        pending.push_back(i);
        return 0;
    }
    int wait() {
        if (waits++ == fail_wait) {
            failed = true;
            return 9;
        }
        for (int64_t i : pending) {
            double h = dt;
            if (!(t < t_end)) {
                log[2 * i] = t;
                log[2 * i + 1] = -1.0;
                continue;
            }
            if (t + h >= t_end) {
                h = t_end - t;
                t = t_end;
            } else {
                t += h;
            }
            log[2 * i] = t;
            log[2 * i + 1] = h;
            ++steps;
            dt *= shrink;
        }
        pending.clear();
        return 0;
    }
};

int main() {
    long runs = 0;
    bool ok = true;
    for (double shrink : {1.0, 0.9, 1.2})
        for (double h0 : {0.0, 0.1})
            for (int64_t max_steps : {int64_t(0), int64_t(1), int64_t(5), int64_t(8), int64_t(9), int64_t(40), int64_t(1) << 40})
                for (int64_t fq = -1; fq < 30; ++fq)
                    for (int64_t fw = -1; fw < 4; ++fw) {
                        Device d;
                        d.t = 0.25;
                        d.t_end = 1.0;
                        d.dt = 0.1;
                        d.shrink = shrink;
                        d.fail_queue = fq;
                        d.fail_wait = fw;
                        double t = d.t;
                        int64_t n = -1;
                        const int rc = trixi_hip::run_steps(&t, d.t_end, h0, max_steps, kChunk, d.log.data(), &n,
                                                            [&](int64_t i) { return d.queue(i); }, [&] { return d.wait(); });
                        const bool wait_failed = fw >= 0 && d.waits > fw;
                        const bool queue_failed = fq >= 0 && d.queued > fq;
                        bool good = rc == (queue_failed ? 7 : (wait_failed ? 9 : 0)) && n <= max_steps && !d.after_error;
                        // what the caller is told is what ran (unless the wait itself failed)
                        good = good && (wait_failed || (t == d.t && n == d.steps && d.pending.empty()));
                        if (rc == 0) good = good && (t == d.t_end || n == max_steps);
                        if (!good) std::printf("shrink %g h0 %g max %ld fq %ld fw %ld: rc %d t %g n %ld\n", shrink, h0,
                                               (long)max_steps, (long)fq, (long)fw, rc, t, (long)n);
                        ok = ok && good;
                        ++runs;
                    }
    std::printf("runs %ld\n%s\n", runs, ok ? "ok" : "FAIL");
    return ok ? 0 : 1;
}
