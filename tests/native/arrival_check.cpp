// The arrival counter of the device reductions (csrc/arrival.hpp) under launches
// that overlap: every order in which the blocks of two launches of one grid size
// can arrive, and random orders of up to four.  Afterwards the counter must be at
// zero, and a launch on its own must take exactly its last block for the last.
// Prints "orders <n>" and "ok" or "FAIL ...".
#include <cstdio>
#include <cstdlib>
#include <random>

#include "arrival.hpp"

using trixi_hip::arrival_is_last;
using trixi_hip::arrival_next;

static bool later_launch_is_right(unsigned count, unsigned blocks) {
    for (unsigned b = 0; b < blocks; ++b) {
        if (arrival_is_last(count, blocks) != (b == blocks - 1)) return false;
        count = arrival_next(count, blocks);
    }
    return count == 0;
}

// Interleavings of two launches with a and b blocks still to come.
static long orders = 0;
static bool walk(unsigned count, unsigned a, unsigned b, unsigned blocks) {
    if (a == 0 && b == 0) {
        ++orders;
        return count == 0 && later_launch_is_right(count, blocks);
    }
    const unsigned next = arrival_next(count, blocks);
    return (a == 0 || walk(next, a - 1, b, blocks)) && (b == 0 || walk(next, a, b - 1, blocks));
}

int main() {
    bool ok = true;
    for (unsigned blocks = 1; blocks <= 7; ++blocks) ok = ok && later_launch_is_right(0, blocks) && walk(0, blocks, blocks, blocks);
    std::mt19937 rng(20261205);
    for (int trial = 0; trial < 20000; ++trial) {
        const unsigned blocks = 1 + rng() % 1024, launches = 1 + rng() % 4;
        unsigned count = 0;
        for (unsigned i = 0; i < blocks * launches; ++i) count = arrival_next(count, blocks);
        ok = ok && count == 0;
    }
    std::printf("orders %ld\n%s\n", orders, ok ? "ok" : "FAIL");
    return ok ? 0 : 1;
}
