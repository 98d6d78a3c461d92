// arrival.hpp -- how the blocks of a reduction find the last one of them.
//
// Every block replaces the counter by arrival_next of it in one atomic step
// (atomicInc with bound blocks - 1), and the block that found blocks - 1 there is
// the last.  The counter is thus at zero before and after every launch, and
// nothing has to clear it.  A counter serves launches of one grid size only:
// then it is at zero whenever no launch is running, also after launches that
// overlapped (n launches add n times the grid size, which is zero modulo the grid
// size), so that an overlap can spoil the overlapping results but no later one.
// A counter shared by grids of several sizes, or one that the last block clears
// with a store, keeps a remainder after an overlap and then takes a block that is
// not the last for it in every later launch.
#pragma once

#if defined(__HIPCC__)
#define TRIXI_ARRIVAL_QUAL __host__ __device__ inline
#else
#define TRIXI_ARRIVAL_QUAL inline
#endif

namespace trixi_hip {

// what atomicInc(counter, blocks - 1) leaves in place of `count`
TRIXI_ARRIVAL_QUAL unsigned arrival_next(unsigned count, unsigned blocks) { return count >= blocks - 1 ? 0 : count + 1; }
// whether the block that found `count` is the last of its launch
TRIXI_ARRIVAL_QUAL bool arrival_is_last(unsigned count, unsigned blocks) { return count >= blocks - 1; }

// The counters of a context, one per grid size of its reductions.
enum ArrivalCounter {
    ARRIVED_ELEMENTS = 0,  // max_dt, max_dt_noalloc and integrals (reduction_blocks)
    ARRIVED_NORMS = 1,     // error norms
    ARRIVED_STATE = 2,     // state check
    ARRIVAL_COUNTERS = 3
};

}  // namespace trixi_hip
