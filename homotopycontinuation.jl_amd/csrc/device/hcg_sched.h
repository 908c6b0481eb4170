// Work distribution of the persistent tracker kernels over the lanes of a wave.
//
// A lane whose path has ended does not close it and start its next path at once: closing a
// path (refinement in double-double, a condition estimate, the record) and starting one
// (tracker and predictor initialization) cost a few tracker steps each, and while one lane
// does it the other 63 lanes of the wave wait.  Idle lanes therefore wait until at least
// `refill` of the wave's live lanes are idle (or all of them are), then close their paths and
// take their next ones from the work queue together, with one atomic per wave.
#pragma once
#include "hcgpu_types.h"

// Measured on the parameter batch (n = 10, 262,144 paths, learned step): 4, 8, 12, 16, 24, 32 idle lanes
// 265.3, 246.3, 240.1, 241.3, 246.8, 256.1 ms; smaller batches have no paths waiting and do not care.
#define HCG_DEFAULT_REFILL 12

__device__ __forceinline__ int refill_threshold(const hcg_options* o) {
    int r = o->refill_idle;
    return r > 0 ? r : HCG_DEFAULT_REFILL;
}

// Called by every live lane of the wave, converged: the mask of the lanes that take a new
// path in this loop iteration (all idle lanes, or none).
__device__ __forceinline__ unsigned long long wave_refill_mask(bool idle, int refill) {
    const unsigned long long im = __ballot(idle ? 1 : 0), lm = __ballot(1);
    return (im != 0ull && (__popcll(im) >= refill || im == lm)) ? im : 0ull;
}

// Called by exactly the lanes of mask m (non-empty, this lane in m): consecutive queue
// indices, in lane order, from one atomicAdd on the queue head.
__device__ __forceinline__ int wave_fetch(unsigned long long m, int32_t* next) {
    const int lane = (int)__lane_id();
    const int leader = __ffsll((unsigned long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(next, __popcll(m));
    base = __shfl(base, leader);
    return base + __popcll(m & ((1ull << lane) - 1ull));
}

// A lane's totals added to the launch counters: summed over the wave first, then one atomic per
// counter and wave.  Every lane of the wave calls it, converged.  (64 atomics on one address per
// counter take about 10 ns each: 2,000 two-variable paths on 1,024 waves spent 3 ms on them.)
__device__ __forceinline__ void wave_add(unsigned long long* counter, unsigned long long v) {
    for (int off = 32; off > 0; off >>= 1) v += (unsigned long long)__shfl_xor((long long)v, off, 64);
    if (__lane_id() == 0) atomicAdd(counter, v);
}
