// Totals of the per-simulation statistics, added on the device.
//
// ctl_sim_run and ctl_batch_run report the sums of eight counters over all
// simulations.  A record is 64 bytes, so 65536 simulations hold 4.2 MB: the
// copy to fresh host memory and the host's loop over it took 3.4 ms of a
// 25 ms pass (and one copy per model in a batch); here the records are read
// once where they are and 64 bytes are copied out.  The sums are of unsigned
// integers, so their order does not show in the result.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/ctl.h"

namespace ctl {

enum { ST_FIRINGS, ST_LEAPS, ST_REJECTIONS, ST_SWITCHES, ST_SSA, ST_POISSON, ST_GAPS, ST_ABSORBED, ST_COUNT };
constexpr int STAT_BLOCK = 256;

// Adds records first, first + stride, ... below n of st to tot, all threads of
// the workgroup together: registers, then a wavefront's lanes, then the four
// wavefronts in LDS, so a workgroup issues eight atomics.
__device__ __forceinline__ void stat_add(const ctl_sim_stat* __restrict__ st, int first, int n, int stride,
                                         unsigned long long* tot) {
    __shared__ unsigned long long part[STAT_BLOCK / 64][ST_COUNT];
    unsigned long long v[ST_COUNT] = {};
    for (long i = first; i < n; i += stride) {        // past n by up to a stride: not an int's sum
        const ctl_sim_stat x = st[i];
        v[ST_FIRINGS] += x.firings;
        v[ST_LEAPS] += x.leaps;
        v[ST_REJECTIONS] += x.rejections;
        v[ST_SWITCHES] += x.switches;
        v[ST_SSA] += x.ssa_steps;
        v[ST_POISSON] += x.poisson;
        v[ST_GAPS] += x.gaps;
        v[ST_ABSORBED] += x.absorbed;
    }
#pragma unroll
    for (int k = 0; k < ST_COUNT; ++k)
        for (int d = 32; d > 0; d >>= 1) v[k] += __shfl_xor(v[k], d, 64);
    if ((threadIdx.x & 63u) == 0)
        for (int k = 0; k < ST_COUNT; ++k) part[threadIdx.x / 64][k] = v[k];
    __syncthreads();
    if (threadIdx.x < ST_COUNT) {
        unsigned long long s = 0;
        for (int w = 0; w < STAT_BLOCK / 64; ++w) s += part[w][threadIdx.x];
        if (s) atomicAdd(tot + threadIdx.x, s);
    }
}

inline void stat_store(ctl_stats& S, const unsigned long long (&t)[ST_COUNT]) {
    S.firings = t[ST_FIRINGS];
    S.leaps = t[ST_LEAPS];
    S.rejections = t[ST_REJECTIONS];
    S.switches = t[ST_SWITCHES];
    S.ssa_steps = t[ST_SSA];
    S.poisson = t[ST_POISSON];
    S.gaps = t[ST_GAPS];
    S.absorbed = t[ST_ABSORBED];
}

}  // namespace ctl
