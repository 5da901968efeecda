// scan.hpp — prefix sums of one workgroup, shared by the ray-group culling, the
// compactions and the BLAS build's sort (gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace luz {

// Exclusive scan in place of n counts (16-byte aligned) by one workgroup of
// 1024 threads: thread t sums its run of `per` consecutive counts (a multiple
// of 4, read as 16-byte vectors so that a run's loads are in flight
// together), the runs' sums are scanned by wave shuffles and one exchange of
// wave totals, and each run is rewritten with its prefixes.  Returns the total
// (to every thread).
__device__ inline uint32_t scan_runs_1024(uint32_t* counts, uint32_t n) {
    __shared__ uint32_t wave_sum[1024 / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t per = (((n + 1023u) / 1024u) + 3u) & ~3u, begin = threadIdx.x * per;
    // the run [begin, end): nv whole vectors, then single counts
    const uint32_t end = begin + per < n ? begin + per : (begin < n ? n : begin);
    const uint32_t nv = (end - begin) >> 2, tail = begin + nv * 4;
    uint4* c4 = reinterpret_cast<uint4*>(counts) + (begin >> 2);
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t k = 0; k < nv; ++k) {
        const uint4 v = c4[k];
        sum += v.x + v.y + v.z + v.w;
    }
    for (uint32_t q = tail; q < end; ++q) sum += counts[q];
    uint32_t incl = sum;
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off);
        if (lane >= off) incl += y;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t w = 0; w < 1024 / 64; ++w) {
        if (w < wave) before += wave_sum[w];
        total += wave_sum[w];
    }
    uint32_t run = before + incl - sum;
#pragma unroll 8
    for (uint32_t k = 0; k < nv; ++k) {
        const uint4 v = c4[k];
        uint4 o;
        o.x = run; run += v.x;
        o.y = run; run += v.y;
        o.z = run; run += v.z;
        o.w = run; run += v.w;
        c4[k] = o;
    }
    for (uint32_t q = tail; q < end; ++q) {
        const uint32_t v = counts[q];
        counts[q] = run;
        run += v;
    }
    return total;
}

}  // namespace luz
