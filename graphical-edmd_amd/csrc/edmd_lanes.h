/*
 * Masks of a wavefront's lanes, and other 64-bit masks, by 32-bit shifts.
 *
 * A 64-bit vector shift by an amount in the last vector register that a kernel
 * has gave wrong results here: a defect of gfx90a, where the compiler keeps the
 * amount out of that register; it does not for gfx950.  Builds of the wide loop
 * that held the lane's number in v127 of 128 took wrong events in 5 to 14% of a
 * batch's systems, each the second on its compute unit; builds of the same
 * source with it in another register did not.  The register is the compiler's
 * choice, so no kernel has such a shift (shifts by a uniform amount are the
 * scalar unit's, a constant amount is no register).  Without them the sweep
 * of 1,048,576 disks takes 1877 us for 1928 and 200 collisions of 400 disks take
 * 567 us for 574.
 */
#ifndef EDMD_LANES_H
#define EDMD_LANES_H

#include <hip/hip_runtime.h>
#include <stdint.h>

/* Whether the running lane's bit is set in m, which is the same on every lane. */
__device__ __forceinline__ bool lane_in(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

/* Bit k alone; none outside 0 .. 63. */
__device__ __forceinline__ uint64_t bit_mask(int k) {
    const uint32_t b = 1u << (k & 31);
    const uint32_t lo = (k >> 5) == 0 ? b : 0u, hi = (k >> 5) == 1 ? b : 0u;
    return (uint64_t)hi << 32 | lo;
}

/* The bits below k: none for k <= 0, all for k >= 64. */
__device__ __forceinline__ uint64_t bits_below(int k) {
    const uint32_t b = (1u << (k & 31)) - 1;
    const uint32_t lo = k <= 0 ? 0u : (k < 32 ? b : ~0u), hi = k <= 32 ? 0u : (k < 64 ? b : ~0u);
    return (uint64_t)hi << 32 | lo;
}

/* How many of m's bits are below the running lane's. */
__device__ __forceinline__ int lanes_before(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

#endif
