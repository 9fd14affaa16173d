/* What the lockstep kernels share on the device (tmc_lock.hip,
 * tmc_lock_prec.hip): a wave's slot of sums, the generator with a
 * wave-uniform absorption count, and the kernel arguments at their use. */
#ifndef TMC_LOCK_DEVICE_H
#define TMC_LOCK_DEVICE_H

#include "tmc_cohort.h"
#include "tmc_device.h"
#include "tmc_philox.h"
#include "tmc_step.h"

namespace tmc {

/* Copies of the overflow shell's sums in a slot (16: 1% slower). */
#define TMC_LOCK_HOT 8u
static_assert(TMC_LOCK_HOT <= TMC_CHECK_HOT, "the shell check covers every overflow copy");

/* Steps of a wave between two flushes of its slot by it: with `waves` waves to
 * the slot a word takes fewer than 2^20 deposits of at most 2^43 each from one
 * flush to the next, so it stays below 2^63. */
__host__ __device__ constexpr uint32_t lock_flush_steps(uint32_t waves) { return (1u << 14) / waves - 1u; }

__host__ __device__ __forceinline__ size_t lock_slot_words(uint32_t shells)
{
    return 2u * ((size_t)shells - 1u + TMC_LOCK_HOT);
}

typedef uint32_t Images __attribute__((ext_vector_type(4)));

/* Philox block (k, 0) of photons with one high counter word and one k (both
 * wave-uniform): what rounds 1 and 2 make of k is scalar.  c3k1: the high
 * counter word ^ key1. */
__device__ __forceinline__ tmc_u32x4 block0_uniform(uint32_t k, uint32_t c3k1, const tmc_philox_photon& pp,
                                                    const tmc_philox_keys& ks)
{
    const uint64_t q0 = (uint64_t)k * TMC_PHILOX_M0;
    const uint64_t p1 = (uint64_t)((uint32_t)(q0 >> 32) ^ c3k1) * TMC_PHILOX_M1;
    uint32_t c0 = pp.c1r1 ^ ((uint32_t)(p1 >> 32) ^ ks.k0[1]), c2 = pp.c2r2k ^ (uint32_t)q0;
    uint64_t a = (uint64_t)c0 * TMC_PHILOX_M0, b = (uint64_t)c2 * TMC_PHILOX_M1;
    c0 = (uint32_t)(b >> 32) ^ ((uint32_t)p1 ^ ks.k0[2]);
    c2 = tmc_xor3((uint32_t)(a >> 32), pp.c3r2, ks.k1[2]);
    uint32_t c1 = (uint32_t)b, c3 = (uint32_t)a;
#pragma unroll
    for (int round = 3; round < 10; ++round) {
        a = (uint64_t)c0 * TMC_PHILOX_M0;
        b = (uint64_t)c2 * TMC_PHILOX_M1;
        c0 = tmc_xor3((uint32_t)(b >> 32), c1, ks.k0[round]);
        c2 = tmc_xor3((uint32_t)(a >> 32), c3, ks.k1[round]);
        c1 = (uint32_t)b;
        c3 = (uint32_t)a;
    }
    return tmc_u32x4{ c0, c1, c2, c3 };
}

/* Moves a slot into a block of the global sums and zeroes it: pairs first,
 * first + stride, ...  SHARED: by atomic swaps, safe while other waves add. */
template <bool SHARED>
__device__ __forceinline__ void lock_flush(unsigned long long* slot, unsigned long long* g, uint32_t shells,
                                           uint32_t first, uint32_t stride)
{
    const uint32_t last = shells - 1u;
    for (uint32_t q = first; q < last + TMC_LOCK_HOT; q += stride) {
        unsigned long long a, b;
        if (SHARED) {
            a = atomicExch(slot + 2u * q, 0ull);
            b = atomicExch(slot + 2u * q + 1u, 0ull);
        } else {
            a = slot[2u * q];
            b = slot[2u * q + 1u];
            slot[2u * q] = 0;
            slot[2u * q + 1u] = 0;
        }
        const uint32_t s = q < last ? q : last;
        unsigned long long oa = 0, ob = 0;
        if (a)
            oa = atomicAdd(g + 2u * s, a);
        if (b)
            ob = atomicAdd(g + 2u * shells + 2u * s, b);
        if (oa + a < oa)
            atomicAdd(g + 2u * s + 1u, 1ull);
        if (ob + b < ob)
            atomicAdd(g + 2u * shells + 2u * s + 1u, 1ull);
    }
}

/* The block of global sums this workgroup flushes into (LockArgs, PrecArgs). */
template <class Args>
__device__ __forceinline__ unsigned long long* lock_block(const Args& a)
{
    return a.work + (size_t)(blockIdx.x % a.copies) * (TMC_COHORT_COUNTERS + 4u * a.shells);
}

/* The end of a lockstep workgroup, called by all its threads: its sums and
 * counts go to its block, by one addition to a word.  (Additions to one word
 * take 7 to 16 ns each, whoever makes them: with a slot and counts a wave, 3e6
 * photons at default physics took 415 us to their first roulette and 76 to the
 * second, with one for eight waves 396 and 28.  Four waves: 2^26 photons 7.69
 * for 7.63 ms; sixteen, whose waves wait for one another at both ends: 7.79.)  `totals`: two zeroed words of LDS. */
template <class Args>
__device__ __forceinline__ void lock_end(const Args& a, unsigned long long* slot, unsigned long long* totals,
                                         uint64_t interactions, uint64_t truncated)
{
    if (__lane_id() == 0u) {
        atomicAdd(totals, (unsigned long long)interactions);
        if (truncated)
            atomicAdd(totals + 1, (unsigned long long)truncated);
    }
    __syncthreads();
    unsigned long long* const block = lock_block(a);
    if (slot)
        lock_flush<false>(slot, block + TMC_COHORT_COUNTERS, a.shells, threadIdx.x, blockDim.x);
    if (threadIdx.x < 2u && totals[threadIdx.x])
        atomicAdd(block + 1u + threadIdx.x, totals[threadIdx.x]);
}

/* The kernel's arguments where a path between two cycles uses them: read
 * through the argument block's pointer passed through an empty asm, so that
 * no load is hoisted into the step loop, whose scalar registers hold the
 * round keys. */
template <class Args>
__device__ __forceinline__ const Args& args_here()
{
    typedef const __attribute__((address_space(4))) Args* ConstArgs;
    ConstArgs p = (ConstArgs)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const Args*)p;
}

} // namespace tmc

#endif
