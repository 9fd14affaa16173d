/* Interface between the host side and the cohort walk (tmc_cohort.hip). */
#ifndef TMC_COHORT_H
#define TMC_COHORT_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tmc {

/* Roulettes a weight table spans at most. */
#define TMC_COHORT_CUTS 30u
/* Entries of the largest weight table the workgroups build in LDS, each for
 * itself; a longer one is converted once, by a launch ahead (8 us, where 256
 * workgroups reading 8 KB each from the host's memory take 25). */
#define TMC_COHORT_BUILD 512u
/* Counter words of a block of sums, and of the result. */
#define TMC_COHORT_COUNTERS 4u
/* Rows of 64 items a drawing wave takes of a round, and the rows a round holds
 * at most. */
#ifndef TMC_COHORT_WAVE_ROWS
#define TMC_COHORT_WAVE_ROWS 2u
#endif
#define TMC_COHORT_ROWS (16u * TMC_COHORT_WAVE_ROWS)

struct CohortArgs {
    uint64_t seed; /* Philox key */
    uint64_t first_photon; /* photon index of cohort 0's first photon */
    uint64_t photons; /* photons in this launch */
    uint32_t groups; /* cohorts: ceil(photons / group) */
    float albedo, spm, shell_max; /* as WalkArgs */
    uint32_t shells;
    uint32_t kcap; /* stop a photon after kcap absorptions */
    uint32_t group; /* photons a cohort starts with (power of two, <= 64) */
    uint32_t drawing; /* waves that draw and tally (<= TMC_COHORT_ROWS / TMC_COHORT_WAVE_ROWS) */
    uint32_t moving; /* waves that move: 3 * group lanes */
    uint32_t build; /* room for the weight table in LDS, in entries (one more wave fills it); 0: it is at `entry` */
    uint32_t entries; /* weights of the table */
    const float* weight; /* host memory: the weight deposited at absorption k < entries */
    const void* entry; /* device memory: the same as pairs of images, where build is 0 */
    uint32_t ncuts; /* roulettes the table spans: the i-th follows absorption cut[i] - 1, and cut[ncuts - 1] = entries */
    uint32_t cut[TMC_COHORT_CUTS];
    float w_end; /* the weight with which a survivor of the last one goes on */
    uint32_t copies; /* copies of the sums the workgroups flush into */
    uint64_t token; /* written to out[0] when the result is there */
    unsigned long long* work; /* `copies` blocks of 4 counters ([0] workgroups done, [1] interactions, [2] truncated,
                                 [3] of the first: blocks done) and 4*shells words of 128-bit sums (lo, hi); zero
                                 before and after the run */
    unsigned long long* out; /* host memory: token, interactions, truncated, 100 MHz ticks, the sums */
};

size_t cohort_lds_bytes(uint32_t shells, uint32_t entries);

/* Converts n weights (host memory) to table entries of 16 bytes. */
hipError_t launch_cohort_table(const float* weight, uint32_t n, void* entry, hipStream_t stream);
hipError_t launch_cohort(uint32_t sampler, uint32_t math, const CohortArgs& a, uint32_t grid, uint32_t block,
                         hipStream_t stream);

} // namespace tmc

#endif
