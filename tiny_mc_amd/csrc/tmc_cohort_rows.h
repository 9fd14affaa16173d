/* Where the cohort walk (tmc_cohort.hip) keeps a round's items in LDS: shared
 * by the kernel and the host's checks of it. */
#ifndef TMC_COHORT_ROWS_H
#define TMC_COHORT_ROWS_H

#include <stdint.h>

#include "tmc_philox.h" /* TMC_HD */

/* Rows of 64 items a drawing wave takes of a round, and the rows a round holds
 * at most. */
#ifndef TMC_COHORT_WAVE_ROWS
#define TMC_COHORT_WAVE_ROWS 2u
#endif
#define TMC_COHORT_ROWS (16u * TMC_COHORT_WAVE_ROWS)

/* A round's items: four arrays (step length, then direction x, y, z, which the
 * movers overwrite with the position), in each a row of absorptions per photon,
 * so that a mover reads and writes four absorptions at a time.  Rows are padded
 * by four floats: 16 lanes' rows then start in 16 different groups of banks. */
#define TMC_COHORT_ARRAY (64u * (TMC_COHORT_ROWS + 4u))
#define TMC_COHORT_ROUND (4u * TMC_COHORT_ARRAY)

namespace tmc {

/* Floats of a photon's row in a round of 2^lg photons. */
TMC_HD uint32_t row_floats(uint32_t lg) { return (TMC_COHORT_ROWS << (6u - lg)) + 4u; }

/* Place of lane `lane` of row `row` in a round's arrays: absorption
 * row (64 >> lg) + (lane >> lg) of photon lane & (2^lg - 1). */
TMC_HD uint32_t item_of(uint32_t row, uint32_t lane, uint32_t lg)
{
    return (lane & ((1u << lg) - 1u)) * row_floats(lg) + (row << (6u - lg)) + (lane >> lg);
}

/* Whether the draws of a round of 2^next_lg photons have to wait until every
 * wave has read the positions of the round of 2^prev_lg photons that the same
 * buffer held: a wave's items are its own words again only if both rounds lay
 * them out alike. */
TMC_HD bool draws_wait(uint32_t prev_lg, uint32_t next_lg) { return prev_lg != next_lg; }

} // namespace tmc

#endif
