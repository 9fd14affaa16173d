// The cohort walk's rounds in LDS (tiny_mc_amd/csrc/tmc_cohort_rows.h), built
// with AddressSanitizer and UndefinedBehaviorSanitizer.  In one pass of the
// walk's loop every drawing wave reads the positions of its items of one round
// and writes the draws of its items of the round two later into the same
// buffer.  For every pair of round sizes and every number of drawing waves:
// every item lies in its array and no two items share a place; and where
// draws_wait() says that the writes need not wait for the other waves' reads,
// no wave writes a place that another one reads.
// Test infrastructure; prints "rounds_check: ok" at the end.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../tiny_mc_amd/csrc/tmc_cohort_rows.h"

#define CHECK(c)                                                                   \
    do {                                                                           \
        if (!(c)) {                                                                \
            std::fprintf(stderr, "rounds_check: %s:%d: %s\n", __FILE__, __LINE__, #c); \
            std::exit(1);                                                          \
        }                                                                          \
    } while (0)

namespace {

// Place -> the wave that takes it (-1: none), for a round of 2^lg photons.
std::vector<int> owners(uint32_t lg, uint32_t drawing)
{
    std::vector<int> own(TMC_COHORT_ARRAY, -1);
    for (uint32_t wave = 0; wave < drawing; ++wave)
        for (uint32_t j = 0; j < TMC_COHORT_WAVE_ROWS; ++j)
            for (uint32_t lane = 0; lane < 64u; ++lane) {
                const uint32_t at = tmc::item_of(wave * TMC_COHORT_WAVE_ROWS + j, lane, lg);
                CHECK(at < TMC_COHORT_ARRAY && own[at] < 0);
                own[at] = (int)wave;
            }
    return own;
}

} // namespace

int main()
{
    uint32_t shared = 0; // pairs of sizes whose waves take each other's places
    for (uint32_t drawing = 1; drawing <= TMC_COHORT_ROWS / TMC_COHORT_WAVE_ROWS; ++drawing)
        for (uint32_t prev = 0; prev <= 6u; ++prev) {
            const std::vector<int> read = owners(prev, drawing);
            for (uint32_t next = 0; next <= 6u; ++next) {
                const std::vector<int> write = owners(next, drawing);
                bool race = false;
                for (uint32_t at = 0; at < TMC_COHORT_ARRAY; ++at)
                    race |= read[at] >= 0 && write[at] >= 0 && read[at] != write[at];
                CHECK(!race || tmc::draws_wait(prev, next));
                shared += race;
            }
        }
    CHECK(shared > 0);
    std::puts("rounds_check: ok");
    return 0;
}
