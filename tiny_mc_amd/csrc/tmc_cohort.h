/* Interface between the host side and the cohort walk (tmc_cohort.hip). */
#ifndef TMC_COHORT_H
#define TMC_COHORT_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tmc {

/* Roulettes a weight table spans at most. */
#define TMC_COHORT_CUTS 30u
/* Roulettes the weight table of n photons spans: three more than the last of
 * them is expected to survive, so that one run in a thousand has a photon that
 * outlives it (and walks on without the table). */
inline uint32_t cuts_for(double n)
{
    uint32_t cuts = 3;
    for (; n >= 1.0 && cuts < TMC_COHORT_CUTS; n *= 0.1)
        ++cuts;
    return cuts;
}
/* Entries of the largest weight table the workgroups build in LDS, each for
 * itself; a longer one is converted once, by a launch ahead (8 us, where 256
 * workgroups reading 8 KB each from the host's memory take 25). */
#define TMC_COHORT_BUILD 512u
/* Counter words of a block of sums, and of the result. */
#define TMC_COHORT_COUNTERS 4u

/* Photons between two roulettes: index in the slice, position and direction. */
struct PhotonList {
    uint32_t* photon;
    float* state[6]; /* x, y, z, then the direction */
};

/* A parameter set of a batch, or a part of its photons, as the set kernels
 * read it.  The photons' high index word is one for all of them. */
struct LockSet {
    uint64_t seed; /* Philox key */
    uint64_t first_photon; /* stream index of its photon 0 */
    uint64_t tally; /* word offset of the set's 4*shells sums */
    uint64_t entry; /* offset of the set's weight table, in entries */
    float albedo, spm, shell_max; /* as WalkArgs */
    uint32_t shells;
    uint32_t head; /* the set's CohortHead */
    uint32_t entries, cuts; /* room of the weight table, and roulettes wanted (0: an earlier part builds it) */
    uint32_t place[2], cap[2]; /* its places in the two survivor lists */
    uint32_t pad;
};
static_assert(sizeof(LockSet) == 80, "LockSet layout");

/* The roulettes of a set's weight table, built on the device: the i-th follows
 * absorption cut[i] - 1; w_end is the weight with which a survivor of the last
 * one goes on. */
struct CohortHead {
    uint32_t ncuts;
    float w_end;
    uint32_t cut[TMC_COHORT_CUTS];
};

/* Photons first .. first + count - 1 of a set (level 0), or of its places in
 * the list of its level. */
struct LockChunk {
    uint32_t set, first, count, pad;
};

/* One level of a batch: sets, queue, and what the launches of a run share. */
struct LockSetArgs {
    const LockSet* sets;
    const CohortHead* heads;
    const void* entry; /* pool of pairs of images */
    const LockChunk* chunks;
    uint32_t nchunks;
    uint32_t cus;
    uint32_t* cursor; /* of this launch */
    uint32_t level; /* roulettes the photons of the queue have survived */
    uint32_t shells_max;
    PhotonList in, out; /* level > 0: the survivors of `level` roulettes; a lock level: those of one more */
    const uint32_t* in_count; /* photons appended to a set's places, TMC_LOCK_LINE words apart */
    uint32_t* out_count;
    unsigned long long* tally; /* tally pool */
    unsigned long long* counters; /* [1] interactions, [2] truncated (TMC_LOCK_OVERFLOW), [4] idle lane-steps */
};

struct CohortArgs {
    uint64_t seed; /* Philox key */
    uint64_t first_photon; /* photon index of cohort 0's first photon */
    uint64_t photons; /* photons in this launch */
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
    uint32_t ncuts; /* roulettes the table spans: the i-th follows absorption cut[i] - 1, and cut[ncuts - 1] = entries
                       (past the cap: ~0u, and entries = kcap) */
    uint32_t cut[TMC_COHORT_CUTS];
    float w_end; /* the weight with which a survivor of the last one goes on */
    uint32_t copies; /* copies of the sums the workgroups flush into */
    /* cohorts from a list (list.photon not null) of photons first_photon + i
     * after their seg0-th roulette, instead of first_photon, first_photon + 1, ... */
    PhotonList list;
    const uint32_t* list_count; /* photons of each stripe of the list (LockArgs), or more if it overflowed */
    uint32_t list_cap, stripes, seg0;
    uint32_t finish; /* this launch ends the run: result to `out` */
    const unsigned long long* start; /* real-time ticks at the run's start; null: this launch's */
    uint64_t token; /* written to out[0] when the result is there */
    unsigned long long* work; /* `copies` blocks of 4 counters ([0] workgroups done, [1] interactions, [2] truncated,
                                 [3] of the first: blocks done) and 4*shells words of 128-bit sums (lo, hi); zero
                                 before and after the run */
    unsigned long long* out; /* host memory: token, interactions, truncated, 100 MHz ticks, the sums */
};

size_t cohort_lds_bytes(uint32_t shells, uint32_t entries);

/* Words between two stripes' counts: a cache line. */
#define TMC_LOCK_LINE 16u
/* Parts of a slice the waves claim from: workgroup b, on XCD b mod 8, claims
 * from part b mod 8. */
#define TMC_LOCK_RANGES 8u

/* Set in a block's truncated photons when a list had no room for a survivor:
 * the run is repeated by the other walk.  (The lists hold an eighth of a stripe's
 * photons and a slack, where a tenth survive: never seen.) */
#define TMC_LOCK_OVERFLOW (1ull << 56)

/* One level of a large run (walk_lock): the photons of a slice, or of the list
 * the level before left, from absorption k0 to k1. */
struct LockArgs {
    uint64_t seed; /* Philox key */
    uint64_t first_photon; /* index of the slice's photon 0 */
    float albedo, spm, shell_max; /* as WalkArgs */
    uint32_t shells;
    uint32_t kcap; /* stop a photon after kcap absorptions */
    uint32_t chunk; /* level 0: photons a wave claims at a time, a multiple of 64, from one of TMC_LOCK_RANGES parts of
                       `range` photons (a multiple of 64 too); 0: the batches go round the waves */
    uint32_t range;
    uint32_t* cursor; /* claims, TMC_LOCK_LINE words apart */
    uint32_t level; /* 0: the slice's photons, else the list's */
    uint32_t photons; /* of the slice (< 2^31) */
    uint32_t k0, k1;
    uint32_t cut_ends, cap_ends; /* whether k1 is a roulette, and the cap */
    const void* entry; /* table of pairs of images, at least two entries beyond k1 */
    /* the lists and their counts are split into stripes, workgroup b reading
     * and appending to stripe b mod `stripes`, of in_cap and out_cap places;
     * counts TMC_LOCK_LINE words apart */
    uint32_t stripes;
    PhotonList in, out;
    const uint32_t* in_count;
    uint32_t* out_count;
    uint32_t in_cap, out_cap;
    uint32_t copies;
    unsigned long long* work; /* as CohortArgs */
};

/* Threads of walk_lock's workgroups, at most. */
#define TMC_LOCK_BLOCK 512u
size_t lock_lds_bytes(uint32_t sampler, uint32_t shells, uint32_t block);
/* LDS of a workgroup that counts the photons of each shell and absorption. */
size_t lock_count_bytes(uint32_t shells, uint32_t absorptions);
/* Resident workgroups of TMC_LOCK_BLOCK threads per CU of walk_lock (counted: the absorptions that are
 * counted by shell, 0: none). */
hipError_t lock_occupancy(uint32_t sampler, uint32_t math, uint32_t counted, uint32_t shells, int* wg_per_cu);
hipError_t launch_lock(uint32_t sampler, uint32_t math, bool counted, const LockArgs& a, uint32_t grid, uint32_t block,
                       hipStream_t stream);

/* The same for the sets of a batch: a level by lockstep waves (0 or 1), and
 * the survivors of a.level roulettes by cohorts, to their end.  Analytic
 * sampler, no cap. */
hipError_t lock_sets_occupancy(uint32_t math, uint32_t block, uint32_t shells_max, int* wg_per_cu);
hipError_t launch_lock_sets(uint32_t math, const LockSetArgs& a, uint32_t grid, uint32_t block, hipStream_t stream);
hipError_t launch_cohort_sets(uint32_t math, const LockSetArgs& a, uint32_t grid, hipStream_t stream);
/* Builds the weight tables of nsets sets. */
hipError_t launch_weigh_sets(const LockSet* sets, uint32_t nsets, CohortHead* heads, void* entry, hipStream_t stream);

/* ---- the precision variants (tmc_lock_prec.hip) ---- */

/* Weight table of a precision variant: cuts as CohortArgs. */
struct PrecHead {
    uint32_t ncuts, pad;
    double w_end;
    uint32_t cut[TMC_COHORT_CUTS];
};

/* A list of photons between two roulettes: index in the slice, and the words of
 * position and direction, word w of place i at state[w * places + i]. */
struct PrecList {
    uint32_t *photon, *state;
    uint32_t places;
};

/* Words of a photon's position and direction. */
__host__ __device__ constexpr uint32_t prec_words(uint32_t precision)
{
    return precision == 3u ? 12u : precision == 2u ? 9u : 6u;
}

/* One launch of a run with a precision variant's arithmetic: the photons of a
 * slice, or of the list the launch before left, through `cycles` roulettes
 * (0: to their end). */
struct PrecArgs {
    uint64_t seed; /* Philox key */
    uint64_t first_photon; /* index of the slice's photon 0 */
    double albedo_d, spm_d; /* as WalkArgs */
    float l2a_hi, l2a_lo, l2s_hi, l2s_lo, spm_w, shell_max;
    uint32_t shells;
    uint32_t level, cycles; /* roulettes survived so far (0: the slice's photons), and to come */
    uint32_t photons; /* of the slice (< 2^31) */
    PrecHead* head;
    void* entry; /* pairs of images, at least one entry beyond the last cut */
    uint32_t entries, cuts; /* room of the table (binary64: its weights), and roulettes wanted */
    const double* weight; /* binary64: host memory, the weights and the table's head */
    const PrecHead* host_head;
    uint32_t stripes; /* of the lists, as LockArgs */
    PrecList in, out;
    const uint32_t* in_count;
    uint32_t* out_count;
    uint32_t in_cap, out_cap;
    uint32_t copies;
    unsigned long long* work; /* as CohortArgs */
};

hipError_t prec_occupancy(uint32_t sampler, uint32_t precision, uint32_t block, uint32_t shells, int* wg_per_cu);
/* Builds the weight table, zeroes `counters` 32-bit words at `counter` and
 * notes the real time at *start. */
hipError_t launch_prec_table(uint32_t precision, const PrecArgs& a, uint32_t* counter, uint32_t counters,
                             unsigned long long* start, hipStream_t stream);
hipError_t launch_prec(uint32_t sampler, uint32_t precision, const PrecArgs& a, uint32_t grid, uint32_t block,
                       hipStream_t stream);
/* Ends a run whose launches have left their sums in a.work (shells, copies,
 * work, start, token and out of CohortArgs). */
hipError_t launch_finish(const CohortArgs& a, hipStream_t stream);

/* Converts n weights (host memory) to table entries of 16 bytes, zeroes
 * `counters` 32-bit words at `counter`, and notes the real time at *start
 * (null: neither). */
hipError_t launch_cohort_table(const float* weight, uint32_t n, void* entry, uint32_t* counter, uint32_t counters,
                               unsigned long long* start, hipStream_t stream);
hipError_t launch_cohort(uint32_t sampler, uint32_t math, const CohortArgs& a, uint32_t grid, uint32_t block,
                         hipStream_t stream);

} // namespace tmc

#endif
