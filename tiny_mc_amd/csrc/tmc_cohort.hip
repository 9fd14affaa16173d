/* The walk of a parameter set by workgroups that carry a cohort of photons
 * in lockstep.
 *
 * In the reference's arithmetic the weight is a function of the absorption
 * count k alone (photon.c:32, 45-49), so photons launched together reach
 * every roulette at the same k, and between two roulettes none of them ends.
 * Nor does anything a photon draws depend on where it is: the step length and
 * direction of absorption k are functions of (photon, k).  Only the positions
 * are a chain, of three FMAs per absorption.  A workgroup therefore walks a
 * cohort of up to 64 photons through T absorptions at a time (a round), in
 * three stages:
 *   draw    (photon, k) -> step length and next direction, any order: the
 *           Philox block, the log, square root, sine and cosine; spread over
 *           the workgroup's drawing waves, 64 (photon, k) pairs a row;
 *   move    the positions, one lane per photon, k after k: one wave (the
 *           mover), which leaves the squared radii;
 *   tally   (photon, k) -> shell, and the weight's images added to the LDS
 *           sums; spread over the drawing waves again.
 * The stages of three successive rounds run at once, with one barrier per
 * round, and a second where the round to be drawn lays its items out otherwise
 * than the one to be tallied, whose buffer it takes.  At a roulette the
 * survivors (a tenth) are packed into the low lanes and go on as a smaller
 * cohort, whose rows then hold several k per wave.
 *
 * What bounds it: the movers' chain, 23 cycles an absorption (a lane that does
 * a whole step by itself takes 740), plus 900 cycles a round to schedule it;
 * with 32 and more photons a cohort, the vector and scalar issue of the
 * drawing waves (16 waves a compute unit, about 3800 cycles a round of 24
 * rows).  Measured on MI355X, whole calls, lane per photon -> this walk: 20
 * photons at default physics 77 -> 22 us, 32,768 173 -> 48 us; 4096 at albedo
 * 0.99 (720 absorptions each) 1147 -> 54 us; 16,384 photons at albedo 0.9999
 * through 20,000 absorptions 1.9 ms, 1.7e11 absorptions/s.
 *
 * Same words, same operations and the same integer sums as step(): results
 * are bit-identical.
 */
#include "tmc_cohort.h"
#include "tmc_cohort_rows.h"
#include "tmc_device.h"
#include "tmc_internal.h"
#include "tmc_math.h"
#include "tmc_philox.h"
#include "tmc_step.h"

namespace tmc {

/* Copies of the overflow shell's sums per workgroup, as walk_f32. */
#define TMC_COHORT_HOT 8u
static_assert(TMC_COHORT_HOT <= TMC_CHECK_HOT, "the shell check covers every overflow copy");

__host__ __device__ __forceinline__ size_t cohort_tally_words(uint32_t shells)
{
    return 2u * ((size_t)shells - 1u + TMC_COHORT_HOT);
}

/* Floats of a hand-over of the movers' state at a roulette: position and
 * direction, three coordinates of 64 photons. */
#define TMC_COHORT_STATE (2u * 3u * 64u)

/* LDS bytes: the weight table (where the kernel builds it), the tallies, two
 * rounds, two hand-overs, the survivor masks, the cuts, and the table
 * builder's words. */
__host__ __device__ __forceinline__ size_t cohort_lds_bytes_of(uint32_t shells, uint32_t entries)
{
    return 16u * (size_t)entries + cohort_tally_words(shells) * 8u + 2u * TMC_COHORT_ROUND * 4u
        + 2u * TMC_COHORT_STATE * 4u + 2u * 8u + 4u * TMC_COHORT_CUTS + 16u;
}

size_t cohort_lds_bytes(uint32_t shells, uint32_t entries) { return cohort_lds_bytes_of(shells, entries); }

/* ------------------------------------------------------------------------ */
/* the weight table of a set: its weights come from the host, which walks the
 * serial recurrence W[k+1] = RN(W[k] a) (tmc::weight_sequence) in 1.3 ns an
 * absorption, where one lane takes 20 to 30                                  */
/* ------------------------------------------------------------------------ */

/* A table entry: the images of w and w*w, low words first. */
typedef uint32_t Images __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Images images_of(float w)
{
    const uint64_t h = fx_heat(w), h2 = fx_heat2(w);
    return Images{ (uint32_t)h, (uint32_t)(h >> 32), (uint32_t)h2, (uint32_t)(h2 >> 32) };
}

/* Converts a set's weights (host memory) to table entries in device memory,
 * for the runs whose table does not fit the LDS or is read by several
 * launches, and clears a run's counters. */
__global__ void __launch_bounds__(256) cohort_table(const float* weight, uint32_t n, Images* entry, uint32_t* counter,
                                                    uint32_t counters, unsigned long long* start)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n)
        entry[i] = images_of(weight[i]);
    if (i < counters)
        counter[i] = 0u;
    if (i == 0u && start)
        *start = __builtin_amdgcn_s_memrealtime();
}

/* ------------------------------------------------------------------------ */
/* the walk                                                                  */
/* ------------------------------------------------------------------------ */

namespace {

/* One round: T absorptions k0 .. k0 + T - 1 of P photons, in rows of 64
 * (photon, k) items, item (kk << lg) + p for photon p and absorption
 * k0 + kk.  Wave-uniform, and the same in every wave of the workgroup. */
struct Round {
    uint32_t k0, T, lg, P, flags;
    uint32_t at; /* the cohort's first photon in the list */
    uint64_t base; /* photon index of the cohort's first photon */
};

enum : uint32_t {
    R_VALID = 1u,
    R_FRESH = 2u, /* the cohort starts here */
    R_CUT = 4u, /* the last absorption is followed by the roulette */
    R_CAP = 8u, /* the photons stop after the last absorption */
    R_LAST = 16u, /* the table's last cut: survivors leave the cohort */
    R_PACKED = 32u, /* the first round after a roulette */
};

/* Smallest lg with 2^lg >= p (1 <= p <= 64). */
__device__ __forceinline__ uint32_t ceil_log2(uint32_t p) { return p <= 1u ? 0u : 32u - (uint32_t)__builtin_clz(p - 1u); }

/* Step length and direction of one absorption from its Philox words. */
template <uint32_t MATH>
__device__ __forceinline__ float4 draw_analytic(const tmc_u32x4& r)
{
    const float t = step_length<MATH>(r.x0);
    const float mu = tmc_u11(r.x1);
    const float s = sin_polar<MATH>(mu);
    float sn, cs;
    sincos_turn<MATH>(r.x2, &sn, &cs);
    return make_float4(t, mu, s * cs, s * sn);
}

/* The same with the rejection sampler: attempt 1 from words 1-2 of block
 * (k, 0), attempts 2b and 2b + 1 from block (k, b), as step_core. */
template <uint32_t MATH>
__device__ __forceinline__ float4 draw_rejection(const tmc_u32x4& r, uint32_t k, const tmc_philox_photon& pp,
                                                 const Physics& ph)
{
    const float t = step_length<MATH>(r.x0);
    float xi1 = tmc_u11(r.x1), xi2 = tmc_u11(r.x2);
    float tt = __builtin_fmaf(xi2, xi2, xi1 * xi1);
    bool accept = tt <= 1.0f && tt > 0.0f;
    uint32_t att = 1u;
    while (!accept) {
        const tmc_u32x4 q = tmc_philox4x32_10_blockb(k, (att + 1u) >> 1, pp, &ph.keys, ph.key0, ph.key1);
        xi1 = tmc_u11(q.x0);
        xi2 = tmc_u11(q.x1);
        tt = __builtin_fmaf(xi2, xi2, xi1 * xi1);
        ++att;
        accept = (tt <= 1.0f && tt > 0.0f) || att >= 64u;
        if (!accept) {
            xi1 = tmc_u11(q.x2);
            xi2 = tmc_u11(q.x3);
            tt = __builtin_fmaf(xi2, xi2, xi1 * xi1);
            ++att;
            accept = (tt <= 1.0f && tt > 0.0f) || att >= 64u;
        }
    }
    const float u = __builtin_fmaf(2.0f, tt, -1.0f);
    const float s = 2.0f * sqrt_cr_walk(1.0f - tt); /* 1 - tt: 0 or >= 2^-24 */
    return make_float4(t, u, xi1 * s, xi2 * s);
}

/* Moves the workgroup's LDS sums into the global ones by atomic swaps (safe
 * while other waves add), words first, first + stride, ... */
__device__ __forceinline__ void cohort_flush(unsigned long long* lds, unsigned long long* g, uint32_t shells,
                                             uint32_t first, uint32_t stride)
{
    const uint32_t last = shells - 1;
    for (uint32_t q = first; q < last + TMC_COHORT_HOT; q += stride) {
        const unsigned long long a = atomicExch(&lds[2 * q], 0ull);
        const unsigned long long b = atomicExch(&lds[2 * q + 1], 0ull);
        const uint32_t s = q < last ? q : last;
        /* both atomics in flight before either's carry is looked at */
        unsigned long long oa = 0, ob = 0;
        if (a)
            oa = atomicAdd(g + 2 * s, a);
        if (b)
            ob = atomicAdd(g + 2 * shells + 2 * s, b);
        if (oa + a < oa)
            atomicAdd(g + 2 * s + 1, 1ull);
        if (ob + b < ob)
            atomicAdd(g + 2 * shells + 2 * s + 1, 1ull);
    }
}

__device__ __forceinline__ uint64_t load_agent(unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void store_agent(unsigned long long* p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* The end of a run: called by every thread of a workgroup.  A workgroup
 * moves its LDS sums into one of `copies` blocks of global words (4 counters,
 * then the sums), with atomics; spread so, because additions to one word
 * from many compute units wait for one another (256 workgroups on one block:
 * 40 us).  The workgroup that finishes last of all adds the blocks up, leaves
 * zeros behind (the next run needs no clearing), and writes the result to
 * the host's memory, its token last: the host reads the result as soon as it
 * sees the token, with no copy queued behind the kernel.  A lone workgroup
 * writes its result as it is.  `flag`: a word of LDS; `flushed`: the
 * workgroup has moved sums into the block before (the same in every thread:
 * there are barriers on either side of the branch). */
__device__ __forceinline__ void finish_run(const CohortArgs& a, unsigned long long* lds, uint32_t* flag, bool counts,
                                           uint64_t interactions, uint64_t truncated, bool flushed)
{
    const uint32_t words = 4u * a.shells, block = TMC_COHORT_COUNTERS + words;
    unsigned long long* const mine = a.work + (size_t)(blockIdx.x % a.copies) * block;
    ulonglong2* const out = (ulonglong2*)(a.out + TMC_COHORT_COUNTERS);
    __syncthreads();
    if (a.finish && !a.list.photon && gridDim.x == 1 && !flushed) {
        const uint32_t last = a.shells - 1u;
        for (uint32_t s = threadIdx.x; s < a.shells; s += blockDim.x) {
            unsigned long long h = lds[2u * s], h2 = lds[2u * s + 1u];
            if (s == last) {
                for (uint32_t c = 1; c < TMC_COHORT_HOT; ++c) {
                    h += lds[2u * (s + c)];
                    h2 += lds[2u * (s + c) + 1u];
                }
            }
            out[s] = ulonglong2{ h, 0ull };
            out[a.shells + s] = ulonglong2{ h2, 0ull };
        }
        if (counts) {
            a.out[1] = interactions;
            a.out[2] = truncated;
            a.out[3] = __builtin_amdgcn_s_memrealtime() - *(volatile unsigned long long*)(flag + 2);
        }
    } else {
        cohort_flush(lds, mine + TMC_COHORT_COUNTERS, a.shells, threadIdx.x, blockDim.x);
        if (counts) {
            atomicAdd(mine + 1, (unsigned long long)interactions);
            if (truncated)
                atomicAdd(mine + 2, (unsigned long long)truncated);
        }
        /* agent-scope atomics: once they have completed, the count may
         * follow (a release fence would write the L2 back, once a wave: 20 us
         * a workgroup) */
        if (!a.finish)
            return;
        wait_vmem();
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t c = blockIdx.x % a.copies;
            const unsigned long long of = (gridDim.x - c + a.copies - 1u) / a.copies; /* workgroups of this copy */
            bool last = __hip_atomic_fetch_add(mine, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1ull == of;
            if (last)
                last = __hip_atomic_fetch_add(a.work + 3, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1ull
                    == (gridDim.x < a.copies ? gridDim.x : a.copies);
            *flag = last;
        }
        __syncthreads();
        if (!*flag)
            return;
        for (uint32_t i = threadIdx.x; i < block / 2u; i += blockDim.x) {
            unsigned long long lo = 0, hi = 0;
            constexpr uint32_t U = 8u; /* copies whose loads are in flight */
            for (uint32_t c = 0; c < a.copies; c += U) {
                unsigned long long l[U], h[U];
#pragma unroll
                for (uint32_t j = 0; j < U; ++j) {
                    unsigned long long* p = a.work + (size_t)(c + j < a.copies ? c + j : c) * block + 2u * i;
                    l[j] = load_agent(p);
                    h[j] = load_agent(p + 1);
                }
#pragma unroll
                for (uint32_t j = 0; j < U; ++j) {
                    if (c + j < a.copies) {
                        unsigned long long* p = a.work + (size_t)(c + j) * block + 2u * i;
                        if (i < TMC_COHORT_COUNTERS / 2u) {
                            /* (done, interactions), (truncated, blocks done) */
                            lo += l[j];
                            hi += h[j];
                        } else {
                            lo += l[j];
                            hi += h[j] + (lo < l[j]);
                        }
                        if (l[j] | h[j]) {
                            store_agent(p, 0ull);
                            store_agent(p + 1, 0ull);
                        }
                    }
                }
            }
            if (i == 0u)
                a.out[1] = hi;
            else if (i == 1u)
                a.out[2] = lo;
            else
                out[i - TMC_COHORT_COUNTERS / 2u] = ulonglong2{ lo, hi };
        }
        if (threadIdx.x == 0)
            a.out[3] = __builtin_amdgcn_s_memrealtime() - (a.start ? *a.start : *(volatile unsigned long long*)(flag + 2));
    }
    wait_vmem(); /* every thread's result words before the token */
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(a.out, (unsigned long long)a.token, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

} // namespace

/* Deposits between two flushes of the LDS sums: a word takes fewer than
 * 2^20 of at most 2^43 each, so it stays below 2^63. */
#define TMC_COHORT_FLUSH (1u << 20)

namespace {

/* Moves one coordinate of one photon through T absorptions: t[i], d[i] are
 * the step length and the next direction of absorption i, and d[i] becomes the
 * coordinate after its step.  Blocks of four, three of them on their way from
 * LDS; reads past the T absorptions stay in the workgroup's LDS and are not
 * used.  (A chain step is an FMA of 8 cycles; with two single reads and a
 * write an absorption it took 28, the LDS instructions of a lone wave
 * issuing every 11.) */
__device__ __forceinline__ void move_chain(float& x, float& u, const float4* t, float4* d, uint32_t T)
{
    constexpr uint32_t D = 4u; /* blocks in registers */
    float4 tt[D], dd[D];
#pragma unroll
    for (uint32_t i = 0; i < D - 1u; ++i) {
        tt[i] = t[i];
        dd[i] = d[i];
    }
    const uint32_t full = T / 4u;
    auto one = [&](float ti, float& di) {
        x = __builtin_fmaf(ti, u, x);
        u = di;
        di = x;
    };
    uint32_t b = 0;
    while (b + D <= full) {
#pragma unroll
        for (uint32_t i = 0; i < D; ++i) {
            tt[(i + D - 1u) % D] = t[b + i + D - 1u];
            dd[(i + D - 1u) % D] = d[b + i + D - 1u];
            one(tt[i].x, dd[i].x);
            one(tt[i].y, dd[i].y);
            one(tt[i].z, dd[i].z);
            one(tt[i].w, dd[i].w);
            d[b + i] = dd[i];
        }
        b += D;
    }
    /* up to D - 1 blocks more, the last one partial */
    const uint32_t left = T - 4u * b;
#pragma unroll
    for (uint32_t i = 0; i < D; ++i) {
        if (4u * i < left) {
            if (i == D - 1u) {
                tt[i] = t[b + i];
                dd[i] = d[b + i];
            }
            one(tt[i].x, dd[i].x);
            if (4u * i + 1u < left)
                one(tt[i].y, dd[i].y);
            if (4u * i + 2u < left)
                one(tt[i].z, dd[i].z);
            if (4u * i + 3u < left)
                one(tt[i].w, dd[i].w);
            d[b + i] = dd[i];
        }
    }
}

} // namespace

/* Weights a round adds to a table built in LDS: read one round, converted
 * the next. */
#define TMC_COHORT_AHEAD 256u

namespace {

/* LDS of a workgroup. */
struct CohortLds {
    Images* built; /* the weight table, where the kernel builds it */
    unsigned long long* tally;
    float *rounds, *states;
    unsigned long long* surv;
    uint32_t *cuts, *flag; /* flag: finish_run's word, then the start time */
    __device__ __forceinline__ CohortLds(unsigned long long* words, uint32_t shells, uint32_t build)
    {
        built = (Images*)words;
        tally = words + 2u * (size_t)build;
        rounds = (float*)(tally + cohort_tally_words(shells));
        states = rounds + 2u * TMC_COHORT_ROUND;
        surv = (unsigned long long*)(states + 2u * TMC_COHORT_STATE);
        cuts = (uint32_t*)(surv + 2);
        flag = cuts + TMC_COHORT_CUTS;
    }
};

/* What a workgroup walks: the cohorts first, first + stride, ... of `photons`
 * photons, at `place` of the list if there is one. */
struct CohortTask {
    uint32_t group, stride, photons, place;
};

/* What a wave counts (the first mover's counts are the workgroup's). */
struct CohortCounts {
    uint64_t interactions, truncated;
    uint64_t idle; /* lanes of the rows without an absorption (batches) */
    bool flushed; /* sums have been moved to `tally` (in every wave alike) */
};

/* Walks a task's cohorts.  a.cut is in LDS (l.cuts); a.build: the weigher's
 * first weights are in `weights`. */
template <uint32_t SAMPLER, uint32_t MATH, bool BATCH>
__device__ __forceinline__ void walk_cohorts(const CohortArgs& a, const PhotonList& list, CohortTask task,
                                             const CohortLds& l,
                                             unsigned long long* tally, float (&weights)[TMC_COHORT_AHEAD / 64u],
                                             CohortCounts& counts)
{
    Images* const built = l.built;
    unsigned long long* const lds = l.tally;
    float *const rounds = l.rounds, *const states = l.states;
    unsigned long long* const surv = l.surv;
    const uint32_t* const cuts = l.cuts;
    const uint32_t lane = __lane_id();
    const uint32_t wave = rfl32(threadIdx.x >> 6);
    const uint32_t drawing = a.drawing;
    const bool weigher = wave >= drawing + a.moving;
    const uint32_t ncuts = a.ncuts;
    uint32_t weighed = 0;

    Physics phys = {};
    phys.albedo = a.albedo;
    phys.spm = a.spm;
    phys.shell_max = a.shell_max;
    phys.key0 = (uint32_t)a.seed;
    phys.key1 = (uint32_t)(a.seed >> 32);
    set_derived(phys);
    const LaneTally lt = { lds, tally_fmax(a.shell_max, lane & (TMC_COHORT_HOT - 1)), ~0ull };

    /* the schedule: every wave steps the same one */
    const bool listed = list.photon != nullptr;
    uint32_t group = task.group; /* next cohort */
    const uint32_t photons = task.photons, place = task.place;
    const uint32_t groups = (photons + a.group - 1u) / a.group;
    Round prev = {}, cur = {}, next = {};
    bool alive = false;
    uint32_t k = 0, seg = 0, cut = 0, P = 0, lg = 0, par = 0;
    uint64_t base = 0;
    uint32_t since_flush = 0;

    /* the lane's photon (offset in its cohort) and, drawing waves, its part
     * of the generator and the images of the lane's item of the round being
     * moved; movers: one coordinate of one photon */
    uint32_t pid = 0;
    tmc_philox_photon pp = {};
    constexpr uint32_t M = TMC_COHORT_WAVE_ROWS;
    Images image[M], image_next[M];
#pragma unroll
    for (uint32_t j = 0; j < M; ++j)
        image[j] = image_next[j] = Images{ 0u, 0u, 0u, 0u };
    float x = 0.0f, u = 0.0f;

    for (;;) {
        /* positions of the lane's item of the previous round, on their way
         * while the next round is scheduled (a buffer serves the rounds of
         * one parity: next and prev) */
        float* const buffer = rounds + (par ^ 1u) * TMC_COHORT_ROUND;
        float px[M], py[M], pz[M];
        if (wave < drawing) {
#pragma unroll
            for (uint32_t j = 0; j < M; ++j) {
                const float* const item = buffer + item_of(wave * M + j, lane, prev.lg);
                px[j] = item[TMC_COHORT_ARRAY];
                py[j] = item[2u * TMC_COHORT_ARRAY];
                pz[j] = item[3u * TMC_COHORT_ARRAY];
            }
        }

        /* ---- schedule the next round ---- */
        uint64_t S = 0; /* photons of cur that outlive its end */
        const uint32_t pid_cur = pid;
        next.flags = next.T = 0;
        bool changed = false;
        if (cur.flags & (R_CUT | R_CAP)) {
            const uint64_t all = cur.P == 64u ? ~0ull : (1ull << cur.P) - 1ull;
            S = cur.flags & R_CUT ? rfl64(surv[par]) : all;
            if (cur.flags & R_CAP) {
                counts.truncated += (uint64_t)__popcll(S);
                S = 0;
            }
            const uint64_t go = cur.flags & R_LAST ? 0ull : S;
            P = rfl32((uint32_t)__popcll(go));
            alive = P != 0u;
            if (alive) {
                /* the survivors take the low lanes, in order */
                const uint32_t rank = mask_rank(go);
                const uint32_t dst = __builtin_amdgcn_inverse_ballot_w64(go) ? rank : P + (lane - rank);
                pid = __builtin_amdgcn_ds_permute((int)(dst * 4u), (int)pid);
                lg = ceil_log2(P);
                pid = __builtin_amdgcn_ds_bpermute((int)((lane & ((1u << lg) - 1u)) * 4u), (int)pid);
                ++seg;
                changed = true;
                next.flags = R_PACKED;
            }
        }
        if (!alive && group < groups) {
            const uint32_t off = group * a.group;
            P = rfl32(photons - off < a.group ? photons - off : a.group);
            lg = ceil_log2(P);
            pid = lane & ((1u << lg) - 1u);
            base = a.first_photon;
            k = 0;
            if (listed) {
                pid = list.photon[place + off + (pid < P ? pid : 0u)];
                k = rfl32(cuts[a.seg0 - 1u]);
            } else {
                base += off;
            }
            next.at = place + off;
            seg = a.seg0;
            group += task.stride;
            next.flags = R_FRESH;
            alive = true;
            changed = true;
        }
        if (changed) {
            cut = rfl32(cuts[seg]);
            const uint64_t photon = base + pid;
            pp = tmc_philox_photon_init((uint32_t)photon, (uint32_t)(photon >> 32), phys.key0, phys.key1);
        }
        if (alive) {
            /* entries the weigher has written by the time this round's images
             * are read, in the next round */
            const uint32_t known = a.build ? weighed + TMC_COHORT_AHEAD : ~0u;
            const uint32_t end = cut < a.kcap ? cut : a.kcap;
            const uint32_t most = (drawing * M) << (6u - lg), left = (end < known ? end : known) - k;
            next.k0 = k;
            next.T = left < most ? left : most;
            next.lg = lg;
            next.P = P;
            next.base = base;
            next.flags |= R_VALID;
            k += next.T;
            if (k == end) {
                if (end == a.kcap)
                    next.flags |= R_CAP;
                if (end == cut)
                    next.flags |= R_CUT | (seg + 1u == ncuts ? R_LAST : 0u);
            }
        }
        if (!((next.flags | cur.flags | prev.flags) & R_VALID))
            break;
        /* (at a roulette and where a cohort of another size starts: two rounds
         * of a cycle) */
        if ((prev.flags & next.flags & R_VALID) && draws_wait(prev.lg, next.lg))
            __syncthreads();

        /* whether the drawing waves flush the sums in this round: counted by
         * every wave, since all of finish_run's threads go by counts.flushed */
        since_flush = rfl32(since_flush + prev.P * prev.T);
        const bool flush = since_flush >= TMC_COHORT_FLUSH - 64u * TMC_COHORT_ROWS;
        if (flush) {
            since_flush = 0;
            counts.flushed = true;
        }

        if (wave < drawing) {
            /* ---- the images of the current round's items ---- */
            if (cur.flags & R_VALID) {
#pragma unroll
                for (uint32_t j = 0; j < M; ++j) {
                    const uint32_t kk = ((wave * M + j) << (6u - cur.lg)) + (lane >> cur.lg);
                    const uint32_t at = cur.k0 + (kk < cur.T ? kk : cur.T - 1u);
                    image_next[j] = a.build ? built[at] : ((const Images*)a.entry)[at];
                }
            }
            /* ---- tally the previous round ---- */
            if (prev.flags & R_VALID) {
                const uint32_t p = lane & ((1u << prev.lg) - 1u);
#pragma unroll
                for (uint32_t j = 0; j < M; ++j) {
                    const uint32_t kk = ((wave * M + j) << (6u - prev.lg)) + (lane >> prev.lg);
                    if (kk < prev.T && p < prev.P) {
                        const float r2 =
                            __builtin_fmaf(pz[j], pz[j], __builtin_fmaf(py[j], py[j], px[j] * px[j]));
                        const uint32_t q = shell_index(r2, phys, lt.fmax);
                        tally_add<false>(lt, q, ((uint64_t)image[j].y << 32) | image[j].x,
                                         ((uint64_t)image[j].w << 32) | image[j].z);
                    }
                }
                if (flush)
                    cohort_flush(lds, tally, a.shells, wave * 64u + lane, drawing * 64u);
            }
            /* ---- draw the next round (lanes past its items draw unused ones) ---- */
            if (next.flags & R_VALID) {
#pragma unroll
                for (uint32_t j = 0; j < M; ++j) {
                    const uint32_t row_k = (wave * M + j) << (6u - next.lg), kk = row_k + (lane >> next.lg);
                    const tmc_u32x4 r = tmc_philox4x32_10_block0_r2(next.k0 + kk, pp, phys.keys);
                    const float4 d = SAMPLER == 1u ? draw_rejection<MATH>(r, next.k0 + kk, pp, phys)
                                                   : draw_analytic<MATH>(r);
                    float* const item = buffer + item_of(wave * M + j, lane, next.lg);
                    item[0] = d.x;
                    item[TMC_COHORT_ARRAY] = d.y;
                    item[2u * TMC_COHORT_ARRAY] = d.z;
                    item[3u * TMC_COHORT_ARRAY] = d.w;
                    const uint32_t last = next.T - 1u - row_k; /* the last item's place in this row */
                    if ((next.flags & R_CUT) && last < (64u >> next.lg)) {
                        const uint64_t m = __ballot(r.x3 < TMC_ROULETTE_KILL_R) >> (last << next.lg);
                        if (lane == 0)
                            surv[par ^ 1u] = next.P == 64u ? m : m & ((1ull << next.P) - 1ull);
                    }
                }
            }
#pragma unroll
            for (uint32_t j = 0; j < M; ++j)
                image[j] = image_next[j];
        } else if (weigher) {
#pragma unroll
            for (uint32_t i = 0; i < TMC_COHORT_AHEAD / 64u; ++i) {
                const uint32_t e = weighed + 64u * i + lane;
                if (e < a.entries)
                    built[e] = images_of(weights[i]);
                weights[i] = e + TMC_COHORT_AHEAD < a.entries ? a.weight[e + TMC_COHORT_AHEAD] : 0.0f;
            }
        } else if (cur.flags & R_VALID) {
            /* ---- move through the current round: lane m of the movers holds
             * coordinate m >> lg of photon m & (2^lg - 1) ---- */
            const uint32_t m = (wave - drawing) * 64u + lane;
            const uint32_t c = m >> cur.lg, p = m & ((1u << cur.lg) - 1u);
            const bool in = c < 3u && p < cur.P;
            const float* const from = states + (par ^ 1u) * TMC_COHORT_STATE;
            if (cur.flags & R_FRESH) {
                x = 0.0f;
                u = c == 2u ? 1.0f : 0.0f;
                if (listed && in) {
                    x = list.state[c][cur.at + p];
                    u = list.state[3u + c][cur.at + p];
                }
            } else if ((cur.flags & R_PACKED) && in) {
                x = from[c * 64u + p];
                u = from[(3u + c) * 64u + p];
            }
            if (wave == drawing) {
                counts.interactions += (uint64_t)cur.P * cur.T;
                if constexpr (BATCH) {
                    const uint32_t rows = (((cur.T - 1u) << cur.lg) >> 6) + 1u;
                    counts.idle += 64ull * rows - (uint64_t)cur.P * cur.T;
                }
            }
            if (in) {
                const float* const t = rounds + par * TMC_COHORT_ROUND + p * row_floats(cur.lg);
                move_chain(x, u, (const float4*)t, (float4*)(t + (1u + c) * TMC_COHORT_ARRAY), cur.T);
                /* the survivors' state, for the lanes they move to */
                if ((S >> p) & 1u) {
                    float* const to = states + par * TMC_COHORT_STATE;
                    const uint32_t rank = (uint32_t)__popcll(S & ((1ull << p) - 1ull));
                    to[c * 64u + rank] = x;
                    to[(3u + c) * 64u + rank] = u;
                }
            }
        }
        __syncthreads();
        if (cur.flags & R_LAST) {
            /* photons that outlive the table (one run in a thousand or
             * fewer) walk on by themselves */
            if (S != 0 && wave == drawing) {
                const float* const from = states + par * TMC_COHORT_STATE;
                const uint32_t rank = mask_rank(S);
                bool live = __builtin_amdgcn_inverse_ballot_w64(S);
                Photon ph;
                launch_photon(ph, cur.base + pid_cur, phys.key0, phys.key1);
                if (live) {
                    ph.x = from[rank];
                    ph.y = from[64u + rank];
                    ph.z = from[128u + rank];
                    ph.u = from[192u + rank];
                    ph.v = from[256u + rank];
                    ph.w = from[320u + rank];
                    ph.k = cur.k0 + cur.T;
                    ph.weight = a.w_end;
                }
                while (__ballot(live) != 0) {
                    const uint32_t n = (uint32_t)__popcll(__ballot(live && absorbs<SAMPLER>(ph)));
                    counts.interactions += n;
                    if constexpr (BATCH)
                        counts.idle += 64u - n;
                    if (live)
                        live = step<SAMPLER, MATH>(ph, phys, lt);
                    counts.truncated += (uint64_t)__popcll(__ballot(live && ph.k >= a.kcap));
                    live = live && ph.k < a.kcap;
                }
            }
        }
        prev = cur;
        cur = next;
        par ^= 1u;
        weighed += TMC_COHORT_AHEAD;
    }
}

} // namespace

template <uint32_t SAMPLER, uint32_t MATH>
__global__ void __launch_bounds__(1024) walk_cohort(CohortArgs a)
{
    extern __shared__ unsigned long long lds_words[];
    const CohortLds l(lds_words, a.shells, a.build);

    const uint32_t lane = __lane_id();
    const uint32_t wave = rfl32(threadIdx.x >> 6);
    const uint32_t drawing = a.drawing; /* waves 0 .. drawing - 1 draw and tally, then come the movers */
    const bool weigher = wave >= drawing + a.moving;
    if (threadIdx.x == 0)
        *(unsigned long long*)(l.flag + 2) = __builtin_amdgcn_s_memrealtime();

    for (uint32_t i = threadIdx.x; i < cohort_tally_words(a.shells); i += blockDim.x)
        l.tally[i] = 0;
    if (threadIdx.x < TMC_COHORT_CUTS)
        l.cuts[threadIdx.x] = a.cut[threadIdx.x];
    /* the weigher's next weights, on their way from the host's memory */
    float weights[TMC_COHORT_AHEAD / 64u];
    if (weigher) {
#pragma unroll
        for (uint32_t i = 0; i < TMC_COHORT_AHEAD / 64u; ++i)
            weights[i] = 64u * i + lane < a.entries ? a.weight[64u * i + lane] : 0.0f;
    }
    __syncthreads();

    CohortTask task = { blockIdx.x, gridDim.x, (uint32_t)a.photons, 0u };
    if (a.list.photon) {
        /* (at least as many workgroups as stripes, or one stripe) */
        const uint32_t stripe = blockIdx.x % a.stripes;
        const uint32_t n = a.list_count[stripe * TMC_LOCK_LINE];
        task.photons = rfl32(n < a.list_cap ? n : a.list_cap);
        task.place = stripe * a.list_cap;
        task.group = blockIdx.x / a.stripes;
        task.stride = (gridDim.x - stripe + a.stripes - 1u) / a.stripes;
    }
    unsigned long long* const tally =
        a.work + (size_t)(blockIdx.x % a.copies) * (TMC_COHORT_COUNTERS + 4u * a.shells) + TMC_COHORT_COUNTERS;
    CohortCounts counts = { 0, 0, 0, false };
    /* the movers' chain is what a round waits for */
    if (wave >= drawing && !weigher)
        __builtin_amdgcn_s_setprio(3);
    walk_cohorts<SAMPLER, MATH, false>(a, a.list, task, l, tally, weights, counts);
    finish_run(a, l.tally, l.flag, wave == drawing && lane == 0, counts.interactions, counts.truncated, counts.flushed);
}

/* One workgroup: adds up the sums that other launches left in a.work, and
 * hands the result over. */
__global__ void __launch_bounds__(1024) finish_kernel(CohortArgs a)
{
    extern __shared__ unsigned long long lds_words[];
    for (uint32_t i = threadIdx.x; i < cohort_tally_words(a.shells); i += blockDim.x)
        lds_words[i] = 0;
    uint32_t* const flag = (uint32_t*)(lds_words + cohort_tally_words(a.shells));
    finish_run(a, lds_words, flag, false, 0, 0, true);
}

/* Waves that draw and that move in a workgroup of a batch: cohorts of 64. */
#define TMC_COHORT_SETS_MOVING 3u
#define TMC_COHORT_SETS_DRAWING 13u

/* The rest of a batch's photons, from their a.level-th roulette to the end:
 * each workgroup claims a run of at most 64 places of a set's part of the
 * list, walks the photons there as one cohort, and adds its sums to the
 * set's. */
template <uint32_t MATH>
__global__ void __launch_bounds__(1024) walk_cohort_sets(LockSetArgs a)
{
    extern __shared__ unsigned long long lds_words[];
    const CohortLds l(lds_words, a.shells_max, 0u);
    const uint32_t lane = __lane_id();
    const uint32_t wave = rfl32(threadIdx.x >> 6);
    for (uint32_t i = threadIdx.x; i < cohort_tally_words(a.shells_max); i += blockDim.x)
        l.tally[i] = 0;
    CohortCounts counts = { 0, 0, 0, false };
    float weights[TMC_COHORT_AHEAD / 64u] = {};
    const uint32_t in = a.level - 1u;
    if (wave >= TMC_COHORT_SETS_DRAWING)
        __builtin_amdgcn_s_setprio(3);
    for (;;) {
        __syncthreads(); /* the last task's flush, and its claim's readers */
        if (threadIdx.x == 0) {
            /* the next chunk with photons in it */
            uint32_t got, n = 0;
            do {
                got = atomicAdd(a.cursor, 1u);
                if (got < a.nchunks) {
                    const LockChunk& ch = a.chunks[got];
                    const uint32_t cap = a.sets[ch.set].cap[in], filled = a.in_count[ch.set * TMC_LOCK_LINE];
                    n = filled < cap ? filled : cap;
                    n = ch.first < n ? n - ch.first : 0u;
                    n = n < ch.count ? n : ch.count;
                }
            } while (got < a.nchunks && n == 0u);
            l.flag[0] = got;
            l.flag[1] = n;
        }
        __syncthreads();
        const uint32_t got = rfl32(l.flag[0]), n = rfl32(l.flag[1]);
        if (got >= a.nchunks)
            break;
        const LockChunk& ch = a.chunks[got];
        const LockSet& s = a.sets[rfl32(ch.set)];
        const CohortHead& h = a.heads[s.head];
        if (threadIdx.x < TMC_COHORT_CUTS)
            l.cuts[threadIdx.x] = h.cut[threadIdx.x];
        CohortArgs c = {};
        c.seed = rfl64(s.seed);
        c.first_photon = rfl64(s.first_photon);
        c.albedo = s.albedo;
        c.spm = s.spm;
        c.shell_max = s.shell_max;
        c.shells = rfl32(s.shells);
        c.kcap = ~0u;
        c.group = 64u;
        c.drawing = TMC_COHORT_SETS_DRAWING;
        c.moving = TMC_COHORT_SETS_MOVING;
        c.entry = (const Images*)a.entry + rfl64(s.entry);
        c.ncuts = rfl32(h.ncuts);
        c.w_end = h.w_end;
        c.seg0 = a.level;
        unsigned long long* const tally = a.tally + rfl64(s.tally);
        __syncthreads();
        walk_cohorts<0u, MATH, true>(c, a.in, { 0u, 1u, n, s.place[in] + ch.first }, l, tally, weights, counts);
        __syncthreads();
        cohort_flush(l.tally, tally, c.shells, threadIdx.x, blockDim.x);
    }
    if (wave == TMC_COHORT_SETS_DRAWING && lane == 0) {
        atomicAdd(a.counters + 1, (unsigned long long)counts.interactions);
        atomicAdd(a.counters + 4, (unsigned long long)counts.idle);
        if (counts.truncated)
            atomicAdd(a.counters + 2, (unsigned long long)counts.truncated);
    }
}

/* The weight table of a set: one lane walks the recurrence W[k+1] = RN(W[k] a),
 * 64 absorptions at a time, and four waves make images of the 256 before.
 * (The chain is a multiplication of 9 cycles an absorption, 4 ns; handing 64 at
 * a time over cost 6 ns an absorption more.  On the host it is 1.3 ns, but for
 * one set after the other.) */
#define TMC_WEIGH_BLOCK 256u

__global__ void __launch_bounds__(64u + TMC_WEIGH_BLOCK) weigh_sets(const LockSet* sets, CohortHead* heads,
                                                                    Images* pool)
{
    __shared__ float4 weights[2][TMC_WEIGH_BLOCK / 4u];
    __shared__ uint32_t valid[2]; /* weights of the block; fewer than it holds: none follow */
    const LockSet& s = sets[blockIdx.x];
    if (s.cuts == 0u)
        return;
    CohortHead& h = heads[s.head];
    Images* const entry = pool + s.entry;
    const float a = s.albedo;
    const uint32_t cuts = s.cuts, entries = s.entries;
    float w = 1.0f;
    uint32_t n = 0;
    for (uint32_t k = 0, par = 0;; k += TMC_WEIGH_BLOCK, par ^= 1u) {
        if (threadIdx.x == 0) {
            uint32_t done = 0;
            while (done < TMC_WEIGH_BLOCK && n < cuts && k + done < entries) {
                const uint32_t left = entries - k - done, room = left < 64u ? left : 64u;
                float4* const out = weights[par] + done / 4u;
                float v = w;
#pragma unroll
                for (uint32_t i = 0; i < 16u; ++i) {
                    float4 q;
                    q.x = v;
                    q.y = q.x * a;
                    q.z = q.y * a;
                    q.w = q.z * a;
                    v = q.w * a;
                    out[i] = q;
                }
                if (v < 0.001f) {
                    /* a roulette among them (the weight never grows between two) */
                    v = w;
                    for (uint32_t i = 0; i < room && n < cuts; ++i) {
                        ((float*)out)[i] = v;
                        v = v * a;
                        if (v < 0.001f) {
                            v = v / 0.1f;
                            h.cut[n++] = k + done + i + 1u;
                        }
                    }
                }
                w = v;
                done += room;
            }
            valid[par] = done;
        }
        /* the block before, on the other side of the barrier */
        const uint32_t i = threadIdx.x - 64u;
        if (k != 0u && threadIdx.x >= 64u && i < valid[par ^ 1u])
            entry[k - TMC_WEIGH_BLOCK + i] = images_of(((const float*)weights[par ^ 1u])[i]);
        __syncthreads();
        if (valid[par] == 0u)
            break;
    }
    if (threadIdx.x == 0) {
        h.ncuts = n;
        h.w_end = w;
    }
}

namespace {

using CohortKernel = void (*)(CohortArgs);

using SetsKernel = void (*)(LockSetArgs);

CohortKernel cohort_kernel(uint32_t sampler, uint32_t math)
{
    if (math == TMC_MATH_OWN)
        return sampler ? walk_cohort<1u, TMC_MATH_OWN> : walk_cohort<0u, TMC_MATH_OWN>;
    return sampler ? walk_cohort<1u, TMC_MATH_HARDWARE> : walk_cohort<0u, TMC_MATH_HARDWARE>;
}

} // namespace

hipError_t launch_cohort_table(const float* weight, uint32_t n, void* entry, uint32_t* counter, uint32_t counters,
                               unsigned long long* start, hipStream_t stream)
{
    const uint32_t most = n > counters ? n : counters;
    hipLaunchKernelGGL(cohort_table, dim3((most + 255u) / 256u), dim3(256), 0, stream, weight, n, (Images*)entry,
                       counter, counters, start);
    return hipGetLastError();
}

hipError_t launch_cohort(uint32_t sampler, uint32_t math, const CohortArgs& a, uint32_t grid, uint32_t block,
                         hipStream_t stream)
{
    hipLaunchKernelGGL(cohort_kernel(sampler, math), dim3(grid), dim3(block), cohort_lds_bytes_of(a.shells, a.build),
                       stream, a);
    return hipGetLastError();
}

hipError_t launch_finish(const CohortArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL(finish_kernel, dim3(1), dim3(1024), cohort_tally_words(a.shells) * 8u + 16u, stream, a);
    return hipGetLastError();
}

hipError_t launch_cohort_sets(uint32_t math, const LockSetArgs& a, uint32_t grid, hipStream_t stream)
{
    const SetsKernel k = math == TMC_MATH_OWN ? walk_cohort_sets<TMC_MATH_OWN> : walk_cohort_sets<TMC_MATH_HARDWARE>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(64u * (TMC_COHORT_SETS_DRAWING + TMC_COHORT_SETS_MOVING)),
                       cohort_lds_bytes_of(a.shells_max, 0u), stream, a);
    return hipGetLastError();
}

hipError_t launch_weigh_sets(const LockSet* sets, uint32_t nsets, CohortHead* heads, void* entry, hipStream_t stream)
{
    hipLaunchKernelGGL(weigh_sets, dim3(nsets), dim3(64u + TMC_WEIGH_BLOCK), 0, stream, sets, heads, (Images*)entry);
    return hipGetLastError();
}

} // namespace tmc
