/* Large binary32 runs with the analytic sampler: waves that carry 64 photons
 * in lockstep from one roulette to the next.
 *
 * Photons launched together reach every roulette at the same absorption
 * (tmc_cohort.hip), so a wave that launches 64 photons at once walks them
 * through a whole cycle with one absorption count: no lane ends on the way,
 * nothing is compared, refilled or masked, and what depends on the count
 * alone leaves the vector unit.  Rounds 1 and 2 of the generator's half that
 * holds the count are scalar (three 32 x 32 products fewer a step), and the
 * weight's images come from the set's table by one load of a single address.
 * At the roulette the tenth that survives is appended to a list in device
 * memory, which the next launch walks through the next cycle, again 64 at a
 * time; when few are left the cohort walk takes the list to its end.
 *
 * What bounds it: vector issue.  66 instructions an absorption of 64 photons
 * (76 in walk_f32), of which the 16 products take 4.6 cycles each on a full
 * SIMD, the 15 three-input XORs, conversions and compares 4.1, the five
 * transcendentals 8, and the additions and multiplications of three vector
 * registers 2.2 (4 with a scalar operand).  Measured on MI355X, whole calls,
 * walk_f32 -> this walk: 2^20 photons at default physics 425 -> 190 us,
 * 3,000,017 638 -> 436 us, 2^26 8.72 -> 7.63 ms; 2^17 at albedo 0.99 1218 -> 257
 * us, at 0.9999 117 -> 22 ms; 2^27 at albedo 0.5 2842 -> 2497 us.
 *
 * Where a first cycle's counts fit LDS (absorptions times shells), a workgroup
 * counts the photons of each (absorption, shell) instead of adding their images:
 * one 32-bit addition for two of 64 bits, and no loads of the table, whose
 * images come in once, when the counts are added up.  2% of a large run
 * (2^30 photons at default physics 126.6 -> 123.9 ms): the LDS additions are
 * not what a step waits for.
 *
 * With the rejection sampler a step is 133 vector instructions, a third
 * of them the second generator block of the quarter of the directions that
 * are drawn again: 2^17 photons at default physics 304 -> 94 us, 2^24 4.24 ->
 * 3.43 ms, 2^20 at albedo 0.99 4.97 -> 2.43 ms.
 *
 * Same words, same operations and the same integer sums as step(): results
 * are bit-identical.
 */
#include "tmc_cohort.h"
#include "tmc_device.h"
#include "tmc_lock_device.h"
#include "tmc_math.h"
#include "tmc_philox.h"
#include "tmc_step.h"

namespace tmc {

/* Absorptions the rejection sampler's waves walk at a time, and the LDS words
 * of the directions they draw again. */
#define TMC_LOCK_GROUP 4u
#define TMC_LOCK_RETRIES (64u * TMC_LOCK_GROUP)

/* LDS of a workgroup: the sums, two totals, and the retries of each wave; or
 * (lock_count_bytes) the totals and the counts. */
size_t lock_lds_bytes(uint32_t sampler, uint32_t shells, uint32_t block)
{
    return 8u * (lock_slot_words(shells) + 2u + (sampler ? block / 64u * TMC_LOCK_RETRIES : 0u));
}

size_t lock_count_bytes(uint32_t shells, uint32_t absorptions)
{
    return 16u + 4ull * absorptions * (shells - 1ull + TMC_LOCK_HOT);
}

namespace {

/* Photon state of a lane. */
struct LockPhoton {
    float x, y, z, u, v, w;
    uint32_t x3; /* the last absorption's roulette word */
};

/* What a photon draws for one absorption. */
struct Drawn {
    float t, u, v, w; /* step length, then the direction it leaves with */
    uint32_t x3;
};

template <uint32_t MATH>
__device__ __forceinline__ Drawn lock_draw(uint32_t k, uint32_t c3k1, const tmc_philox_photon& pp,
                                           const Physics& phys)
{
    const tmc_u32x4 r = block0_uniform(k, c3k1, pp, phys.keys);
    Drawn d;
    d.t = step_length<MATH>(r.x0);
    d.u = tmc_u11(r.x1);
    const float s = sin_polar<MATH>(d.u);
    float sn, cs;
    sincos_turn<MATH>(r.x2, &sn, &cs);
    d.v = s * cs;
    d.w = s * sn;
    d.x3 = r.x3;
    return d;
}

/* Moves the photon by its direction and the step length of d, and takes d's
 * direction; returns the squared radius. */
__device__ __forceinline__ float lock_move(LockPhoton& p, const Drawn& d)
{
    p.x = __builtin_fmaf(d.t, p.u, p.x);
    p.y = __builtin_fmaf(d.t, p.v, p.y);
    p.z = __builtin_fmaf(d.t, p.w, p.z);
    p.u = d.u;
    p.v = d.v;
    p.w = d.w;
    p.x3 = d.x3;
    return __builtin_fmaf(p.z, p.z, __builtin_fmaf(p.y, p.y, p.x * p.x));
}

__device__ __forceinline__ void lock_add(const LaneTally& lt, uint32_t q, const Images& e)
{
    tally_add(lt, q, ((uint64_t)e.y << 32) | e.x, ((uint64_t)e.w << 32) | e.z);
}

/* Absorption k (wave-uniform) of every lane, its images in e. */
template <uint32_t MATH>
__device__ __forceinline__ void lock_step(LockPhoton& p, uint32_t k, uint32_t c3k1, const tmc_philox_photon& pp,
                                          const Physics& phys, const LaneTally& lt, const Images& e)
{
    const float r2 = lock_move(p, lock_draw<MATH>(k, c3k1, pp, phys));
    lock_add(lt, shell_index(r2, phys, lt.fmax), e);
}

/* Absorptions k and k + 1 up to the shells' pairs *qa and *qb: both draws ahead
 * of both moves, so that a wave has four independent chains of products to
 * issue from (with few waves on a SIMD the products' latency is what a step
 * costs). */
template <uint32_t MATH>
__device__ __forceinline__ void lock_walk2(LockPhoton& p, uint32_t k, uint32_t c3k1, const tmc_philox_photon& pp,
                                           const Physics& phys, float fmax, uint32_t* qa, uint32_t* qb)
{
    const Drawn a = lock_draw<MATH>(k, c3k1, pp, phys), b = lock_draw<MATH>(k + 1u, c3k1, pp, phys);
    const float ra = lock_move(p, a), rb = lock_move(p, b);
    bool sa, sb;
    float fa = shell_coord_short(ra, phys, fmax, &sa), fb = shell_coord_short(rb, phys, fmax, &sb);
    if (__builtin_expect(__ballot(!(sa && sb)) != 0, 0)) {
        fa = (float)shell_index(ra, phys, fmax);
        fb = (float)shell_index(rb, phys, fmax);
    }
    *qa = (uint32_t)fa;
    *qb = (uint32_t)fb;
}

template <uint32_t MATH>
__device__ __forceinline__ void lock_step2(LockPhoton& p, uint32_t k, uint32_t c3k1, const tmc_philox_photon& pp,
                                           const Physics& phys, const LaneTally& lt, const Images& e0,
                                           const Images& e1)
{
    uint32_t qa, qb;
    lock_walk2<MATH>(p, k, c3k1, pp, phys, lt.fmax, &qa, &qb);
    lock_add(lt, qa, e0);
    lock_add(lt, qb, e1);
}

/* The wave's photons from their launch to absorption k1, counted: `row` holds
 * a count for every pair and absorption, `pairs` to an absorption. */
template <uint32_t MATH>
__device__ __forceinline__ void lock_cycle_counted(LockPhoton& p, uint32_t k1, uint32_t c3k1,
                                                   const tmc_philox_photon& pp, const Physics& phys,
                                                   const LaneTally& lt, uint32_t* row, uint32_t pairs)
{
    uint32_t k = 0;
    for (; k + 2u <= k1; k += 2u, row += 2u * pairs) {
        uint32_t qa, qb;
        lock_walk2<MATH>(p, k, c3k1, pp, phys, lt.fmax, &qa, &qb);
        if (__builtin_amdgcn_inverse_ballot_w64(lt.deposit)) {
            atomicAdd(row + qa, 1u);
            atomicAdd(row + pairs + qb, 1u);
        }
    }
    if (k != k1) {
        const float r2 = lock_move(p, lock_draw<MATH>(k, c3k1, pp, phys));
        const uint32_t q = shell_index(r2, phys, lt.fmax);
        if (__builtin_amdgcn_inverse_ballot_w64(lt.deposit))
            atomicAdd(row + q, 1u);
    }
}

/* Adds a workgroup's counts, each times its absorption's images, to a block of
 * the global sums.  A pair's absorptions go to four threads, or to one for each
 * 32: every thread adds to the pair's words, and additions to one word take 7 to
 * 16 ns each.  (With all threads at work on few shells 2^22 photons at default
 * physics took 1994 us with one shell, 1354 with 8 and 884 with 24; so they take
 * 782, 607 and 593, and 581 with 101 either way.) */
__device__ __forceinline__ void count_flush(const uint32_t* counts, const Images* entry, uint32_t k1,
                                            unsigned long long* g, uint32_t shells)
{
    const uint32_t last = shells - 1u, pairs = last + TMC_LOCK_HOT;
    const uint32_t most = k1 / 32u > 4u ? k1 / 32u : 4u, room = pairs < blockDim.x ? blockDim.x / pairs : 1u;
    const uint32_t parts = room < most ? room : most; /* threads to a pair */
    for (uint32_t i = threadIdx.x; i < pairs * parts; i += blockDim.x) {
        const uint32_t q = i % pairs;
        unsigned __int128 h = 0, h2 = 0;
        for (uint32_t k = i / pairs; k < k1; k += parts) {
            const uint32_t n = counts[k * pairs + q];
            const Images e = entry[k];
            h += (unsigned __int128)(((uint64_t)e.y << 32) | e.x) * n;
            h2 += (unsigned __int128)(((uint64_t)e.w << 32) | e.z) * n;
        }
        const uint32_t s = q < last ? q : last;
        for (uint32_t w = 0; w < 2u; ++w) {
            const unsigned __int128 v = w ? h2 : h;
            if (v == 0)
                continue;
            unsigned long long* const at = g + 2u * (w * shells + s);
            const unsigned long long lo = (unsigned long long)v, old = atomicAdd(at, lo);
            const unsigned long long hi = (unsigned long long)(v >> 64) + (old + lo < old);
            if (hi)
                atomicAdd(at + 1, hi);
        }
    }
}

/* Orders a wave's LDS accesses across its lanes (the LDS serves them in the
 * order of the instructions). */
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* Absorptions k .. k + G - 1 with the rejection sampler (photon.c:34-43), as
 * step_core makes its attempts: the first from words 1-2 of block (k, 0),
 * attempts 2b and 2b + 1 from block (k, b).  Of 64 lanes some always reject
 * (14 on average), so the (photon, absorption) pairs of G absorptions whose
 * first attempt fails are gathered, through LDS, into as few passes over a
 * further block as hold them: 55 pairs for G = 4, one pass with its lanes
 * nearly full, and a second for the twentieth part that fails again.
 * `images`: the table's entry of absorption k. */
template <uint32_t MATH, uint32_t G>
__device__ __forceinline__ void lock_group_rejection(LockPhoton& p, uint32_t k, uint32_t hi, uint32_t plo,
                                                     const tmc_philox_photon& pp, const Physics& phys,
                                                     const LaneTally& lt, const char* images, uint32_t zero,
                                                     unsigned long long* retries)
{
    float t[G], a[G], b[G];
    uint32_t at[G]; /* the lane's pair j among the gathered */
    uint64_t again[G];
    uint32_t n = 0;
#pragma unroll
    for (uint32_t j = 0; j < G; ++j) {
        const tmc_u32x4 r = block0_uniform(k + j, hi ^ phys.key1, pp, phys.keys);
        t[j] = step_length<MATH>(r.x0);
        a[j] = tmc_u11(r.x1);
        b[j] = tmc_u11(r.x2);
        if (j == G - 1u)
            p.x3 = r.x3;
        const float tt = __builtin_fmaf(b[j], b[j], a[j] * a[j]);
        again[j] = lt.deposit & ~__ballot(tt <= 1.0f && tt > 0.0f);
        at[j] = n + mask_rank(again[j]);
        n += (uint32_t)__popcll(again[j]);
        if (__builtin_amdgcn_inverse_ballot_w64(again[j]))
            retries[at[j]] = __lane_id() | j << 6;
    }
    n = rfl32(n);
    wave_order();
    for (uint32_t first = 0; first < n; first += 64u) {
        const uint32_t i = first + __lane_id();
        bool open = i < n;
        const uint32_t pair = open ? (uint32_t)retries[i] : 0u;
        const uint32_t from = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((pair & 63u) << 2), (int)plo);
        const tmc_philox_photon q = tmc_philox_photon_init(from, hi, phys.key0, phys.key1);
        float x = 0.0f, y = 0.0f;
        for (uint32_t block = 1u; __ballot(open) != 0; ++block) {
            const tmc_u32x4 r = tmc_philox4x32_10_blockb(k + (pair >> 6), block, q, &phys.keys, phys.key0, phys.key1);
            const float x0 = tmc_u11(r.x0), y0 = tmc_u11(r.x1), x1 = tmc_u11(r.x2), y1 = tmc_u11(r.x3);
            const float t0 = __builtin_fmaf(y0, y0, x0 * x0), t1 = __builtin_fmaf(y1, y1, x1 * x1);
            const bool ok0 = (t0 <= 1.0f && t0 > 0.0f) || block == 32u; /* (the 64th attempt is taken) */
            if (open) {
                x = ok0 ? x0 : x1;
                y = ok0 ? y0 : y1;
            }
            open = open && !(ok0 || (t1 <= 1.0f && t1 > 0.0f));
        }
        if (i < n)
            retries[i] = (uint64_t)__float_as_uint(y) << 32 | __float_as_uint(x);
    }
    wave_order();
    Images e[G];
#pragma unroll
    for (uint32_t j = 0; j < G; ++j)
        e[j] = *(const Images*)(images + 16u * j + zero);
    float r2[G];
#pragma unroll
    for (uint32_t j = 0; j < G; ++j) {
        if (__builtin_amdgcn_inverse_ballot_w64(again[j])) {
            const uint64_t xy = retries[at[j]];
            a[j] = __uint_as_float((uint32_t)xy);
            b[j] = __uint_as_float((uint32_t)(xy >> 32));
        }
        const float tt = __builtin_fmaf(b[j], b[j], a[j] * a[j]);
        Drawn d;
        d.t = t[j];
        d.u = __builtin_fmaf(2.0f, tt, -1.0f);
        const float s = 2.0f * sqrt_cr_walk(1.0f - tt); /* 1 - tt: 0 or >= 2^-24 */
        d.v = a[j] * s;
        d.w = b[j] * s;
        d.x3 = p.x3;
        r2[j] = lock_move(p, d);
    }
#pragma unroll
    for (uint32_t j = 0; j < G; ++j)
        lock_add(lt, shell_index(r2[j], phys, lt.fmax), e[j]);
}

/* lock_cycle with the rejection sampler. */
template <uint32_t MATH, class Flush>
__device__ __forceinline__ void lock_cycle_rejection(LockPhoton& p, uint32_t k0, uint32_t k1, const char* table,
                                                     uint32_t zero, uint32_t hi, uint32_t plo,
                                                     const tmc_philox_photon& pp, const Physics& phys,
                                                     const LaneTally& lt, unsigned long long* retries, uint32_t& room,
                                                     uint32_t every, const Flush& flush)
{
    constexpr uint32_t G = TMC_LOCK_GROUP;
    for (uint32_t k = k0; k != k1;) {
        const uint32_t left = k1 - k, n = rfl32(left < room ? left : room);
        room -= n;
        const char* from = table + 16ull * k;
        const uint32_t stop = k + n;
        for (; k + G <= stop; k += G, from += 16u * G)
            lock_group_rejection<MATH, G>(p, k, hi, plo, pp, phys, lt, from, zero, retries);
        for (; k != stop; ++k, from += 16u)
            lock_group_rejection<MATH, 1u>(p, k, hi, plo, pp, phys, lt, from, zero, retries);
        if (room == 0u) {
            flush();
            room = every;
        }
    }
}

/* The wave's photons from absorption k0 to k1 (lanes without one walk a stale
 * one, their deposits masked).  `table`: the set's weight table; `room`: steps
 * to the next flush of the slot, which `flush` does, `every` so many. */
template <uint32_t MATH, class Flush>
__device__ __forceinline__ void lock_cycle(LockPhoton& p, uint32_t k0, uint32_t k1, const char* table, uint32_t zero,
                                           uint32_t c3k1, const tmc_philox_photon& pp, const Physics& phys,
                                           const LaneTally& lt, uint32_t& room, uint32_t every, const Flush& flush)
{
    for (uint32_t k = k0; k != k1;) {
        const uint32_t left = k1 - k, n = rfl32(left < room ? left : room);
        room -= n;
        const char* from = table + 16ull * k;
        Images e0 = *(const Images*)(from + zero), e1 = *(const Images*)(from + 16u + zero);
        const uint32_t stop = k + (n & ~1u);
        for (; k != stop; k += 2u) {
            from += 32u;
            lock_step2<MATH>(p, k, c3k1, pp, phys, lt, e0, e1);
            e0 = *(const Images*)(from + zero);
            e1 = *(const Images*)(from + 16u + zero);
        }
        if (n & 1u) {
            lock_step<MATH>(p, k, c3k1, pp, phys, lt, e0);
            ++k;
        }
        if (room == 0u) {
            flush();
            room = every;
        }
    }
}

/* Loads the lane's photon from place i of a list; returns its index. */
__device__ __forceinline__ uint32_t lock_load(LockPhoton& p, const PhotonList& l, uint32_t i)
{
    p.x = l.state[0][i];
    p.y = l.state[1][i];
    p.z = l.state[2][i];
    p.u = l.state[3][i];
    p.v = l.state[4][i];
    p.w = l.state[5][i];
    return l.photon[i];
}

/* Appends the photons of the lanes in S (not empty), of index `off`, to the
 * `cap` places from `place` of a list; false if not all of them had room. */
__device__ __forceinline__ bool lock_append(uint64_t S, uint32_t off, const LockPhoton& p, const PhotonList& l,
                                            uint32_t* count, uint32_t place, uint32_t cap, uint32_t lane)
{
    const uint32_t n = (uint32_t)__popcll(S);
    uint32_t base = 0;
    if (lane == 0)
        base = atomicAdd(count, n);
    base = rfl32(base);
    const uint32_t to = base + mask_rank(S);
    if (__builtin_amdgcn_inverse_ballot_w64(S) && to < cap) {
        const uint32_t i = place + to;
        l.photon[i] = off;
        l.state[0][i] = p.x;
        l.state[1][i] = p.y;
        l.state[2][i] = p.z;
        l.state[3][i] = p.u;
        l.state[4][i] = p.v;
        l.state[5][i] = p.w;
    }
    return base + n <= cap;
}

} // namespace

/* (LockArgs must stay the only parameter: args_here) */
template <uint32_t SAMPLER, uint32_t MATH, bool COUNTED = false>
__global__ void __launch_bounds__(TMC_LOCK_BLOCK, SAMPLER ? 6 : 1) walk_lock(LockArgs a)
{
    extern __shared__ unsigned long long lds[];
    const uint32_t lane = __lane_id();
    const uint32_t wave = rfl32(threadIdx.x >> 6);
    unsigned long long *const totals = lds, *const slot = lds + 2;
    uint32_t* const counts = (uint32_t*)slot;
    const uint32_t pairs = a.shells - 1u + TMC_LOCK_HOT;
    for (uint32_t i = threadIdx.x; i < (COUNTED ? a.k1 * pairs : 4u * pairs); i += blockDim.x)
        counts[i] = 0u; /* (a pair of sums is four words) */
    if (threadIdx.x < 2u)
        totals[threadIdx.x] = 0ull;
    __syncthreads();

    Physics phys = {};
    phys.albedo = a.albedo;
    phys.spm = a.spm;
    phys.shell_max = a.shell_max;
    phys.key0 = (uint32_t)a.seed;
    phys.key1 = (uint32_t)(a.seed >> 32);
    set_derived<true>(phys);
    LaneTally lt = { slot, tally_fmax(a.shell_max, lane & (TMC_LOCK_HOT - 1u)), ~0ull };
    /* the photons' high index word is the launch's */
    const uint32_t c3k1 = (uint32_t)(a.first_photon >> 32) ^ phys.key1;
    const uint32_t k0 = a.k0, k1 = a.k1;
    /* images: loaded with a vector offset of zero, so that they arrive in the
     * registers the atomics want, and not through scalar ones */
    const char* const table = (const char*)a.entry;
    uint32_t zero = 0;
    asm volatile("" : "+v"(zero));

    /* photons of this level: the slice's, or this stripe's part of the list.
     * A stripe's counts and photons are those of one XCD's workgroups, and few
     * enough waves append to one count: additions to one address take 7 to
     * 16 ns each (with one count, albedo 0.5 ran at a tenth of the rate).
     * The batches of 64 go round the waves, which take about the same time for
     * one; where a wave has many of them, it claims a few at a time, from the
     * part of the slice of its XCD's waves (2^26 photons at default physics:
     * 8.6 ms round the waves, 8.2 claimed; 2^20: 0.22 and 0.37 ms). */
    const uint32_t stripe = blockIdx.x % a.stripes, waves_per_wg = blockDim.x >> 6;
    uint32_t photons = a.photons, place = 0, at = 64u * (blockIdx.x * waves_per_wg + wave),
             stride = 64u * waves_per_wg * gridDim.x, claimed = 0;
    const bool claims = a.chunk != 0u;
    if (a.level) {
        const uint32_t n = a.in_count[stripe * TMC_LOCK_LINE];
        photons = rfl32(n < a.in_cap ? n : a.in_cap);
        place = stripe * a.in_cap;
        at = 64u * (blockIdx.x / a.stripes * waves_per_wg + wave);
        stride = 64u * waves_per_wg * ((gridDim.x - stripe + a.stripes - 1u) / a.stripes);
    }
    uint64_t interactions = 0, truncated = 0;
    constexpr uint32_t every = lock_flush_steps(TMC_LOCK_BLOCK / 64u);
    uint32_t room = every; /* steps to the next flush */

    if (claims) {
        /* range of this XCD's claims; `claimed`: where the current one ends */
        const uint32_t x = blockIdx.x % TMC_LOCK_RANGES;
        place = x * a.range;
        photons = place >= a.photons ? 0u : a.photons - place < a.range ? a.photons - place : a.range;
        stride = 64u;
        at = 0;
    }
    for (;; at += stride) {
        if (claims && at >= claimed) {
            const LockArgs& c = args_here<LockArgs>();
            uint32_t got = 0;
            if (lane == 0)
                got = atomicAdd(c.cursor + blockIdx.x % TMC_LOCK_RANGES * TMC_LOCK_LINE, c.chunk);
            at = rfl32(got);
            claimed = at + c.chunk;
        }
        if (at >= photons)
            break;
        const uint64_t in = photons - at >= 64u ? ~0ull : (1ull << (photons - at)) - 1ull;
        lt.deposit = in;
        LockPhoton p = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f, ~0u };
        tmc_philox_photon pp;
        uint32_t plo; /* low index word */
        {
            const LockArgs& c = args_here<LockArgs>();
            uint32_t off = place + at + lane;
            if (c.level && __builtin_amdgcn_inverse_ballot_w64(in))
                off = lock_load(p, c.in, off);
            const uint64_t photon = c.first_photon + off;
            plo = (uint32_t)photon;
            pp = tmc_philox_photon_init((uint32_t)photon, (uint32_t)(photon >> 32), phys.key0, phys.key1);
        }
        const auto flush = [&]() {
            const LockArgs& c = args_here<LockArgs>();
            lock_flush<true>(slot, lock_block(c) + TMC_COHORT_COUNTERS, c.shells, lane, 64u);
        };
        if constexpr (COUNTED)
            lock_cycle_counted<MATH>(p, k1, c3k1, pp, phys, lt, counts, pairs);
        else if constexpr (SAMPLER == 1u)
            lock_cycle_rejection<MATH>(p, k0, k1, table, zero, c3k1 ^ phys.key1, plo, pp, phys, lt,
                                       slot + lock_slot_words(a.shells) + wave * TMC_LOCK_RETRIES, room, every, flush);
        else
            lock_cycle<MATH>(p, k0, k1, table, zero, c3k1, pp, phys, lt, room, every, flush);
        interactions += (uint64_t)__popcll(in) * (k1 - k0);
        const LockArgs& c = args_here<LockArgs>();
        uint64_t S = c.cut_ends ? in & __ballot(p.x3 < TMC_ROULETTE_KILL_R) : in;
        if (c.cap_ends) {
            truncated += (uint64_t)__popcll(S);
            S = 0;
        }
        if (S != 0) {
            uint32_t off = place + at + lane;
            if (c.level && __builtin_amdgcn_inverse_ballot_w64(S))
                off = c.in.photon[off];
            if (!lock_append(S, off, p, c.out, c.out_count + stripe * TMC_LOCK_LINE, stripe * c.out_cap, c.out_cap, lane)
                && lane == 0)
                atomicOr(lock_block(c) + 2, TMC_LOCK_OVERFLOW);
        }
    }
    const LockArgs& c = args_here<LockArgs>();
    lock_end(c, COUNTED ? nullptr : slot, totals, interactions, truncated);
    if constexpr (COUNTED)
        count_flush(counts, (const Images*)c.entry, c.k1, lock_block(c) + TMC_COHORT_COUNTERS, c.shells);
}

/* A level of a batch: each wave claims chunks of the queue, each a run of
 * photons of one set, longest first, and moves its slot's sums into the set's
 * when the next chunk is of another set.
 *
 * A wave's first chunk is its own: the queue in rows of a wave for every SIMD,
 * every second row backwards, since a row's first workgroup sits beside the
 * first of the others, and with all rows forwards the SIMDs with the longest
 * chunk had the longest of each row (a batch of 64 sets, 17,000 batches of
 * photons for 6144 waves: 2.60 and 2.25 ms).  (LockSetArgs must stay the only
 * parameter: args_here) */
template <uint32_t MATH>
__global__ void __launch_bounds__(256) walk_lock_sets(LockSetArgs a)
{
    extern __shared__ unsigned long long lds[];
    const uint32_t lane = __lane_id();
    const uint32_t wave = rfl32(threadIdx.x >> 6);
    unsigned long long *const totals = lds, *const slot = lds + 2u + wave * lock_slot_words(a.shells_max);
    for (uint32_t i = lane; i < lock_slot_words(a.shells_max); i += 64u)
        slot[i] = 0;
    if (threadIdx.x < 2u)
        totals[threadIdx.x] = 0ull;
    __syncthreads();
    uint32_t zero = 0;
    asm volatile("" : "+v"(zero));

    Physics phys = {};
    LaneTally lt = { slot, 0.0f, ~0ull };
    uint32_t set = ~0u, k0 = 0, k1 = 0, hi = 0;
    const char* table = nullptr;
    uint64_t interactions = 0, idle = 0;
    constexpr uint32_t every = lock_flush_steps(1u);
    uint32_t room = every;
    const uint32_t waves_per_wg = blockDim.x >> 6;
    bool begun = false;
    auto flush = [&]() {
        const LockSetArgs& c = args_here<LockSetArgs>();
        const LockSet& s = c.sets[set];
        lock_flush<false>(slot, c.tally + s.tally, s.shells, lane, 64u);
    };

    for (;;) {
        uint32_t first, count;
        {
            const LockSetArgs& c = args_here<LockSetArgs>();
            uint32_t got = 0;
            if (begun) {
                if (lane == 0)
                    got = atomicAdd(c.cursor, 1u);
                got = rfl32(got) + gridDim.x * waves_per_wg;
                if (got >= c.nchunks)
                    break;
            } else {
                begun = true;
                const uint32_t row = blockIdx.x / c.cus, left = gridDim.x - row * c.cus;
                const uint32_t n = waves_per_wg * (left < c.cus ? left : c.cus); /* waves of this row */
                const uint32_t i = waves_per_wg * (blockIdx.x % c.cus) + wave;
                got = waves_per_wg * c.cus * row + (row & 1u ? n - 1u - i : i);
                if (got >= c.nchunks)
                    continue;
            }
            const LockChunk& ch = c.chunks[got];
            const uint32_t next = rfl32(ch.set);
            first = rfl32(ch.first);
            count = rfl32(ch.count);
            if (c.level) {
                /* of the set's places, those that were filled */
                const uint32_t cap = c.sets[next].cap[c.level - 1u], n = c.in_count[next * TMC_LOCK_LINE];
                const uint32_t have = rfl32(n < cap ? n : cap);
                if (first >= have)
                    continue;
                count = have - first < count ? have - first : count;
            }
            if (next != set) {
                if (set != ~0u)
                    flush();
                set = next;
                const LockSet& s = c.sets[set];
                phys.key0 = rfl32((uint32_t)s.seed);
                phys.key1 = rfl32((uint32_t)(s.seed >> 32));
                phys.albedo = s.albedo;
                phys.spm = s.spm;
                phys.shell_max = s.shell_max;
                set_derived<true>(phys);
                lt.fmax = tally_fmax(s.shell_max, lane & (TMC_LOCK_HOT - 1u));
                const CohortHead& h = c.heads[s.head];
                k0 = rfl32(c.level ? h.cut[c.level - 1u] : 0u);
                k1 = rfl32(h.cut[c.level]);
                hi = rfl32((uint32_t)(s.first_photon >> 32));
                table = (const char*)c.entry + 16ull * rfl64(s.entry);
                room = every;
            }
        }
        for (uint32_t at = 0; at < count; at += 64u) {
            const uint64_t in = count - at >= 64u ? ~0ull : (1ull << (count - at)) - 1ull;
            lt.deposit = in;
            LockPhoton p = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f, ~0u };
            tmc_philox_photon pp;
            uint32_t off = first + at + lane;
            {
                const LockSetArgs& c = args_here<LockSetArgs>();
                const LockSet& s = c.sets[set];
                if (c.level && __builtin_amdgcn_inverse_ballot_w64(in))
                    off = lock_load(p, c.in, s.place[c.level - 1u] + off);
                const uint64_t photon = s.first_photon + off;
                pp = tmc_philox_photon_init((uint32_t)photon, hi, phys.key0, phys.key1);
            }
            lock_cycle<MATH>(p, k0, k1, table, zero, hi ^ phys.key1, pp, phys, lt, room, every, flush);
            const uint32_t n = (uint32_t)__popcll(in);
            interactions += (uint64_t)n * (k1 - k0);
            idle += (uint64_t)(64u - n) * (k1 - k0);
            const uint64_t S = in & __ballot(p.x3 < TMC_ROULETTE_KILL_R);
            if (S != 0) {
                const LockSetArgs& c = args_here<LockSetArgs>();
                const LockSet& s = c.sets[set];
                if (!lock_append(S, off, p, c.out, c.out_count + set * TMC_LOCK_LINE, s.place[c.level],
                                 s.cap[c.level], lane)
                    && lane == 0)
                    atomicOr(c.counters + 2, TMC_LOCK_OVERFLOW);
            }
        }
    }
    if (set != ~0u)
        flush();
    /* (one addition a workgroup to a word, as lock_end) */
    if (lane == 0) {
        atomicAdd(totals, (unsigned long long)interactions);
        atomicAdd(totals + 1, (unsigned long long)idle);
    }
    __syncthreads();
    if (threadIdx.x < 2u)
        atomicAdd(args_here<LockSetArgs>().counters + 1u + 3u * threadIdx.x, totals[threadIdx.x]);
}

namespace {

using LockKernel = void (*)(LockArgs);

LockKernel lock_kernel(uint32_t sampler, uint32_t math, bool counted)
{
    if (counted) /* (analytic sampler) */
        return math == TMC_MATH_OWN ? walk_lock<0u, TMC_MATH_OWN, true> : walk_lock<0u, TMC_MATH_HARDWARE, true>;
    if (math == TMC_MATH_OWN)
        return sampler ? walk_lock<1u, TMC_MATH_OWN> : walk_lock<0u, TMC_MATH_OWN>;
    return sampler ? walk_lock<1u, TMC_MATH_HARDWARE> : walk_lock<0u, TMC_MATH_HARDWARE>;
}

} // namespace

hipError_t launch_lock(uint32_t sampler, uint32_t math, bool counted, const LockArgs& a, uint32_t grid, uint32_t block,
                       hipStream_t stream)
{
    const size_t lds = counted ? lock_count_bytes(a.shells, a.k1) : lock_lds_bytes(sampler, a.shells, block);
    hipLaunchKernelGGL(lock_kernel(sampler, math, counted), dim3(grid), dim3(block), lds, stream, a);
    return hipGetLastError();
}

hipError_t lock_occupancy(uint32_t sampler, uint32_t math, uint32_t counted, uint32_t shells, int* wg_per_cu)
{
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        wg_per_cu, lock_kernel(sampler, math, counted), (int)TMC_LOCK_BLOCK,
        counted ? lock_count_bytes(shells, counted) : lock_lds_bytes(sampler, shells, TMC_LOCK_BLOCK));
}

namespace {

using LockSetsKernel = void (*)(LockSetArgs);

size_t lock_sets_lds_bytes(uint32_t shells_max, uint32_t block)
{
    return 16u + (block / 64u) * lock_slot_words(shells_max) * 8u;
}

LockSetsKernel lock_sets_kernel(uint32_t math)
{
    return math == TMC_MATH_OWN ? walk_lock_sets<TMC_MATH_OWN> : walk_lock_sets<TMC_MATH_HARDWARE>;
}

} // namespace

hipError_t launch_lock_sets(uint32_t math, const LockSetArgs& a, uint32_t grid, uint32_t block, hipStream_t stream)
{
    hipLaunchKernelGGL(lock_sets_kernel(math), dim3(grid), dim3(block), lock_sets_lds_bytes(a.shells_max, block), stream, a);
    return hipGetLastError();
}

hipError_t lock_sets_occupancy(uint32_t math, uint32_t block, uint32_t shells_max, int* wg_per_cu)
{
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(wg_per_cu, lock_sets_kernel(math), (int)block,
                                                        lock_sets_lds_bytes(shells_max, block));
}

} // namespace tmc
