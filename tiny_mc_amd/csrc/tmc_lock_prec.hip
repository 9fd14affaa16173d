/* Runs of the precision variants (tmc_step_prec.h) in lockstep.
 *
 * In each of them the weight is, as in the binary32 walk, a function of the
 * absorption count alone: a product of binary64 factors, or 2^x of the counts
 * of absorptions and of roulettes survived.  So 64 photons launched together
 * stay together from roulette to roulette (tmc_lock.hip), the weight's images
 * come from a table that a workgroup builds ahead, and the part of the generator
 * that holds the count is scalar.  While there are more survivors than a photon
 * for every lane of a wave on each SIMD, they are appended to a list and packed
 * into full waves for the next cycle; fewer walk on where they are.
 *
 * What bounds it: the binary64 logarithm, square roots, sine and cosine (200
 * binary64 instructions of an absorption's 300, 4 cycles and more each), and
 * with few photons a lane's chain through them.  Measured on MI355X, whole
 * calls at default physics, lane per photon -> this walk: binary64 4096 photons
 * 327 -> 107 us, 2^20 1176 -> 754 us, 2^22 2.85 -> 2.56 ms (1.2e11
 * absorptions/s; the shape does not matter: 4 to 6 waves a SIMD 9.7 to 10.2 ms
 * at 2^24); weight from counts 242 -> 93, 543 -> 368 us and 1.30 -> 1.08 ms.
 *
 * Same words, same operations and the same integer sums as step(): results
 * are bit-identical.
 */
#include "tmc_step_prec.h"
#include "tmc_lock_device.h"

namespace tmc {

static size_t prec_lds_bytes(uint32_t shells) { return (lock_slot_words(shells) + 2u) * 8u; }

namespace {

/* Photon and physics of a variant. */
template <uint32_t PREC>
struct Variant {
    using PhotonT = PhotonW;
    using PhysicsT = PhysicsW;
};
template <>
struct Variant<3u> {
    using PhotonT = Photon64;
    using PhysicsT = Physics64;
};

template <uint32_t PREC>
__device__ __forceinline__ typename Variant<PREC>::PhysicsT physics_of(const PrecArgs& a)
{
    if constexpr (PREC == 3u)
        return Physics64{ a.albedo_d, a.spm_d, (double)(a.shells - 1u), a.shells - 1u, (uint32_t)a.seed,
                          (uint32_t)(a.seed >> 32) };
    else
        return PhysicsW{ a.l2a_hi, a.l2a_lo, a.l2s_hi, a.l2s_lo, a.spm_w, a.shell_max, a.shells - 1u, (uint32_t)a.seed,
                         (uint32_t)(a.seed >> 32) };
}

/* f(word, value) for the words of a photon's position and direction. */
template <uint32_t PREC, class F>
__device__ __forceinline__ void each_word(PhotonW& p, const F& f)
{
    f(0u, p.x);
    f(1u, p.y);
    f(2u, p.z);
    f(3u, p.u);
    f(4u, p.v);
    f(5u, p.w);
    if constexpr (PREC == 2u) {
        f(6u, p.xl);
        f(7u, p.yl);
        f(8u, p.zl);
    }
}

template <uint32_t PREC, class F>
__device__ __forceinline__ void each_word(Photon64& p, const F& f)
{
    f(0u, p.x);
    f(2u, p.y);
    f(4u, p.z);
    f(6u, p.u);
    f(8u, p.v);
    f(10u, p.w);
}

struct LoadWords {
    const PrecList& l;
    uint32_t i;
    __device__ __forceinline__ uint32_t word(uint32_t w) const { return l.state[(size_t)w * l.places + i]; }
    __device__ __forceinline__ void operator()(uint32_t w, float& v) const { v = __uint_as_float(word(w)); }
    __device__ __forceinline__ void operator()(uint32_t w, double& v) const
    {
        v = __hiloint2double((int)word(w + 1u), (int)word(w));
    }
};

struct StoreWords {
    const PrecList& l;
    uint32_t i;
    __device__ __forceinline__ void operator()(uint32_t w, float& v) const
    {
        l.state[(size_t)w * l.places + i] = __float_as_uint(v);
    }
    __device__ __forceinline__ void operator()(uint32_t w, double& v) const
    {
        l.state[(size_t)w * l.places + i] = (uint32_t)__double2loint(v);
        l.state[(size_t)(w + 1u) * l.places + i] = (uint32_t)__double2hiint(v);
    }
};

__device__ __forceinline__ Images pair_of(uint64_t h, uint64_t h2)
{
    return Images{ (uint32_t)h, (uint32_t)(h >> 32), (uint32_t)h2, (uint32_t)(h2 >> 32) };
}

template <uint32_t SAMPLER, uint32_t PREC, class PhotonT, class PhysicsT>
__device__ __forceinline__ bool step_of(PhotonT& p, const PhysicsT& ph, const LaneTally& lt)
{
    if constexpr (PREC == 3u)
        return step<SAMPLER>(p, ph, lt);
    else
        return step<SAMPLER, PREC == 2u>(p, ph, lt);
}

} // namespace

/* The weight table, and what a run starts from: workgroup 0 builds the table,
 * the others clear the counters. */
#define TMC_PREC_BLOCK 1024u

template <uint32_t PREC>
__global__ void __launch_bounds__(TMC_PREC_BLOCK) prec_table(PrecArgs a, uint32_t* counter, uint32_t counters,
                                                             unsigned long long* start)
{
    __shared__ uint32_t first;
    const uint32_t i = threadIdx.x;
    Images* const entry = (Images*)a.entry;
    const uint32_t at = blockIdx.x * TMC_PREC_BLOCK + i;
    if (at < counters)
        counter[at] = 0u;
    if (at == 0u)
        *start = __builtin_amdgcn_s_memrealtime();
    if constexpr (PREC == 3u) {
        /* the host has walked the products (on the device 93 ns an absorption
         * for a lane with its comparisons) */
        if (at < a.entries) {
            const double w = a.weight[at];
            entry[at] = pair_of(fx_heat64(w), fx_heat2_64(w));
        }
        if (at < sizeof(PrecHead) / 4u)
            ((uint32_t*)a.head)[at] = ((const uint32_t*)a.host_head)[at];
    } else {
        if (blockIdx.x != 0u)
            return;
        const auto phys = physics_of<PREC>(a);
        uint32_t n = 0; /* cuts so far */
        float w = 1.0f;
        /* 1024 absorptions of a cycle at a time, up to the first that ends it */
        if (i == 0u)
            entry[0] = pair_of(fx_heat(1.0f), fx_heat2(1.0f));
        for (uint32_t k = 1; k < a.entries && n < a.cuts;) {
            __syncthreads();
            if (i == 0u)
                first = ~0u;
            __syncthreads();
            const float v = weight_from_counts(k + i, n, phys);
            if (v < 0.001f)
                atomicMin(&first, k + i);
            __syncthreads();
            const uint32_t f = first;
            if (k + i < f && k + i < a.entries)
                entry[k + i] = pair_of(fx_heat(v), fx_heat2(v));
            if (f == ~0u) {
                k += TMC_PREC_BLOCK;
                continue;
            }
            if (f >= a.entries)
                break;
            if (i == 0u)
                a.head->cut[n] = f;
            ++n;
            w = weight_from_counts(f, n, phys);
            if (i == 0u)
                entry[f] = pair_of(fx_heat(w), fx_heat2(w));
            k = f + 1u;
        }
        if (i == 0u) {
            a.head->ncuts = n;
            a.head->w_end = w;
        }
    }
}

/* (PrecArgs must stay the only parameter: args_here) */
template <uint32_t SAMPLER, uint32_t PREC>
__global__ void __launch_bounds__(256) walk_lock_prec(PrecArgs a)
{
    extern __shared__ unsigned long long lds[];
    const uint32_t lane = __lane_id();
    const uint32_t wave = rfl32(threadIdx.x >> 6);
    unsigned long long *const totals = lds, *const slot = lds + 2;
    for (uint32_t i = threadIdx.x; i < lock_slot_words(a.shells) + 2u; i += blockDim.x)
        lds[i] = 0;
    __syncthreads();

    using PhotonT = typename Variant<PREC>::PhotonT;
    const auto phys = physics_of<PREC>(a);
    const tmc_philox_keys keys = tmc_philox_key_schedule(phys.key0, phys.key1);
    LaneTally lt = { slot, tally_fmax(a.shell_max, lane & (TMC_LOCK_HOT - 1u)), ~0ull };
    const uint32_t hi = (uint32_t)(a.first_photon >> 32), c3k1 = hi ^ phys.key1;
    uint32_t zero = 0;
    asm volatile("" : "+v"(zero));
    const char* const table = (const char*)a.entry;

    /* this wave's batches, as walk_lock */
    const uint32_t stripe = blockIdx.x % a.stripes, waves_per_wg = blockDim.x >> 6;
    uint32_t photons = a.photons, place = 0, at = 64u * (blockIdx.x * waves_per_wg + wave),
             stride = 64u * waves_per_wg * gridDim.x;
    if (a.level) {
        const uint32_t n = a.in_count[stripe * TMC_LOCK_LINE];
        photons = rfl32(n < a.in_cap ? n : a.in_cap);
        place = stripe * a.in_cap;
        at = 64u * (blockIdx.x / a.stripes * waves_per_wg + wave);
        stride = 64u * waves_per_wg * ((gridDim.x - stripe + a.stripes - 1u) / a.stripes);
    }
    const uint32_t ncuts = rfl32(a.head->ncuts);
    bool failed = ncuts < a.cuts; /* (the table has room for them: never seen) */
    uint64_t interactions = 0;
    const uint32_t every = lock_flush_steps(waves_per_wg);
    uint32_t room = every;
    for (; at < photons && !failed; at += stride) {
        uint64_t in = photons - at >= 64u ? ~0ull : (1ull << (photons - at)) - 1ull;
        PhotonT p;
        uint32_t off = place + at + lane;
        {
            const PrecArgs& c = args_here<PrecArgs>();
            const bool listed = c.level && __builtin_amdgcn_inverse_ballot_w64(in);
            const uint32_t i = off;
            if (listed)
                off = c.in.photon[i];
            launch_photon(p, c.first_photon + off, phys.key0, phys.key1);
            if (listed)
                each_word<PREC>(p, LoadWords{ c.in, i });
        }
        uint32_t level, stop;
        {
            const PrecArgs& c = args_here<PrecArgs>();
            level = c.level;
            stop = c.cycles ? c.level + c.cycles : ~0u;
        }
        uint32_t k = level ? rfl32(args_here<PrecArgs>().head->cut[level - 1u]) : 0u;
        while (in != 0 && level < ncuts) {
            const uint32_t k1 = rfl32(args_here<PrecArgs>().head->cut[level]);
            lt.deposit = in;
            interactions += (uint64_t)__popcll(in) * (k1 - k);
            uint32_t x3 = 0;
            Images e = *(const Images*)(table + 16ull * k + zero);
            while (k != k1) {
                const uint32_t left = k1 - k, n = rfl32(left < room ? left : room), end = k + n;
                room -= n;
                const char* from = table + 16ull * k;
                for (; k != end; ++k) {
                    from += 16u;
                    const Images next = *(const Images*)(from + zero);
                    const tmc_u32x4 r = block0_uniform(k, c3k1, p.pp, keys);
                    p.k = k;
                    uint32_t q;
                    if constexpr (PREC == 3u)
                        q = move(p, r, phys, lt);
                    else
                        q = move<PREC == 2u>(p, r, phys, lt);
                    tally_add(lt, q, ((uint64_t)e.y << 32) | e.x, ((uint64_t)e.w << 32) | e.z);
                    turn<SAMPLER>(p, r, phys);
                    x3 = r.x3;
                    e = next;
                }
                if (room == 0u) {
                    const PrecArgs& c = args_here<PrecArgs>();
                    lock_flush<true>(slot, lock_block(c) + TMC_COHORT_COUNTERS, c.shells, lane, 64u);
                    room = every;
                }
            }
            in &= __ballot(x3 < TMC_ROULETTE_KILL_R);
            ++level;
            if (level == stop && in != 0) {
                const PrecArgs& c = args_here<PrecArgs>();
                const uint32_t n = (uint32_t)__popcll(in);
                uint32_t base = 0;
                if (lane == 0)
                    base = atomicAdd(c.out_count + stripe * TMC_LOCK_LINE, n);
                base = rfl32(base);
                const uint32_t to = base + mask_rank(in);
                if (__builtin_amdgcn_inverse_ballot_w64(in) && to < c.out_cap) {
                    const uint32_t i = stripe * c.out_cap + to;
                    c.out.photon[i] = off;
                    each_word<PREC>(p, StoreWords{ c.out, i });
                }
                failed |= base + n > c.out_cap;
                in = 0;
            }
        }
        if (in != 0) {
            /* past the table */
            bool live = __builtin_amdgcn_inverse_ballot_w64(in);
            lt.deposit = ~0ull;
            p.k = k;
            p.weight = args_here<PrecArgs>().head->w_end;
            if constexpr (PREC != 3u) {
                p.e = k;
                p.r = ncuts;
            }
            for (uint32_t steps = 0; __ballot(live) != 0; ++steps) {
                interactions += (uint64_t)__popcll(__ballot(live));
                if (live)
                    live = step_of<SAMPLER, PREC>(p, phys, lt);
                if (steps % every == every - 1u) {
                    const PrecArgs& c = args_here<PrecArgs>();
                    lock_flush<true>(slot, lock_block(c) + TMC_COHORT_COUNTERS, c.shells, lane, 64u);
                }
            }
            /* (the slot has taken at most two intervals' deposits, below 2^64) */
        }
    }
    const PrecArgs& c = args_here<PrecArgs>();
    if (failed && lane == 0)
        atomicOr(lock_block(c) + 2, TMC_LOCK_OVERFLOW);
    lock_end(c, slot, totals, interactions, 0);
}

namespace {

using PrecKernel = void (*)(PrecArgs);

PrecKernel prec_kernel(uint32_t sampler, uint32_t precision)
{
    const bool rej = sampler == 1u;
    switch (precision) {
    case 1u: return rej ? walk_lock_prec<1u, 1u> : walk_lock_prec<0u, 1u>;
    case 2u: return rej ? walk_lock_prec<1u, 2u> : walk_lock_prec<0u, 2u>;
    default: return rej ? walk_lock_prec<1u, 3u> : walk_lock_prec<0u, 3u>;
    }
}

} // namespace

hipError_t prec_occupancy(uint32_t sampler, uint32_t precision, uint32_t block, uint32_t shells, int* wg_per_cu)
{
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(wg_per_cu, prec_kernel(sampler, precision), (int)block,
                                                        prec_lds_bytes(shells));
}

hipError_t launch_prec_table(uint32_t precision, const PrecArgs& a, uint32_t* counter, uint32_t counters,
                             unsigned long long* start, hipStream_t stream)
{
    const uint32_t most = precision == 3u && a.entries > counters ? a.entries : counters;
    const uint32_t grid = 1u + most / TMC_PREC_BLOCK;
    if (precision == 3u)
        hipLaunchKernelGGL(prec_table<3u>, dim3(grid), dim3(TMC_PREC_BLOCK), 0, stream, a, counter, counters, start);
    else
        hipLaunchKernelGGL(prec_table<1u>, dim3(grid), dim3(TMC_PREC_BLOCK), 0, stream, a, counter, counters, start);
    return hipGetLastError();
}

hipError_t launch_prec(uint32_t sampler, uint32_t precision, const PrecArgs& a, uint32_t grid, uint32_t block,
                       hipStream_t stream)
{
    hipLaunchKernelGGL(prec_kernel(sampler, precision), dim3(grid), dim3(block), prec_lds_bytes(a.shells), stream,
                       a);
    return hipGetLastError();
}

} // namespace tmc
