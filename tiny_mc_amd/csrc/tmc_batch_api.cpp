/* Host side of the batched sweep (include/tiny_mc_gpu.h, tmc_batch_*).
 *
 * A plan owns the device copies of the set table and the chunk queue, the
 * tally pool and, optionally, a HIP graph of the steady launch sequence
 * (clear kernel, persistent walk kernel, copy-back), so repeated runs of the
 * same batch cost one graph launch.
 *
 * Scheduling: each set's expected absorptions per photon L follow from the
 * binary32 weight cadence (tmc::expected_interactions).  A set of N photons
 * is cut into chunks of 64 * P photons with P = ceil(chunk_work / (64 L)),
 * so every chunk carries about chunk_work absorptions and a wave drains (its
 * lanes run out of the set's photons) once per ~P photons per lane.  Chunks
 * are sorted by expected duration, longest first, which keeps the long
 * high-albedo chunks off the end of the launch.
 *
 * Passes: a wave's LDS slot holds the largest shell count of its launch, so
 * a few sets with many shells would lower every wave's occupancy.  Sets are
 * grouped by the launch shape their shell count allows (classes with under a
 * tenth of the work join the next larger class), and each group runs as a
 * launch of its own, one after the other on the same stream, with its own
 * chunk queue and cursor; the tallies and counters are shared.
 *
 * Lockstep: with the analytic sampler and automatic options the launches are
 * those of tmc_lock.hip and tmc_cohort.hip instead, unless the sets' first
 * cycles are too short for that (tmc::lockstep_batch): waves carry 64 photons of
 * a set in lockstep to the first roulette, and append the tenth that survives
 * to the set's places in a list; where a batch leaves enough of them they are
 * walked to the second roulette the same way, and workgroups carry what is
 * left to its end as cohorts.  Measured on MI355X, walk_multi -> this:
 * 64 sets, 1.1e6 photons, planned, run and released 11.1 -> 3.1 ms; a kept
 * plan of 512 sets, 5.6e7 photons 232 -> 140 ms, of 4096 sets, 4.1e9 photons
 * 11.9 -> 9.9 s (its lanes idle 0.02% of the steps, 1.1% before; making it 16
 * -> 141 ms).
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "../../include/tiny_mc_gpu.h"
#include "tmc_batch_internal.h"
#include "tmc_cohort.h"
#include "tmc_context.h"
#include "tmc_internal.h"

#define TMC_EXPORT extern "C" __attribute__((visibility("default")))

static_assert(TMC_BATCH_CURSOR0 + TMC_BATCH_MAX_PASSES <= TMC_BATCH_COUNTERS, "pass cursors beyond the counters");

namespace {

/* One launch of a batch: the sets of one LDS size class. */
struct PassPlan {
    uint32_t grid = 0, block = 0, wps = 0, shells_max = 1;
    uint64_t nchunks = 0;
    uint64_t chunk_work = 0;
    double work = 0.0;
    tmc::BatchArgs args;
};

/* The lockstep launches of a batch: its sets in parts of at most kPart
 * photons, the parts in slices that share the lists. */
struct LockSlice {
    uint32_t first[3] = { 0, 0, 0 }, chunks[3] = { 0, 0, 0 }; /* queue of the first cycle, of the second, of the cohorts */
};

struct LockPlan {
    bool on = false;
    std::vector<LockSlice> slices;
    uint32_t cycles = 1; /* walked in lockstep before the cohorts */
    uint32_t grid = 0, cus = 0; /* workgroups of the lockstep launches and of the cohorts */
    void* d = nullptr; /* parts, heads, chunks, lists and tables */
    uint32_t* counts = nullptr; /* per part and list, then the cursors: TMC_LOCK_LINE words each */
    uint64_t count_words = 0; /* of 64 bits */
    uint32_t parts = 0;
    tmc::LockSetArgs args;
    tmc::PhotonList list[2];
};

/* Photons of a part (its survivors' places fit a slice). */
constexpr uint64_t kPart = 1ull << 26;
/* Parts of a batch: 100 MB in the host's memory (a set may have 2^63 photons). */
constexpr size_t kParts = 1u << 20;
/* Places of a slice's first list: 0.9 GB. */
constexpr uint64_t kSlicePlaces = 1ull << 25;
/* Entries of the weight tables of a batch: 1 GB. */
constexpr uint64_t kBatchEntries = 1ull << 26;
/* Expected survivors of a roulette from which on the next cycle is walked by
 * lockstep waves too: with fewer, their 64-photon batches leave most of the
 * chip's 8192 waves without one. */
constexpr double kSecondCycle = 200000.0;
constexpr uint32_t kLockBlock = 256;

/* Absorptions to a set's first roulette, and from there to the second (0: the
 * first is further than is walked out, tmc::expected_interactions). */
struct Cadence {
    uint32_t k1 = 0, k2 = 0;
};

} // namespace

struct tmc_batch_plan {
    uint32_t nsets = 0;
    uint64_t tally_words = 0;
    uint64_t nchunks = 0;
    uint64_t photons = 0;
    double expected = 0.0;
    /* shape of the pass with the most work (reported in the statistics) */
    uint64_t chunk_work = 0;
    uint32_t sampler = 0, math = 0, grid = 0, block = 0, copies = 1, wps = 0, shells_max = 1;
    uint32_t npasses = 0;
    PassPlan pass[TMC_BATCH_MAX_PASSES];
    bool use_graph = false;
    tmc::BatchSet* d_sets = nullptr;
    tmc::BatchChunk* d_chunks = nullptr;
    unsigned long long* d_tally = nullptr;
    unsigned long long* d_done = nullptr;
    unsigned long long* d_counters = nullptr;
    unsigned long long* h_tally = nullptr; /* pinned */
    unsigned long long* h_counters = nullptr; /* pinned, TMC_BATCH_COUNTERS words */
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    LockPlan lock;
};

namespace {

/* Device and pinned memory, and the graph, go through tmc::release, which
 * defers them while a serving kernel is resident (hipFree and hipHostFree
 * would wait for it). */
void plan_free(tmc_batch_plan* p)
{
    if (!p)
        return;
    if (p->exec || p->graph) {
        hipGraphExec_t exec = p->exec;
        hipGraph_t graph = p->graph;
        tmc::release([exec, graph]() {
            if (exec)
                (void)hipGraphExecDestroy(exec);
            if (graph)
                (void)hipGraphDestroy(graph);
        });
    }
    for (void* d : { (void*)p->d_sets, (void*)p->d_chunks, (void*)p->d_tally, (void*)p->d_done, (void*)p->d_counters,
                     p->lock.d })
        tmc::release_device(d);
    tmc::release_host(p->h_tally);
    tmc::release_host(p->h_counters);
    delete p;
}

/* Enqueues the lockstep launches. */
hipError_t enqueue_lock(const tmc_batch_plan* p, hipStream_t stream)
{
    const LockPlan& l = p->lock;
    uint32_t* cursor = l.counts + 2ull * l.parts * TMC_LOCK_LINE;
    for (const LockSlice& s : l.slices) {
        for (uint32_t level = 0; level < 3u; ++level, cursor += TMC_LOCK_LINE) {
            if (!s.chunks[level])
                continue;
            tmc::LockSetArgs a = l.args;
            a.chunks += s.first[level];
            a.nchunks = s.chunks[level];
            a.cursor = cursor;
            a.level = std::min(level, l.cycles);
            if (a.level) {
                a.in = l.list[a.level - 1u];
                a.in_count = l.counts + (uint64_t)(a.level - 1u) * l.parts * TMC_LOCK_LINE;
            }
            hipError_t e;
            if (level < 2u) {
                a.out = l.list[level];
                a.out_count = l.counts + (uint64_t)level * l.parts * TMC_LOCK_LINE;
                const uint32_t per = kLockBlock / 64u;
                e = tmc::launch_lock_sets(p->math, a, std::min(l.grid, (a.nchunks + per - 1u) / per), kLockBlock, stream);
            } else {
                e = tmc::launch_cohort_sets(p->math, a, std::min(l.cus, a.nchunks), stream);
            }
            if (e != hipSuccess)
                return e;
        }
    }
    return hipSuccess;
}

/* Enqueues clear + walk + copies on `stream`. */
hipError_t enqueue_run(tmc_batch_plan* p, bool lock, hipStream_t stream)
{
    hipError_t e = tmc::launch_batch_clear(p->d_tally, p->tally_words, p->d_done, p->nsets, p->d_counters, stream);
    if (e != hipSuccess)
        return e;
    if (lock) {
        e = tmc::launch_clear((unsigned long long*)p->lock.counts, p->lock.count_words, stream);
        if (e == hipSuccess)
            e = enqueue_lock(p, stream);
        if (e != hipSuccess)
            return e;
    }
    for (uint32_t j = 0; j < p->npasses && !lock; ++j) {
        const PassPlan& q = p->pass[j];
        if (!q.nchunks)
            continue;
        e = tmc::launch_batch(p->sampler, p->math, q.args, q.grid, q.block, stream);
        if (e != hipSuccess)
            return e;
    }
    e = hipMemcpyAsync(p->h_tally, p->d_tally, p->tally_words * sizeof(uint64_t), hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess)
        return e;
    return hipMemcpyAsync(p->h_counters, p->d_counters, TMC_BATCH_COUNTERS * sizeof(uint64_t), hipMemcpyDeviceToHost,
                          stream);
}

/* Launch shape for per-wave LDS slots of shells_max shells: the requested
 * block, or the largest of 256/128/64 whose slots fit on a CU, with the
 * resident workgroups capped by waves_per_simd when requested.  *fits is
 * false when no block fits. */
hipError_t launch_shape(const tmc_batch_plan* p, const tmc_batch_options* o, uint32_t cus, uint32_t shells_max,
                        PassPlan* q, bool* fits)
{
    *fits = false;
    std::vector<uint32_t> cand;
    if (o->block)
        cand.push_back(o->block);
    else
        cand = { 256u, 128u, 64u };
    for (uint32_t b : cand) {
        int n = 0;
        if (tmc::batch_lds_bytes(b, shells_max, p->copies) <= 160u * 1024u) {
            const hipError_t e = tmc::batch_occupancy(p->sampler, p->math, b, shells_max, p->copies, &n);
            if (e != hipSuccess)
                return e;
        }
        if (n <= 0)
            continue;
        const uint32_t waves_per_wg = b / 64u;
        if (o->waves_per_simd)
            n = std::min<int>(n, (int)std::max(1u, o->waves_per_simd * 4u / waves_per_wg));
        q->block = b;
        q->grid = (uint32_t)n * cus;
        q->wps = (uint32_t)n * waves_per_wg / 4u;
        q->shells_max = shells_max;
        *fits = true;
        return hipSuccess;
    }
    return hipSuccess;
}

/* Plans the lockstep launches of a batch; leaves p->lock off where they don't
 * apply: with the rejection sampler, with a cap on the absorptions, where the
 * caller chose a launch shape, with more than TMC_LOCK_SHELLS shells, where the weight tables or a first
 * cycle are longer than is worth laying out, where walk_multi is faster (tmc::lockstep_batch), and beside a server
 * that has the device.  `once`: the plan is made for one run.  TMC_OK, or TMC_E_HIP. */
int plan_lock(tmc::Context* c, const tmc_set* sets, uint32_t nsets, const tmc_batch_options* o, bool once, uint64_t kcap,
              const std::vector<tmc::BatchSet>& hs, const std::vector<Cadence>& cad, tmc_batch_plan* p)
{
    LockPlan& l = p->lock;
    if (o->sampler != TMC_SAMPLER_ANALYTIC || o->block || o->waves_per_simd || o->copies || o->chunk_work
        || kcap != 0xFFFFFFFFull || p->shells_max > TMC_LOCK_SHELLS || p->photons == 0 || tmc::serving())
        return TMC_OK;

    /* launch shape */
    int per_cu = 0;
    if (tmc::lock_sets_occupancy(p->math, kLockBlock, p->shells_max, &per_cu) != hipSuccess)
        return TMC_E_HIP;
    if (per_cu <= 0)
        return TMC_OK;
    l.cus = (uint32_t)c->compute_units;
    l.grid = (uint32_t)per_cu * l.cus;
    const double waves = (double)l.grid * (kLockBlock / 64u);

    std::vector<tmc::LockLoad> load;
    for (uint32_t i = 0; i < nsets; ++i) {
        if (!sets[i].params.photons)
            continue;
        if (cad[i].k1 == 0)
            return TMC_OK;
        load.push_back({ (double)sets[i].params.photons, (double)cad[i].k1 });
    }
    if (!tmc::lockstep_batch(load, waves, once))
        return TMC_OK;

    /* the sets' cadences and tables, and their parts */
    struct Part {
        uint32_t set;
        uint64_t first, count; /* photons of the set */
    };
    std::vector<tmc::LockSet> ls;
    std::vector<Part> parts;
    l.cycles = 0.1 * (double)p->photons >= kSecondCycle ? 2u : 1u;
    uint64_t entries = 0;
    for (uint32_t i = 0; i < nsets; ++i) {
        const uint64_t n = sets[i].params.photons;
        if (n == 0)
            continue;
        const uint32_t cuts = std::max(tmc::cuts_for((double)n), l.cycles + 2u);
        /* (later cycles can be a step longer than the second; two entries are
         * read ahead of the last) */
        const uint64_t room = cad[i].k1 + (uint64_t)(cuts - 1u) * (cad[i].k2 + 2u) + 64u;
        tmc::LockSet s;
        std::memset(&s, 0, sizeof s);
        s.seed = hs[i].seed;
        s.tally = hs[i].tally_offset;
        s.entry = entries;
        s.albedo = hs[i].albedo;
        s.spm = hs[i].spm;
        s.shell_max = hs[i].shell_max;
        s.shells = hs[i].shells;
        s.head = i;
        s.entries = (uint32_t)room;
        s.cuts = cuts;
        entries += room + 2u;
        if (entries > kBatchEntries)
            return TMC_OK;
        for (uint64_t done = 0; done < n;) {
            s.first_photon = hs[i].first_photon + done;
            const uint64_t count =
                std::min<uint64_t>(std::min<uint64_t>(kPart, n - done), (1ull << 32) - (s.first_photon & 0xFFFFFFFFull));
            if (parts.size() == kParts)
                return TMC_OK;
            parts.push_back({ i, done, count });
            ls.push_back(s);
            s.cuts = 0; /* the first part builds the table */
            done += count;
        }
    }
    l.parts = (uint32_t)parts.size();

    /* slices, places and queues: chunks of a wave's 32nd of a launch's work,
     * longest first */
    struct Run { /* chunks of a part, of one length */
        double steps;
        uint32_t part, first, each, chunks;
    };
    std::vector<tmc::LockChunk> queue;
    uint64_t places[2] = { 0, 0 };
    for (size_t i = 0; i < parts.size();) {
        LockSlice slice;
        uint64_t used[2] = { 0, 0 };
        std::vector<Run> runs[3];
        auto cut = [&](uint32_t level, uint32_t part, uint64_t n, double cycle, double each) {
            const uint64_t batches = std::max<uint64_t>(1, (uint64_t)std::min(1e6, std::ceil(each / cycle)));
            const uint32_t full = (uint32_t)(n / (64u * batches)), rest = (uint32_t)(n - 64u * batches * full);
            if (full)
                runs[level].push_back({ cycle * (double)batches, part, 0u, (uint32_t)(64u * batches), full });
            if (rest)
                runs[level].push_back({ cycle * std::ceil((double)rest / 64.0), part, (uint32_t)(n - rest), rest, 1u });
        };
        const size_t begin = i;
        double steps[2] = { 0.0, 0.0 }; /* of 64 photons, in the first and the second cycles */
        for (; i < parts.size(); ++i) {
            /* places for an eighth of the photons and a slack, where a tenth
             * survive, and for a 64th after the second roulette */
            const uint64_t n = parts[i].count;
            const uint32_t cap[2] = { (uint32_t)(n / 8u + 64u), (uint32_t)(n / 64u + 64u) };
            if (used[0] && used[0] + cap[0] > kSlicePlaces)
                break;
            for (uint32_t w = 0; w < 2u; ++w) {
                ls[i].place[w] = (uint32_t)used[w];
                ls[i].cap[w] = cap[w];
                used[w] += cap[w];
            }
            const Cadence& k = cad[parts[i].set];
            steps[0] += (double)k.k1 * std::ceil((double)n / 64.0);
            steps[1] += (double)k.k2 * std::ceil((double)n / 640.0);
        }
        for (size_t j = begin; j < i; ++j) {
            const Cadence& k = cad[parts[j].set];
            cut(0, (uint32_t)j, parts[j].count, (double)k.k1, std::max(tmc::kLockChunkSteps, steps[0] / waves / 32.0));
            if (l.cycles > 1u)
                cut(1, (uint32_t)j, ls[j].cap[0], (double)k.k2, std::max(tmc::kLockChunkSteps, steps[1] / waves / 32.0));
            cut(2, (uint32_t)j, ls[j].cap[l.cycles - 1u], (double)k.k2, 1.0);
        }
        for (uint32_t level = 0; level < 3u; ++level) {
            std::stable_sort(runs[level].begin(), runs[level].end(),
                             [](const Run& x, const Run& y) { return x.steps > y.steps; });
            slice.first[level] = (uint32_t)queue.size();
            for (const Run& r : runs[level]) {
                if (queue.size() + r.chunks > 1u << 26)
                    return TMC_OK;
                for (uint32_t j = 0; j < r.chunks; ++j)
                    queue.push_back({ r.part, r.first + j * r.each, r.each, 0u });
            }
            slice.chunks[level] = (uint32_t)queue.size() - slice.first[level];
        }
        for (uint32_t w = 0; w < 2u; ++w)
            places[w] = std::max(places[w], used[w]);
        l.slices.push_back(slice);
    }
    if (l.cycles < 2u)
        places[1] = 0;

    /* one block of device memory; what the host writes comes first */
    uint64_t bytes = 0;
    auto take = [&](uint64_t n) {
        const uint64_t at = bytes;
        bytes += (n + 255u) / 256u * 256u;
        return at;
    };
    const uint64_t at_sets = take(ls.size() * sizeof(tmc::LockSet));
    const uint64_t at_queue = take(queue.size() * sizeof(tmc::LockChunk));
    const uint64_t written = bytes;
    const uint64_t at_heads = take(nsets * sizeof(tmc::CohortHead));
    l.count_words = (2ull * l.parts + 3ull * l.slices.size()) * TMC_LOCK_LINE / 2u;
    const uint64_t at_counts = take(l.count_words * 8u);
    const uint64_t at_entries = take(entries * 16u);
    const uint64_t at_lists = take(28u * (places[0] + places[1]));
    if (hipMalloc(&l.d, bytes) != hipSuccess) {
        l.d = nullptr;
        (void)hipGetLastError();
        return TMC_OK;
    }
    std::vector<char> stage(written);
    std::memcpy(stage.data() + at_sets, ls.data(), ls.size() * sizeof(tmc::LockSet));
    std::memcpy(stage.data() + at_queue, queue.data(), queue.size() * sizeof(tmc::LockChunk));
    char* const d = (char*)l.d;
    float* at = (float*)(d + at_lists);
    for (uint32_t w = 0; w < 2u; ++w) {
        l.list[w].photon = (uint32_t*)at;
        at += places[w];
        for (float*& f : l.list[w].state) {
            f = at;
            at += places[w];
        }
    }
    l.counts = (uint32_t*)(d + at_counts);
    tmc::LockSetArgs& a = l.args;
    std::memset(&a, 0, sizeof a);
    a.sets = (const tmc::LockSet*)(d + at_sets);
    a.heads = (const tmc::CohortHead*)(d + at_heads);
    a.chunks = (const tmc::LockChunk*)(d + at_queue);
    a.entry = d + at_entries;
    a.cus = l.cus;
    a.shells_max = p->shells_max;
    a.tally = p->d_tally;
    a.counters = p->d_counters;
    hipError_t e = hipMemcpyAsync(d, stage.data(), written, hipMemcpyHostToDevice, c->stream);
    /* (a server may have taken the device since: the plan is made without
     * waiting for it, and keeps to walk_multi) */
    const tmc::LockstepRun run;
    l.on = (bool)run;
    if (e == hipSuccess && l.on)
        e = tmc::launch_weigh_sets(a.sets, l.parts, (tmc::CohortHead*)(d + at_heads), d + at_entries, c->stream);
    if (e != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    return TMC_OK;
}

int plan_create_locked(tmc::Context* c, const tmc_set* sets, uint32_t nsets, const tmc_batch_options* o, bool once,
                       tmc_batch_plan** out)
{
    if (o->sampler > TMC_SAMPLER_REJECTION || o->math > TMC_MATH_OWN)
        return TMC_E_INVALID;
    if (o->block && (o->block < 64u || o->block > 1024u || o->block % 64u))
        return TMC_E_INVALID;
    const uint32_t copies = o->copies ? o->copies : 1u;
    if (copies != 1u && copies != 2u)
        return TMC_E_INVALID;
    if (o->waves_per_simd > 8u)
        return TMC_E_INVALID;

    tmc_batch_plan* p = new (std::nothrow) tmc_batch_plan;
    if (!p)
        return TMC_E_NOMEM;
    p->nsets = nsets;
    p->sampler = o->sampler;
    p->math = o->math;
    p->copies = copies;
    p->use_graph = o->use_graph != 0;

    /* set table */
    std::vector<tmc::BatchSet> hs(nsets);
    std::vector<tmc::PlanSet> ps(nsets);
    std::vector<Cadence> cad(nsets);
    uint64_t off = 0;
    double work = 0.0;
    uint32_t shells_max = 1;
    uint64_t kcap = o->max_interactions ? o->max_interactions : 0xFFFFFFFFull;
    if (kcap > 0xFFFFFFFFull)
        kcap = 0xFFFFFFFFull;
    for (uint32_t i = 0; i < nsets; ++i) {
        const tmc_params& q = sets[i].params;
        tmc::BatchSet& d = hs[i];
        std::memset(&d, 0, sizeof d);
        d.seed = sets[i].seed;
        d.first_photon = sets[i].first_photon;
        d.tally_offset = off;
        d.albedo = tmc::derived_albedo(&q);
        d.spm = tmc::derived_spm(&q);
        d.shell_max = (float)(q.shells - 1);
        d.shells = q.shells;
        d.kcap = (uint32_t)kcap;
        off += 4 * (uint64_t)q.shells;
        shells_max = std::max(shells_max, q.shells);
        ps[i] = { q.shells, q.photons, tmc::expected_interactions(&q, kcap, &cad[i].k1, &cad[i].k2) };
        work += ps[i].L * (double)q.photons;
        p->photons += q.photons;
    }
    p->tally_words = off;
    p->shells_max = shells_max;
    p->expected = work;

    /* launch passes and chunk queues */
    const uint32_t cus = (uint32_t)c->compute_units;
    const tmc::ShapeFn shape_of = [&](uint32_t shells, tmc::PlanShape* shape) {
        PassPlan s;
        bool fits = false;
        if (launch_shape(p, o, cus, shells, &s, &fits) != hipSuccess)
            return (int)TMC_E_HIP;
        if (!fits)
            return (int)TMC_E_INVALID; /* LDS slots of this many shells do not fit */
        *shape = { s.grid, s.block, s.wps };
        return (int)TMC_OK;
    };
    std::vector<tmc::PlanPass> passes;
    std::vector<tmc::PlanChunk> pc;
    const int prc = tmc::plan_passes(ps, o->chunk_work, TMC_BATCH_MAX_PASSES, shape_of, &passes, &pc);
    if (prc != TMC_OK) {
        plan_free(p);
        return prc;
    }
    std::vector<tmc::BatchChunk> hc(pc.size());
    for (size_t k = 0; k < pc.size(); ++k)
        hc[k] = { pc[k].set, pc[k].count, pc[k].first };
    p->npasses = (uint32_t)passes.size();
    std::vector<uint64_t> first_chunk(passes.size());
    for (size_t j = 0; j < passes.size(); ++j) {
        PassPlan& q = p->pass[j];
        q.grid = passes[j].shape.grid;
        q.block = passes[j].shape.block;
        q.wps = passes[j].shape.wps;
        q.shells_max = passes[j].hi;
        q.work = passes[j].work;
        q.chunk_work = passes[j].chunk_work;
        q.nchunks = passes[j].nchunks;
        first_chunk[j] = passes[j].first_chunk;
    }
    p->nchunks = hc.size();
    uint32_t main_pass = 0;
    for (uint32_t j = 1; j < p->npasses; ++j)
        if (p->pass[j].work > p->pass[main_pass].work)
            main_pass = j;
    if (p->npasses) {
        p->grid = p->pass[main_pass].grid;
        p->block = p->pass[main_pass].block;
        p->wps = p->pass[main_pass].wps;
        p->chunk_work = p->pass[main_pass].chunk_work;
    }

    /* device memory */
    if (hipMalloc((void**)&p->d_sets, std::max<size_t>(1, nsets) * sizeof(tmc::BatchSet)) != hipSuccess
        || hipMalloc((void**)&p->d_chunks, std::max<size_t>(1, hc.size()) * sizeof(tmc::BatchChunk)) != hipSuccess
        || hipMalloc((void**)&p->d_tally, std::max<uint64_t>(1, p->tally_words) * sizeof(uint64_t)) != hipSuccess
        || hipMalloc((void**)&p->d_done, std::max<size_t>(1, 2 * (size_t)nsets) * sizeof(uint64_t)) != hipSuccess
        || hipMalloc((void**)&p->d_counters, TMC_BATCH_COUNTERS * sizeof(uint64_t)) != hipSuccess
        || hipHostMalloc((void**)&p->h_tally, std::max<uint64_t>(1, p->tally_words) * sizeof(uint64_t), 0)
            != hipSuccess
        || hipHostMalloc((void**)&p->h_counters, TMC_BATCH_COUNTERS * sizeof(uint64_t), 0) != hipSuccess) {
        plan_free(p);
        return TMC_E_NOMEM;
    }
    if ((nsets
         && hipMemcpyAsync(p->d_sets, hs.data(), nsets * sizeof(tmc::BatchSet), hipMemcpyHostToDevice, c->stream)
             != hipSuccess)
        || (!hc.empty()
            && hipMemcpyAsync(p->d_chunks, hc.data(), hc.size() * sizeof(tmc::BatchChunk), hipMemcpyHostToDevice,
                              c->stream)
                != hipSuccess)
        || hipStreamSynchronize(c->stream) != hipSuccess) {
        plan_free(p);
        return TMC_E_HIP;
    }

    for (uint32_t j = 0; j < p->npasses; ++j) {
        tmc::BatchArgs& a = p->pass[j].args;
        std::memset(&a, 0, sizeof a);
        a.sets = p->d_sets;
        a.chunks = p->d_chunks + first_chunk[j];
        a.nchunks = (uint32_t)p->pass[j].nchunks;
        a.shells_max = p->pass[j].shells_max;
        a.copies = copies;
        a.counters = p->d_counters;
        a.cursor = TMC_BATCH_CURSOR0 + j;
        a.tally = p->d_tally;
        a.done = p->d_done;
    }

    int lrc = TMC_OK;
    try {
        lrc = plan_lock(c, sets, nsets, o, once, kcap, hs, cad, p);
    } catch (const std::bad_alloc&) {
        p->lock.on = false; /* (its queue is the largest of the host's tables) */
    }
    if (!p->lock.on) {
        tmc::release_device(p->lock.d);
        p->lock = LockPlan();
    }
    if (lrc != TMC_OK) {
        plan_free(p);
        return lrc;
    }

    if (p->use_graph) {
        hipStream_t s = c->stream;
        if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) {
            plan_free(p);
            return TMC_E_HIP;
        }
        const hipError_t e1 = enqueue_run(p, p->lock.on, s);
        const hipError_t e2 = hipStreamEndCapture(s, &p->graph);
        if (e1 != hipSuccess || e2 != hipSuccess
            || hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0) != hipSuccess) {
            plan_free(p);
            return TMC_E_HIP;
        }
    }
    *out = p;
    return TMC_OK;
}

/* Runs the plan's launches once, by the lockstep walk or the other. */
int plan_launch(tmc::Context* c, tmc_batch_plan* p, bool lock)
{
    if (hipEventRecord(c->ev_start, c->stream) != hipSuccess)
        return TMC_E_HIP;
    if (p->use_graph && lock == p->lock.on) {
        if (hipGraphLaunch(p->exec, c->stream) != hipSuccess)
            return TMC_E_HIP;
    } else if (enqueue_run(p, lock, c->stream) != hipSuccess) {
        return TMC_E_HIP;
    }
    if (hipEventRecord(c->ev_stop, c->stream) != hipSuccess)
        return TMC_E_HIP;
    return TMC_OK;
}

int plan_run_locked(tmc::Context* c, tmc_batch_plan* p, uint64_t* tallies, tmc_batch_stats* st)
{
    const auto t0 = std::chrono::steady_clock::now();
    bool walked = false;
    if (p->lock.on) {
        /* (the cohorts' workgroups need whole compute units) */
        const tmc::LockstepRun run;
        if (run) {
            const int rc = plan_launch(c, p, true);
            if (hipStreamSynchronize(c->stream) != hipSuccess || rc != TMC_OK)
                return TMC_E_HIP;
            walked = p->h_counters[2] < TMC_LOCK_OVERFLOW; /* else a list had no room for a survivor */
        }
    }
    if (!walked) {
        const int rc = plan_launch(c, p, false);
        if (rc != TMC_OK)
            return rc;
        if (hipStreamSynchronize(c->stream) != hipSuccess)
            return TMC_E_HIP;
    }
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, c->ev_start, c->ev_stop) != hipSuccess)
        return TMC_E_HIP;
    if (tallies)
        std::memcpy(tallies, p->h_tally, p->tally_words * sizeof(uint64_t));
    if (st) {
        st->sets = p->nsets;
        st->photons = p->photons;
        st->interactions = p->h_counters[1];
        st->truncated = p->h_counters[2];
        st->idle_lane_steps = p->h_counters[4];
        st->chunks = p->nchunks;
        st->chunk_work = p->chunk_work;
        st->expected_interactions = p->expected;
        st->kernel_ms = ms;
        st->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        st->grid = p->grid;
        st->block = p->block;
        st->copies = p->copies;
        st->waves_per_simd = p->wps;
        st->passes = p->npasses;
        st->reserved = 0;
    }
    return TMC_OK;
}

int check_sets(const tmc_set* sets, uint32_t nsets)
{
    if (!sets && nsets)
        return TMC_E_INVALID;
    for (uint32_t i = 0; i < nsets; ++i) {
        const int rc = tmc::check_params(&sets[i].params);
        if (rc != TMC_OK)
            return rc;
        if (!tmc::photon_range_ok(sets[i].first_photon, sets[i].params.photons))
            return TMC_E_RANGE;
    }
    return TMC_OK;
}

} // namespace

TMC_EXPORT void tmc_batch_options_default(tmc_batch_options* opt)
{
    if (opt)
        std::memset(opt, 0, sizeof *opt);
}

TMC_EXPORT uint64_t tmc_batch_tally_words(const tmc_set* sets, uint32_t nsets)
{
    uint64_t w = 0;
    for (uint32_t i = 0; sets && i < nsets; ++i)
        w += 4 * (uint64_t)sets[i].params.shells;
    return w;
}

namespace {

int plan_create(const tmc_set* sets, uint32_t nsets, const tmc_batch_options* opt, bool once, tmc_batch_plan** plan)
{
    if (!plan)
        return TMC_E_INVALID;
    *plan = nullptr;
    int rc = check_sets(sets, nsets);
    if (rc != TMC_OK)
        return rc;
    tmc_batch_options o;
    if (opt)
        o = *opt;
    else
        tmc_batch_options_default(&o);
    std::lock_guard<std::mutex> lock(tmc::api_mutex());
    tmc::Context* c = nullptr;
    rc = tmc::acquire_context(&c);
    if (rc != TMC_OK)
        return rc;
    return plan_create_locked(c, sets, nsets, &o, once, plan);
}

} // namespace

TMC_EXPORT int tmc_batch_plan_create(const tmc_set* sets, uint32_t nsets, const tmc_batch_options* opt,
                                     tmc_batch_plan** plan)
{
    return plan_create(sets, nsets, opt, false, plan);
}

TMC_EXPORT int tmc_batch_plan_run(tmc_batch_plan* plan, uint64_t* tallies, tmc_batch_stats* stats)
{
    if (!plan)
        return TMC_E_INVALID;
    std::lock_guard<std::mutex> lock(tmc::api_mutex());
    tmc::Context* c = nullptr;
    const int rc = tmc::acquire_context(&c);
    if (rc != TMC_OK)
        return rc;
    return plan_run_locked(c, plan, tallies, stats);
}

TMC_EXPORT void tmc_batch_plan_destroy(tmc_batch_plan* plan)
{
    if (!plan)
        return;
    std::lock_guard<std::mutex> lock(tmc::api_mutex());
    plan_free(plan);
}

TMC_EXPORT int tmc_batch_run(const tmc_set* sets, uint32_t nsets, const tmc_batch_options* opt, uint64_t* tallies,
                             tmc_batch_stats* stats)
{
    tmc_batch_plan* plan = nullptr;
    int rc = plan_create(sets, nsets, opt, true, &plan);
    if (rc != TMC_OK)
        return rc;
    rc = tmc_batch_plan_run(plan, tallies, stats);
    tmc_batch_plan_destroy(plan);
    return rc;
}

TMC_EXPORT int tmc_batch_autotune(const tmc_set* sets, uint32_t nsets, const tmc_batch_options* base,
                                  uint32_t sample_divisor, tmc_batch_options* best)
{
    if (!best)
        return TMC_E_INVALID;
    int rc = check_sets(sets, nsets);
    if (rc != TMC_OK)
        return rc;
    tmc_batch_options b0;
    if (base)
        b0 = *base;
    else
        tmc_batch_options_default(&b0);
    b0.use_graph = 0;
    if (sample_divisor == 0)
        sample_divisor = 1;
    auto reduced = [&](uint32_t divisor) {
        std::vector<tmc_set> r(sets, sets + nsets);
        for (auto& s : r)
            if (s.params.photons)
                s.params.photons = std::max<uint64_t>(64, s.params.photons / divisor);
        return r;
    };
    const std::vector<tmc_set> sample = reduced(sample_divisor);

    /* the automatic chunk work of the full batch on the default shape */
    tmc_batch_plan* probe = nullptr;
    rc = tmc_batch_plan_create(sets, nsets, &b0, &probe);
    if (rc != TMC_OK)
        return rc;
    const uint64_t auto_cw = probe->chunk_work;
    const double full_work = probe->expected;
    tmc_batch_plan_destroy(probe);
    /* chunk work is tuned as a multiple of the automatic value, scaled to a
     * reduced copy so that it sees the same chunk count per wave */
    auto scale_of = [&](const std::vector<tmc_set>& r, double* scale) -> int {
        tmc_batch_plan* sp = nullptr;
        const int e = tmc_batch_plan_create(r.data(), nsets, &b0, &sp);
        if (e != TMC_OK)
            return e;
        *scale = full_work > 0 ? sp->expected / full_work : 1.0;
        tmc_batch_plan_destroy(sp);
        return TMC_OK;
    };
    double scale = 1.0;
    rc = scale_of(sample, &scale);
    if (rc != TMC_OK)
        return rc;

    /* each candidate: the best of `reps` runs after a warm-up run */
    auto time_on = [&](const std::vector<tmc_set>& r, double sc, const tmc_batch_options& o, double mult,
                       int reps) -> double {
        tmc_batch_options t = o;
        /* (the automatic value as such: with automatic options throughout, the
         * lockstep walk is the candidate that the others have to beat) */
        if (mult != 1.0 || b0.chunk_work)
            t.chunk_work = (uint64_t)std::max(4096.0, mult * (double)auto_cw * sc);
        tmc_batch_plan* plan = nullptr;
        if (tmc_batch_plan_create(r.data(), nsets, &t, &plan) != TMC_OK)
            return 1e300;
        tmc_batch_stats st;
        double best_ms = 1e300;
        for (int rep = 0; rep <= reps; ++rep) /* first run warms the code object */
            if (tmc_batch_plan_run(plan, nullptr, &st) == TMC_OK && rep > 0)
                best_ms = std::min(best_ms, st.kernel_ms);
        tmc_batch_plan_destroy(plan);
        return best_ms;
    };
    auto time_of = [&](const tmc_batch_options& o, double mult) { return time_on(sample, scale, o, mult, 3); };
    /* a candidate replaces the current options only when it is faster by
     * kMargin on the sample: the sample's shorter queues favour shapes that
     * do not carry over to the full batch, and the automatic options already
     * keep nearly every lane busy */
    constexpr double kMargin = 0.97;

    tmc_batch_options cur = b0;
    double cur_mult = 1.0;
    double cur_ms = time_of(cur, cur_mult);
    for (double m : { 0.25, 4.0 }) {
        const double ms = time_of(cur, m);
        if (ms < kMargin * cur_ms) {
            cur_ms = ms;
            cur_mult = m;
        }
    }
    for (uint32_t copies : { 2u }) {
        tmc_batch_options t = cur;
        t.copies = copies;
        const double ms = time_of(t, cur_mult);
        if (ms < kMargin * cur_ms) {
            cur_ms = ms;
            cur = t;
        }
    }
    for (uint32_t block : { 64u, 512u }) {
        tmc_batch_options t = cur;
        t.block = block;
        const double ms = time_of(t, cur_mult);
        if (ms < kMargin * cur_ms) {
            cur_ms = ms;
            cur = t;
        }
    }
    for (uint32_t wps : { 6u, 4u }) {
        tmc_batch_options t = cur;
        t.waves_per_simd = wps;
        const double ms = time_of(t, cur_mult);
        if (ms < kMargin * cur_ms) {
            cur_ms = ms;
            cur = t;
        }
    }
    if (cur_ms >= 1e300)
        return TMC_E_HIP;
    /* a choice other than *base must also win on a copy four times larger
     * (the whole batch for divisors up to 4): on the 4096-set sweep the
     * 1/16 sample once picked 4x chunk work and 6 waves per SIMD, 2.4% slower
     * than the defaults on the full batch */
    const bool changed = cur_mult != 1.0 || cur.block != b0.block || cur.waves_per_simd != b0.waves_per_simd
        || cur.copies != b0.copies;
    if (changed) {
        const uint32_t div2 = sample_divisor / 4u > 1u ? sample_divisor / 4u : 1u;
        const std::vector<tmc_set> confirm = div2 > 1u ? reduced(div2) : std::vector<tmc_set>(sets, sets + nsets);
        double sc2 = 1.0;
        rc = scale_of(confirm, &sc2);
        if (rc != TMC_OK)
            return rc;
        const double base_ms = time_on(confirm, sc2, b0, 1.0, 2);
        const double pick_ms = time_on(confirm, sc2, cur, cur_mult, 2);
        if (!(pick_ms < kMargin * base_ms)) {
            cur = b0;
            cur_mult = 1.0;
        }
    }
    *best = cur;
    /* unchanged chunk work stays automatic (the plan derives it per pass) */
    best->chunk_work = cur_mult == 1.0 ? b0.chunk_work : (uint64_t)std::max(4096.0, cur_mult * (double)auto_cw);
    best->use_graph = base ? base->use_graph : 0;
    return TMC_OK;
}
