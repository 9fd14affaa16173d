/* Host planning with no HIP in it (tmc_plan.h). */
#include "tmc_plan.h"

#include <algorithm>
#include <cmath>
#include <iterator>

/* Parameter checks.  The reference has none (params.h:14 only warns that
 * MU_A must be non-zero: with mu_a = 0 the weight never reaches the cutoff
 * and photon() never returns). */
int tmc::check_params(const tmc_params* p)
{
    if (!p)
        return TMC_E_INVALID;
    if (!std::isfinite(p->mu_a) || !std::isfinite(p->mu_s) || !std::isfinite(p->microns_per_shell))
        return TMC_E_INVALID;
    if (!(p->mu_a > 0.0f) || !(p->mu_s >= 0.0f) || !(p->microns_per_shell > 0.0f))
        return TMC_E_INVALID;
    if (p->shells < 1 || p->shells > TMC_MAX_SHELLS)
        return TMC_E_INVALID;
    /* binary32 albedo must stay below 1, or the weight never decays */
    const volatile float sum = p->mu_s + p->mu_a;
    const volatile float albedo = p->mu_s / sum;
    if (!(albedo < 1.0f))
        return TMC_E_INVALID;
    const double spm = 1e4 / (double)p->microns_per_shell / (double)sum;
    if (!std::isfinite((float)spm) || !((float)spm > 0.0f))
        return TMC_E_INVALID;
    return TMC_OK;
}

/* photon.c:8: albedo evaluated in float. */
float tmc::derived_albedo(const tmc_params* p)
{
    const volatile float sum = p->mu_s + p->mu_a;
    return p->mu_s / sum;
}

/* photon.c:9: 1e4 is a double literal, so the quotient is formed in double
 * from the float sum mu_a + mu_s, then stored as float. */
float tmc::derived_spm(const tmc_params* p)
{
    const volatile float sum = p->mu_a + p->mu_s;
    return (float)(1e4 / (double)p->microns_per_shell / (double)sum);
}

/* The weight after k absorptions is a deterministic binary32 sequence
 * (photon.c:32, 45-49): it falls below 0.001 after k1 steps, then after k2
 * steps of each later cycle (the first of them; later cycles can differ by
 * a step).  False if the first cycle is longer than `limit` steps. */
bool tmc::weight_cadence(const tmc_params* p, uint32_t limit, uint32_t* k1_out, uint32_t* k2_out)
{
    const float a = derived_albedo(p);
    float w = 1.0f;
    uint32_t k1 = 0;
    while (w >= 0.001f && k1 < limit) {
        w = w * a;
        ++k1;
    }
    if (!(w < 0.001f))
        return false;
    /* later cycles start from the cutoff weight / 0.1 */
    float v = w / 0.1f;
    uint32_t k2 = 0;
    while (v >= 0.001f && k2 < limit) {
        v = v * a;
        ++k2;
    }
    *k1_out = k1;
    *k2_out = k2 ? k2 : 1;
    return true;
}

uint32_t tmc::weight_sequence(const tmc_params* p, uint32_t room, uint32_t max_cuts, float* weight, uint32_t* cut,
                              float* w_end)
{
    const float a = derived_albedo(p);
    float w = 1.0f;
    uint32_t k = 0, n = 0;
    while (n < max_cuts && k < room) {
        weight[k++] = w;
        w = w * a;
        if (w < 0.001f) {
            w = w / 0.1f;
            cut[n++] = k;
        }
    }
    *w_end = w;
    return n;
}

/* Mean absorptions k1 + k2 p / (1 - p) with p the survival probability
 * 1677721 / 2^24 of the (0,1] uniform. */
double tmc::expected_interactions(const tmc_params* p, uint64_t kcap, uint32_t* k1_out, uint32_t* k2_out)
{
    const double pr = 1677721.0 / 16777216.0;
    uint32_t k1 = 0, k2 = 0;
    double c1, c2;
    if (weight_cadence(p, 1u << 20, &k1, &k2)) {
        c1 = (double)k1;
        c2 = (double)k2;
    } else {
        /* albedo so close to 1 that the cadence is long: continuous estimate */
        const double a = (double)derived_albedo(p);
        c1 = std::log(0.001) / std::log(a);
        c2 = std::log(0.1) / std::log(a);
        k1 = k2 = 0;
    }
    if (k1_out)
        *k1_out = k1;
    if (k2_out)
        *k2_out = k2;
    double mean = c1 + c2 * pr / (1.0 - pr);
    if (kcap && mean > (double)kcap)
        mean = (double)kcap;
    return mean < 1.0 ? 1.0 : mean;
}

bool tmc::cohort_shape(uint64_t photons, uint64_t most, double L, uint32_t shells, uint32_t cus, CohortShape* shape)
{
    if (photons == 0 || photons > most || cus == 0)
        return false;
    /* one workgroup per compute unit, and cohorts as small as that allows: a
     * round of fewer photons is more absorptions of each, and costs little
     * more.  But every workgroup has its sums to add to the others' at the
     * end, 8 us for 256 of them, so short walks keep 16 photons together
     * (1000 photons at default physics: 4 photons a cohort 30.8 us, 16: 29.3,
     * 64: 34.2; 512 at albedo 0.99: 2: 68.9, 16: 83.2), and a handful of them
     * in one workgroup, which has nobody to add to. */
    const bool shortwalk = L < 200.0;
    uint32_t group = shortwalk ? (photons <= 64 ? 64u : 16u) : 2u;
    while (group < 64u && (photons + group - 1) / group > cus)
        group *= 2u;
    shape->group = group;
    shape->groups = (uint32_t)((photons + group - 1) / group);
    /* three coordinates of each photon, a lane each; with a weigher 16 waves */
    shape->moving = (3u * group + 63u) / 64u;
    shape->drawing = 15u - shape->moving;
    shape->grid = std::min(shape->groups, cus);
    /* blocks of sums: 8 take 256 workgroups' additions without much waiting
     * (1: 40 us more, 32: 4 us more, for adding them up) */
    shape->copies = std::min(8u, std::max(1u, shape->grid / 4u));
    const uint64_t room = ((uint64_t)TMC_MAX_SHELLS * 4 + 4) / (4ull * shells + 4);
    if (shape->copies > room)
        shape->copies = (uint32_t)room;
    return true;
}

/* Measured on MI355X, equal sets, a run of a kept plan by walk_multi and by the
 * lockstep launches.  Launching 64 photons and appending their survivors costs
 * about 17 ps a photon, which a cycle of 30 absorptions (1.95 and 1.65 ps each)
 * earns back: 131e6 photons in 2000 sets, first cycles of 2, 5, 10, 31 and, 20e6
 * in 300 sets, 73 absorptions: 1.46 and 2.84, 2.20 and 3.26, 3.22 and 4.26, 8.66
 * and 8.53, 3.26 and 2.83 ms.  In shorter cycles it is for the batches that
 * walk_multi's lanes walk in one claim each, 0.5 ms however few they are
 * (cycles of 10: 64 sets of 2^16 photons 603 and 553 us, 8 of 2^18 582 and 533,
 * of 2^20 659 and 789; 2000 of one photon 381 and 417), down to cycles of 8 (of 2:
 * 8 sets of 2^14 386 and 449 us, of 2^18 621 and 1098).
 *
 * All waves append to the count of the set they walk, and additions to one
 * address take more than 11 ns each, while 8192 waves end a batch of 64 photons
 * every 0.1 k1 ns: with not enough sets under way at a time they wait for one
 * another, and more so where lockstep has little to gain (eight sets of 2^22
 * photons, cycles of 31: 2.60 and 4.62 ms, of 73: 5.61 and 6.57, of 2^20, 73:
 * 1.65 and 1.69; four of 2^21, 31: 1.03 and 1.29, 54: 1.47 and 1.65, 73: 1.71 and
 * 1.92, 211: 4.85 and 3.92).
 *
 * A plan made for one run has to earn what laying it out and releasing it takes
 * more, 0.1 ms and 0.1 us a set, and 0.3 ms for large lists (planned, run and
 * released, default physics: one set of 64 photons 222 and 231 us, of 1000 561
 * and 338; 2000 sets of 64 863 and 920, of 1000 1394 and 1296; 10,000 of 1000 4816
 * and 5670; 8 of 2^20 1845 and 1981; cycles of 31, one of 2^20 655 and 718, 64 of
 * 2^16 856 and 810; of 10, 64 of 2^14 681 and 519, of 2^16 706 and 792; albedo
 * 0.99, 2000 of 1000 7022 and 5655, 8 of 2^18 4701 and 3568). */
bool tmc::lockstep_batch(const std::vector<LockLoad>& sets, double waves, bool once)
{
    double photons = 0.0, steps = 0.0;
    for (const LockLoad& s : sets) {
        photons += s.photons;
        steps += s.photons * s.k1;
    }
    const double n = (double)sets.size(), mean = photons > 0.0 ? steps / photons : 0.0;
    constexpr double many = 4194304.0;
    if (mean < 8.0 || (mean < 30.0 && (photons >= many || n > 1000.0)))
        return false;
    if (once && (steps < 40.0 * n * n || (mean < 100.0 && (steps < 30000.0 || photons >= many))
                 || (mean < 30.0 && photons > many / 4.0)
                 || (mean >= 30.0 && mean < 100.0 && photons >= many / 4.0 && photons >= many / 16.0 * n)))
        return false;
    /* work of the sets whose waves wait for their count: a wave's 32nd of a
     * launch is a chunk */
    const double each = std::max(kLockChunkSteps, steps / 64.0 / waves / 32.0);
    double waits = 0.0;
    for (const LockLoad& s : sets) {
        const double chunks = s.photons / 64.0 / std::ceil(each / s.k1);
        if (s.k1 * std::max(1.0, waves / chunks) < (s.k1 < 100.0 ? 200.0 : 120.0))
            waits += s.photons * s.k1;
    }
    return waits <= steps / 8.0;
}

/* Entries of the binary32 walk's weight table (0: the walk multiplies).
 * The table is built per workgroup when the launch starts, so small runs
 * multiply; it must span the first cycle and eight more (a photon survives
 * eight roulettes with probability 1e-8), or the lanes past its end would
 * run the arithmetic beside it on most steps.  Automatic for both samplers
 * (measured at default physics, 2^30 photons: analytic 157.0 -> 150.6 ms,
 * rejection 260.0 -> 257.1 ms, whose retry iterations read an entry they do
 * not use). */
uint32_t tmc::weight_table_entries(const tmc_params* p, uint32_t precision, uint64_t photons, uint32_t request)
{
    if (precision != TMC_PRECISION_FP32 || request == TMC_WEIGHT_TABLE_OFF)
        return 0;
    if (request)
        return std::min<uint32_t>(request, TMC_WALK_TABLE_MAX);
    if (photons < (1ull << 20))
        return 0;
    uint32_t k1 = 0, k2 = 0;
    if (!weight_cadence(p, TMC_WALK_TABLE_MAX, &k1, &k2) || (uint64_t)k1 + 8ull * k2 > TMC_WALK_TABLE_MAX)
        return 0;
    return (uint32_t)std::min<uint64_t>(TMC_WALK_TABLE_MAX, (uint64_t)k1 + 24ull * k2);
}

int tmc::plan_passes(const std::vector<PlanSet>& sets, uint64_t chunk_work, uint32_t max_passes,
                     const ShapeFn& shape_of, std::vector<PlanPass>* passes, std::vector<PlanChunk>* chunks)
{
    passes->clear();
    chunks->clear();
    const size_t nsets = sets.size();
    double work = 0.0;
    for (const PlanSet& s : sets)
        work += s.L * (double)s.photons;

    /* LDS size classes: the distinct shell counts, ascending, grouped by the
     * launch shape they allow */
    std::vector<uint32_t> svals;
    for (const PlanSet& s : sets)
        svals.push_back(s.shells);
    std::sort(svals.begin(), svals.end());
    svals.erase(std::unique(svals.begin(), svals.end()), svals.end());
    std::vector<double> swork(svals.size(), 0.0);
    for (const PlanSet& s : sets) {
        const size_t k = (size_t)(std::lower_bound(svals.begin(), svals.end(), s.shells) - svals.begin());
        swork[k] += s.L * (double)s.photons;
    }
    std::vector<PlanPass> groups;
    for (size_t k = 0; k < svals.size(); ++k) {
        PlanShape shape;
        const int rc = shape_of(svals[k], &shape);
        if (rc != TMC_OK)
            return rc;
        if (!groups.empty() && groups.back().shape.grid == shape.grid && groups.back().shape.block == shape.block) {
            groups.back().hi = svals[k];
            groups.back().work += swork[k];
        } else {
            PlanPass g;
            g.lo = g.hi = svals[k];
            g.shape = shape;
            g.work = swork[k];
            groups.push_back(g);
        }
    }
    /* a class with under a tenth of the work joins its neighbour with more
     * shells (whose slots hold both), and there are at most max_passes */
    while (groups.size() > 1) {
        size_t m = 0;
        for (size_t k = 1; k < groups.size(); ++k)
            if (groups[k].work < groups[m].work)
                m = k;
        if (groups[m].work >= 0.1 * work && groups.size() <= max_passes)
            break;
        const size_t lo_i = m + 1 < groups.size() ? m : m - 1, hi_i = lo_i + 1;
        PlanPass g = groups[hi_i];
        g.lo = groups[lo_i].lo;
        g.work += groups[lo_i].work;
        groups[lo_i] = g;
        groups.erase(groups.begin() + (ptrdiff_t)hi_i);
    }

    /* chunk queues, one per pass */
    struct Item {
        PlanChunk ch;
        double dur;
    };
    std::vector<std::vector<Item>> items(groups.size());
    for (PlanPass& g : groups) {
        const double waves = (double)g.shape.grid * (g.shape.block / 64u);
        g.chunk_work = chunk_work ? chunk_work : (uint64_t)std::max(65536.0, g.work / (16.0 * std::max(waves, 1.0)));
    }
    for (size_t i = 0; i < nsets; ++i) {
        const uint64_t N = sets[i].photons;
        if (!N)
            continue;
        size_t g = 0;
        while (sets[i].shells > groups[g].hi)
            ++g;
        const double L = sets[i].L;
        double per_lane = std::ceil((double)groups[g].chunk_work / (64.0 * L));
        per_lane = std::min(std::max(per_lane, 1.0), (double)(1u << 24));
        uint64_t C = 64u * (uint64_t)per_lane;
        /* keep the queue below 2^24 chunks */
        const uint64_t min_c = (N >> 24) + 1;
        if (C < min_c)
            C = (min_c + 63) / 64 * 64;
        if (C > (1ull << 31))
            C = 1ull << 31;
        for (uint64_t first = 0; first < N; first += C) {
            const uint64_t cnt = std::min(C, N - first);
            items[g].push_back({ { (uint32_t)i, (uint32_t)cnt, first }, (double)((cnt + 63) / 64) * L });
        }
    }
    for (auto& v : items)
        std::stable_sort(v.begin(), v.end(), [](const Item& x, const Item& y) { return x.dur > y.dur; });
    /* the pass with the longest chunk first, so that the launch sequence ends
     * on short chunks */
    std::vector<size_t> order(groups.size());
    for (size_t g = 0; g < order.size(); ++g)
        order[g] = g;
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) {
        const double dx = items[x].empty() ? 0.0 : items[x][0].dur, dy = items[y].empty() ? 0.0 : items[y][0].dur;
        return dx > dy;
    });
    for (size_t g : order) {
        if (items[g].size() > UINT32_MAX)
            return TMC_E_RANGE; /* a pass's queue length is a 32-bit kernel argument */
        PlanPass q = groups[g];
        q.first_chunk = chunks->size();
        q.nchunks = items[g].size();
        for (const Item& it : items[g])
            chunks->push_back(it.ch);
        passes->push_back(q);
    }
    return TMC_OK;
}

void tmc::Arena::init(uint64_t words)
{
    free_.clear();
    if (words)
        free_[0] = words;
}

bool tmc::Arena::alloc(uint64_t n, uint64_t* off)
{
    for (auto it = free_.begin(); it != free_.end(); ++it) {
        if (it->second >= n) {
            *off = it->first;
            const uint64_t rest = it->second - n, at = it->first + n;
            free_.erase(it);
            if (rest)
                free_[at] = rest;
            return true;
        }
    }
    return false;
}

void tmc::Arena::release(uint64_t off, uint64_t n)
{
    auto it = free_.emplace(off, n).first;
    auto nx = std::next(it);
    if (nx != free_.end() && it->first + it->second == nx->first) {
        it->second += nx->second;
        free_.erase(nx);
    }
    if (it != free_.begin()) {
        auto pv = std::prev(it);
        if (pv->first + pv->second == it->first) {
            pv->second += it->second;
            free_.erase(it);
        }
    }
}

uint64_t tmc::chunk_photons(double work, double L, uint64_t max_per_lane, uint64_t left)
{
    double per_lane = std::floor(work / (64.0 * L));
    per_lane = std::min(std::max(per_lane, 1.0), (double)max_per_lane);
    return std::max<uint64_t>(1, std::min<uint64_t>(left, 64u * (uint64_t)per_lane));
}

double tmc::backlog_share(uint64_t photons, double L, double cap)
{
    return std::min((double)photons * L, cap);
}

double tmc::serve_chunk_scale(double backlog, double base_work, uint32_t waves, double chunks_per_wave,
                              uint32_t max_scale)
{
    return std::min(std::max(1.0, backlog / (chunks_per_wave * base_work * (double)waves)), (double)max_scale);
}
