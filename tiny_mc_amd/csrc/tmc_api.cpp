/* C ABI of the photon-transport path (include/tiny_mc_gpu.h).
 *
 * Host side of one run: validate the params.h-style parameters, derive the
 * binary32 constants exactly as photon.c:8-9 does, form the weights, and launch
 * the lockstep walks, whose last workgroup writes the 128-bit integer tallies
 * into host memory; or, where those don't apply, clear the device words, launch
 * the persistent walk kernel once, and copy the tallies back.  The conversion to
 * the reference's heat / heat2 units is done in double on the host.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <mutex>
#include <vector>

#include "../../include/tiny_mc_gpu.h"
#include "tmc_cohort.h"
#include "tmc_context.h"
#include "tmc_internal.h"

#define TMC_EXPORT extern "C" __attribute__((visibility("default")))

using tmc::Context;

namespace {

std::mutex g_mutex;
Context* g_ctx = nullptr;

int destroy_context(Context* c)
{
    if (!c)
        return TMC_OK;
    (void)hipSetDevice(c->device);
    if (c->d_work)
        tmc::release_device(c->d_work);
    tmc::release_device(c->d_table);
    tmc::release_device(c->d_lists);
    tmc::release_host(c->h_out);
    tmc::release_host(c->h_weight);
    if (c->ev_start)
        (void)hipEventDestroy(c->ev_start);
    if (c->ev_stop)
        (void)hipEventDestroy(c->ev_stop);
    if (c->stream)
        (void)hipStreamDestroy(c->stream);
    delete c;
    return TMC_OK;
}

/* Creates the context on `device` (-1: the current device). */
int create_context(int device, Context** out)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0)
        return TMC_E_NODEVICE;
    if (device < 0) {
        if (hipGetDevice(&device) != hipSuccess)
            return TMC_E_NODEVICE;
    }
    if (device >= count)
        return TMC_E_NODEVICE;
    if (hipSetDevice(device) != hipSuccess)
        return TMC_E_HIP;
    Context* c = new (std::nothrow) Context;
    if (!c)
        return TMC_E_NOMEM;
    c->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
        delete c;
        return TMC_E_HIP;
    }
    c->compute_units = prop.multiProcessorCount;
    std::snprintf(c->arch, sizeof c->arch, "%s", prop.gcnArchName);
    /* default-priority stream (never a prioritised one); no device memory
     * yet: the single-run words are allocated at the first run, so that the
     * no-allocation entry point can create the context too */
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess
        || hipEventCreate(&c->ev_start) != hipSuccess || hipEventCreate(&c->ev_stop) != hipSuccess) {
        destroy_context(c);
        return TMC_E_HIP;
    }
    /* the static scratch's address on this device; a failure here is
     * reported by tiny_mc_gpu_run_noalloc, the only user */
    (void)tmc::scratch_setup(device);
    *out = c;
    return TMC_OK;
}

} // namespace

std::mutex& tmc::api_mutex() { return g_mutex; }

int tmc::acquire_context(Context** out)
{
    if (!g_ctx) {
        int rc = create_context(-1, &g_ctx);
        if (rc != TMC_OK)
            return rc;
    }
    if (hipSetDevice(g_ctx->device) != hipSuccess)
        return TMC_E_HIP;
    *out = g_ctx;
    return TMC_OK;
}

namespace {

/* An allocation that failed: its error must not meet the next launch, which
 * returns the last one. */
bool no_memory()
{
    (void)hipGetLastError();
    return false;
}

/* The single-run words at the largest shell count, once per context. */
int ensure_work(Context* c)
{
    if (!c->d_work
        && hipMalloc((void**)&c->d_work, tmc::run_work_words(TMC_MAX_SHELLS) * sizeof(unsigned long long))
            != hipSuccess) {
        c->d_work = nullptr;
        no_memory();
        return TMC_E_NOMEM;
    }
    return TMC_OK;
}

/* n values of host-coherent memory, the first of them zero, and their device
 * address, once. */
template <class T>
bool host_values(T** host, T** device, size_t n)
{
    if (*host)
        return true;
    T *h = nullptr, *d = nullptr;
    if (hipHostMalloc((void**)&h, n * sizeof(T), hipHostMallocCoherent) != hipSuccess)
        return no_memory();
    if (hipHostGetDevicePointer((void**)&d, h, 0) != hipSuccess) {
        tmc::release_host(h);
        return no_memory();
    }
    h[0] = 0;
    *host = h;
    *device = d;
    return true;
}

/* What the cohort and lockstep walks need beside those words (20 MB): each
 * piece is allocated once, and without one of them the run is lane per
 * photon. */
bool ensure_lockstep(Context* c)
{
    if (!host_values(&c->h_out, &c->d_out, tmc::run_work_words(TMC_MAX_SHELLS))
        || !host_values(&c->h_weight, &c->d_weight, tmc::kTableEntries))
        return false;
    if (!c->d_table && hipMalloc(&c->d_table, 16ull * tmc::kTableEntries) != hipSuccess) {
        c->d_table = nullptr;
        return no_memory();
    }
    return true;
}

/* Releases made while a serving kernel is resident (tmc_context.h). */
std::mutex g_release_mutex;
int g_serving_kernels = 0, g_serving_waiting = 0, g_lockstep_runs = 0;
std::vector<std::function<void()>> g_deferred;

} // namespace

void tmc::release(std::function<void()> fn)
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    if (g_serving_kernels > 0)
        g_deferred.push_back(std::move(fn));
    else
        fn();
}

void tmc::release_device(void* p)
{
    if (p)
        release([p]() { (void)hipFree(p); });
}

void tmc::release_host(void* p)
{
    if (p)
        release([p]() { (void)hipHostFree(p); });
}

tmc::LockstepRun::LockstepRun()
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    on_ = g_serving_kernels == 0 && g_serving_waiting == 0;
    g_lockstep_runs += on_;
}

tmc::LockstepRun::~LockstepRun()
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    g_lockstep_runs -= on_;
}

bool tmc::serving()
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    return g_serving_kernels > 0 || g_serving_waiting > 0;
}

bool tmc::serving_kernel_started(bool* waiting)
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    const bool wait = g_lockstep_runs > 0;
    g_serving_waiting += (int)wait - (int)*waiting;
    *waiting = wait;
    g_serving_kernels += !wait;
    return !wait;
}

void tmc::serving_kernel_waived(bool* waiting)
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    g_serving_waiting -= *waiting;
    *waiting = false;
}

void tmc::serving_kernel_left()
{
    std::lock_guard<std::mutex> lock(g_release_mutex);
    if (--g_serving_kernels > 0)
        return;
    std::vector<std::function<void()>> todo;
    todo.swap(g_deferred);
    for (auto& fn : todo)
        fn();
}

namespace {

double u128_to_double(uint64_t lo, uint64_t hi)
{
    /* hi * 2^64 + lo, with one rounding of the 128-bit value in the common
     * case hi == 0 */
    return std::ldexp((double)hi, 64) + (double)lo;
}

} // namespace

namespace {

/* Longest time a run spins on its result's token before it waits for the
 * stream: the token comes 10 us before hipStreamSynchronize returns, which
 * matters to runs of tens of microseconds. */
constexpr std::chrono::microseconds kSpin(500);

/* The weight table of a run and the arguments its launches share.  `cuts`:
 * roulettes the table is to span.  False if it does not fit.  A capped run's
 * table ends with the cap, and its roulettes with ones that are never reached
 * (100 photons stopped after 100 absorptions, the whole table and this: albedo
 * 0.9999 161 and 25 us; 1 - 1e-6, which does not fit, 1376 and 22 us). */
bool weigh(Context* c, const tmc_params* p, uint64_t seed, uint64_t kcap, uint32_t cuts, tmc::CohortArgs* a)
{
    std::memset(a, 0, sizeof *a);
    constexpr uint32_t room = (uint32_t)tmc::kTableEntries - 2u;
    a->ncuts = tmc::weight_sequence(p, (uint32_t)std::min<uint64_t>(room, kcap), cuts, c->h_weight, a->cut, &a->w_end);
    if (a->ncuts < cuts && kcap > room)
        return false;
    a->entries = a->ncuts < cuts ? (uint32_t)kcap : a->cut[a->ncuts - 1];
    while (a->ncuts < cuts)
        a->cut[a->ncuts++] = ~0u;
    a->weight = c->d_weight;
    a->entry = c->d_table;
    a->seed = seed;
    a->albedo = tmc::derived_albedo(p);
    a->spm = tmc::derived_spm(p);
    a->shell_max = (float)(p->shells - 1);
    a->shells = p->shells;
    a->kcap = (uint32_t)kcap;
    a->work = c->d_work;
    a->out = c->d_out;
    return true;
}

/* About the absorptions of a photon's first cycle (the weight falls to a
 * thousandth), at most kcap. */
double first_cycle(const tmc_params* p, uint64_t kcap)
{
    const double a = (double)tmc::derived_albedo(p);
    const double k = a > 0.0 ? std::log(0.001) / std::log(a) : 1.0;
    return std::min(std::max(k, 1.0), (double)kcap);
}

void use_shape(const tmc::CohortShape& s, tmc::CohortArgs* a)
{
    a->group = s.group;
    a->drawing = s.drawing;
    a->moving = s.moving;
    a->copies = s.copies;
}

/* Enqueues a run by `launches` behind what clears the device words, unless a
 * server has the device (TMC_E_UNSUPPORTED), and waits for its result. */
int finish_enqueued(Context* c, uint64_t token, uint32_t shells, uint64_t* tally, tmc_run_stats* st,
                    const std::function<bool()>& launches)
{
    const tmc::LockstepRun run;
    if (!run)
        return TMC_E_UNSUPPORTED;
    const bool zero = c->work_zero;
    c->work_zero = false;
    if ((!zero && tmc::launch_clear(c->d_work, tmc::run_work_words(TMC_MAX_SHELLS), c->stream) != hipSuccess)
        || !launches()) {
        (void)hipStreamSynchronize(c->stream); /* h_weight may still be read */
        return TMC_E_HIP;
    }
    const auto t0 = std::chrono::steady_clock::now();
    while (__atomic_load_n(&c->h_out[0], __ATOMIC_ACQUIRE) != token) {
        if (std::chrono::steady_clock::now() - t0 > kSpin) {
            if (hipStreamSynchronize(c->stream) != hipSuccess
                || __atomic_load_n(&c->h_out[0], __ATOMIC_ACQUIRE) != token)
                return TMC_E_HIP;
        }
    }
    c->work_zero = true;
    std::memcpy(tally, c->h_out + TMC_COHORT_COUNTERS, 4 * (size_t)shells * sizeof(uint64_t));
    if (st) {
        st->interactions = c->h_out[1];
        st->truncated = c->h_out[2];
        st->kernel_ms = 1e-5 * (double)c->h_out[3]; /* 100 MHz ticks */
    }
    return TMC_OK;
}

/* Photons of the largest run for the cohort walk. */
uint64_t cohort_most(const tmc_params* p, const tmc_options* o)
{
    if (p->shells > TMC_LOCK_SHELLS)
        return TMC_COHORT_PHOTONS_WIDE;
    return o->sampler == TMC_SAMPLER_ANALYTIC ? TMC_COHORT_PHOTONS : TMC_COHORT_PHOTONS_REJECTION;
}

/* One binary32 run by the cohort walk.  TMC_E_UNSUPPORTED: not one for it. */
int run_cohort(Context* c, const tmc_params* p, uint64_t seed, const tmc_options* o, uint64_t kcap, uint64_t* tally,
               tmc_run_stats* st)
{
    tmc::CohortShape shape;
    const uint64_t most = cohort_most(p, o);
    if (!tmc::cohort_shape(p->photons, most, first_cycle(p, kcap), p->shells, (uint32_t)c->compute_units, &shape))
        return TMC_E_UNSUPPORTED;
    tmc::CohortArgs a;
    if (!weigh(c, p, seed, kcap, tmc::cuts_for((double)p->photons), &a))
        return TMC_E_UNSUPPORTED;
    a.build = a.entries <= TMC_COHORT_BUILD ? a.entries : 0u;
    if (tmc::cohort_lds_bytes(p->shells, a.build) > 160u * 1024u)
        return TMC_E_UNSUPPORTED;
    a.first_photon = o->first_photon;
    a.photons = p->photons;
    a.finish = 1;
    a.token = ++c->token;
    use_shape(shape, &a);
    const uint32_t block = 64u * (a.drawing + a.moving + (a.build ? 1u : 0u));
    const int rc = finish_enqueued(c, a.token, p->shells, tally, st, [&]() {
        return (a.build
                || tmc::launch_cohort_table(a.weight, a.entries, c->d_table, nullptr, 0, nullptr, c->stream)
                    == hipSuccess)
            && tmc::launch_cohort(o->sampler, o->math, a, shape.grid, block, c->stream) == hipSuccess;
    });
    if (rc == TMC_OK && st) {
        st->grid = shape.grid;
        st->block = block;
        st->chunk = a.group;
    }
    return rc;
}

/* Survivors of a large run that the cohort walk takes over: with fewer, the
 * lockstep waves leave most of the chip idle.  Flat from 40,000 to 250,000 (2^20
 * photons 236 and 233 us, 2^26 8.59 and 8.61 ms); 15,000 cost 2^20 photons 5 us. */
constexpr uint32_t kHandOver = 40000;

/* Photons whose survivors share one of `stripes` stripes, at most: those of
 * every stripes-th workgroup, with room for waves that claim more than
 * others. */
uint32_t list_photons(uint32_t photons, uint32_t stripes)
{
    const uint32_t share = photons / stripes;
    return share + share / 8u + 4096u;
}

/* Places of a stripe of a survivor list, for n photons that share it: a tenth
 * survive a roulette, so an eighth and a slack of 256 for the first list, an
 * eighth of that for the second. */
uint32_t list_cap(uint32_t which, uint32_t n) { return (which ? n / 64u : n / 8u) + 256u; }

/* Constants of the precision variants (WalkArgs, PrecArgs): formed in FP64,
 * each rounded once. */
template <class Args>
void precision_constants(const tmc_params* p, Args* a)
{
    const double mu_a = p->mu_a, mu_s = p->mu_s;
    a->albedo_d = mu_s / (mu_s + mu_a);
    a->spm_d = 1e4 / (double)p->microns_per_shell / (mu_a + mu_s);
    const double l2a = std::log2(a->albedo_d), l2s = -std::log2((double)0.1f);
    a->l2a_hi = (float)l2a;
    a->l2a_lo = (float)(l2a - (double)a->l2a_hi);
    a->l2s_hi = (float)l2s;
    a->l2s_lo = (float)(l2s - (double)a->l2s_hi);
    a->spm_w = (float)a->spm_d;
}

/* Room for lists of `bytes` bytes beside the start time and the counters of a
 * large run, kept for the next one. */
bool keep_lists(Context* c, size_t bytes)
{
    bytes += 4ull * tmc::kRunCounters + 8;
    if (c->d_lists && c->lists_bytes >= bytes)
        return true;
    tmc::release_device(c->d_lists);
    c->d_lists = nullptr;
    if (hipMalloc(&c->d_lists, bytes) != hipSuccess) {
        c->d_lists = nullptr;
        return no_memory();
    }
    c->lists_bytes = bytes;
    return true;
}

/* Photons of a run in slices: at most `most` in each, none across a multiple of
 * 2^32. */
struct Slice {
    uint64_t first;
    uint32_t photons;
};

std::vector<Slice> slices_of(uint64_t first, uint64_t photons, uint64_t most)
{
    std::vector<Slice> slices;
    for (uint64_t done = 0; done < photons;) {
        const uint64_t at = first + done;
        const uint64_t n = std::min<uint64_t>(std::min<uint64_t>(most, photons - done),
                                              (1ull << 32) - (at & 0xFFFFFFFFull));
        slices.push_back({ at, (uint32_t)n });
        done += n;
    }
    return slices;
}

/* Threads of a lockstep launch's workgroups for `waves` waves of work: half of
 * TMC_LOCK_BLOCK where that leaves fewer waves on the fullest compute unit, if
 * the waves are all resident (half as large, at least twice as many workgroups
 * are: 8 of them take 60 KB of LDS, with the rejection sampler 6 take 90), else
 * TMC_LOCK_BLOCK, with half as many sums to add up, which is what a cycle of
 * fewer than 64 steps takes.  (Albedo 0.99: 50,000 photons, 98 workgroups of
 * eight waves or 196 of four, 237 and 198 us; 180,000 421 and 352 us; 2^17
 * photons at default physics 58 and 61 us.) */
uint32_t lock_block_for(double waves, uint32_t steps, uint32_t grid_most, uint32_t cus)
{
    const auto fullest = [=](double per_wg) { return per_wg * std::ceil(std::ceil(waves / per_wg) / (double)cus); };
    constexpr double per_wg = TMC_LOCK_BLOCK / 64u;
    return steps >= 64u && waves <= per_wg * (double)grid_most && fullest(per_wg / 2.0) < fullest(per_wg)
        ? TMC_LOCK_BLOCK / 2u
        : TMC_LOCK_BLOCK;
}

/* One large binary32 run by lockstep waves, level by level, and the cohort
 * walk for the last survivors.  TMC_E_UNSUPPORTED: not one for it. */
int run_lock(Context* c, const tmc_params* p, uint64_t seed, const tmc_options* o, uint64_t kcap, uint64_t* tally,
             tmc_run_stats* st)
{
    if (p->photons <= cohort_most(p, o) || p->photons > (1ull << 40) || p->shells > TMC_LOCK_SHELLS)
        return TMC_E_UNSUPPORTED;
    /* many photons of short walks: launching them 64 at a time and appending
     * the survivors costs what the step saves (2^27 photons, lane per photon
     * and here: albedo 1/6 1548 and 1685 us, with the rejection sampler 2216
     * and 2290 us; albedo 0.5 2849 and 2784 us, 4885 and 4696 us; 2^26 at 1/6
     * 1049 and 850 us; rejection sampler at 0.01 and 0.09, 4 * 2^23 photons 663
     * and 485, 684 and 635 us, 6 * 2^23 685 and 687, 814 and 909, 2^26 773 and
     * 868, 970 and 1176; at 0.2, 2^26 1399 and 1306) */
    const double first = first_cycle(p, kcap);
    if (first < 8.0
        && p->photons > (o->sampler == TMC_SAMPLER_REJECTION && first < 4.0 ? 5ull << 23 : 1ull << 26))
        return TMC_E_UNSUPPORTED;
    const uint64_t slice = std::min<uint64_t>(p->photons, 1ull << tmc::kSliceLog);
    uint32_t levels = 1;
    double rest = 0.1 * (double)slice; /* survivors the cohort walk takes over */
    for (; rest > (double)kHandOver; rest *= 0.1)
        ++levels;
    tmc::CohortArgs a;
    if (!weigh(c, p, seed, kcap, levels + tmc::cuts_for(rest), &a))
        return TMC_E_UNSUPPORTED;
    if (tmc::cohort_lds_bytes(p->shells, 0) > 160u * 1024u)
        return TMC_E_UNSUPPORTED;
    /* the lists, counters and start time */
    uint32_t log = 20;
    while ((1ull << log) < slice)
        ++log;
    const uint32_t most = list_photons(1u << log, tmc::kStripes);
    const size_t places[2] = { (size_t)tmc::kStripes * list_cap(0, most), (size_t)tmc::kStripes * list_cap(1, most) };
    if (!keep_lists(c, 28 * (places[0] + places[1])))
        return TMC_E_UNSUPPORTED;
    unsigned long long* const start = (unsigned long long*)c->d_lists;
    uint32_t* const counters = (uint32_t*)(start + 1);
    tmc::PhotonList lists[2];
    float* at = (float*)(counters + tmc::kRunCounters);
    for (uint32_t w = 0; w < 2; ++w) {
        lists[w].photon = (uint32_t*)at;
        at += places[w];
        for (float*& f : lists[w].state) {
            f = at;
            at += places[w];
        }
    }
    const std::vector<Slice> slices = slices_of(o->first_photon, p->photons, slice);
    const uint32_t words = tmc::kStripes * TMC_LOCK_LINE; /* of a level's counts */
    const uint32_t per_slice = levels * words + TMC_LOCK_RANGES * TMC_LOCK_LINE;
    if (slices.size() * per_slice > tmc::kRunCounters)
        return TMC_E_UNSUPPORTED;

    const uint32_t cus = (uint32_t)c->compute_units;
    /* (the batches go round the resident waves, so a workgroup that had to wait
     * for another to end would double the launch's time) */
    int per_cu = 0;
    if (tmc::lock_occupancy(o->sampler, o->math, 0u, p->shells, &per_cu) != hipSuccess || per_cu <= 0)
        return TMC_E_HIP;
    const uint32_t grid_most = (uint32_t)per_cu * cus;
    /* the first cycle counted: where the counts of four workgroups fit a CU's
     * LDS, and a slice has the work to make up for adding them up at the end
     * (first cycles of 1.6e8 absorptions: 508 us summed, 536 counted; 2.2e8
     * 528 and 528; 6e8 1231 and 1159; 4.8e9 7.93 and 7.75 ms) */
    const uint32_t k_first = std::min(a.cut[0], a.kcap);
    const bool counted = o->sampler == TMC_SAMPLER_ANALYTIC && (double)slice * (double)k_first >= 3e8
        && tmc::lock_count_bytes(p->shells, k_first) <= 40u * 1024u;
    int counted_cu = 0;
    if (counted
        && (tmc::lock_occupancy(o->sampler, o->math, k_first, p->shells, &counted_cu) != hipSuccess
            || counted_cu <= 0))
        return TMC_E_HIP;
    tmc::CohortShape shape;
    tmc::cohort_shape((uint64_t)std::max(1.0, rest), kHandOver + 1u, first_cycle(p, kcap), p->shells, cus, &shape);
    use_shape(shape, &a);
    a.copies = 8; /* (at most 450 shells: they fit) */
    a.token = ++c->token;
    a.start = start;
    a.list = lists[(levels - 1) & 1u];
    a.seg0 = levels;

    tmc::LockArgs l;
    std::memset(&l, 0, sizeof l);
    l.seed = seed;
    l.albedo = a.albedo;
    l.spm = a.spm;
    l.shell_max = a.shell_max;
    l.shells = a.shells;
    l.kcap = a.kcap;
    l.entry = c->d_table;
    l.work = c->d_work;
    l.copies = a.copies;
    uint32_t grid0 = 0, block0 = 0;
    auto launches = [&]() {
        /* two more entries than the steps read ahead of the last cut */
        if (tmc::launch_cohort_table(a.weight, a.entries, c->d_table, counters, (uint32_t)slices.size() * per_slice,
                                     start, c->stream)
            != hipSuccess)
            return false;
        for (size_t si = 0; si < slices.size(); ++si) {
            uint32_t* const count = counters + si * per_slice; /* survivors by level */
            double n = (double)slices[si].photons;
            bool capped = false;
            const uint32_t wgs = (uint32_t)std::min<double>(grid_most, std::ceil(n / TMC_LOCK_BLOCK));
            /* at least eight workgroups a stripe, or one stripe */
            l.stripes = std::min(std::min(tmc::kStripes, cus), std::max(1u, wgs / 8u));
            const uint32_t per = list_photons(slices[si].photons, l.stripes);
            l.first_photon = slices[si].first;
            l.photons = slices[si].photons;
            for (uint32_t lv = 0; lv < levels && !capped; ++lv, n *= 0.1) {
                l.level = lv;
                l.k0 = lv ? a.cut[lv - 1] : 0u;
                l.k1 = std::min(a.cut[lv], a.kcap);
                l.cut_ends = a.cut[lv] <= a.kcap;
                l.cap_ends = a.kcap <= a.cut[lv];
                capped = l.cap_ends;
                l.in = lists[(lv + 1) & 1u];
                l.out = lists[lv & 1u];
                l.in_count = count + (lv ? lv - 1 : 0) * words;
                l.in_cap = l.out_cap;
                l.out_count = count + lv * words;
                l.out_cap = list_cap(lv & 1u, per);
                const double waves = std::ceil(n / 64.0);
                const bool by_count = counted && lv == 0;
                const uint32_t block = by_count ? TMC_LOCK_BLOCK : lock_block_for(waves, l.k1 - l.k0, grid_most, cus);
                const uint32_t per_wg = block / 64u;
                /* (of half the size twice as many, with the rejection sampler:
                 * its waves' passes over retries differ, and one that takes a
                 * second batch ends late.  262,145 to 327,680 photons, albedo
                 * 0.99, capped as the large ones and all at once: 826 and 765
                 * to 957 and 888 us; analytic 490 and 495 at 300,000, default
                 * physics 93 and 96 us, for the sums) */
                const uint32_t most = by_count ? (uint32_t)counted_cu * cus
                    : o->sampler == TMC_SAMPLER_REJECTION ? grid_most * (TMC_LOCK_BLOCK / block)
                                                          : grid_most;
                const uint32_t grid =
                    std::max(l.stripes, (uint32_t)std::min<double>(most, std::ceil(waves / (double)per_wg)));
                l.chunk = 0;
                if (lv == 0) {
                    grid0 = grid;
                    block0 = block;
                    const uint64_t each = (uint64_t)waves / (per_wg * grid); /* batches a wave */
                    if (each >= 8) {
                        /* a wave's 32nd, but (short cycles) not less than 128
                         * absorptions: a range's claims take 7 to 16 ns each,
                         * one after the other (2^24 photons at albedo 0.5 854
                         * and 509 us, at 1/6 878 and 406 us) */
                        const uint64_t least = std::min<uint64_t>((127u + l.k1) / l.k1, each / 4);
                        l.chunk = 64u * (uint32_t)std::min<uint64_t>(32, std::max<uint64_t>(least, each / 32));
                        l.range = (slices[si].photons / TMC_LOCK_RANGES + 64u) / 64u * 64u;
                        l.cursor = count + levels * words;
                    }
                }
                if (tmc::launch_lock(o->sampler, o->math, by_count, l, grid, block, c->stream) != hipSuccess)
                    return false;
            }
            a.finish = si + 1 == slices.size();
            a.first_photon = slices[si].first;
            a.list_count = count + (levels - 1) * words;
            a.list_cap = list_cap((levels - 1) & 1u, per);
            a.stripes = l.stripes;
            if (tmc::launch_cohort(o->sampler, o->math, a, cus, 64u * (a.drawing + a.moving), c->stream)
                != hipSuccess)
                return false;
        }
        return true;
    };
    const int rc = finish_enqueued(c, a.token, p->shells, tally, st, launches);
    if (rc == TMC_OK && c->h_out[2] >= TMC_LOCK_OVERFLOW)
        return TMC_E_UNSUPPORTED;
    if (rc == TMC_OK && st) {
        st->grid = grid0;
        st->block = block0;
        st->chunk = 64;
    }
    return rc;
}

/* Photons from which on the survivors of a roulette are packed into full waves:
 * a wave on each SIMD. */
constexpr double kPackPhotons = 65536.0;

/* Photons of the largest run of a precision variant for the lockstep waves.
 * Short cycles end there for the reason they do in binary32, and the passes of a
 * wave over the directions that the rejection sampler draws again cost more than
 * lockstep saves on a full chip, which fewer photons of long walks fill.
 * Measured, lane per photon and here: weight from counts, albedo 0.01, 2^26
 * photons 804 and 776 us, 2^27 1222 and 1477; binary64 2^25 766 and 773, 2^26 1306
 * and 1509; albedo 0.5 2^27 4.50 and 4.28, 11.13 and 11.35 ms.  Rejection sampler,
 * weight from counts: albedo 0.2 2^25 1117 and 1118, 2^26 2025 and 2141 us; 0.5
 * 2^24 1122 and 1089, 2^25 1988 and 2071 us; 0.8 2^23 1543 and 1553, 2^24 2895 and
 * 2973 us; default 2^22 1904 and 1873, 2^23 3447 and 3509, 2^24 6470 and 6772 us;
 * albedo 0.97 2^23 9780 and 9875 us. */
uint64_t prec_most(const tmc_options* o, double first)
{
    const bool rejection = o->sampler == TMC_SAMPLER_REJECTION;
    if (first < 8.0)
        return rejection || o->precision == TMC_PRECISION_FP64 ? 1ull << 25 : 1ull << 26;
    return !rejection ? 1ull << 36 : first < 25.0 ? 1ull << 24 : 1ull << 22;
}

/* One run with a precision variant's arithmetic by lockstep waves.
 * TMC_E_UNSUPPORTED: not one for them. */
int run_prec(Context* c, const tmc_params* p, uint64_t seed, const tmc_options* o, uint64_t kcap, uint64_t* tally,
             tmc_run_stats* st)
{
    if (p->photons == 0 || p->shells > TMC_LOCK_SHELLS || kcap != 0xFFFFFFFFull
        || p->photons > prec_most(o, first_cycle(p, kcap)))
        return TMC_E_UNSUPPORTED;
    tmc::PrecArgs a;
    std::memset(&a, 0, sizeof a);
    precision_constants(p, &a);
    if (!(a.albedo_d > 0.0 && a.albedo_d < 1.0))
        return TMC_E_UNSUPPORTED;
    a.seed = seed;
    a.shell_max = (float)(p->shells - 1);
    a.shells = p->shells;
    const uint64_t slice = std::min<uint64_t>(p->photons, 1ull << tmc::kSliceLog);
    /* the table: the cuts that the last survivors are expected to need, each
     * cycle's length from its logarithm, and slack for the roundings on the way */
    const double l = -std::log(a.albedo_d), first = std::log(1000.0) / l, later = std::log(10.0) / l;
    a.cuts = tmc::cuts_for((double)slice);
    const double room = 1.001 * (first + a.cuts * later) + 3.0 * a.cuts + 64.0;
    if (room > (double)tmc::kTableEntries - 16.0)
        return TMC_E_UNSUPPORTED;
    a.entries = (uint32_t)room;
    a.entry = c->d_table;
    if (o->precision == TMC_PRECISION_FP64) {
        /* the weights and cuts themselves, in the memory that holds a binary32
         * run's weights: its products, one after the other, as the walk's */
        constexpr size_t kHead = 32; /* of its doubles */
        static_assert(sizeof(tmc::PrecHead) <= 8 * kHead, "head");
        const uint32_t most = (uint32_t)(tmc::kTableEntries / 2 - kHead);
        double* const weight = (double*)c->h_weight;
        tmc::PrecHead* const head = (tmc::PrecHead*)(weight + most);
        head->ncuts = head->pad = 0;
        uint32_t k = 0;
        double w = 1.0;
        while (head->ncuts < a.cuts && k < most) {
            weight[k++] = w;
            w *= a.albedo_d;
            if (w < (double)0.001f) {
                w /= (double)0.1f;
                head->cut[head->ncuts++] = k;
            }
        }
        if (head->ncuts < a.cuts)
            return TMC_E_UNSUPPORTED;
        head->w_end = w;
        a.entries = k;
        a.weight = (const double*)c->d_weight;
        a.host_head = (const tmc::PrecHead*)(a.weight + most);
    }

    /* launches: through one roulette each, while the survivors fill the chip */
    uint32_t packs = 0;
    for (double rest = (double)slice; rest > kPackPhotons; rest *= 0.1)
        ++packs;
    const uint32_t most = list_photons((uint32_t)slice, tmc::kStripes);
    const uint32_t planes = 1u + tmc::prec_words(o->precision);
    const size_t places[2] = { packs > 0 ? (size_t)tmc::kStripes * list_cap(0, most) : 0,
                               packs > 1 ? (size_t)tmc::kStripes * list_cap(1, most) : 0 };
    if (!keep_lists(c, sizeof(tmc::PrecHead) + 4ull * planes * (places[0] + places[1])))
        return TMC_E_UNSUPPORTED;
    unsigned long long* const start = (unsigned long long*)c->d_lists;
    uint32_t* const counters = (uint32_t*)(start + 1);
    a.head = (tmc::PrecHead*)(counters + tmc::kRunCounters);
    uint32_t* at = (uint32_t*)(a.head + 1);
    tmc::PrecList lists[2];
    for (uint32_t w = 0; w < 2; ++w) {
        lists[w] = { at, at + places[w], (uint32_t)places[w] };
        at += planes * places[w];
    }
    const std::vector<Slice> slices = slices_of(o->first_photon, p->photons, slice);
    const uint32_t words = tmc::kStripes * TMC_LOCK_LINE; /* of a list's counts */
    if (slices.size() * packs * words > tmc::kRunCounters)
        return TMC_E_UNSUPPORTED;

    const uint32_t block = 256, cus = (uint32_t)c->compute_units;
    int per_cu = 0;
    if (tmc::prec_occupancy(o->sampler, o->precision, block, p->shells, &per_cu) != hipSuccess || per_cu <= 0)
        return TMC_E_HIP;
    const uint32_t grid_most = (uint32_t)per_cu * cus;
    a.copies = 8;
    a.work = c->d_work;
    tmc::CohortArgs f;
    std::memset(&f, 0, sizeof f);
    f.shells = p->shells;
    f.copies = a.copies;
    f.finish = 1;
    f.list.photon = counters; /* (the sums are others', even with one workgroup) */
    f.start = start;
    f.token = ++c->token;
    f.work = c->d_work;
    f.out = c->d_out;
    uint32_t grid0 = 0;
    const int rc = finish_enqueued(c, f.token, p->shells, tally, st, [&]() {
        if (tmc::launch_prec_table(o->precision, a, counters, (uint32_t)slices.size() * packs * words, start, c->stream)
            != hipSuccess)
            return false;
        for (size_t si = 0; si < slices.size(); ++si) {
            uint32_t* const count = counters + si * packs * words;
            double n = (double)slices[si].photons;
            const uint32_t wgs = (uint32_t)std::min<double>(grid_most, std::ceil(n / 256.0));
            a.stripes = std::min(std::min(tmc::kStripes, cus), std::max(1u, wgs / 8u));
            const uint32_t per = list_photons(slices[si].photons, a.stripes);
            a.first_photon = slices[si].first;
            a.photons = slices[si].photons;
            for (uint32_t level = 0; level <= packs; ++level, n *= 0.1) {
                a.level = level;
                a.cycles = level < packs ? 1u : 0u;
                a.in = lists[(level + 1) & 1u];
                a.out = lists[level & 1u];
                a.in_count = count + (level ? level - 1 : 0) * words;
                a.in_cap = a.out_cap;
                a.out_count = count + level * words;
                a.out_cap = list_cap(level & 1u, per);
                const uint32_t grid = std::max(a.stripes, (uint32_t)std::min<double>(grid_most, std::ceil(n / 256.0)));
                if (level == 0)
                    grid0 = grid;
                if (tmc::launch_prec(o->sampler, o->precision, a, grid, block, c->stream) != hipSuccess)
                    return false;
            }
        }
        return tmc::launch_finish(f, c->stream) == hipSuccess;
    });
    if (rc == TMC_OK && c->h_out[2] >= TMC_LOCK_OVERFLOW)
        return TMC_E_UNSUPPORTED;
    if (rc == TMC_OK && st) {
        st->grid = grid0;
        st->block = block;
        st->chunk = 64;
    }
    return rc;
}

} // namespace

int tmc::run_walk(Context* c, const tmc_params* p, uint64_t seed, const tmc_options* o, unsigned long long* work,
                  uint64_t* tally, tmc_run_stats* st)
{
    const auto t0 = std::chrono::steady_clock::now();
    const uint32_t S = p->shells;
    if (o->sampler > TMC_SAMPLER_REJECTION || o->precision > TMC_PRECISION_FP64 || o->math > TMC_MATH_OWN)
        return TMC_E_INVALID;
    if (!tmc::photon_range_ok(o->first_photon, p->photons))
        return TMC_E_RANGE;

    uint32_t block = o->block ? o->block : 256u;
    if (block < 64u || block > 1024u || (block % 64u) != 0u)
        return TMC_E_INVALID;
    uint32_t chunk = o->chunk;
    if (chunk && (chunk < 64u || (chunk % 64u) != 0u || chunk > (1u << 24)))
        return TMC_E_INVALID;
    uint64_t kcap = o->max_interactions ? o->max_interactions : 0xFFFFFFFFull;
    if (kcap > 0xFFFFFFFFull)
        kcap = 0xFFFFFFFFull;
    if (o->reserved)
        return TMC_E_INVALID;
    const uint32_t table_k = tmc::weight_table_entries(p, o->precision, p->photons, o->weight_table);
    /* the cohort and lockstep walks: runs of the allocating entry point with no
     * launch shape or table asked for (cohort_shape has the sizes), unless a
     * server has the device */
    if (work == c->d_work && !o->block && !o->grid && !o->chunk && !o->weight_table && p->photons && !tmc::serving()
        && ensure_lockstep(c)) {
        int rc = TMC_E_UNSUPPORTED;
        try {
            if (o->precision == TMC_PRECISION_FP32) {
                rc = run_cohort(c, p, seed, o, kcap, tally, st);
                if (rc == TMC_E_UNSUPPORTED)
                    rc = run_lock(c, p, seed, o, kcap, tally, st);
            } else {
                rc = run_prec(c, p, seed, o, kcap, tally, st);
            }
        } catch (const std::bad_alloc&) {
            /* (all that they allocate is there before the first launch) */
        }
        if (rc == TMC_OK && st) {
            st->photons = p->photons;
            st->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
            st->sampler = o->sampler;
            st->precision = o->precision;
            st->math = o->math;
            st->weight_table = table_k;
        }
        if (rc != TMC_E_UNSUPPORTED)
            return rc;
    }
    uint32_t grid = o->grid;
    if (grid == 0) {
        int per_cu = 0;
        if (tmc::walk_occupancy(o->sampler, o->precision, o->math, block, S, table_k, &per_cu) != hipSuccess
            || per_cu <= 0)
            return TMC_E_HIP;
        grid = (uint32_t)per_cu * (uint32_t)c->compute_units;
    }
    /* Do not launch far more waves than photons to walk. */
    const uint64_t waves_needed = (p->photons + 63u) / 64u;
    const uint32_t waves_per_wg = block / 64u;
    const uint64_t wg_needed = (waves_needed + waves_per_wg - 1) / waves_per_wg;
    if (wg_needed < grid)
        grid = (uint32_t)(wg_needed ? wg_needed : 1u);
    if (!chunk) {
        /* photons a wave claims at a time (64 per lane-photon): about 256
         * expected absorptions per lane between two claims, as a wave waits
         * for its claim's device-scope atomic (short walks would otherwise
         * claim every few steps, all waves on one counter), at least 4 per
         * lane, and few enough that each wave gets about 4 claims, so the
         * waves finish together */
        const double L = std::max(1.0, tmc::expected_interactions(p, kcap));
        const double waves = (double)grid * waves_per_wg;
        double per_lane = std::ceil(256.0 / L);
        per_lane = std::min(per_lane, std::floor((double)p->photons / (64.0 * 4.0 * waves)));
        per_lane = std::min(std::max(per_lane, 4.0), (double)(1u << 18));
        chunk = 64u * (uint32_t)per_lane;
    }

    unsigned long long* const d_counters = work;
    unsigned long long* const d_tally = work + tmc::kRunCounterWords;
    tmc::WalkArgs a;
    std::memset(&a, 0, sizeof a);
    a.seed = seed;
    a.first_photon = o->first_photon;
    a.photons = p->photons;
    a.albedo = tmc::derived_albedo(p);
    a.spm = tmc::derived_spm(p);
    a.shell_max = (float)(S - 1);
    a.shells = S;
    a.chunk = chunk;
    precision_constants(p, &a);
    /* Each wave swaps the workgroup's LDS sums out at least every
     * flush_interval steps, so between two swaps of one entry at most
     * waves_per_wg * 64 * flush_interval deposits of at most 2^43 (heat2
     * image of w = 1) accumulate: keep that below 2^63. */
    a.flush_interval = (1u << 14) / waves_per_wg;
    a.kcap = (uint32_t)kcap;
    a.table_k = table_k;
    a.counters = d_counters;
    a.tally = d_tally;

    if (work == c->d_work)
        c->work_zero = false;

    float kernel_ms = 0.0f;
    /* a fill kernel, not a memset: the same sequence serves callers that
     * cannot have memset nodes in their streams */
    if (tmc::launch_clear(work, tmc::run_work_words(S), c->stream) != hipSuccess)
        return TMC_E_HIP;
    unsigned long long counters[4] = { 0, 0, 0, 0 };
    if (p->photons > 0) {
        if (hipEventRecord(c->ev_start, c->stream) != hipSuccess)
            return TMC_E_HIP;
        if (tmc::launch_walk(o->sampler, o->precision, o->math, a, grid, block, c->stream) != hipSuccess)
            return TMC_E_HIP;
        if (hipEventRecord(c->ev_stop, c->stream) != hipSuccess)
            return TMC_E_HIP;
    }
    if (hipMemcpyAsync(tally, d_tally, 4 * (size_t)S * sizeof(uint64_t), hipMemcpyDeviceToHost, c->stream)
            != hipSuccess
        || hipMemcpyAsync(counters, d_counters, sizeof counters, hipMemcpyDeviceToHost, c->stream) != hipSuccess)
        return TMC_E_HIP;
    if (hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    if (p->photons > 0 && hipEventElapsedTime(&kernel_ms, c->ev_start, c->ev_stop) != hipSuccess)
        return TMC_E_HIP;
    if (st) {
        st->photons = p->photons;
        st->interactions = counters[1];
        st->truncated = counters[2];
        st->kernel_ms = kernel_ms;
        st->total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        st->grid = grid;
        st->block = block;
        st->chunk = chunk;
        st->sampler = o->sampler;
        st->precision = o->precision;
        st->math = o->math;
        st->weight_table = table_k;
    }
    return TMC_OK;
}

TMC_EXPORT void tmc_options_default(tmc_options* opt)
{
    if (!opt)
        return;
    std::memset(opt, 0, sizeof *opt);
    opt->sampler = TMC_SAMPLER_ANALYTIC;
}

TMC_EXPORT int tiny_mc_gpu_run_ex(const tmc_params* p, uint64_t seed, const tmc_options* opt, uint64_t* tally,
                                  tmc_run_stats* stats)
{
    int rc = tmc::check_params(p);
    if (rc != TMC_OK)
        return rc;
    if (!tally)
        return TMC_E_INVALID;
    tmc_options o;
    if (opt)
        o = *opt;
    else
        tmc_options_default(&o);
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    rc = tmc::acquire_context(&c);
    if (rc != TMC_OK)
        return rc;
    rc = ensure_work(c);
    if (rc != TMC_OK)
        return rc;
    return tmc::run_walk(c, p, seed, &o, c->d_work, tally, stats);
}

TMC_EXPORT int tiny_mc_gpu_tally_to_heat(const tmc_params* p, const uint64_t* tally, double* heat, double* heat2)
{
    int rc = tmc::check_params(p);
    if (rc != TMC_OK)
        return rc;
    if (!tally || !heat || !heat2)
        return TMC_E_INVALID;
    const uint32_t S = p->shells;
    /* (1 - albedo) in double from the parameters; the FP32 transport's
     * albedo (photon.c:8) only drives the weight decay. */
    const double albedo = (double)p->mu_s / ((double)p->mu_s + (double)p->mu_a);
    const double oma = 1.0 - albedo;
    const double s1 = std::ldexp(oma, -TMC_HEAT_FRAC_BITS);
    const double s2 = std::ldexp(oma * oma, -TMC_HEAT2_FRAC_BITS);
    for (uint32_t s = 0; s < S; ++s) {
        heat[s] = s1 * u128_to_double(tally[2 * s], tally[2 * s + 1]);
        heat2[s] = s2 * u128_to_double(tally[2 * S + 2 * s], tally[2 * S + 2 * s + 1]);
    }
    return TMC_OK;
}

TMC_EXPORT int tiny_mc_gpu_run(const tmc_params* p, uint64_t seed, double* heat, double* heat2)
{
    int rc = tmc::check_params(p);
    if (rc != TMC_OK)
        return rc;
    if (!heat || !heat2)
        return TMC_E_INVALID;
    uint64_t* tally = new (std::nothrow) uint64_t[4 * (size_t)p->shells];
    if (!tally)
        return TMC_E_NOMEM;
    rc = tiny_mc_gpu_run_ex(p, seed, nullptr, tally, nullptr);
    if (rc == TMC_OK)
        rc = tiny_mc_gpu_tally_to_heat(p, tally, heat, heat2);
    delete[] tally;
    return rc;
}

TMC_EXPORT int tiny_mc_gpu_init(int device)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_ctx) {
        if (device >= 0 && device != g_ctx->device)
            return TMC_E_INVALID;
        return TMC_OK;
    }
    return create_context(device, &g_ctx);
}

TMC_EXPORT void tiny_mc_gpu_shutdown(void)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    destroy_context(g_ctx);
    g_ctx = nullptr;
}

TMC_EXPORT int tiny_mc_gpu_device_info(char* name, size_t cap, int* compute_units)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    int rc = tmc::acquire_context(&c);
    if (rc != TMC_OK)
        return rc;
    if (name && cap)
        std::snprintf(name, cap, "%s", c->arch);
    if (compute_units)
        *compute_units = c->compute_units;
    return TMC_OK;
}

TMC_EXPORT double tiny_mc_gpu_expected_interactions(const tmc_params* p)
{
    if (tmc::check_params(p) != TMC_OK)
        return 0.0;
    return tmc::expected_interactions(p, 0);
}

TMC_EXPORT const char* tiny_mc_gpu_strerror(int status)
{
    switch (status) {
    case TMC_OK: return "ok";
    case TMC_E_INVALID: return "invalid argument";
    case TMC_E_NODEVICE: return "no usable HIP device";
    case TMC_E_HIP: return "HIP runtime error";
    case TMC_E_NOMEM: return "out of memory";
    case TMC_E_RANGE: return "photon index range exceeds 2^63";
    case TMC_E_UNSUPPORTED: return "unsupported option";
    case TMC_E_TOO_LARGE: return "more shells than the no-allocation scratch holds";
    case TMC_PENDING: return "pending";
    default: return "unknown status";
    }
}

namespace {

/* Device buffers of a diagnostic call, freed on every path. */
struct DevBufs {
    void* p[5] = { nullptr, nullptr, nullptr, nullptr, nullptr };
    ~DevBufs()
    {
        for (void* q : p)
            tmc::release_device(q);
    }
};

} // namespace

TMC_EXPORT int tiny_mc_gpu_philox(const uint32_t* ctr, const uint32_t* key, uint32_t n, uint32_t* out)
{
    if ((!ctr || !key || !out) && n)
        return TMC_E_INVALID;
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    int rc = tmc::acquire_context(&c);
    if (rc != TMC_OK || n == 0)
        return rc;
    DevBufs b;
    if (hipMalloc(&b.p[0], 16 * (size_t)n) != hipSuccess || hipMalloc(&b.p[1], 8 * (size_t)n) != hipSuccess
        || hipMalloc(&b.p[2], 16 * (size_t)n) != hipSuccess)
        return TMC_E_NOMEM;
    if (hipMemcpyAsync(b.p[0], ctr, 16 * (size_t)n, hipMemcpyHostToDevice, c->stream) != hipSuccess
        || hipMemcpyAsync(b.p[1], key, 8 * (size_t)n, hipMemcpyHostToDevice, c->stream) != hipSuccess
        || tmc::launch_philox((const uint32_t*)b.p[0], (const uint32_t*)b.p[1], n, (uint32_t*)b.p[2], c->stream)
            != hipSuccess
        || hipMemcpyAsync(out, b.p[2], 16 * (size_t)n, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    return TMC_OK;
}

TMC_EXPORT int tiny_mc_gpu_eval_step_math(uint32_t math, const float* in, uint32_t n, float* step_out,
                                          float* sin_out, float* cos_out, float* polar_out)
{
    if (((!in || !step_out || !sin_out || !cos_out || !polar_out) && n) || math > TMC_MATH_OWN)
        return TMC_E_INVALID;
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    int rc = tmc::acquire_context(&c);
    if (rc != TMC_OK || n == 0)
        return rc;
    DevBufs b;
    const size_t bytes = 4 * (size_t)n;
    for (int i = 0; i < 5; ++i)
        if (hipMalloc(&b.p[i], bytes) != hipSuccess)
            return TMC_E_NOMEM;
    if (hipMemcpyAsync(b.p[0], in, bytes, hipMemcpyHostToDevice, c->stream) != hipSuccess
        || tmc::launch_eval_step_math(math, (const float*)b.p[0], n, (float*)b.p[1], (float*)b.p[2],
                                      (float*)b.p[3], (float*)b.p[4], c->stream)
            != hipSuccess
        || hipMemcpyAsync(step_out, b.p[1], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipMemcpyAsync(sin_out, b.p[2], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipMemcpyAsync(cos_out, b.p[3], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipMemcpyAsync(polar_out, b.p[4], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    return TMC_OK;
}

TMC_EXPORT int tiny_mc_gpu_eval_math(const float* in, uint32_t n, float* log_out, float* sin_out, float* cos_out)
{
    if ((!in || !log_out || !sin_out || !cos_out) && n)
        return TMC_E_INVALID;
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    int rc = tmc::acquire_context(&c);
    if (rc != TMC_OK || n == 0)
        return rc;
    DevBufs b;
    const size_t bytes = 4 * (size_t)n;
    for (int i = 0; i < 4; ++i)
        if (hipMalloc(&b.p[i], bytes) != hipSuccess)
            return TMC_E_NOMEM;
    if (hipMemcpyAsync(b.p[0], in, bytes, hipMemcpyHostToDevice, c->stream) != hipSuccess
        || tmc::launch_eval_math((const float*)b.p[0], n, (float*)b.p[1], (float*)b.p[2], (float*)b.p[3], c->stream)
            != hipSuccess
        || hipMemcpyAsync(log_out, b.p[1], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipMemcpyAsync(sin_out, b.p[2], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipMemcpyAsync(cos_out, b.p[3], bytes, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    return TMC_OK;
}

TMC_EXPORT int tiny_mc_gpu_check_short_op(uint32_t op, uint32_t first_bits, uint64_t count, uint64_t* mismatches,
                                          uint32_t* first_mismatch)
{
    if (!mismatches || !first_mismatch || op > TMC_CHECK_DIV_TENTH || count > (1ull << 32)
        || (uint64_t)first_bits + count > (1ull << 32))
        return TMC_E_INVALID;
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    int rc = tmc::acquire_context(&c);
    if (rc != TMC_OK)
        return rc;
    DevBufs b;
    unsigned long long h[2] = { 0ull, ~0ull };
    if (hipMalloc(&b.p[0], sizeof h) != hipSuccess)
        return TMC_E_NOMEM;
    if (hipMemcpyAsync(b.p[0], h, sizeof h, hipMemcpyHostToDevice, c->stream) != hipSuccess
        || tmc::launch_check_short_op(op, first_bits, count, (unsigned long long*)b.p[0], c->stream) != hipSuccess
        || hipMemcpyAsync(h, b.p[0], sizeof h, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    *mismatches = h[0];
    *first_mismatch = h[0] ? (uint32_t)h[1] : 0u;
    return TMC_OK;
}

TMC_EXPORT int tiny_mc_gpu_check_shell_index(const tmc_params* p, uint32_t first_bits, uint64_t count,
                                             uint64_t* violations, uint32_t* first_violation, uint64_t* unsure)
{
    if (!violations || !first_violation || !unsure || count > (1ull << 32)
        || (uint64_t)first_bits + count > (1ull << 32))
        return TMC_E_INVALID;
    int rc = tmc::check_params(p);
    if (rc != TMC_OK)
        return rc;
    std::lock_guard<std::mutex> lock(g_mutex);
    Context* c = nullptr;
    rc = tmc::acquire_context(&c);
    if (rc != TMC_OK)
        return rc;
    DevBufs b;
    unsigned long long h[3] = { 0ull, ~0ull, 0ull };
    if (hipMalloc(&b.p[0], sizeof h) != hipSuccess)
        return TMC_E_NOMEM;
    if (hipMemcpyAsync(b.p[0], h, sizeof h, hipMemcpyHostToDevice, c->stream) != hipSuccess
        || tmc::launch_check_shell(tmc::derived_spm(p), (float)(p->shells - 1), first_bits, count,
                                   (unsigned long long*)b.p[0], c->stream)
            != hipSuccess
        || hipMemcpyAsync(h, b.p[0], sizeof h, hipMemcpyDeviceToHost, c->stream) != hipSuccess
        || hipStreamSynchronize(c->stream) != hipSuccess)
        return TMC_E_HIP;
    *violations = h[0];
    *first_violation = h[0] ? (uint32_t)h[1] : 0u;
    *unsure = h[2];
    return TMC_OK;
}

TMC_EXPORT int tiny_mc_gpu_check_sqrt(uint32_t first_bits, uint64_t count, uint64_t* mismatches,
                                      uint32_t* first_mismatch)
{
    return tiny_mc_gpu_check_short_op(TMC_CHECK_SQRT, first_bits, count, mismatches, first_mismatch);
}
