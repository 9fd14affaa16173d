// The library's host code (tmc_api.cpp, tmc_batch_api.cpp, tmc_serve_api.cpp)
// over the fake device, with AddressSanitizer and UndefinedBehaviorSanitizer:
// failed allocations, calls beside servers, repeats after a full list.  The
// argument names the check to run.  Test infrastructure; prints "<name>: ok".
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "../../include/tiny_mc_gpu.h"
#include "fake_device.h"

#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c)) {                                                               \
            std::fprintf(stderr, "host_check: %s:%d: %s\n", __FILE__, __LINE__, #c); \
            std::_Exit(1);                                                        \
        }                                                                         \
    } while (0)

static size_t g_largest = 0; // of the host's allocations
static long g_fail_new = -1; // the one that fails (0: the next)

void* operator new(size_t n)
{
    if (n > g_largest)
        g_largest = n;
    if (g_fail_new >= 0 && g_fail_new-- == 0)
        throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1))
        return p;
    throw std::bad_alloc();
}
void* operator new(size_t n, const std::nothrow_t&) noexcept { return std::malloc(n ? n : 1); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

tmc_params params(uint64_t photons, float mu_a = 2.0f, float mu_s = 20.0f, uint32_t shells = 101)
{
    tmc_params p;
    std::memset(&p, 0, sizeof p);
    p.mu_a = mu_a;
    p.mu_s = mu_s;
    p.shells = shells;
    p.microns_per_shell = 50.0f;
    p.photons = photons;
    return p;
}

int run(const tmc_params& p, uint32_t precision = TMC_PRECISION_FP32, uint32_t block = 0,
        uint64_t max_interactions = 0, uint32_t sampler = TMC_SAMPLER_ANALYTIC)
{
    tmc_options o;
    tmc_options_default(&o);
    o.precision = precision;
    o.block = block;
    o.max_interactions = max_interactions;
    o.sampler = sampler;
    std::vector<uint64_t> tally(4 * (size_t)p.shells);
    tmc_run_stats st;
    return tiny_mc_gpu_run_ex(&p, 1, &o, tally.data(), &st);
}

struct Form {
    uint64_t photons;
    uint32_t precision;
    int fake::Launches::*kernel;
};
const Form kForms[] = { { 3000, TMC_PRECISION_FP32, &fake::Launches::cohort },
                        { 300000, TMC_PRECISION_FP32, &fake::Launches::lock },
                        { 3000, TMC_PRECISION_FP32_WEIGHT, &fake::Launches::prec },
                        { 300000, TMC_PRECISION_FP64, &fake::Launches::prec } };

// Each allocation of a first run fails in turn: that call is refused or takes
// the lane-per-photon walk, and the next one, with the memory there, is an
// ordinary one.
void failed_allocations()
{
    for (const Form& f : kForms)
        for (long n = 0; n < 6; ++n) {
            fake::reset();
            fake::fail_alloc = n;
            const int first = run(params(f.photons), f.precision);
            CHECK(first == TMC_OK || (first == TMC_E_NOMEM && n == 0));
            fake::fail_alloc = -1;
            fake::reset();
            CHECK(run(params(f.photons), f.precision) == TMC_OK);
            CHECK(fake::launched().*f.kernel > 0 && fake::launched().walk == 0);
            tiny_mc_gpu_shutdown();
            CHECK(fake::live_bytes() == 0);
        }
    // 256 KiB are all that the lane-per-photon walk needs
    for (uint32_t block : { 0u, 256u }) {
        fake::reset();
        fake::alloc_limit = 1u << 19;
        for (int i = 0; i < 2; ++i)
            CHECK(run(params(3000), TMC_PRECISION_FP32, block) == TMC_OK);
        CHECK(fake::launched().walk == 2 && fake::launched().cohort == 0);
        fake::alloc_limit = SIZE_MAX;
        CHECK(run(params(3000)) == TMC_OK && fake::launched().cohort == 1);
        tiny_mc_gpu_shutdown();
    }
}

tmc_server* open_server()
{
    tmc_serve_options o;
    tmc_serve_options_default(&o);
    o.max_requests = 8;
    o.ring_chunks = 1u << 12;
    o.idle_ms = 60000; // the kernel stays
    tmc_server* s = nullptr;
    CHECK(tmc_serve_open(&o, &s) == TMC_OK);
    return s;
}

uint64_t submit(tmc_server* s, uint64_t photons)
{
    tmc_set q;
    std::memset(&q, 0, sizeof q);
    q.params = params(photons);
    uint64_t id = 0;
    CHECK(tmc_serve_submit(s, &q, &id) == TMC_OK);
    return id;
}

int batch(uint64_t photons, uint32_t nsets = 3, float mu_a = 2.0f, bool keep = false)
{
    std::vector<tmc_set> sets(nsets);
    for (tmc_set& q : sets) {
        std::memset(&q, 0, sizeof q);
        q.params = params(photons, mu_a);
    }
    std::vector<uint64_t> tally(tmc_batch_tally_words(sets.data(), nsets));
    tmc_batch_stats st;
    if (!keep)
        return tmc_batch_run(sets.data(), nsets, nullptr, tally.data(), &st);
    tmc_batch_plan* plan = nullptr;
    int rc = tmc_batch_plan_create(sets.data(), nsets, nullptr, &plan);
    if (rc == TMC_OK)
        rc = tmc_batch_plan_run(plan, tally.data(), &st);
    tmc_batch_plan_destroy(plan);
    return rc;
}

// A request that arrives while a run's launches are queued: the serving kernel
// is not launched before the last of them has ended, the server's callers do
// not wait for it, and the next run does not take the device again.
void server_during_run()
{
    constexpr size_t forms = sizeof kForms / sizeof kForms[0];
    for (size_t i = 0; i <= forms; ++i) {
        const bool sets = i == forms;
        int fake::Launches::*const kernel = sets ? &fake::Launches::cohort_sets
            : kForms[i].precision               ? &fake::Launches::prec
                                                : &fake::Launches::cohort;
        auto once = [&]() { return sets ? batch(50000) : run(params(kForms[i].photons), kForms[i].precision); };
        fake::reset();
        tmc_server* s = open_server();
        fake::hold(true);
        int first = 1, second = 1;
        std::thread caller([&]() {
            first = once();
            second = once();
        });
        while (!(fake::launched().*kernel))
            std::this_thread::sleep_for(std::chrono::milliseconds(1));
        const uint64_t id = submit(s, 1000);
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        const int launched = fake::launched().*kernel;
        CHECK(fake::launched().serve == 0);
        CHECK(tmc_serve_poll(s, id, nullptr, nullptr) == TMC_PENDING);
        fake::hold(false);
        caller.join();
        CHECK(first == TMC_OK && second == TMC_OK);
        CHECK(fake::launched().*kernel == launched);
        CHECK((sets ? fake::launched().batch : fake::launched().walk) > 0);
        std::vector<uint64_t> tally(4 * 101);
        CHECK(tmc_serve_wait(s, id, 60.0, tally.data(), nullptr) == TMC_OK);
        CHECK(fake::launched().serve == 1);
        tmc_serve_close(s);
        // without the server the runs are in lockstep again
        CHECK(once() == TMC_OK && fake::launched().*kernel > launched);
        tiny_mc_gpu_shutdown();
        CHECK(fake::live_bytes() == 0);
    }
}

// Runs and plans beside a resident serving kernel take no memory for the walks
// that they cannot use there.
void memory_beside_server()
{
    fake::reset();
    tmc_server* s = open_server();
    const uint64_t id = submit(s, 1000);
    std::vector<uint64_t> tally(4 * 101);
    CHECK(tmc_serve_wait(s, id, 60.0, tally.data(), nullptr) == TMC_OK && fake::launched().serve == 1);
    const size_t before = fake::live_bytes();
    for (const Form& f : kForms)
        CHECK(run(params(f.photons), f.precision) == TMC_OK);
    CHECK(fake::launched().walk == 4 && fake::live_bytes() - before < 1u << 20);
    tmc_set q;
    std::memset(&q, 0, sizeof q);
    q.params = params(1u << 24, 0.2f);
    tmc_batch_plan* plan = nullptr;
    CHECK(tmc_batch_plan_create(&q, 1, nullptr, &plan) == TMC_OK);
    CHECK(fake::live_bytes() - before < 2u << 20);
    CHECK(tmc_batch_plan_run(plan, tally.data(), nullptr) == TMC_OK && fake::launched().batch == 1);
    tmc_batch_plan_destroy(plan);
    tmc_serve_close(s);
    CHECK(fake::launched().lock + fake::launched().lock_sets + fake::launched().cohort + fake::launched().prec == 0);
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

// A set with more photons than a plan's lockstep launches are laid out for: it
// is planned, and what the host lays out before it leaves them is bounded.
void enormous_set()
{
    fake::reset();
    tmc_set q;
    std::memset(&q, 0, sizeof q);
    q.params = params(1ull << 48, 0.2f);
    tmc_batch_plan* plan = nullptr;
    g_largest = 0;
    CHECK(tmc_batch_plan_create(&q, 1, nullptr, &plan) == TMC_OK);
    tmc_batch_plan_destroy(plan);
    CHECK(g_largest <= 100u << 20);
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

// A run stopped after a few absorptions takes no longer weight table than that,
// whatever the albedo, and a table of its own for one that would not fit.
void capped_runs()
{
    for (const float mu_a : { 2.0f, 2e-3f, 2e-5f })
        for (const uint64_t cap : { 1ull, 7ull, 1000ull, 50000ull })
            for (const Form& f : { kForms[0], kForms[1] }) {
                fake::reset();
                CHECK(run(params(f.photons, mu_a), f.precision, 0, cap) == TMC_OK);
                CHECK(fake::launched().*f.kernel > 0 && fake::launched().walk == 0);
                CHECK(fake::table_entries <= cap);
            }
    tiny_mc_gpu_shutdown();
}

// Lockstep waves of the rejection sampler in long cycles: where they fit the
// chip, in workgroups of either size, every one of them is launched.
void all_waves_at_once()
{
    for (uint64_t n = 50000; n <= 400000; n += 9973) { // one level
        fake::reset();
        CHECK(run(params(n, 0.5f, 50.0f), TMC_PRECISION_FP32, 0, 0, TMC_SAMPLER_REJECTION) == TMC_OK);
        CHECK(fake::launched().lock == 1);
        const uint64_t waves = (n + 63) / 64; // fake: four workgroups of eight a CU
        CHECK((uint64_t)fake::lock_grid * fake::lock_block / 64 >= std::min<uint64_t>(waves, 8192));
    }
    tiny_mc_gpu_shutdown();
}

// Batches of short cycles, and one-off batches of many small sets, by the
// lane-per-photon walk; others in lockstep.
void batch_walks()
{
    const struct {
        uint32_t nsets;
        uint64_t photons;
        float mu_a;
        bool keep, lock;
    } forms[] = { { 3, 50000, 2.0f, false, true },  { 2000, 64, 2.0f, false, false }, { 2000, 64, 2.0f, true, true },
                  { 64, 1 << 18, 2000.0f, true, false }, { 64, 1 << 18, 20.0f, true, false },
                  { 64, 1 << 14, 20.0f, true, true }, { 2, 1 << 22, 2.0f, true, false },
                  { 2, 1 << 22, 0.2f, false, true } };
    for (const auto& f : forms) {
        fake::reset();
        CHECK(batch(f.photons, f.nsets, f.mu_a, f.keep) == TMC_OK);
        CHECK((fake::launched().lock_sets > 0) == f.lock && (fake::launched().batch > 0) == !f.lock);
    }
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

// Each of the host's own allocations of a run fails in turn: the run takes the
// lane-per-photon walk, and nothing is thrown at the caller.
void failed_host_allocations()
{
    for (const Form& f : kForms) {
        fake::reset();
        CHECK(run(params(f.photons), f.precision) == TMC_OK && fake::launched().*f.kernel > 0);
        const int ordinary = fake::launched().*f.kernel;
        for (long n = 0;; ++n) {
            fake::reset();
            const tmc_params p = params(f.photons);
            std::vector<uint64_t> tally(4 * (size_t)p.shells);
            tmc_options o;
            tmc_options_default(&o);
            o.precision = f.precision;
            g_fail_new = n;
            CHECK(tiny_mc_gpu_run_ex(&p, 1, &o, tally.data(), nullptr) == TMC_OK);
            const bool failed = g_fail_new < 0;
            g_fail_new = -1;
            CHECK(failed ? fake::launched().walk == 1 : fake::launched().*f.kernel == ordinary);
            if (!failed)
                break;
        }
    }
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

// A survivor that finds no room in its list: the call is repeated by the other
// walk, and the next one is in lockstep again.
void full_lists()
{
    const Form lock[] = { kForms[1], { 300000, TMC_PRECISION_FP32_WEIGHT, &fake::Launches::prec }, kForms[3] };
    for (const Form& f : lock) {
        fake::reset();
        fake::overflow = true;
        CHECK(run(params(f.photons), f.precision) == TMC_OK);
        CHECK(fake::launched().*f.kernel > 0 && fake::launched().walk == 1);
        fake::reset();
        CHECK(run(params(f.photons), f.precision) == TMC_OK);
        CHECK(fake::launched().*f.kernel > 0 && fake::launched().walk == 0);
    }
    for (const bool keep : { false, true }) {
        fake::reset();
        fake::overflow = true;
        CHECK(batch(50000, 3, 2.0f, keep) == TMC_OK);
        CHECK(fake::launched().lock_sets > 0 && fake::launched().batch == 1);
        fake::reset();
        CHECK(batch(50000, 3, 2.0f, keep) == TMC_OK);
        CHECK(fake::launched().lock_sets > 0 && fake::launched().batch == 0);
    }
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

// The slices of a large run: all its photons in order, at most 2^27 in each and
// one high index word, and lists whose places the launches find there.
void slices()
{
    const uint64_t photons[] = { 1u << 17, 3000017, 1ull << 27, (1ull << 27) + 1, (1ull << 28) - 1, 5ull << 27 };
    const uint64_t firsts[] = { 0, 1, (1ull << 32) - 1, (1ull << 32) - (1ull << 26), (7ull << 32) - 40000 };
    for (const uint32_t precision : { TMC_PRECISION_FP32, TMC_PRECISION_FP32_COMPENSATED, TMC_PRECISION_FP64 })
        for (const uint64_t n : photons)
            for (const uint64_t first : firsts) {
                fake::reset();
                const tmc_params p = params(n);
                std::vector<uint64_t> tally(4 * (size_t)p.shells);
                tmc_options o;
                tmc_options_default(&o);
                o.precision = precision;
                o.first_photon = first;
                CHECK(tiny_mc_gpu_run_ex(&p, 1, &o, tally.data(), nullptr) == TMC_OK && fake::launched().walk == 0);
                uint64_t at = first;
                for (const auto& s : fake::slices) {
                    CHECK(s.first == at && s.second > 0 && s.second <= 1ull << 27);
                    CHECK(s.first >> 32 == (s.first + s.second - 1) >> 32);
                    at += s.second;
                }
                CHECK(at == first + n);
            }
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

// Large runs of short cycles and of the precision variants with the rejection
// sampler by the lane-per-photon walk; the sizes up to there in lockstep.
void run_walks()
{
    const uint32_t rej = TMC_SAMPLER_REJECTION;
    const struct {
        float mu_a, mu_s;
        uint32_t precision, sampler;
        uint64_t most; // in lockstep
    } lines[] = { { 100.0f, 1.0f, TMC_PRECISION_FP32, 0, 1ull << 26 },
                  { 100.0f, 1.0f, TMC_PRECISION_FP32, rej, 5ull << 23 },
                  { 20.0f, 5.0f, TMC_PRECISION_FP32, rej, 1ull << 26 },
                  { 20.0f, 5.0f, TMC_PRECISION_FP32_WEIGHT, 0, 1ull << 26 },
                  { 20.0f, 5.0f, TMC_PRECISION_FP32_COMPENSATED, rej, 1ull << 25 },
                  { 20.0f, 5.0f, TMC_PRECISION_FP64, 0, 1ull << 25 },
                  { 10.0f, 10.0f, TMC_PRECISION_FP64, rej, 1ull << 24 },
                  { 2.0f, 20.0f, TMC_PRECISION_FP32_WEIGHT, rej, 1ull << 22 } };
    for (const auto& l : lines)
        for (const uint64_t over : { 0u, 1u }) {
            fake::reset();
            CHECK(run(params(l.most + over, l.mu_a, l.mu_s), l.precision, 0, 0, l.sampler) == TMC_OK);
            CHECK(fake::launched().walk == (int)over);
            CHECK((fake::launched().lock + fake::launched().prec > 0) == !over);
        }
    for (const uint32_t precision : { TMC_PRECISION_FP32, TMC_PRECISION_FP32_WEIGHT, TMC_PRECISION_FP64 }) {
        fake::reset();
        CHECK(run(params(1ull << 27, 10.0f, 10.0f), precision) == TMC_OK && fake::launched().walk == 0);
    }
    tiny_mc_gpu_shutdown();
    CHECK(fake::live_bytes() == 0);
}

const struct {
    const char* name;
    void (*check)();
} kChecks[] = {
    { "failed_allocations", failed_allocations },
    { "server_during_run", server_during_run },
    { "memory_beside_server", memory_beside_server },
    { "enormous_set", enormous_set },
    { "capped_runs", capped_runs },
    { "all_waves_at_once", all_waves_at_once },
    { "batch_walks", batch_walks },
    { "failed_host_allocations", failed_host_allocations },
    { "full_lists", full_lists },
    { "slices", slices },
    { "run_walks", run_walks },
};

} // namespace

int main(int argc, char** argv)
{
    for (const auto& c : kChecks)
        if (argc == 2 && !std::strcmp(argv[1], c.name)) {
            c.check();
            std::printf("%s: ok\n", c.name);
            return 0;
        }
    std::fprintf(stderr, "host_check: no such check\n");
    return 2;
}
