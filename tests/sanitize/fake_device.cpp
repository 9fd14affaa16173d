// See fake_device.h.
#include "fake_device.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/tiny_mc_gpu.h"
#include "../../tiny_mc_amd/csrc/tmc_batch_internal.h"
#include "../../tiny_mc_amd/csrc/tmc_cohort.h"
#include "../../tiny_mc_amd/csrc/tmc_context.h"
#include "../../tiny_mc_amd/csrc/tmc_internal.h"

namespace fake {

std::vector<std::pair<uint64_t, uint64_t>> slices;
long fail_alloc = -1;
size_t alloc_limit = SIZE_MAX;
bool overflow = false;
uint32_t lock_grid = 0, lock_block = 0, table_entries = 0;

namespace {

std::mutex m;
std::condition_variable cv;
std::map<void*, size_t> blocks;
size_t bytes = 0;
hipError_t last = hipSuccess; // as hipGetLastError gives it
Launches count;
bool held = false;
std::map<hipStream_t, std::vector<std::thread>> running; // kernels that have not ended, by stream
std::map<hipStream_t, int> busy;

hipError_t fail(hipError_t e)
{
    std::lock_guard<std::mutex> l(m);
    last = e;
    return e;
}

// hipGetLastError as the launches return it.
hipError_t launch_status()
{
    std::lock_guard<std::mutex> l(m);
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}

hipError_t alloc(void** p, size_t n)
{
    *p = nullptr;
    bool no;
    {
        std::lock_guard<std::mutex> l(m);
        no = fail_alloc == 0 || n > alloc_limit;
        if (fail_alloc >= 0)
            --fail_alloc;
    }
    void* const b = no ? nullptr : std::malloc(n ? n : 1);
    if (!b)
        return fail(hipErrorOutOfMemory);
    std::lock_guard<std::mutex> l(m);
    blocks[b] = n;
    bytes += n;
    *p = b;
    return hipSuccess;
}

hipError_t release(void* p)
{
    std::lock_guard<std::mutex> l(m);
    if (!p)
        return hipSuccess;
    auto it = blocks.find(p);
    if (it == blocks.end())
        std::abort();
    bytes -= it->second;
    blocks.erase(it);
    std::free(p);
    return hipSuccess;
}

// Runs `kernel` on the stream: at once, or (held) in a thread that first waits
// for hold(false).
template <class F>
void enqueue(hipStream_t s, bool wait, const F& kernel)
{
    {
        std::lock_guard<std::mutex> l(m);
        if (!wait || !held)
            wait = false;
        else
            ++busy[s];
    }
    if (!wait) {
        kernel();
        return;
    }
    std::thread t([s, kernel]() {
        {
            std::unique_lock<std::mutex> l(m);
            cv.wait(l, []() { return !held; });
        }
        kernel();
        std::lock_guard<std::mutex> l(m);
        --busy[s];
    });
    std::lock_guard<std::mutex> l(m);
    running[s].push_back(std::move(t));
}

void touch(void* p, size_t at, size_t n) { std::memset((char*)p + at, 0, n); }

void touch(const tmc::PhotonList& l, size_t places)
{
    if (!places)
        return;
    l.photon[0] = l.photon[places - 1] = 0;
    for (float* f : l.state)
        f[0] = f[places - 1] = 0.0f;
}

} // namespace

size_t live_bytes()
{
    std::lock_guard<std::mutex> l(m);
    return bytes;
}

Launches launched()
{
    std::lock_guard<std::mutex> l(m);
    return count;
}

void reset()
{
    std::lock_guard<std::mutex> l(m);
    count = Launches{};
    fail_alloc = -1;
    alloc_limit = SIZE_MAX;
    overflow = false;
    slices.clear();
}

void hold(bool on)
{
    std::lock_guard<std::mutex> l(m);
    held = on;
    cv.notify_all();
}

namespace {

void counted(int Launches::*what)
{
    std::lock_guard<std::mutex> l(m);
    ++(count.*what);
}

// The result of a run that ends with `a`: the sums that the launches left.
void end_run(const tmc::CohortArgs& a, uint64_t interactions)
{
    unsigned long long truncated = 0;
    const size_t block = TMC_COHORT_COUNTERS + 4ull * a.shells;
    for (uint32_t c = 0; c < a.copies; ++c) {
        truncated += a.work[c * block + 2];
        touch(a.work + c * block, 0, block * 8);
    }
    touch(a.out + TMC_COHORT_COUNTERS, 0, 32ull * a.shells);
    a.out[1] = interactions;
    a.out[2] = truncated;
    a.out[3] = 1;
    __atomic_store_n(a.out, a.token, __ATOMIC_RELEASE);
}

} // namespace
} // namespace fake

using namespace fake;

extern "C" {
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)
{
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return launch_status(); }
hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { return alloc(p, n); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned int)
{
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int)
{
    *s = (hipStream_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::vector<std::thread> t;
    {
        std::lock_guard<std::mutex> l(m);
        t.swap(running[s]);
    }
    for (std::thread& k : t)
        k.join();
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s)
{
    {
        std::lock_guard<std::mutex> l(m);
        if (busy[s])
            return hipErrorNotReady;
    }
    return hipStreamSynchronize(s);
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    (void)hipStreamSynchronize(s);
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
}

namespace tmc {

int scratch_setup(int) { return TMC_OK; }

// ---- single runs ----

hipError_t launch_clear(unsigned long long* p, size_t n, hipStream_t)
{
    touch(p, 0, 8 * n);
    return launch_status();
}
hipError_t launch_walk(uint32_t, uint32_t, uint32_t, const WalkArgs& a, uint32_t, uint32_t, hipStream_t)
{
    counted(&Launches::walk);
    a.counters[1] = a.photons;
    touch(a.tally, 0, 32ull * a.shells);
    return launch_status();
}
hipError_t walk_occupancy(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, int* n)
{
    *n = 4;
    return hipSuccess;
}
size_t cohort_lds_bytes(uint32_t shells, uint32_t entries) { return 16ull * shells + 16ull * entries + 80000u; }
hipError_t launch_cohort_table(const float* weight, uint32_t n, void* entry, uint32_t* counter, uint32_t counters,
                               unsigned long long* start, hipStream_t)
{
    table_entries = n;
    volatile float last_weight = weight[n - 1];
    (void)last_weight;
    touch(entry, 0, 16ull * (n + 2u)); /* two entries more are read */
    if (counters)
        touch(counter, 0, 4ull * counters);
    if (start)
        *start = 1;
    return launch_status();
}
hipError_t launch_cohort(uint32_t, uint32_t, const CohortArgs& a, uint32_t, uint32_t, hipStream_t s)
{
    counted(&Launches::cohort);
    if (a.build)
        table_entries = a.entries;
    if (a.list.photon)
        touch(a.list, (size_t)a.stripes * a.list_cap);
    enqueue(s, a.finish, [a]() {
        if (a.finish)
            end_run(a, a.photons);
    });
    return launch_status();
}
hipError_t launch_finish(const CohortArgs& a, hipStream_t s)
{
    enqueue(s, true, [a]() { end_run(a, a.photons); });
    return launch_status();
}
size_t lock_count_bytes(uint32_t shells, uint32_t absorptions) { return 16u + 4ull * absorptions * (shells + 7ull); }
hipError_t lock_occupancy(uint32_t, uint32_t, uint32_t, uint32_t, int* n)
{
    *n = 4;
    return hipSuccess;
}
hipError_t launch_lock(uint32_t, uint32_t, bool, const LockArgs& a, uint32_t grid, uint32_t block, hipStream_t)
{
    counted(&Launches::lock);
    lock_grid = grid;
    lock_block = block;
    if (!a.level)
        slices.push_back({ a.first_photon, a.photons });
    if (!a.cap_ends)
        touch(a.out, (size_t)a.stripes * a.out_cap);
    if (a.level)
        touch(a.in, (size_t)a.stripes * a.in_cap);
    a.out_count[(a.stripes - 1u) * TMC_LOCK_LINE] = 0;
    if (a.chunk)
        a.cursor[(TMC_LOCK_RANGES - 1u) * TMC_LOCK_LINE] = 0;
    if (overflow)
        a.work[2] |= TMC_LOCK_OVERFLOW;
    return launch_status();
}
hipError_t prec_occupancy(uint32_t, uint32_t, uint32_t, uint32_t, int* n)
{
    *n = 4;
    return hipSuccess;
}
hipError_t launch_prec_table(uint32_t precision, const PrecArgs& a, uint32_t* counter, uint32_t counters,
                             unsigned long long* start, hipStream_t)
{
    touch(a.entry, 0, 16ull * (a.entries + 1u));
    touch(a.head, 0, sizeof *a.head);
    if (precision == TMC_PRECISION_FP64) {
        volatile double last_weight = a.weight[a.entries - 1];
        (void)last_weight;
        *a.head = *a.host_head;
    }
    if (counters)
        touch(counter, 0, 4ull * counters);
    *start = 1;
    return launch_status();
}
hipError_t launch_prec(uint32_t, uint32_t, const PrecArgs& a, uint32_t, uint32_t, hipStream_t)
{
    counted(&Launches::prec);
    if (!a.level)
        slices.push_back({ a.first_photon, a.photons });
    if (a.cycles)
        touch(a.out.photon, 4ull * a.stripes * a.out_cap - 4u, 4);
    if (overflow)
        a.work[2] |= TMC_LOCK_OVERFLOW;
    return launch_status();
}

// ---- batches ----

size_t batch_lds_bytes(uint32_t block, uint32_t shells, uint32_t copies) { return 4ull * block / 16u * shells * copies; }
hipError_t batch_occupancy(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, int* n)
{
    *n = 4;
    return hipSuccess;
}
hipError_t launch_batch_clear(unsigned long long* tally, uint64_t words, unsigned long long* done, uint32_t nsets,
                              unsigned long long* counters, hipStream_t)
{
    touch(tally, 0, 8 * words);
    touch(done, 0, 16ull * nsets);
    touch(counters, 0, 8 * TMC_BATCH_COUNTERS);
    return launch_status();
}
hipError_t launch_batch(uint32_t, uint32_t, const BatchArgs& a, uint32_t, uint32_t, hipStream_t)
{
    counted(&Launches::batch);
    for (uint32_t i = 0; i < a.nchunks; ++i)
        a.counters[1] += a.chunks[i].count;
    return launch_status();
}
hipError_t lock_sets_occupancy(uint32_t, uint32_t, uint32_t, int* n)
{
    *n = 4;
    return hipSuccess;
}
hipError_t launch_weigh_sets(const LockSet* sets, uint32_t nsets, CohortHead* heads, void* entry, hipStream_t)
{
    for (uint32_t i = 0; i < nsets; ++i)
        if (sets[i].cuts) {
            touch(&heads[sets[i].head], 0, sizeof *heads);
            touch(entry, 16 * sets[i].entry, 16ull * (sets[i].entries + 2u));
        }
    return launch_status();
}
hipError_t launch_lock_sets(uint32_t, const LockSetArgs& a, uint32_t, uint32_t, hipStream_t)
{
    counted(&Launches::lock_sets);
    for (uint32_t i = 0; i < a.nchunks; ++i) {
        const LockSet& s = a.sets[a.chunks[i].set];
        touch(&a.out.photon[s.place[a.level]], 0, 4ull * s.cap[a.level]);
        a.out_count[a.chunks[i].set * TMC_LOCK_LINE] = 0;
        if (!a.level)
            a.counters[1] += a.chunks[i].count;
    }
    if (overflow)
        a.counters[2] |= TMC_LOCK_OVERFLOW;
    return launch_status();
}
hipError_t launch_cohort_sets(uint32_t, const LockSetArgs& a, uint32_t, hipStream_t s)
{
    counted(&Launches::cohort_sets);
    a.cursor[0] = 0;
    enqueue(s, true, []() {});
    return launch_status();
}

// ---- serving ----

hipError_t serve_occupancy(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, int* n)
{
    *n = 4;
    return hipSuccess;
}

namespace {

// The resident kernel: takes every published entry, and finishes a request
// once all its photons were in entries; leaves when it is asked to.
void serve_kernel(BatchArgs a)
{
    uint64_t at = a.ticket_base;
    std::map<uint32_t, uint64_t> done;
    for (;;) {
        const uint64_t tail = __atomic_load_n(&a.hctl->tail, __ATOMIC_ACQUIRE);
        for (; at < tail; ++at) {
            RingEntry& e = a.ring[at & a.ring_mask];
            const uint32_t slot = e.set & ((1u << TMC_SERVE_SLOT_BITS) - 1u);
            done[slot] += e.count ? e.count : e.first;
            __atomic_store_n(&e.seq, at | TMC_RING_CONSUMED, __ATOMIC_RELEASE);
            if (done[slot] == a.sets[slot].photons) {
                done[slot] = 0;
                a.flags[2 * slot + 1] = a.sets[slot].photons;
                __atomic_store_n(&a.flags[2 * slot], (unsigned long long)a.sets[slot].token, __ATOMIC_RELEASE);
            }
        }
        __atomic_store_n(&a.hctl->claimed, at, __ATOMIC_RELEASE);
        if (__atomic_load_n(&a.hctl->stop, __ATOMIC_ACQUIRE) == a.launch_id)
            return;
        std::this_thread::sleep_for(std::chrono::microseconds(100));
    }
}

} // namespace

hipError_t launch_serve(uint32_t, uint32_t, const BatchArgs& a, uint32_t, uint32_t, hipStream_t s)
{
    counted(&Launches::serve);
    std::lock_guard<std::mutex> l(m);
    ++busy[s];
    running[s].push_back(std::thread([a, s]() {
        serve_kernel(a);
        std::lock_guard<std::mutex> l2(m);
        --busy[s];
    }));
    return hipSuccess;
}

// ---- diagnostics: not under test ----

hipError_t launch_philox(const uint32_t*, const uint32_t*, uint32_t, uint32_t*, hipStream_t) { return hipSuccess; }
hipError_t launch_check_shell(float, float, uint32_t, uint64_t, unsigned long long*, hipStream_t) { return hipSuccess; }
hipError_t launch_check_short_op(uint32_t, uint32_t, uint64_t, unsigned long long*, hipStream_t) { return hipSuccess; }
hipError_t launch_eval_step_math(uint32_t, const float*, uint32_t, float*, float*, float*, float*, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_eval_math(const float*, uint32_t, float*, float*, float*, hipStream_t) { return hipSuccess; }

} // namespace tmc
