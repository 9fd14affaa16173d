/* The library's implicit per-process context and the parameter helpers
 * shared by the single-run, batched and serving entry points. */
#ifndef TMC_CONTEXT_H
#define TMC_CONTEXT_H

#include <hip/hip_runtime.h>

#include <functional>
#include <mutex>

#include "../../include/tiny_mc_gpu.h"
#include "tmc_plan.h"

namespace tmc {

/* Device words of one single run: the walk's counters ([0] claim offset,
 * [1] absorptions, [2] truncated photons, [3] unused), then the 4 * shells
 * tally words.  The context allocates them once at the largest shell count
 * (run_work_words(TMC_MAX_SHELLS) words, 256 KiB) and keeps them until
 * shutdown, so no run of the lane-per-photon walk allocates or frees device
 * memory.  The lockstep walks' 20 MB are kept in the same way from the first run
 * on, and their lists, which grow with the largest run so far (to 0.6 GB, a
 * precision variant's to 1.1 GB). */
constexpr size_t kRunCounterWords = 4;
constexpr size_t run_work_words(uint32_t shells) { return kRunCounterWords + 4 * (size_t)shells; }

/* Entries of the cohort walk's weight table (16 bytes each). */
constexpr size_t kTableEntries = 1u << 20;

/* Photons of a slice of a large run (log2), and the counters of all its slices.
 * (A slice's last launches leave the chip idle for 70 us: 2^27 photons at
 * albedo 0.5 in slices of 2^26 2658 us, in one of 2^27 2497; the lists of 2^27
 * take 0.6 GB.) */
constexpr uint32_t kSliceLog = 27;
constexpr uint32_t kRunCounters = 1u << 21;
constexpr uint32_t kStripes = 64; /* parts of a slice and of the survivor lists */

struct Context {
    int device = -1;
    int compute_units = 0;
    char arch[64] = { 0 };
    hipStream_t stream = nullptr; /* default priority */
    hipEvent_t ev_start = nullptr, ev_stop = nullptr;
    void* d_table = nullptr; /* weight table of the cohort walk (kTableEntries entries), allocated at the first run */
    unsigned long long* h_out = nullptr; /* host-coherent result words of the cohort walk, and their device address */
    unsigned long long* d_out = nullptr;
    float* h_weight = nullptr; /* weights of the run's table (host-coherent memory), and their device address */
    float* d_weight = nullptr;
    void* d_lists = nullptr; /* survivor lists and counters of large runs */
    size_t lists_bytes = 0;
    uint64_t token = 0; /* of the last cohort walk */
    bool work_zero = false; /* d_work holds zeros */
    unsigned long long* d_work = nullptr; /* run_work_words(TMC_MAX_SHELLS) words, allocated at the first run */
};

/* Serialises every entry point that touches the context. */
std::mutex& api_mutex();

/* The context, created on the current device at first use.  Call with
 * api_mutex() held. */
int acquire_context(Context** out);

/* One single run (tiny_mc_gpu_run_ex) with its counters and tallies in the
 * device words `work` (run_work_words(p->shells) of them): clears them with
 * a kernel, launches the walk, copies the tallies to `tally` (host) and
 * synchronises the context's stream.  Allocates nothing, but for the lockstep
 * walks, which are for the context's own words only.  Call with api_mutex()
 * held; p is checked. */
int run_walk(Context* c, const tmc_params* p, uint64_t seed, const tmc_options* o, unsigned long long* work,
             uint64_t* tally, tmc_run_stats* st);

/* The static scratch of tiny_mc_gpu_run_noalloc on `device` (current):
 * looks its address up once per device.  TMC_OK or a negative status. */
int scratch_setup(int device);

/* Releases of device resources while a serving kernel may be resident.
 * hipFree and hipHostFree synchronise the whole device, so under load they
 * would wait for a resident serving kernel that never becomes idle.  A
 * release made while any server's kernel runs is queued and performed once
 * no serving kernel runs; otherwise it happens at once.  A server calls
 * serving_kernel_started() before it launches its kernel (which waits for
 * a release in progress) and serving_kernel_left() once the kernel has
 * ended (which performs the queued releases when it was the last one). */
void release(std::function<void()> fn);
void release_device(void* p); /* hipFree */
void release_host(void* p); /* hipHostFree */
/* Launches that need whole compute units, from before the first of them is
 * enqueued until the last has ended.  Beside a resident serving kernel they
 * would wait for it, where a kernel of small workgroups finds room beside a
 * server that reserves some: false, for the whole life of the object, if one is
 * resident or waits to be launched.  While one of these objects is true, no
 * serving kernel is launched. */
class LockstepRun {
public:
    LockstepRun();
    ~LockstepRun();
    LockstepRun(const LockstepRun&) = delete;
    LockstepRun& operator=(const LockstepRun&) = delete;
    explicit operator bool() const { return on_; }

private:
    bool on_;
};
/* Whether a LockstepRun would be off: nothing need be prepared for it. */
bool serving();
/* False while a LockstepRun is on: the caller asks again later, *waiting (false
 * at first) is set, and from then on every new LockstepRun is off. */
bool serving_kernel_started(bool* waiting);
void serving_kernel_left();
/* A server that ends without its kernel. */
void serving_kernel_waived(bool* waiting);

} // namespace tmc

#endif
