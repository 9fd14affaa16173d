// A device for the library's host code on the CPU: the HIP calls and the
// kernel launches that tmc_api.cpp, tmc_batch_api.cpp and tmc_serve_api.cpp
// make, over ordinary memory.  Launches touch the ends of what their kernels
// would read and write (so that AddressSanitizer sees a null or short buffer)
// and leave results of the right form; they walk no photons.
// Test infrastructure.
#ifndef FAKE_DEVICE_H
#define FAKE_DEVICE_H

#include <cstddef>
#include <cstdint>
#include <utility>
#include <vector>

namespace fake {

// Allocations (device and pinned host): the one that fails (0: the next one,
// -1: none), the largest that succeeds, and the bytes held.
extern long fail_alloc;
extern size_t alloc_limit;
extern size_t live_bytes();

// What was launched since reset().
struct Launches {
    int walk, cohort, lock, prec, batch, lock_sets, cohort_sets, serve;
};
extern Launches launched();
extern void reset();

// The last launch of a single run or of a batch in lockstep ends only once
// this is false again.
extern void hold(bool on);
// A survivor list of the next lockstep launch has no room.
extern bool overflow;

// A launch of lockstep waves: workgroups and threads of the last one.
extern uint32_t lock_grid, lock_block;
// First photon and photons of each first level since reset().
extern std::vector<std::pair<uint64_t, uint64_t>> slices;
// Entries of the last weight table.
extern uint32_t table_entries;

} // namespace fake

#endif
