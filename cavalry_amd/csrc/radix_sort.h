// Stable LSD radix sort of (key, u32 value) pairs; see radix_sort.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"

namespace cav {

// Sort of the first min(cap, *n_dev) pairs.
// Digit counts and tile counters of up to 8 passes, and the failure word:
// nonzero after the sort when a look-back wait exceeded its bound (what the
// sort left is no order then).
constexpr int kCountedSortErr = 8 * 256 + 8;
constexpr int kCountedSortWords = kCountedSortErr + 1;
template <typename K>
struct CountedSort {
    K* keys[2] = {nullptr, nullptr};              // keys[0] holds the input
    uint32_t* vals[2] = {nullptr, nullptr};       // vals[0] holds the input
    uint32_t* work = nullptr;                     // kCountedSortWords, zero before the sort
    uint64_t* status[2] = {nullptr, nullptr};     // counted_sort_status_bytes(cap) each
    const uint32_t* n_dev = nullptr;
    int result = 0;                               // index of the buffer holding the output
};

// Onesweep sort (one kernel per 8-bit digit pass, decoupled look-back).
template <typename K>
struct OnesweepBuffers {
    K* keys[2] = {nullptr, nullptr};         // keys[0] holds the input
    uint32_t* vals[2] = {nullptr, nullptr};  // vals[0] holds the input
    const uint32_t* hist = nullptr;          // passes * 256 digit counts of the keys
    uint32_t* status = nullptr;              // passes * 256 * onesweep_tiles look-back words, zero before the sort
    uint32_t* tile_ctr = nullptr;            // passes tile counters, zero before the sort
    uint32_t* err = nullptr;                 // nonzero: a look-back wait exceeded its bound
    int result = 0;                          // index of the buffer holding the output
};

struct Marker;
int64_t sort_tiles(int64_t n);
int64_t onesweep_tiles(int64_t n);  // look-back tiles of the onesweep sort (at most sort_tiles)
int64_t counted_sort_status_bytes(int64_t cap);
hipError_t onesweep_sort_pairs(OnesweepBuffers<uint32_t>& b, int64_t n, int key_bits, hipStream_t s,
                               Marker* mk);
hipError_t onesweep_sort_pairs(OnesweepBuffers<uint64_t>& b, int64_t n, int key_bits, hipStream_t s,
                               Marker* mk);
// launched through a sink (a stream or a graph under construction)
hipError_t sort_pairs_counted(CountedSort<uint32_t>& b, int64_t cap, int key_bits, LaunchSink& ls);
hipError_t sort_pairs_counted(CountedSort<uint64_t>& b, int64_t cap, int key_bits, LaunchSink& ls);

}  // namespace cav
