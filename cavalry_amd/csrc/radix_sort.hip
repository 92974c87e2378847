// Stable LSD radix sort of (key, u32 value) pairs: one kernel per 8-bit digit
// pass (onesweep).
//
// Replaces thrust::stable_sort_by_key at BVH/BVH.cu:335. Keys are 30-bit
// Morton codes in u32 or 63-bit codes in u64; values start as the original
// triangle index, so the output order equals sorting (key, index) pairs. The
// build's digit histograms are accumulated by the kernel that makes the codes.
// The renderers sort as many pairs as a word in device memory says (guided
// paths' shading order and table updates); there k_hist makes the histograms.
#include "dev_common.h"
#include "lbvh.h"
#include "radix_sort.h"

namespace cav {
namespace {

constexpr int kBlock = 256;
constexpr int kRadix = 256;

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K k, int shift) {
    return (uint32_t)(k >> shift) & (kRadix - 1);
}

// element count: n, or the smaller count held on the device
__device__ __forceinline__ int64_t live_n(int64_t n, const uint32_t* n_dev) {
    if (!n_dev) return n;
    const int64_t d = (int64_t)*n_dev;
    return d < n ? d : n;
}

// One read of the keys: digit histograms for every pass at once; zeroes in
// the first pass's look-back words (`zero`, words_per_tile for every `tile` pairs).
template <typename K>
__global__ __launch_bounds__(kBlock) void k_hist(const K* __restrict__ keys, int64_t n,
                                                 const uint32_t* __restrict__ n_dev, int passes,
                                                 uint32_t* __restrict__ hist, int tile, int words_per_tile,
                                                 uint32_t* __restrict__ zero) {
    __shared__ uint32_t h[8 * kRadix];
    n = live_n(n, n_dev);
    const int64_t first = (int64_t)blockIdx.x * kBlock + threadIdx.x, stride = (int64_t)gridDim.x * kBlock;
    if (first - threadIdx.x >= n) return;  // the whole block
    for (int i = threadIdx.x; i < passes * kRadix; i += kBlock) h[i] = 0;
    const int64_t nzero = (n + tile - 1) / tile * words_per_tile;
    for (int64_t i = first; i < nzero; i += stride < n ? stride : (n + kBlock - 1) / kBlock * kBlock) zero[i] = 0u;
    __syncthreads();
    for (int64_t i = first; i < n; i += stride) {
        const K k = keys[i];
        for (int p = 0; p < passes; ++p) atomicAdd(&h[p * kRadix + digit_of(k, 8 * p)], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < passes * kRadix; i += kBlock)
        if (h[i]) atomicAdd(&hist[i], h[i]);
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
}

// ---------------------------------------------------------------- onesweep
// One kernel per digit pass (Merrill & Garland's single-pass radix sort with
// decoupled look-back). Workgroups take tiles in launch order from a counter,
// so every tile a workgroup waits on belongs to a workgroup already running.
// Per tile: rank the keys by digit (the ballot multisplit above), publish the
// tile's per-digit counts, add up predecessors' counts back to the first
// published inclusive prefix, publish this tile's inclusive prefix, and
// scatter the tile through LDS so each digit run is written contiguously
// (the keys, then the values through the same LDS buffer).
// Look-back words: flag << 30 | count (flag 1: this tile's count, 2: count
// of this and all earlier tiles), read and written as agent-scope atomics.
// The global start of every digit comes from the pass's digit histogram,
// which the key producer accumulated beforehand.
// The shape (512 threads x 16 keys, 4 predecessors per look-back step) was
// the fastest of a sweep over 256..1024 threads, 16..32 keys per thread and
// windows of 1..32 predecessors on 2^24 Morton codes: larger windows load
// the look-back words faster than they are published.
// Sorts of a count held on the device take 256 threads (half the tile: their
// 0.1M to 1M pairs are few tiles) and 64-bit look-back words (a render may
// hold more than 2^30 update records).
constexpr int kOsBlock = 512;
constexpr int kOsItems = 16;
constexpr int kOsTile = kOsBlock * kOsItems;
constexpr int kOsSmall = 256;
constexpr int kSpinLimit = 1 << 24;  // bounded wait; exceeding it flags *err (never expected)
constexpr int kLookback = 4;          // predecessors read per look-back step

// Exclusive scan over the workgroup of one value per thread (threads past
// the first 256 pass 0); returns the total too.
template <int kOsWaves>
__device__ __forceinline__ uint32_t os_excl_scan(uint32_t v, uint32_t* wsum, uint32_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan(v);
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint32_t off = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kOsWaves; ++w) {
        const uint32_t s = wsum[w];
        if (w < wave) off += s;
        total += s;
    }
    __syncthreads();
    return off + inc - v;
}

// S: the look-back word, two flag bits above its count. zero: the look-back
// words of another pass that this pass's tiles clear (null: none).
template <typename K, typename S, int kOsBlock>
__global__ __launch_bounds__(kOsBlock) void k_onesweep(const K* __restrict__ kin,
                                                       const uint32_t* __restrict__ vin,
                                                       K* __restrict__ kout, uint32_t* __restrict__ vout,
                                                       int64_t n, const uint32_t* __restrict__ n_dev, int shift,
                                                       const uint32_t* __restrict__ phist,
                                                       S* status, S* zero, uint32_t* tile_ctr,
                                                       uint32_t* err) {
    constexpr int kOsWaves = kOsBlock / 64, kOsTile = kOsBlock * kOsItems;
    constexpr S kAgg = (S)1 << (8 * sizeof(S) - 2), kIncl = (S)2 << (8 * sizeof(S) - 2), kCountMask = kAgg - 1;
    __shared__ uint32_t wh[kOsWaves][kRadix];
    __shared__ uint32_t tstart[kRadix];
    __shared__ uint32_t gbase[kRadix];
    __shared__ uint32_t wsum[kOsWaves];
    __shared__ uint32_t stile;
    __shared__ K stage[kOsTile];  // the tile's keys in digit order, then its values

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    n = live_n(n, n_dev);
    if ((int64_t)blockIdx.x * kOsTile >= n) return;  // as many workgroups stay as there are tiles
    if (threadIdx.x == 0) stile = atomicAdd(tile_ctr, 1u);
    for (int i = threadIdx.x; i < kOsWaves * kRadix; i += kOsBlock) (&wh[0][0])[i] = 0;
    __syncthreads();
    const int tile = (int)stile;
    const int64_t tbase = (int64_t)tile * kOsTile;
    const int tile_n = (int)((n - tbase) < kOsTile ? (n - tbase) : kOsTile);

    // wave w owns elements [w*64*kOsItems, (w+1)*64*kOsItems) of the tile;
    // item j of lane l is element w*64*kOsItems + j*64 + l, so (w, j, l) is
    // element order. Loads go through one uniform base per wave.
    K key[kOsItems];
    uint32_t val[kOsItems];
    uint32_t rank[kOsItems];
    const int wbase = wave * 64 * kOsItems;
    const K* kb = kin + tbase + wbase;
    const uint32_t* vb = vin + tbase + wbase;
    if (tile_n == kOsTile) {
#pragma unroll
        for (int j = 0; j < kOsItems; ++j) {
            key[j] = kb[j * 64 + lane];
            val[j] = vb[j * 64 + lane];
        }
    } else {
#pragma unroll
        for (int j = 0; j < kOsItems; ++j) {
            const bool in = wbase + j * 64 + lane < tile_n;
            key[j] = in ? kb[j * 64 + lane] : (K)0;
            val[j] = in ? vb[j * 64 + lane] : 0u;
        }
    }

    // lanes with equal digits: eight ballots; a lane keeps the lanes that
    // agree with it on every bit (m XNOR its own bit, spread over 64 lanes)
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int j = 0; j < kOsItems; ++j) {
        const bool valid = wbase + j * 64 + lane < tile_n;
        const uint32_t d = valid ? digit_of(key[j], shift) : 0u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int32_t sb = -(int32_t)((d >> b) & 1u);
            const uint64_t m = __ballot(sb != 0);
            const uint64_t sm = (uint64_t)(uint32_t)sb | ((uint64_t)(uint32_t)sb << 32);
            peers &= ~(m ^ sm);
        }
        uint32_t r = 0;
        if (valid) {
            const uint32_t before = (uint32_t)__popcll(peers & lt);
            const uint32_t base = wh[wave][d];
            if (before == 0) wh[wave][d] = base + (uint32_t)__popcll(peers);
            r = base + before;
        }
        rank[j] = r;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    if (threadIdx.x < kRadix) {
        const int d = threadIdx.x;
        uint32_t run = 0;
#pragma unroll
        for (int w = 0; w < kOsWaves; ++w) {
            const uint32_t c = wh[w][d];
            wh[w][d] = run;
            run += c;
        }
        tstart[d] = run;  // the tile's count of digit d, until the scan below
        // look-back for digit d: publish, then sum predecessors' counts
        S* my = status + (int64_t)tile * kRadix + d;
        if (zero) zero[(int64_t)tile * kRadix + d] = 0;
        uint32_t excl = 0;
        if (tile == 0) {
            __hip_atomic_store(my, kIncl | (S)run, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            __hip_atomic_store(my, kAgg | (S)run, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // predecessors are read kLookback at a time (independent loads in
            // flight), then added newest first up to the first inclusive
            // count or the first one not yet published, which is read again
            int t = tile - 1;
            int spins = 0;
            bool done = false;
            while (!done) {
                S w[kLookback];
#pragma unroll
                for (int q = 0; q < kLookback; ++q)
                    w[q] = t - q >= 0 ? __hip_atomic_load(status + (int64_t)(t - q) * kRadix + d, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT)
                                      : kIncl;
                int used = 0;
#pragma unroll
                for (int q = 0; q < kLookback; ++q) {
                    const S f = w[q] & ~kCountMask;
                    if (f == 0) break;
                    excl += (uint32_t)(w[q] & kCountMask);
                    used = q + 1;
                    if (f == kIncl) { done = true; break; }
                }
                t -= used;
                if (!done && used == 0) {
                    if (++spins > kSpinLimit) { atomicAdd(err, 1u); break; }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            __hip_atomic_store(my, kIncl | ((S)excl + (S)run), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        gbase[d] = excl;
    }
    __syncthreads();
    {
        // start of digit d in the output: digits below d, then earlier tiles;
        // in the tile: digits below d
        const bool dt = threadIdx.x < kRadix;
        uint32_t tot;
        const uint32_t below = os_excl_scan<kOsWaves>(dt ? phist[threadIdx.x] : 0u, wsum, tot);
        const uint32_t ts = os_excl_scan<kOsWaves>(dt ? tstart[threadIdx.x] : 0u, wsum, tot);
        if (dt) {
            gbase[threadIdx.x] += below;
            tstart[threadIdx.x] = ts;
        }
    }
    __syncthreads();

#pragma unroll
    for (int j = 0; j < kOsItems; ++j) {
        if (wbase + j * 64 + lane < tile_n) {
            const uint32_t d = digit_of(key[j], shift);
            rank[j] += tstart[d] + wh[wave][d];  // the item's position in the tile's digit order
            stage[rank[j]] = key[j];
        }
    }
    __syncthreads();
    uint32_t o[kOsItems];
#pragma unroll
    for (int j = 0; j < kOsItems; ++j) {
        const int i = threadIdx.x + j * kOsBlock;
        if (i < tile_n) {
            const K k = stage[i];
            const uint32_t d = digit_of(k, shift);
            o[j] = gbase[d] + (uint32_t)(i - (int)tstart[d]);
            kout[o[j]] = k;
        }
    }
    __syncthreads();
    uint32_t* sval = reinterpret_cast<uint32_t*>(stage);
#pragma unroll
    for (int j = 0; j < kOsItems; ++j)
        if (wbase + j * 64 + lane < tile_n) sval[rank[j]] = val[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kOsItems; ++j) {
        const int i = threadIdx.x + j * kOsBlock;
        if (i < tile_n) vout[o[j]] = sval[i];
    }
}

template <typename K>
hipError_t onesweep_impl(OnesweepBuffers<K>& b, int64_t n, int key_bits, hipStream_t s, Marker* mk) {
    const int passes = (key_bits + 7) / 8;
    const int64_t tiles = onesweep_tiles(n);
    int cur = 0;
    for (int p = 0; p < passes; ++p) {
        hipLaunchKernelGGL((k_onesweep<K, uint32_t, kOsBlock>), dim3((unsigned)tiles), dim3(kOsBlock), 0, s,
                           b.keys[cur], b.vals[cur], b.keys[cur ^ 1], b.vals[cur ^ 1], n, (const uint32_t*)nullptr,
                           8 * p, b.hist + p * kRadix, b.status + (int64_t)p * kRadix * tiles, (uint32_t*)nullptr,
                           b.tile_ctr + p, b.err);
        mark(mk, "sort_onesweep");
        cur ^= 1;
    }
    b.result = cur;
    return hipGetLastError();
}

// One pass uses one of the two sets of look-back words and clears the other.
// Three kernels per pass (counts, scan, scatter) and a clear took 26 launches
// for 64-bit keys where this takes 9: 175 us a step of a served burst before, 102
// now (0.3M records); the shading order of 2M hits (18 bits) 98 us and 91.
template <typename K>
hipError_t counted_impl(CountedSort<K>& b, int64_t cap, int key_bits, LaunchSink& ls) {
    using S = uint64_t;
    const int passes = (key_bits + 7) / 8;
    int64_t hblocks = (cap + kBlock * 16 - 1) / (kBlock * 16);
    hblocks = hblocks > 2048 ? 2048 : (hblocks < 1 ? 1 : hblocks);
    ls.launch("k_hist", &k_hist<K>, dim3((unsigned)hblocks), dim3(kBlock), b.keys[0], cap, b.n_dev, passes, b.work,
              kOsSmall * kOsItems, kRadix * (int)(sizeof(S) / 4), (uint32_t*)b.status[0]);
    int cur = 0;
    for (int p = 0; p < passes; ++p) {
        ls.launch("k_onesweep", &k_onesweep<K, S, kOsSmall>, dim3((unsigned)sort_tiles(cap)), dim3(kOsSmall),
                  b.keys[cur], b.vals[cur], b.keys[cur ^ 1], b.vals[cur ^ 1], cap, b.n_dev, 8 * p,
                  b.work + p * kRadix, b.status[p & 1], b.status[(p & 1) ^ 1], b.work + kRadix * 8 + p, b.work + kCountedSortErr);
        cur ^= 1;
    }
    b.result = cur;
    return ls.err;
}

}  // namespace

int64_t sort_tiles(int64_t n) { return (n + kOsSmall * kOsItems - 1) / (kOsSmall * kOsItems); }
int64_t onesweep_tiles(int64_t n) { return (n + kOsTile - 1) / kOsTile; }
int64_t counted_sort_status_bytes(int64_t cap) { return 8 * kRadix * sort_tiles(cap); }

hipError_t onesweep_sort_pairs(OnesweepBuffers<uint32_t>& b, int64_t n, int key_bits, hipStream_t s,
                               Marker* mk) {
    return onesweep_impl<uint32_t>(b, n, key_bits, s, mk);
}
hipError_t onesweep_sort_pairs(OnesweepBuffers<uint64_t>& b, int64_t n, int key_bits, hipStream_t s,
                               Marker* mk) {
    return onesweep_impl<uint64_t>(b, n, key_bits, s, mk);
}
hipError_t sort_pairs_counted(CountedSort<uint32_t>& b, int64_t cap, int key_bits, LaunchSink& ls) {
    return counted_impl(b, cap, key_bits, ls);
}
hipError_t sort_pairs_counted(CountedSort<uint64_t>& b, int64_t cap, int key_bits, LaunchSink& ls) {
    return counted_impl(b, cap, key_bits, ls);
}

}  // namespace cav
