// Build of the wide traversal tree: an 8-wide tree with 8-bit child boxes
// (after Ylitie, Karras and Laine, "Efficient Incoherent Ray Traversal on
// GPUs Through Compressed Wide BVHs", 2017), collapsed from a binary radix
// tree over Morton codes of its own.
//
// The reference's codes keep their quirk (BVH/BVH.cu:79-92: centroids below
// the scene's centre saturate to 0, so up to seven eighths of the scene share
// a code prefix), and its tree is what every export and test compares. A ray
// over that tree fetched thousands of records (bounce rays over a 1M-triangle
// interior: 7500 each). What a trace returns does not depend on the tree
// except through the order of equally near hits (wide_trace.hip), so the
// traces walk this tree instead, whose codes span the whole scene box.
// Tried and dropped, in records fetched per ray on interiors of 1M triangles
// (camera / bounce / shadow) and soups of 4M: cubic cells 26 / 64 / 32 and 90
// against 21 / 59 / 23 and 59 here, 42-bit codes 23 / 62 / 34 and 90 (with the
// classes that follow), triangles 8 (32) times larger than the typical one in
// trees of their own 23 / 63 / 36 and 90 (19 / 60 / 30 and 63).
#include "dev_common.h"
#include "lbvh.h"
#include "wide.h"

namespace cav {
namespace {

constexpr int kBlock = 256;
constexpr int kCodeBits = 30;
constexpr int kCtrTris = 80, kCtrTop = 81;  // words past the level counts
constexpr int kMaxWideLevels = 78;

__device__ __forceinline__ uint32_t spread10(uint32_t x) {
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}
__device__ __forceinline__ uint32_t cell10(float v) {  // NaN -> 0
    return (uint32_t)(int)fmn(fmx(v * 1024.f, 0.f), 1023.f);
}

// Codes of the triangle boxes' centres, the digit counts of the four sort
// passes, and zeroes in the sort's look-back words (as k_morton does for the
// reference's codes). 36 B read and 8 B written per triangle.
constexpr int kCodeBlocks = 1024;
__global__ __launch_bounds__(kBlock) void k_wide_codes(const float* __restrict__ tris, int64_t n,
                                                       const uint32_t* __restrict__ ob, uint32_t* __restrict__ keys,
                                                       uint32_t* __restrict__ vals, uint32_t* __restrict__ hist,
                                                       uint32_t* __restrict__ zero, int64_t nzero) {
    __shared__ uint32_t h[4 * 256];
    for (int j = threadIdx.x; j < 4 * 256; j += kBlock) h[j] = 0u;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    const int64_t first = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    for (int64_t j = first; j < nzero; j += stride) zero[j] = 0u;
    __syncthreads();
    const v3 slo = mk3(ord2f(ob[0]), ord2f(ob[1]), ord2f(ob[2]));
    const v3 shi = mk3(ord2f(ob[3]), ord2f(ob[4]), ord2f(ob[5]));
    const v3 se = sub3(shi, slo);
    const v3 inv = mk3(1.f / fmx(se.x, 1e-30f), 1.f / fmx(se.y, 1e-30f), 1.f / fmx(se.z, 1e-30f));
    for (int64_t i = first; i < n; i += stride) {
        const float* p = tris + i * 9;
        const v3 a = mk3(p[0], p[1], p[2]), b = mk3(p[3], p[4], p[5]), c = mk3(p[6], p[7], p[8]);
        const v3 lo = mk3(fmn(a.x, fmn(b.x, c.x)), fmn(a.y, fmn(b.y, c.y)), fmn(a.z, fmn(b.z, c.z)));
        const v3 hi = mk3(fmx(a.x, fmx(b.x, c.x)), fmx(a.y, fmx(b.y, c.y)), fmx(a.z, fmx(b.z, c.z)));
        const v3 m = sub3(scale3(add3(lo, hi), 0.5f), slo);
        const uint32_t key = (spread10(cell10(m.x * inv.x)) << 2) | (spread10(cell10(m.y * inv.y)) << 1) |
                             spread10(cell10(m.z * inv.z));
        keys[i] = key;
        vals[i] = (uint32_t)i;
#pragma unroll
        for (int q = 0; q < 4; ++q) atomicAdd(&h[q * 256 + ((key >> (8 * q)) & 255u)], 1u);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < 4 * 256; j += kBlock)
        if (h[j]) atomicAdd(&hist[j], h[j]);
}

// Sort histograms, tile counters and level counts to zero; the root's item.
// (The failure word stays: where b's own sort failed, its gates may hold
// arrivals and nothing is built.)
__global__ void k_wide_init(uint32_t* hist, int nhist, uint32_t* ctr, uint4* nodes, int n) {
    for (int i = threadIdx.x; i < nhist; i += blockDim.x) hist[i] = 0u;
    for (int i = threadIdx.x; i < kWideCtrWords; i += blockDim.x) ctr[i] = i == 0 ? 1u : 0u;
    if (threadIdx.x == 0) nodes[5] = make_uint4(0u, 0u, (uint32_t)n - 1u, 0u);
}

struct WideBuild {
    const NodeBox* nbox;  // binary tree over the sorted codes (ids as the reference's)
    const int4* topo;
    const uint32_t* order;
    const float* tris;
    const int32_t* mesh;
    const uint32_t* bounds;  // the triangles' box (order-preserving ints)
    const uint32_t* err;     // set: the sort failed, nothing is built
    uint4* nodes;
    float4* wtris;
    uint32_t* ctr;
    int n;
};

__device__ __forceinline__ void lds_sync() {  // LDS written and read by one wave
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint32_t group_max(uint32_t v) {  // over 8 lanes
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) v = max(v, (uint32_t)__shfl_xor((int)v, d, 64));
    return v;
}
__device__ __forceinline__ uint32_t group_or(uint32_t v) {
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) v |= (uint32_t)__shfl_xor((int)v, d, 64);
    return v;
}

// One wide node per group of 8 lanes, one child per lane. Starts from the
// binary node's two children and opens the inner one of largest area until
// eight are held; children of more than kWideLeaf triangles become nodes of
// the next level, the rest leaf slots. A child's slot is the octant of the
// node that its centre lies towards (the best free one, best fits first), so
// that slots in the order slot ^ ray octant go front to back. A wave's eight
// nodes take their children's places with one atomic. Every lane of the wave
// calls it; groups without a node pass valid = false.
__device__ void wide_collapse(const WideBuild& w, uint32_t idx, bool valid, uint32_t next_start, uint32_t* next_ctr,
                              uint32_t min_unit, uint4* stage) {
    const int lane = threadIdx.x & 63, g = lane >> 3, sl = lane & 7;
    const int n = w.n;
    uint4 it = make_uint4(0u, 0u, 0u, 0u);
    if (valid) it = w.nodes[(int64_t)idx * kWideWords + 5];
    const NodeBox nb = w.nbox[it.x];
    const int4 tp0 = w.topo[it.x];
    const auto split_of = [n](int left) { return left < n - 1 ? left : left - (n - 1); };
    bool have = valid && sl < 2;
    int cid = 0, cl = 0, cr = 0;
    float4 ba = make_float4(0, 0, 0, 0), bb = ba;
    int4 tp = make_int4(0, 0, 0, 0);
    if (have) {
        const int sp = split_of(tp0.x);
        cid = sl == 0 ? tp0.x : tp0.y;
        cl = sl == 0 ? (int)it.y : sp + 1;
        cr = sl == 0 ? sp : (int)it.z;
        const NodeBox b = w.nbox[cid];
        ba = b.a; bb = b.b;
        tp = w.topo[cid];
    }
    int nch = 2;
#pragma unroll 1
    for (int k = 2; k < 8; ++k) {
        const bool inner = have && cid < n - 1;
        const uint32_t key =
            group_max(inner ? (0x80000000u | (__float_as_uint(ba.w) & 0x7ffffff8u) | (uint32_t)(7 - sl)) : 0u);
        if (__ballot(key != 0u) == 0ull) break;
        const bool open = key != 0u;
        const int src = (lane & 56) | (7 - (int)(key & 7u));
        const int lc = __shfl(tp.x, src, 64), rc = __shfl(tp.y, src, 64);
        const int wl = __shfl(cl, src, 64), wr = __shfl(cr, src, 64);
        const int sp = split_of(lc);
        const bool isw = open && lane == src, isn = open && sl == nch;
        if (isw || isn) {
            have = true;
            cid = isw ? lc : rc;
            cl = isw ? wl : sp + 1;
            cr = isw ? sp : wr;
            const NodeBox b = w.nbox[cid];
            ba = b.a; bb = b.b;
            tp = w.topo[cid];
        }
        nch += open ? 1 : 0;
    }
    const int cnt = cr - cl + 1;
    const bool inner = have && cnt > kWideLeaf;
    const bool leaf = have && !inner;

    // slots: every child asks for the best free one; where several ask for
    // the same, the best fit has it and the others ask again
    int slot = 0;
    {
        const float cx = (ba.x + bb.x) - (nb.a.x + nb.b.x), cy = (ba.y + bb.y) - (nb.a.y + nb.b.y),
                    cz = (ba.z + bb.z) - (nb.a.z + nb.b.z);
        uint32_t free_slots = 0xffu;
        bool todo = have;
        while (__ballot(todo)) {
            float bv = -INFINITY;
            int bs = __ffs((int)free_slots) - 1;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const float v = (s & 1 ? cx : -cx) + (s & 2 ? cy : -cy) + (s & 4 ? cz : -cz);
                if (((free_slots >> s) & 1u) && v > bv) { bv = v; bs = s; }
            }
            // wish: the fit in order, then the lane (so that none are equal), the slot in the low bits
            const uint32_t wish = todo ? (f2ord(bv) & ~127u) | (uint32_t)(8 | sl) << 3 | (uint32_t)bs : 0u;
            bool mine = todo;
#pragma unroll
            for (int d = 1; d < 8; ++d) {
                const uint32_t o = (uint32_t)__shfl_xor((int)wish, d, 64);
                mine = mine && !(o > wish && (o & 7u) == (uint32_t)bs);
            }
            if (mine) { slot = bs; todo = false; }
            free_slots &= ~group_or(mine ? 1u << bs : 0u);
        }
    }

    // places of the inner children and of the triangles
    const uint64_t innb = __ballot(inner);
    const uint32_t imask = group_or(inner ? 1u << slot : 0u);
    const uint32_t counts = group_or(leaf ? (uint32_t)cnt << (2 * slot) : 0u);
    const auto count_of = [](uint32_t c) { return (uint32_t)(__popc(c & 0x5555u) + 2 * __popc(c & 0xaaaau)); };
    const uint32_t ntri = count_of(counts);
    uint32_t tpre = ntri;
#pragma unroll
    for (int d = 8; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)tpre, d, 64);
        if (lane >= d) tpre += o;
    }
    uint32_t base_n = 0, base_t = 0;
    if (lane == 63) {
        const uint32_t ni = (uint32_t)__popcll(innb);
        if (ni) base_n = atomicAdd(next_ctr, ni);
        if (tpre) base_t = atomicAdd(w.ctr + kCtrTris, tpre);
    }
    base_n = (uint32_t)__shfl((int)base_n, 63, 64);
    base_t = (uint32_t)__shfl((int)base_t, 63, 64);
    const uint32_t child_base = next_start + base_n + (uint32_t)__popcll(innb & ((1ull << (lane & 56)) - 1ull));
    const uint32_t tri_base = base_t + tpre - ntri;

    // the node's origin, a step of its coordinates (and the smallest unit)
    // below the box, and its scale: the smallest power of two with the box
    // inside 254 units
    uint32_t ex[3];
    float org[3], isc[3];
    const float blo[3] = {nb.a.x, nb.a.y, nb.a.z}, bhi[3] = {nb.b.x, nb.b.y, nb.b.z};
    const float least = __uint_as_float(min_unit << 23);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        org[k] = blo[k] - fmx(fabsf(blo[k]) * 0x1p-23f, least);
        uint32_t e = (__float_as_uint(fmx(bhi[k] - org[k], 0.f) * (1.0001f / 254.f)) >> 23) + 1u;
        e = e < min_unit ? min_unit : (e > 230u ? 230u : e);  // (coordinates up to 2^40 are traced: 161 at most)
        ex[k] = e + kPlaneBits;
        isc[k] = __uint_as_float((254u - e) << 23);
    }
    uint8_t* mine = reinterpret_cast<uint8_t*>(stage + g * 5);
    if (sl < 5) stage[g * 5 + sl] = make_uint4(0u, 0u, 0u, 0u);
    lds_sync();
    if (have) {
        const float lo[3] = {ba.x, ba.y, ba.z}, hi[3] = {bb.x, bb.y, bb.z};
        // rounded outwards; the 1e-4 units cover the rounding of the two
        // operations (255 units times 2^-23 at most)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float ql = floorf((lo[k] - org[k]) * isc[k] - 1e-4f), qh = ceilf((hi[k] - org[k]) * isc[k] + 1e-4f);
            mine[wide_plane(k, slot)] = (uint8_t)(int)fmn(fmx(ql, 0.f), 255.f);
            mine[wide_plane(k, slot) + 2] = (uint8_t)(int)fmn(fmx(qh, 0.f), 255.f);
        }
        const uint32_t below = counts & ((1u << (2 * slot)) - 1u);
        mine[24 + slot] = inner ? (uint8_t)((1u << 5) | (24u + (uint32_t)slot))
                                : (uint8_t)((((1u << cnt) - 1u) << 5) | count_of(below));
    }
    if (sl == 0) {
        uint32_t* hd = reinterpret_cast<uint32_t*>(mine);
        hd[0] = __float_as_uint(org[0]);
        hd[1] = __float_as_uint(org[1]);
        hd[2] = __float_as_uint(org[2]);
        hd[3] = ex[0] | (ex[1] << 8) | (ex[2] << 16) | (imask << 24);
        hd[4] = child_base;
        hd[5] = tri_base;
    }
    lds_sync();
    if (valid && sl < 5) w.nodes[(int64_t)idx * kWideWords + sl] = stage[g * 5 + sl];
    lds_sync();
    if (inner) {
        const uint32_t ci = child_base + (uint32_t)__popc(imask & ((1u << slot) - 1u));
        w.nodes[(int64_t)ci * kWideWords + 5] = make_uint4((uint32_t)cid, (uint32_t)cl, (uint32_t)cr, 0u);
    }
    if (leaf) {
        const uint32_t at = tri_base + count_of(counts & ((1u << (2 * slot)) - 1u));
        for (int t = 0; t < cnt; ++t) {
            const uint32_t prim = w.order[cl + t];
            const float* p = w.tris + (int64_t)prim * 9;
            float4* o = w.wtris + (int64_t)(at + t) * 3;
            o[0] = make_float4(p[0], p[1], p[2], __uint_as_float(prim));
            o[1] = make_float4(p[3], p[4], p[5], __int_as_float(w.mesh ? w.mesh[prim] : 0));
            o[2] = make_float4(p[6], p[7], p[8], 0.f);
        }
    }
}

__device__ __forceinline__ uint32_t min_unit_of(const uint32_t* bounds) {
    float box[6];
    for (int k = 0; k < 6; ++k) box[k] = ord2f(bounds[k]);
    return wide_scale(box).min_unit;
}

__device__ __forceinline__ uint32_t ctr_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Levels from *(ctr + kCtrTop) + skip on in one workgroup (1024 threads, 128
// nodes at a time), while they hold at most `limit` nodes; leaves the level
// it stopped at in kCtrTop. The first levels are a few dependent loads each,
// so one workgroup's barriers are cheaper than launches, and a scene of a few
// thousand triangles needs no other launch.
__global__ __launch_bounds__(1024) void k_wide_levels(WideBuild w, int skip, uint32_t limit) {
    __shared__ uint4 stage[16][40];
    const int wave = threadIdx.x >> 6, g = (threadIdx.x & 63) >> 3;
    if (*w.err) return;
    const uint32_t min_unit = min_unit_of(w.bounds);
    int lvl = (int)ctr_load(w.ctr + kCtrTop) + skip;
    uint32_t start = 0;
    for (int k = 0; k < lvl; ++k) start += ctr_load(w.ctr + k);
    for (; lvl < kMaxWideLevels; ++lvl) {
        const uint32_t cnt = ctr_load(w.ctr + lvl);
        if (cnt == 0u || cnt > limit) break;
        for (uint32_t b = 0; b < cnt; b += 128u) {
            const uint32_t i = b + (uint32_t)(wave * 8 + g);
            wide_collapse(w, start + (i < cnt ? i : 0u), i < cnt, start + cnt, w.ctr + lvl + 1, min_unit, stage[wave]);
        }
        __syncthreads();
        start += cnt;
    }
    __syncthreads();
    if (threadIdx.x == 0) w.ctr[kCtrTop] = (uint32_t)lvl;
}

// One level over the device: level kCtrTop + j.
__global__ __launch_bounds__(kBlock) void k_wide_level(WideBuild w, int j) {
    __shared__ uint4 stage[kBlock / 64][40];
    const int wave = threadIdx.x >> 6, g = (threadIdx.x & 63) >> 3;
    const int lvl = (int)w.ctr[kCtrTop] + j;
    if (lvl >= kMaxWideLevels || *w.err) return;
    uint32_t start = 0;
    for (int k = 0; k < lvl; ++k) start += w.ctr[k];
    const uint32_t cnt = w.ctr[lvl], min_unit = min_unit_of(w.bounds);
    const uint32_t per = gridDim.x * (kBlock / 8);
    for (uint32_t b = blockIdx.x * (kBlock / 8) + (uint32_t)(wave * 8); b < cnt; b += per) {
        const uint32_t i = b + (uint32_t)g;
        wide_collapse(w, start + (i < cnt ? i : 0u), i < cnt, start + cnt, w.ctr + lvl + 1, min_unit, stage[wave]);
    }
}

size_t up256(size_t b) { return (b + 255) / 256 * 256; }

}  // namespace

size_t wide_bytes(int n) {
    const size_t N = (size_t)n;
    return up256(4 * kWideCtrWords) + 256 + up256(16 * kWideWords * (size_t)wide_node_capacity(n)) + up256(48 * N) +
           up256(4 * N) + (n <= kWideApart ? wide_scratch_bytes(n) : 0);
}
size_t wide_scratch_bytes(int n) {
    const size_t N = (size_t)n, M = 2 * N - 1;
    return 4 * up256(4 * N) + up256(sizeof(NodeBox) * M) + up256(sizeof(int4) * M);
}

namespace {
struct Carver {
    unsigned char* p;
    template <typename T>
    void take(T*& out, size_t bytes) {
        out = reinterpret_cast<T*>(p);
        p += up256(bytes);
    }
};
}  // namespace

void wide_carve(WideBuffers& w, void* base, int n) {
    const size_t N = (size_t)n;
    Carver c{static_cast<unsigned char*>(base)};
    w.base = base;
    c.take(w.ctr, 4 * kWideCtrWords);
    c.take(w.bounds, 64);
    c.take(w.nodes, 16 * kWideWords * (size_t)wide_node_capacity(n));
    c.take(w.tris, 48 * N);
    c.take(w.leaf_of, 4 * N);
    w.scratch = n <= kWideApart ? c.p : nullptr;
}

hipError_t wide_build(WideBuffers& w, LbvhBuffers& b, void* scratch, const float* tris, const int32_t* mesh, int n,
                      const uint32_t* bounds, hipStream_t s, Marker* mk) {
    const size_t N = (size_t)n, M = 2 * N - 1;
    const int64_t tiles = onesweep_tiles(n);
    OnesweepBuffers<uint32_t> ob;
    Carver c{static_cast<unsigned char*>(scratch)};
    for (int k = 0; k < 2; ++k) {
        c.take(ob.keys[k], 4 * N);
        c.take(ob.vals[k], 4 * N);
    }
    NodeBox* nbox;
    int4* topo;
    c.take(nbox, sizeof(NodeBox) * M);
    c.take(topo, sizeof(int4) * M);
    ob.hist = b.hist;
    ob.status = b.counts;
    ob.tile_ctr = b.hist + kSortHistWords;
    ob.err = b.hist + kSortHistWords + 8;
    int nb = (n + kBlock - 1) / kBlock;
    if (nb > kCodeBlocks) nb = kCodeBlocks;
    hipLaunchKernelGGL(k_wide_init, dim3(1), dim3(1024), 0, s, b.hist, kSortHistWords + 8, w.ctr, w.nodes, n);
    hipLaunchKernelGGL(k_wide_codes, dim3(nb), dim3(kBlock), 0, s, tris, (int64_t)n, bounds, ob.keys[0], ob.vals[0],
                       b.hist, b.counts, 4 * 256 * tiles);
    mark(mk, "wide_codes");
    hipError_t e = onesweep_sort_pairs(ob, n, kCodeBits, s, nullptr);
    if (e != hipSuccess) return e;
    mark(mk, "wide_sort");
    const uint32_t* order = ob.vals[ob.result];
    // (the heights go to the level list, which only the treelet rounds use)
    const BottomUpOut out{order, nbox, topo, b.lvl_list, b.gate64, ob.err};
    e = bottom_up_tree(ob.keys[ob.result], kCodeBits, tris, n, out, s, nullptr);
    if (e != hipSuccess) return e;
    mark(mk, "wide_tree");
    const WideBuild wb{nbox, topo, order, tris, mesh, bounds, ob.err, w.nodes, w.tris, w.ctr, n};
    // up to 512 nodes per level in one workgroup; then a launch per level
    // until all but a skewed tree's last few nodes are done; then those
    const bool small = n <= 4096;
    hipLaunchKernelGGL(k_wide_levels, dim3(1), dim3(1024), 0, s, wb, 0, small ? 0xffffffffu : 512u);
    if (!small) {
        int levels = 6;  // (an empty one costs 3 us; a skewed tree left to one workgroup cost 1.2 ms)
        for (int64_t left = (int64_t)n / 512; left > 0; left /= 8) ++levels;
        int64_t blocks = (wide_node_capacity(n) + kBlock / 8 - 1) / (kBlock / 8);
        if (blocks > 2048) blocks = 2048;
        for (int j = 0; j < levels; ++j)
            hipLaunchKernelGGL(k_wide_level, dim3((unsigned)blocks), dim3(kBlock), 0, s, wb, j);
        hipLaunchKernelGGL(k_wide_levels, dim3(1), dim3(1024), 0, s, wb, levels, 0xffffffffu);
    }
    mark(mk, "wide_nodes");
    return hipGetLastError();
}

}  // namespace cav
