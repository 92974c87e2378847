// Closest-hit and any-hit traces over the wide tree (wide.h), with the
// reference's answers bit for bit (BVH::intersect and BVH::testVisibility,
// BVH/BVH.h:23-189).
//
// Why another tree gives the same answers. A triangle is a candidate when the
// reference can reach its leaf: when the ray hits the leaf's own box. The slab
// test (Core/BoundingBox.h:55-74) is monotone under box inclusion -- the
// subtraction, the product with the ray's reciprocal direction, min and max
// all are -- so a ray that hits the leaf's box hits every box above it, and
// starts in them no later -- unless the ray runs exactly along a plane of the
// leaf's box (0 * inf = NaN in the slab test, which then can fail further up):
// such a hit counts only after every box above it has been tested (grazes,
// leaf_path). The triangle's vertices are in the wide tree's
// record, so its leaf box is tested here exactly as the reference tests it.
//
// Any-hit: the answer is whether any candidate blocks the ray before its
// limit, which no order changes.
//
// Closest-hit: the nearest candidate M is the reference's answer unless it
// skips M, and it skips a box only at or beyond a hit X found before: every
// box on M's path starts at or before M's own (e_M), so such an X lies at or
// before max(t_M, e_M). A ray that met another hit X with t_X <= max(t_M,
// e_M) -- coincident surfaces, a box standing on a floor -- goes to
// k_wide_finish, which collects all hits that close and replays the
// reference's order among them from the reference's tree. The trace keeps the
// nearest triangle hit and the second's distance and looks at the nearest's
// own box at the end; where that hit turns out to be no candidate, or a
// grazing one, the finishing pass decides too (an any-hit ray likewise, by
// the first triangle hit that blocks it).
//
// The wide boxes only have to contain the exact ones. They are rounded
// outwards, their planes' distances carry a slack of 2^-20 of their terms
// (the two roundings are 2^-23 each), and boxes are skipped only beyond
// kReach = 1 + 2^-5 times the nearest hit (any-hit: times the limit) and a
// slack of 2^-16 of the scene's largest coordinate. A triangle beyond that
// could matter only if Moller-Trumbore put its t about as far short of the
// start of its own box (the assumption, with a margin 16 times wider, that
// the cooperative passes over the reference's tree make, traverse.hip). It does where its determinant is
// little more than rounding: a triangle met edge on, a needle, products near
// the smallest floats. Such a triangle rarely comes alone -- a ray in the
// plane of a tessellated floor meets dozens -- so a closest-hit ray that
// tests one (thin_test), or whose nearest hit is one (thin_hit), goes to the
// finishing pass, which then walks the ray's whole line without skipping any
// box: its answer assumes nothing about distances. Of 140 million rays in the
// plane of turned floors with walls and at needles none was answered wrongly
// (and on a model of 460,000, none down to an eighth of thin_test's limit);
// what remains open is a ray whose only thin triangles all lie behind its
// nearest hit. Random rays go that way once in 20,000 (interiors, soups of
// 20,000 triangles); where half of the triangles are needles of 1:30, one in
// 200 does (1M rays over 400K triangles 3.0 to 3.3 ms), of 1:300 one in 25
// (4.0 to 7.2; in the reference's order 22).
//
// Per node and lane: five 16-byte loads from one line and 198 VALU
// instructions for eight children, against four loads and 90 instructions
// for the two children of a reference node; a stack entry holds all of a
// node's remaining children. The instructions are what bounds the traces
// (bounce rays over 1M triangles: 91% of the issue slots, 47% of the lanes at
// work; a tree of 2^24 triangles: 66%, and 4.3 TB/s past L2). Planes
// read as half floats instead of converted bytes, and the nearest hit's own
// box tested once when the ray is through instead of at every hit (an
// iteration of 64 rays met some hit three times in four): 2M camera rays 0.56
// to 0.50 ms, 1M bounce rays 0.97 to 0.89,
// 2M shadow rays 0.84 to 0.79.
// Tried and dropped: a second set of pending triangles per lane, tested once
// 20 to 40 lanes have some (bounce rays 1.34 to 1.52 ms: lanes wait), and all
// triangles of an iteration before its next node (0.90 to 0.92).
#include <algorithm>
#include <cfloat>

#include "dev_common.h"
#include "launch.h"
#include "lbvh.h"
#include "trace_common.h"
#include "wide.h"
#include "wide_trace.h"

namespace cav {
namespace {

constexpr float kReach = 1.0f + 1.0f / 32.0f;
constexpr float kOwnBox = 1.0f + 1.0f / 64.0f;  // a box starting further beyond its hit: the reference decides
constexpr float kSlack = 1.0f / 1048576.0f;     // 2^-20
// Limits of a determinant against the sizes of its factors:
constexpr float kThinTest = 0x1p-18f;  // of a tested triangle (largest components)
constexpr float kThinHit = 0x1p-20f;   // of a hit: the error of its t against what boxes are visited beyond it
constexpr float kTiny = 0x1p-100f;     // below: products in the triangle test may have lost bits to underflow
constexpr int kWideStack = 12;                  // stack entries in LDS
constexpr int kWideDeep = 68;                   // entries in all: more than a tree over 32-bit codes has levels
// Idle lanes a wave collects before it hands out rays: setting a ray up costs
// as much as a third of a node test for however few lanes (Cornell path
// 8.17 ms at 1, 7.92 at 8, 7.90 at 16; bounce rays 1.23, 1.20, 1.23).
constexpr int kRefill = 12;
constexpr int kUndecided = -2;                  // hit id of a ray that the finishing pass still has to find by scanning

// selector of the near planes of an axis (a byte, a zero, a byte, a zero); the far ones' is ^ kFarPlanes
__device__ __forceinline__ uint32_t near_planes(float inv) { return inv < 0.f ? 0x0c030c02u : 0x0c010c00u; }
constexpr uint32_t kFarPlanes = 0x00020002u;

// The ray as the node tests use it: direction scaled to a largest component
// in [1, 2) (a power of two, exact), reciprocals bounded so that an axis the
// ray runs along gives huge distances instead of infinities (WideScale).
struct WideRay {
    v3 o, inv;
    float scale;  // true t * scale = t in the scaled direction
    uint32_t oct;
    uint32_t nx, ny, nz;  // selectors of the near planes (near_planes)
};
__device__ __forceinline__ float wide_rcp(float d, float most) {
    const float r = __builtin_amdgcn_rcpf(d);
    return __builtin_copysignf(fmn(fabsf(r), most), d);
}
enum RayKind {
    kRayFine,
    kRayOdd,  // only the reference's traversal takes it: from far beyond the scene, or a direction near float's limits
    kRayDead  // hits nothing: a zero direction (every determinant is 0) or one that is not finite, or a NaN
              // origin (Moller-Trumbore's t is 0 or NaN for every finite triangle)
};
__device__ __forceinline__ RayKind wide_ray(v3 o, v3 d, float farthest, float rcp_max, WideRay& r) {
    const float m = fmx(fabsf(d.x), fmx(fabsf(d.y), fabsf(d.z)));
    const uint32_t e = __float_as_uint(m) >> 23;
    const bool dead = !(fabsf(d.x) <= FLT_MAX && fabsf(d.y) <= FLT_MAX && fabsf(d.z) <= FLT_MAX) || m == 0.f ||
                      !(o.x == o.x && o.y == o.y && o.z == o.z);
    const bool fine = fabsf(o.x) <= farthest && fabsf(o.y) <= farthest && fabsf(o.z) <= farthest && e >= 2u &&
                      e <= 252u;
    r.o = o;
    r.scale = __uint_as_float(e << 23);
    const float down = __uint_as_float((254u - e) << 23);
    r.inv = mk3(wide_rcp(d.x * down, rcp_max), wide_rcp(d.y * down, rcp_max), wide_rcp(d.z * down, rcp_max));
    r.nx = near_planes(r.inv.x); r.ny = near_planes(r.inv.y); r.nz = near_planes(r.inv.z);
    r.oct = (r.inv.x < 0.f ? 1u : 0u) | (r.inv.y < 0.f ? 2u : 0u) | (r.inv.z < 0.f ? 4u : 0u);
    return dead ? kRayDead : (fine ? kRayFine : kRayOdd);
}

// Bits of a node's eight slot bytes, four at a time: the inner ones get the
// ray's octant xored into their slot, so that ascending bits go front to back.
__device__ __forceinline__ uint32_t order_slots(uint32_t meta, uint32_t oct4) {
    const uint32_t inner = (meta & (meta << 1)) & 0x10101010u;  // 24 + slot: bits 3 and 4
    return meta ^ (oct4 & ((inner >> 1) - (inner >> 4)));  // 7 in the low bits of the inner ones' bytes
}

// One axis of one node: plane distances are (the byte's half float) * a + b.
struct AxisPlanes {
    float an, af, bn, bf;
};
__device__ __forceinline__ AxisPlanes axis_planes(float p, uint32_t e, float o, float inv) {
    const float a = __uint_as_float(e << 23) * inv, b = (p - o) * inv;
    AxisPlanes r;
    r.an = __builtin_fmaf(-kSlack, fabsf(a), a);
    r.af = __builtin_fmaf(kSlack, fabsf(a), a);
    r.bn = __builtin_fmaf(-kSlack, fabsf(b), b);
    r.bf = __builtin_fmaf(kSlack, fabsf(b), b);
    return r;
}

// The planes of two slots as two half floats, near or far ones by the
// selector: one byte permutation in place of two conversions and half a
// select, and the fused multiply-add takes halves as they are (denormal ones
// included: byte * 2^-24 exactly, as the exponents are kPlaneBits up).
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ half2v plane_pair(uint32_t word, uint32_t sel) {
    return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(word, word, sel));
}
// Tests a node's children against the ray up to `cut` (scaled units): bits
// 0..23 the triangles of hit leaf slots, 24..31 the hit inner children in
// front-to-back order.
__device__ __forceinline__ uint32_t test_children(const uint4& w0, const uint4& w1, const uint4& w2, const uint4& w3,
                                                  const uint4& w4, const WideRay& r, float cut) {
    const AxisPlanes x = axis_planes(__uint_as_float(w0.x), w0.w & 255u, r.o.x, r.inv.x);
    const AxisPlanes y = axis_planes(__uint_as_float(w0.y), (w0.w >> 8) & 255u, r.o.y, r.inv.y);
    const AxisPlanes z = axis_planes(__uint_as_float(w0.z), (w0.w >> 16) & 255u, r.o.z, r.inv.z);
    const uint32_t fx = r.nx ^ kFarPlanes, fy = r.ny ^ kFarPlanes, fz = r.nz ^ kFarPlanes;
    const uint32_t oct4 = r.oct * 0x01010101u;
    const uint32_t px[4] = {w2.x, w2.y, w2.z, w2.w}, py[4] = {w3.x, w3.y, w3.z, w3.w}, pz[4] = {w4.x, w4.y, w4.z, w4.w};
    uint32_t mask = 0;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const uint32_t meta = order_slots(half ? w1.w : w1.z, oct4);
#pragma unroll
        for (int pair = 0; pair < 2; ++pair) {
            const int w = 2 * half + pair;
            const half2v xn = plane_pair(px[w], r.nx), xf = plane_pair(px[w], fx);
            const half2v yn = plane_pair(py[w], r.ny), yf = plane_pair(py[w], fy);
            const half2v zn = plane_pair(pz[w], r.nz), zf = plane_pair(pz[w], fz);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float tn =
                    fmx(fmx(__builtin_fmaf((float)xn[c], x.an, x.bn), __builtin_fmaf((float)yn[c], y.an, y.bn)),
                        fmx(__builtin_fmaf((float)zn[c], z.an, z.bn), 0.f));
                const float tf =
                    fmn(fmn(__builtin_fmaf((float)xf[c], x.af, x.bf), __builtin_fmaf((float)yf[c], y.af, y.bf)),
                        fmn(__builtin_fmaf((float)zf[c], z.af, z.bf), cut));
                const uint32_t m = meta >> (8 * (2 * pair + c));
                const uint32_t bits = ((m >> 5) & 7u) << (m & 31u);
                mask |= tn <= tf ? bits : 0u;
            }
        }
    }
    return mask;
}

// Whether a slab test divides 0 by 0 on an axis: the ray does not move along
// it and starts on one of the box's two planes.
__device__ __forceinline__ bool grazes(float inv, float o, float lo, float hi) {
    return fabsf(inv) == INFINITY && (o == lo || o == hi);
}

// The triangle's own box as the reference's leaf has it (Core/Triangle.h:242-268)
// and where the ray enters it (-1: never). touch: the ray runs along a plane of
// the box (see grazes).
__device__ __forceinline__ float leaf_entry(const float4& a, const float4& b, const float4& c, v3 o, v3 d, bool& touch) {
    const v3 inv = div3(mk3(1.f, 1.f, 1.f), d);
    const v3 lo = mk3(fmn(a.x, fmn(b.x, c.x)), fmn(a.y, fmn(b.y, c.y)), fmn(a.z, fmn(b.z, c.z)));
    const v3 hi = mk3(fmx(a.x, fmx(b.x, c.x)), fmx(a.y, fmx(b.y, c.y)), fmx(a.z, fmx(b.z, c.z)));
    touch = grazes(inv.x, o.x, lo.x, hi.x) || grazes(inv.y, o.y, lo.y, hi.y) || grazes(inv.z, o.z, lo.z, hi.z);
    return slab(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, o, inv);
}
__device__ __forceinline__ TTri edges(const float4& a, const float4& b, const float4& c) {
    return TTri{a, make_float4(b.x - a.x, b.y - a.y, b.z - a.z, 0.f), make_float4(c.x - a.x, c.y - a.y, c.z - a.z, 0.f)};
}
__device__ __forceinline__ bool wide_tri_hit(const float4& a, const float4& b, const float4& c, v3 o, v3 d, float& t,
                                             float& u, float& v) {
    return tri_hit(edges(a, b, c), o, d, t, u, v);
}
__device__ __forceinline__ float det_of(const TTri& tr, v3 d) {
    return dot3(mk3(tr.b.x, tr.b.y, tr.b.z), cross3(d, mk3(tr.c.x, tr.c.y, tr.c.z)));
}
__device__ __forceinline__ float size_of(v3 v) { return fabsf(v.x) + fabsf(v.y) + fabsf(v.z); }
__device__ __forceinline__ float sizes_of(const TTri& tr) {
    return size_of(mk3(tr.b.x, tr.b.y, tr.b.z)) * size_of(mk3(tr.c.x, tr.c.y, tr.c.z));
}
// Whether a triangle's determinant is too small to trust its t. An exact 0 is
// never a hit, but where it is the sum of terms that are not, the triangle lies
// in the ray's plane, and others of the same floor may round to something.
__device__ __forceinline__ bool thin_test(const float4& a, const float4& b, const float4& c, v3 d, float scale) {
    const TTri tr = edges(a, b, c);
    const float det = det_of(tr, d);
    const float m1 = fmx(fabsf(tr.b.x), fmx(fabsf(tr.b.y), fabsf(tr.b.z)));
    const float m2 = fmx(fabsf(tr.c.x), fmx(fabsf(tr.c.y), fabsf(tr.c.z)));
    if (det != 0.f) return fabsf(det) < fmx(m1 * m2 * (scale * kThinTest), kTiny);
    const v3 p = cross3(d, mk3(tr.c.x, tr.c.y, tr.c.z));
    return tr.b.x * p.x != 0.f || tr.b.y * p.y != 0.f;  // (the third term then is not 0 either)
}
// The same for a hit at t, its numerator looked at too: whether t is off by
// more than a good part of `past`, the distance beyond it that boxes are visited to.
__device__ __forceinline__ bool thin_hit(const float4& a, const float4& b, const float4& c, v3 o, v3 d, float t,
                                         float past) {
    const TTri tr = edges(a, b, c);
    const float num = fabsf(det_of(tr, d)) * past;
    const float err = sizes_of(tr) * (size_of(d) * t + size_of(sub3(o, mk3(a.x, a.y, a.z)))) * kThinHit;
    return !(err <= num) || num < kTiny;
}
// 1 / r.scale, the distance in true units of one in scaled ones
__device__ __forceinline__ float unscale(const WideRay& r) {
    return __uint_as_float((254u - (__float_as_uint(r.scale) >> 23)) << 23);
}

// A wave's next rays for the lanes that need one (wave-uniform control flow).
// The first seven eighths of a batch are dealt out beforehand, 64 rays to a
// wave in turn: with a counter alone, a batch of short rays waits for it (one
// atomic costs 5 ns there; Cornell path 8.3 ms with all but a wave's first 64
// from the counter, 7.3 now; 2M camera rays 0.78 and 0.56). The rest comes from the counter, two chunks
// a wave or more (`most` rays at most), so that waves with short rays end up
// tracing more.
struct Dispenser {
    int64_t base, stride, first, chunk;  // first: rays dealt out without the counter
    int avail, turns;                    // turns: of the wave's own 64 rays, still to come
    __device__ __forceinline__ Dispenser(int64_t nrays, int most) {
        const int64_t per = blockDim.x >> 6;
        stride = (int64_t)gridDim.x * per * 64;
        base = ((int64_t)blockIdx.x * per + (threadIdx.x >> 6)) * 64;
        avail = 64;
        const int64_t own = nrays * 7 / 8 / stride;
        turns = own > 1 ? (int)own - 1 : 0;
        first = stride * (turns + 1);
        const int64_t c = (nrays - first) / (stride / 64 * 2) / 64 * 64;
        chunk = c < 64 ? 64 : (c < most ? c : most);
    }
    __device__ __forceinline__ int64_t next(uint64_t need, int lane, unsigned long long* counter) {
        const int cnt = __popcll(need), rank = __popcll(need & ((1ull << lane) - 1ull));
        int64_t mine;
        if (avail < cnt) {
            int64_t nb;
            int got = 64;
            if (turns > 0) {
                --turns;
                // (base has moved on by 64 - avail within this turn)
                nb = base - (64 - avail) + stride;
            } else {
                unsigned long long taken = 0;
                const int who = __ffsll((long long)need) - 1;
                if (lane == who) taken = atomicAdd(counter, (unsigned long long)chunk);
                nb = (int64_t)__shfl(taken, who, 64) + first;
                got = (int)chunk;
            }
            mine = rank < avail ? base + rank : nb + (rank - avail);
            base = nb + (cnt - avail);
            avail = got - (cnt - avail);
        } else {
            mine = base + rank;
            base += cnt;
            avail -= cnt;
        }
        return mine;
    }
    // every ray has been dealt out
    __device__ __forceinline__ bool drained(const unsigned long long* counter, int64_t nrays) const {
        return (int64_t)__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + first >= nrays;
    }
};

// Stack of a lane: entry {first inner child, mask of inner slots << 8 |
// remaining children's bits}; the first kWideStack in LDS, the rest (skewed
// trees only) in scratch.
template <int B>
struct WideStackLds {
    uint32_t base[kWideStack][B];
    uint16_t bits[kWideStack][B];
};

// A lane of the trace counts in one register (a second one cost camera rays
// 1%): records, and triangles from bit kTriShift. Counts that come near their
// fields' ends are added between rays.
constexpr int kTriShift = 17;
constexpr uint32_t kFetchesFull = 1u << 31 | 1u << (kTriShift - 1);
__device__ __forceinline__ uint64_t packed_fetches(uint32_t n) {  // triangles << 32 | records
    return (uint64_t)(n >> kTriShift) << 32 | (n & ((1u << kTriShift) - 1u));
}
__device__ __forceinline__ void add_fetches_lane(unsigned long long* fetched, uint64_t n) {
    atomicAdd(fetched, (unsigned long long)(uint32_t)n);
    atomicAdd(fetched + kFetchTris, (unsigned long long)(n >> 32));
}
// A wave's counts into the launch's words (fetch_word).
__device__ __forceinline__ void add_fetches(unsigned long long* fetched, uint64_t n) {
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) n += __shfl_xor(n, dd, 64);
    if ((threadIdx.x & 63) == 0 && n > 0) add_fetches_lane(fetched, n);
}

struct WideList {           // rays left to the finishing pass
    uint32_t* ids = nullptr;
    uint32_t* n = nullptr;  // rays listed (past cap: the rest are marked in the hit ids)
    uint32_t cap = 0;
    int after = 0;          // steps before a ray still in flight at the batch's end is listed (0: never)
    uint32_t mark = 0;      // whole_mark
};
// The bit of a closest-hit ray's id that says it has to be taken over its
// whole line, where ids leave one for it (0: the pass finds out by itself).
inline uint32_t whole_mark(int64_t nrays) { return nrays <= (int64_t(1) << 31) ? 1u << 31 : 0u; }

// kAny: any-hit (limit, src, dst, ovis) instead of closest-hit (oprim ...).
template <bool kAny, int B>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(6))) void k_wide_trace(const uint4* __restrict__ nodes, const float4* __restrict__ tris,
                                                  const float* __restrict__ rays, int64_t nrays_arg,
                                                  const uint32_t* __restrict__ nrays_dev,
                                                  int32_t* __restrict__ oprim, float* __restrict__ ot,
                                                  float* __restrict__ ou, float* __restrict__ ov,
                                                  const float* __restrict__ limit, const int32_t* __restrict__ src,
                                                  const int32_t* __restrict__ dst, uint8_t* __restrict__ ovis,
                                                  uint32_t* __restrict__ overflow,
                                                  unsigned long long* __restrict__ next_ray,
                                                  unsigned long long* __restrict__ fetched, WideList wl,
                                                  float farthest, float rcp_max, float slack, int most) {
    __shared__ WideStackLds<B> lds;
    const int lane = threadIdx.x & 63;
    const int64_t nrays = nrays_dev ? (int64_t)*nrays_dev : nrays_arg;

    int64_t ri = -1;  // ray held by this lane; -1 = needs one, -2 = none left
    WideRay r;
    r.o = r.inv = mk3(0, 0, 0);
    r.scale = 1.f;
    r.oct = r.nx = r.ny = r.nz = 0;
    v3 d = mk3(0, 0, 0);
    float best = FLT_MAX, rival = FLT_MAX, bu = 0.f, bv = 0.f, cut = 0.f;  // rival: the second nearest hit
    int bt = -1, sm = -1, dm = -1, steps = 0;  // bt: the nearest hit's triangle record
    bool odd = false, over = false, may_list = false, drained = false;  // over: traversed, result still to be written
    bool thin = false;  // has tested a triangle whose t is not to be trusted
    uint32_t cbase = 0, group = 0;  // the current node's inner children: first one, slot mask << 8 | bits to visit
    uint32_t tbase = 0, tbits = 0;  // triangles to test
    int sp = 0, maxsp = 0;
    uint32_t deep[2 * (kWideDeep - kWideStack)];
    uint32_t nfetch = 0;  // records fetched, triangles among them << kTriShift
    Dispenser disp(nrays, most);

    while (true) {
        const uint64_t idle = __ballot(ri == -1 || over);
        if (idle && (__popcll(idle) >= kRefill || !__ballot(ri >= 0 && !over))) {
            if (over) {
                bool ask = odd, whole = false;  // the finishing pass has to decide; over the whole line
                int prim = -1;
                if (bt >= 0) {
                    const float4* tp = tris + (int64_t)bt * 3;
                    const float4 a = tp[0], b = tp[1], c = tp[2];
                    prim = __float_as_int(a.w);
                    bool touch;
                    const float e = leaf_entry(a, b, c, r.o, d, touch);
                    ask = ask || touch || !(e >= 0.f);
                    if (!kAny) {
                        const float near = slack * unscale(r);
                        whole = thin || thin_hit(a, b, c, r.o, d, best, best * (kReach - 1.f) + near);
                        ask = ask || whole || rival <= fmx(best, e) || e > best * kOwnBox + 0.5f * near ||
                              !(best < FLT_MAX);
                    }
                }
                if (kAny) {
                    ovis[ri] = prim >= 0 ? 0 : 1;
                } else {
                    oprim[ri] = prim;
                    ot[ri] = prim >= 0 ? best : 0.f;
                    if (ou) ou[ri] = bu;
                    if (ov) ov[ri] = bv;
                }
                if (ask) {
                    const uint32_t slot = atomicAdd(wl.n, 1u);
                    if (slot < wl.cap) wl.ids[slot] = (uint32_t)ri | (whole ? wl.mark : 0u);
                    else if (kAny) ovis[ri] = 255;
                    else oprim[ri] = kUndecided;
                }
                if (nfetch & kFetchesFull) {
                    add_fetches_lane(fetched, packed_fetches(nfetch));
                    nfetch = 0;
                }
                over = false;
                ri = -1;
            }
            const uint64_t need = __ballot(ri == -1);
            if (need) {
                const int64_t mine = disp.next(need, lane, next_ray);
                if (ri == -1) {
                    ri = mine < nrays ? mine : -2;
                    if (ri >= 0) {
                        v3 o;
                        load_ray(rays, ri, o, d);
                        const RayKind kind = wide_ray(o, d, farthest, rcp_max, r);
                        best = rival = FLT_MAX; bt = -1; bu = 0.f; bv = 0.f;
                        odd = kind == kRayOdd;
                        thin = false;
                        may_list = wl.after > 0;
                        steps = 0; sp = 0; tbits = 0;
                        cbase = 0;
                        group = (1u << 8) | (1u << r.oct);  // the root, as slot 0 of a node of one child
                        cut = FLT_MAX;
                        if (kAny) {
                            best = limit[ri];
                            const bool use = !(best == INFINITY);
                            if (use) cut = __builtin_fmaf(best * r.scale, kReach, slack);
                            if (use && !(best > 0.f)) group = 0;  // nothing lies before it
                            sm = src ? src[ri] : -1;
                            dm = dst ? dst[ri] : -1;
                        }
                        if (kind != kRayFine) group = 0;
                    }
                }
            }
        }
        if (!__ballot(ri >= 0)) break;  // every lane is out of rays
        if (ri < 0 || over) continue;

        bool done = false, listed = false;
        if (may_list && steps >= wl.after) {
            if (!drained && ((steps - wl.after) & 255) == 0)
                drained = disp.drained(next_ray, nrays);
            if (drained) {  // a long ray at the end: a whole wave finishes it
                const uint32_t slot = atomicAdd(wl.n, 1u);
                if (slot < wl.cap) {
                    wl.ids[slot] = (uint32_t)ri;
                    done = listed = true;
                }
                may_list = false;
            }
        }
        ++steps;

        if (!done && tbits == 0) {
            if ((group & 255u) == 0u) {
                if (sp == 0) {
                    done = true;
                } else {
                    --sp;
                    if (sp < kWideStack) {
                        cbase = lds.base[sp][threadIdx.x];
                        group = lds.bits[sp][threadIdx.x];
                    } else {
                        cbase = deep[2 * (sp - kWideStack)];
                        group = deep[2 * (sp - kWideStack) + 1];
                    }
                }
            }
            if (!done) {
                const int bit = __ffs((int)(group & 255u)) - 1;
                group &= group - 1u;
                const uint32_t slot = (uint32_t)bit ^ r.oct;
                const uint32_t child = cbase + (uint32_t)__popc((group >> 8) & ((1u << slot) - 1u));
                if (group & 255u) {
                    if (sp < kWideStack) {
                        lds.base[sp][threadIdx.x] = cbase;
                        lds.bits[sp][threadIdx.x] = (uint16_t)group;
                    } else {
                        deep[2 * (sp - kWideStack)] = cbase;
                        deep[2 * (sp - kWideStack) + 1] = group;
                    }
                    ++sp;
                    maxsp = max(maxsp, sp);
                }
                const uint4* nd = nodes + (int64_t)child * kWideWords;
                const uint4 w0 = nd[0], w1 = nd[1], w2 = nd[2], w3 = nd[3], w4 = nd[4];
                ++nfetch;
                const uint32_t mask = test_children(w0, w1, w2, w3, w4, r, cut);
                cbase = w1.x;
                tbase = w1.y;
                tbits = mask & 0xffffffu;
                group = ((w0.w >> 24) << 8) | (mask >> 24);
            }
        }
        if (!done && tbits != 0) {
            const uint32_t k = (uint32_t)__ffs((int)tbits) - 1u;
            tbits &= tbits - 1u;
            const float4* tp = tris + (int64_t)(tbase + k) * 3;
            const float4 a = tp[0], b = tp[1], c = tp[2];
            nfetch += 1u + (1u << kTriShift);
            float t, u, v;
            if (kAny) {
                const int mesh = __float_as_int(b.w);
                if (mesh != sm && mesh != dm && wide_tri_hit(a, b, c, r.o, d, t, u, v) &&
                    (best == INFINITY || t < best)) {
                    bt = (int)(tbase + k);
                    done = true;
                }
            } else {
                thin = thin || thin_test(a, b, c, d, r.scale);
                if (wide_tri_hit(a, b, c, r.o, d, t, u, v)) {
                    rival = fmn(rival, fmx(t, best));
                    if (bt < 0 || t < best) {  // (the first hit counts at any distance, infinity included)
                        best = t; bu = u; bv = v; bt = (int)(tbase + k);
                        cut = __builtin_fmaf(t * r.scale, kReach, slack);
                    }
                }
            }
        }
        if (done) {
            if (listed) ri = -1;
            else over = true;
        }
    }
    // (an atomic per workgroup and word: they serialise, 5 ns each, and a wave's
    // made each launch of the Cornell box 20 us longer)
    __shared__ uint64_t wfetch[B / 64];
    __shared__ int wdeep[B / 64];
    uint64_t fetches = packed_fetches(nfetch);
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) {
        maxsp = max(maxsp, __shfl_xor(maxsp, dd, 64));
        fetches += __shfl_xor(fetches, dd, 64);
    }
    if (lane == 0) {
        wfetch[threadIdx.x >> 6] = fetches;
        wdeep[threadIdx.x >> 6] = maxsp;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < B / 64; ++w) {
            fetches += wfetch[w];
            maxsp = max(maxsp, wdeep[w]);
        }
        if (maxsp > 0) atomicMax(overflow + 6, (uint32_t)maxsp);
        if (fetches > 0) add_fetches_lane(fetched, fetches);
    }
}

// ------------------------------------------------------------- finishing pass
// One wave per listed ray, from the wide tree's root: pending nodes in LDS,
// eight at a time, one child per lane. Closest-hit collects every hit within
// reach of the nearest (64 at most) and, when several lie close enough for
// the reference's order to decide, replays that order; any-hit stops at the
// first blocker. A closest-hit ray that meets a thin triangle is left to the
// whole workgroup, which collects every hit on its line. A ray that does not
// fit goes through the reference's tree on one lane of the wave.
//
// Few rays go over their whole line (5 of 2M camera rays, 86 of 1M random
// ones), but one holds up the launch: by one wave it took 130 us in an
// interior and 190 in a soup of 0.5M triangles, a microsecond for each eight
// nodes. By a workgroup's eight waves, and without the wave's own attempt
// where the trace already knows (WideList::mark), 39 and 36.
constexpr int kPend = 1024;
constexpr int kCands = 64;
constexpr int kFinishWaves = 8;       // closest-hit: waves of a workgroup
constexpr int kFinishTurn = 16;       // rays a wave takes before the workgroup's whole lines
constexpr int kWholePend = 4096, kWholeCands = 512;
constexpr int kRefStack = 64;  // BVH/BVH.h:41,122

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Where a leaf comes in the reference's depth-first traversal of a ray: its
// path from the root, bit 63 first, 1 where it goes to the child taken second
// (the farther one, the right one on ties; BVH/BVH.h:83-94). The leaf earlier
// in that order has the smaller path, and two paths part at their leaves'
// lowest common ancestor. reach: the ray hits every box on the path below the
// root's. The tree has at most 64 levels; false: the walk did not end (never
// for a valid tree).
__device__ bool leaf_path(const WideDev& w, int leaf, v3 o, v3 inv, uint64_t& path, int& depth, bool& reach) {
    path = 0;
    depth = 0;
    reach = true;
    for (int x = leaf; x != 0;) {
        if (depth >= kRefStack) return false;
        const int p = w.topo[x].z;
        const int4 t = w.topo[p];
        const NodeBox l = w.nbox[t.x], r = w.nbox[t.y];
        const float dl = slab(l.a.x, l.a.y, l.a.z, l.b.x, l.b.y, l.b.z, o, inv);
        const float dr = slab(r.a.x, r.a.y, r.a.z, r.b.x, r.b.y, r.b.z, o, inv);
        reach = reach && (t.x == x ? dl : dr) >= 0.f;
        const bool second = (dl > dr) == (t.x == x);
        path = (path >> 1) | (second ? 1ull << 63 : 0ull);
        x = p;
        ++depth;
    }
    return true;
}

// Whether the ray hits every box above a triangle's leaf (but the root's).
__device__ bool reached(const WideDev& w, int prim, v3 o, v3 d, bool& bad) {
    uint64_t path;
    int depth;
    bool reach;
    if (!leaf_path(w, w.leaf_of[prim], o, div3(mk3(1.f, 1.f, 1.f), d), path, depth, reach)) bad = true;
    return reach;
}

// The reference's traversal of one ray by one lane (k_trace / k_trace_any).
__device__ void reference_closest(const TRec* recs, const float* root, v3 o, v3 d, int max_steps, int* stack,
                                  int& prim, float& t, float& u, float& v, uint32_t& ovf) {
    const v3 inv = div3(mk3(1.f, 1.f, 1.f), d);
    float best = FLT_MAX, bu = 0.f, bv = 0.f;
    bool hit = false;
    int bp = -1, cur = 0, sp = 0;
    prim = -1; t = u = v = 0.f;
    if (slab(root[0], root[1], root[2], root[3], root[4], root[5], o, inv) < 0.f) return;
    for (int steps = 0;; ++steps) {
        if (steps >= max_steps) { ++ovf; break; }
        const float4* rec = reinterpret_cast<const float4*>(recs + (cur >= 0 ? cur : ~cur));
        const float4 q0 = rec[0], q1 = rec[1], q2 = rec[2];
        bool next = false;
        if (cur >= 0) {
            const int4 refs = reinterpret_cast<const int4*>(rec)[3];
            const float dl = slab(q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, o, inv);
            const float dr = slab(q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, o, inv);
            const bool hl = dl >= 0 && dl < best, hr = dr >= 0 && dr < best;
            if (hl && hr) {
                const bool lfar = dl > dr;
                if (sp < kRefStack) stack[sp++] = lfar ? refs.x : refs.y; else ++ovf;
                if (sp < kRefStack) { cur = lfar ? refs.y : refs.x; next = true; } else ++ovf;
            } else if (hl || hr) {
                if (sp < kRefStack) { cur = hl ? refs.x : refs.y; next = true; } else ++ovf;
            }
        } else {
            float ht, hu, hv;
            if (tri_hit(TTri{q0, q1, q2}, o, d, ht, hu, hv) && (!hit || ht < best)) {
                hit = true; best = ht; bu = hu; bv = hv; bp = __float_as_int(q0.w);
            }
        }
        if (!next) {
            if (sp == 0) break;
            cur = stack[--sp];
        }
    }
    if (hit) { prim = bp; t = best; u = bu; v = bv; }
}
__device__ bool reference_blocked(const TRec* recs, v3 o, v3 d, float lim, int sm, int dm, int max_steps, int* stack,
                                  uint32_t& ovf) {
    const v3 inv = div3(mk3(1.f, 1.f, 1.f), d);
    const bool use = !(lim == INFINITY);
    int cur = 0, sp = 0;
    for (int steps = 0;; ++steps) {
        if (steps >= max_steps) { ++ovf; return false; }
        const float4* rec = reinterpret_cast<const float4*>(recs + (cur >= 0 ? cur : ~cur));
        const float4 q0 = rec[0], q1 = rec[1], q2 = rec[2];
        bool next = false;
        if (cur >= 0) {
            const int4 refs = reinterpret_cast<const int4*>(rec)[3];
            const float dl = slab(q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, o, inv);
            const float dr = slab(q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, o, inv);
            const bool hl = dl >= 0, hr = dr >= 0;
            if (hl && hr) {
                const bool lfar = dl > dr;
                if (sp < kRefStack) stack[sp++] = lfar ? refs.x : refs.y; else ++ovf;
                if (sp < kRefStack) { cur = lfar ? refs.y : refs.x; next = true; } else ++ovf;
            } else if (hl || hr) {
                if (sp < kRefStack) { cur = hl ? refs.x : refs.y; next = true; } else ++ovf;
            }
        } else {
            const int mesh = __float_as_int(q1.w);
            float t, u, v;
            if (mesh != sm && mesh != dm && tri_hit(TTri{q0, q1, q2}, o, d, t, u, v) && (!use || t < lim)) return true;
        }
        if (!next) {
            if (sp == 0) return false;
            cur = stack[--sp];
        }
    }
}

struct FinishLds {
    uint32_t pend[kPend];
    float t[kCands], u[kCands], v[kCands], e[kCands];
    int32_t p[kCands];
    int stack[kRefStack];
};
struct WholeLds {
    uint32_t pend[kWholePend];
    float t[kWholeCands], u[kWholeCands], v[kWholeCands], e[kWholeCands];
    int32_t p[kWholeCands];
    int stack[kRefStack];
    uint32_t npend, ncands, bad, endless;
};

// A lane's child of a pending node: its wide box against the ray. Returns the
// slot byte's meaning: inner child index (inner set) or first triangle and
// count; count 0 and !inner: nothing hit.
__device__ __forceinline__ void lane_child(const uint4* nd, int slot, const WideRay& r, float cut, bool& inner,
                                           uint32_t& at, int& count) {
    const uint4 w0 = nd[0], w1 = nd[1];
    const uint8_t* by = reinterpret_cast<const uint8_t*>(nd);
    const uint32_t m = by[24 + slot];
    uint32_t plane[6];  // (all loads before the first branch)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        plane[2 * k] = by[wide_plane(k, slot)];
        plane[2 * k + 1] = by[wide_plane(k, slot) + 2];
    }
    inner = false;
    at = 0;
    count = 0;
    if (m == 0u) return;
    float tn = 0.f, tf = cut;
    const float org[3] = {__uint_as_float(w0.x), __uint_as_float(w0.y), __uint_as_float(w0.z)};
    const float ro[3] = {r.o.x, r.o.y, r.o.z}, ri[3] = {r.inv.x, r.inv.y, r.inv.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const AxisPlanes ap = axis_planes(org[k], (w0.w >> (8 * k)) & 255u, ro[k], ri[k]);
        constexpr float kByte = 1.f / (float)(1 << kPlaneBits);
        const float lo = (float)plane[2 * k] * kByte, hi = (float)plane[2 * k + 1] * kByte;
        tn = fmx(tn, __builtin_fmaf(ri[k] < 0.f ? hi : lo, ap.an, ap.bn));
        tf = fmn(tf, __builtin_fmaf(ri[k] < 0.f ? lo : hi, ap.af, ap.bf));
    }
    if (!(tn <= tf)) return;
    const uint32_t imask = w0.w >> 24;
    if ((imask >> slot) & 1u) {
        inner = true;
        at = w1.x + (uint32_t)__popc(imask & ((1u << slot) - 1u));
    } else {
        at = w1.y + (m & 31u);
        count = __popc(m >> 5);
    }
}

struct FinishArgs {
    WideDev w;
    const TRec* recs;
    const float* root;
    const float* rays;
    int64_t nrays;
    const uint32_t* nrays_dev;
    const uint32_t* ids;
    const uint32_t* n;
    uint32_t cap;
    uint32_t* fails;  // rays that took the reference's traversal
    uint32_t* overflow;
    unsigned long long* fetched;
    int ntris;
    uint32_t mark;
};

// Which of the hits of a wave's lanes (rival, two or more) the reference's
// traversal ends with: its order among them, one lane each. A hit is skipped
// when its path, below the box that was pending before an earlier hit was
// met, starts at or beyond that hit. -1: a walk up the tree did not end.
__device__ int replay(const WideDev& w, v3 o, v3 d, bool rival, float ct, float ce, int prim) {
    const int lane = threadIdx.x & 63;
    const v3 inv = div3(mk3(1.f, 1.f, 1.f), d);
    uint64_t path = ~0ull;
    int depth = 0;
    bool reach;
    const bool ok = !rival || leaf_path(w, w.leaf_of[prim], o, inv, path, depth, reach);
    if (__ballot(!ok)) return -1;
    float near = FLT_MAX;
    bool visited = false;
    int win = -1;
    for (uint64_t left = __ballot(rival); left != 0ull;) {
        uint64_t first = (left >> lane) & 1ull ? path : ~0ull;
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) {
            const uint64_t other = (uint64_t)__shfl_xor((unsigned long long)first, dd, 64);
            first = other < first ? other : first;
        }
        const uint64_t at = __ballot(((left >> lane) & 1ull) && path == first);
        const int c = __ffsll((long long)at) - 1;
        left &= ~(1ull << c);
        const float ec = __shfl(ce, c, 64), tc = __shfl(ct, c, 64);
        const int dc = __shfl(depth, c, 64);
        const bool skips = visited && ec >= ct && dc > __clzll((long long)(path ^ first)) + 1;
        if (__ballot(skips)) continue;
        if (lane == c) visited = true;
        if (tc < near) {
            near = tc;
            win = c;
        }
    }
    return win;
}
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) v = fmn(v, __shfl_xor(v, dd, 64));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) v = fmx(v, __shfl_xor(v, dd, 64));
    return v;
}

struct ClosestOut {
    int32_t* prim;
    float *t, *u, *v;
};
__device__ void write_hit(const ClosestOut& out, int64_t ri, int prim, float t, float u, float v) {
    out.prim[ri] = prim;
    out.t[ri] = t;
    if (out.u) out.u[ri] = u;
    if (out.v) out.v[ri] = v;
}
// One lane: the ray over the reference's tree.
__device__ void reference_ray(const FinishArgs& A, int64_t ri, v3 o, v3 d, int* stack, const ClosestOut& out) {
    uint32_t ovf = 0;
    int prim;
    float t, u, v;
    reference_closest(A.recs, A.root, o, d, 2 * A.ntris - 1, stack, prim, t, u, v, ovf);
    if (ovf) atomicAdd(A.overflow, ovf);
    atomicAdd(A.fails, 1u);
    write_hit(out, ri, prim, t, u, v);
}
__device__ __forceinline__ bool root_hit(const FinishArgs& A, v3 o, v3 d) {
    return slab(A.root[0], A.root[1], A.root[2], A.root[3], A.root[4], A.root[5], o, div3(mk3(1.f, 1.f, 1.f), d)) >= 0.f;
}

// A ray by a wave. false: it has to be taken over its whole line.
__device__ bool finish_closest(const FinishArgs& A, int64_t ri, FinishLds& L, const ClosestOut& out, uint64_t& nfetch) {
    const int lane = threadIdx.x & 63;
    v3 o, d;
    load_ray(A.rays, ri, o, d);
    WideRay r;
    const RayKind kind = wide_ray(o, d, A.w.far_origin, A.w.rcp_max, r);
    bool failed = kind == kRayOdd;
    bool bad = false;      // a walk up the reference's tree did not end
    bool endless = false;  // a hit at a distance that overflowed (counts where there is no other)
    bool thin = false;
    const bool in_root = root_hit(A, o, d);
    const float near = A.w.near_slack * unscale(r);
    float best = FLT_MAX;
    int count = kind == kRayFine ? 1 : 0, nc = 0;
    if (lane == 0) L.pend[0] = 0u;
    wave_fence();
    while (count > 0) {
        const int k = count < 8 ? count : 8;
        const int g = lane >> 3;
        bool inner = false;
        uint32_t at = 0;
        int nt = 0;
        if (g < k) {
            const uint32_t node = L.pend[count - 1 - g];
            const float cut = best == FLT_MAX ? FLT_MAX : __builtin_fmaf(best * r.scale, kReach, A.w.near_slack);
            lane_child(A.w.nodes + (int64_t)node * kWideWords, lane & 7, r, cut, inner, at, nt);
            nfetch += (lane & 7) == 0 ? 1u : 0u;
        }
        count -= k;
        wave_fence();
        for (int j = 0; j < kWideLeaf; ++j) {
            float t = 0.f, u = 0.f, v = 0.f, e = -1.f;
            int p = -1;
            bool hit = false;
            if (j < nt) {
                const float4* tp = A.w.tris + (int64_t)(at + (uint32_t)j) * 3;
                const float4 a = tp[0], b = tp[1], c = tp[2];
                nfetch += (1ull << 32) + 1u;
                thin = thin || thin_test(a, b, c, d, r.scale);
                if (wide_tri_hit(a, b, c, o, d, t, u, v)) {
                    thin = thin || thin_hit(a, b, c, o, d, t, t * (kReach - 1.f) + near);
                    bool touch;
                    e = leaf_entry(a, b, c, o, d, touch);
                    hit = e >= 0.f && e < FLT_MAX;
                    p = __float_as_int(a.w);
                    if (hit && touch) hit = in_root && reached(A.w, p, o, d, bad);
                    endless = endless || (hit && !(t < FLT_MAX));
                    hit = hit && t < FLT_MAX;
                }
            }
            best = fmn(best, wave_min(hit ? t : FLT_MAX));
            const bool add = hit && t <= best * kReach + near;
            const uint64_t am = __ballot(add);
            if (am == 0ull) continue;
            const int na = __popcll(am);
            const uint64_t lt = (1ull << lane) - 1ull;
            if (nc + na > kCands) {  // keep those still near the nearest
                const float ct = L.t[lane], cu = L.u[lane], cv = L.v[lane], ce = L.e[lane];
                const int cp = L.p[lane];
                const bool keep = lane < nc && ct <= best * kReach + near;
                const uint64_t km = __ballot(keep);
                wave_fence();
                if (keep) {
                    const int i = __popcll(km & lt);
                    L.t[i] = ct; L.u[i] = cu; L.v[i] = cv; L.e[i] = ce; L.p[i] = cp;
                }
                nc = __popcll(km);
                wave_fence();
            }
            if (nc + na > kCands) {
                failed = true;
            } else {
                if (add) {
                    const int i = nc + __popcll(am & lt);
                    L.t[i] = t; L.u[i] = u; L.v[i] = v; L.e[i] = e; L.p[i] = p;
                }
                nc += na;
            }
        }
        const uint64_t im = __ballot(inner);
        const int ni = __popcll(im);
        if (count + ni > kPend) failed = true;
        if (failed || __ballot(thin)) break;
        if (inner) L.pend[count + __popcll(im & ((1ull << lane) - 1ull))] = at;
        count += ni;
        wave_fence();
    }
    wave_fence();
    if (!failed && __ballot(thin)) return false;
    if (__ballot(bad) || (nc == 0 && __ballot(endless))) failed = true;
    int win = -1;
    if (!failed && nc > 0) {
        // the hits whose order could matter: at or before the farthest of
        // their own boxes' starts
        const float ct = lane < nc ? L.t[lane] : FLT_MAX, ce = lane < nc ? L.e[lane] : 0.f;
        float bound = best;
        for (bool grew = true; grew;) {
            const float m = wave_max(ct <= bound ? fmx(ct, ce) : 0.f);
            grew = m > bound;
            if (grew) bound = m;
        }
        if (bound > best * kOwnBox + 0.5f * near) return false;
        const bool rival = ct <= bound;
        const uint64_t rm = __ballot(rival);
        win = __popcll(rm) == 1 ? __ffsll((long long)rm) - 1 : replay(A.w, o, d, rival, ct, ce, rival ? L.p[lane] : 0);
        if (win < 0) failed = true;
    }
    if (lane == 0) {
        if (failed) reference_ray(A, ri, o, d, L.stack, out);
        else if (win >= 0) write_hit(out, ri, L.p[win], L.t[win], L.u[win], L.v[win]);
        else write_hit(out, ri, -1, 0.f, 0.f, 0.f);
    }
    wave_fence();
    return true;
}

// A ray over its whole line by all waves of the workgroup, 64 nodes at a
// time: no box of the line is skipped, so that the answer does not rest on
// where the hits' distances lie.
__device__ void finish_whole(const FinishArgs& A, int64_t ri, WholeLds& W, const ClosestOut& out, uint64_t& nfetch) {
    const int lane = threadIdx.x & 63;
    v3 o, d;
    load_ray(A.rays, ri, o, d);
    WideRay r;
    const RayKind kind = wide_ray(o, d, A.w.far_origin, A.w.rcp_max, r);  // (fine: others are not sent here)
    const bool in_root = root_hit(A, o, d);
    if (threadIdx.x == 0) {
        W.pend[0] = 0u;
        W.npend = kind == kRayFine ? 1u : 0u;
        W.ncands = W.bad = W.endless = 0u;
    }
    __syncthreads();
    while (true) {
        const int count = (int)W.npend;
        if (count == 0 || W.bad != 0u || W.ncands > (uint32_t)kWholeCands) break;  // (alike in all threads)
        const int k = count < 8 * kFinishWaves ? count : 8 * kFinishWaves;
        const int g = (int)(threadIdx.x >> 3);
        const uint32_t node = g < k ? W.pend[count - 1 - g] : 0u;
        __syncthreads();
        if (threadIdx.x == 0) W.npend = (uint32_t)(count - k);
        __syncthreads();
        bool inner = false;
        uint32_t at = 0;
        int nt = 0;
        if (g < k) {
            lane_child(A.w.nodes + (int64_t)node * kWideWords, lane & 7, r, FLT_MAX, inner, at, nt);
            nfetch += (lane & 7) == 0 ? 1u : 0u;
        }
        const uint64_t im = __ballot(inner);
        if (im != 0ull) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(&W.npend, (uint32_t)__popcll(im));
            base = (uint32_t)__shfl((int)base, 0, 64) + (uint32_t)__popcll(im & ((1ull << lane) - 1ull));
            if (inner && base < (uint32_t)kWholePend) W.pend[base] = at;
            if (inner && base >= (uint32_t)kWholePend) W.bad = 1u;
        }
        for (int j = 0; j < nt; ++j) {
            const float4* tp = A.w.tris + (int64_t)(at + (uint32_t)j) * 3;
            const float4 a = tp[0], b = tp[1], c = tp[2];
            nfetch += (1ull << 32) + 1u;
            float t, u, v;
            if (!wide_tri_hit(a, b, c, o, d, t, u, v)) continue;
            bool touch, bad = false;
            const float e = leaf_entry(a, b, c, o, d, touch);
            bool hit = e >= 0.f && e < FLT_MAX;
            const int p = __float_as_int(a.w);
            if (hit && touch) hit = in_root && reached(A.w, p, o, d, bad);
            if (bad) W.bad = 1u;
            if (!hit) continue;
            if (!(t < FLT_MAX)) {
                W.endless = 1u;
                continue;
            }
            const uint32_t i = atomicAdd(&W.ncands, 1u);
            if (i < (uint32_t)kWholeCands) {
                W.t[i] = t; W.u[i] = u; W.v[i] = v; W.e[i] = e; W.p[i] = p;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 64) {
        const int nc = (int)W.ncands;
        bool failed = W.bad != 0u || nc > kWholeCands || (nc == 0 && W.endless != 0u);
        int win = -1;
        if (!failed && nc > 0) {
            // as in finish_closest, and the hits that could matter in its lanes
            float best = FLT_MAX;
            for (int i = lane; i < nc; i += 64) best = fmn(best, W.t[i]);
            best = wave_min(best);
            float bound = best;
            for (bool grew = true; grew;) {
                float m = 0.f;
                for (int i = lane; i < nc; i += 64)
                    if (W.t[i] <= bound) m = fmx(m, fmx(W.t[i], W.e[i]));
                m = wave_max(m);
                grew = m > bound;
                if (grew) bound = m;
            }
            int mine = -1, n = 0;
            for (int b = 0; b < nc && n <= 64; b += 64) {
                uint64_t m = __ballot(b + lane < nc && W.t[b + lane < nc ? b + lane : 0] <= bound);
                for (; m != 0ull; m &= m - 1ull, ++n)
                    if (lane == n) mine = b + __ffsll((long long)m) - 1;
            }
            if (n > 64) {
                failed = true;
            } else {
                const bool rival = mine >= 0;
                const int c = n == 1 ? 0
                                     : replay(A.w, o, d, rival, rival ? W.t[mine] : FLT_MAX, rival ? W.e[mine] : 0.f,
                                              rival ? W.p[mine] : 0);
                if (c < 0) failed = true;
                else win = __shfl(mine, c, 64);
            }
        }
        if (lane == 0) {
            if (failed) reference_ray(A, ri, o, d, W.stack, out);
            else if (win >= 0) write_hit(out, ri, W.p[win], W.t[win], W.u[win], W.v[win]);
            else write_hit(out, ri, -1, 0.f, 0.f, 0.f);
        }
    }
    __syncthreads();
}

__device__ void finish_any(const FinishArgs& A, int64_t ri, FinishLds& L, const float* limit, const int32_t* src,
                           const int32_t* dst, uint8_t* ovis, uint64_t& nfetch) {
    const int lane = threadIdx.x;
    v3 o, d;
    load_ray(A.rays, ri, o, d);
    WideRay r;
    const RayKind kind = wide_ray(o, d, A.w.far_origin, A.w.rcp_max, r);
    bool failed = kind == kRayOdd;
    const float lim = limit[ri];
    const bool use = !(lim == INFINITY);
    const float cut = use ? __builtin_fmaf(lim * r.scale, kReach, A.w.near_slack) : FLT_MAX;
    const int sm = src ? src[ri] : -1, dm = dst ? dst[ri] : -1;
    int count = kind != kRayFine || (use && !(lim > 0.f)) ? 0 : 1;
    bool blocked = false, bad = false;
    if (lane == 0) L.pend[0] = 0u;
    wave_fence();
    while (count > 0) {
        const int k = count < 8 ? count : 8;
        const int g = lane >> 3;
        bool inner = false, hit = false;
        uint32_t at = 0;
        int nt = 0;
        if (g < k) {
            const uint32_t node = L.pend[count - 1 - g];
            lane_child(A.w.nodes + (int64_t)node * kWideWords, lane & 7, r, cut, inner, at, nt);
            nfetch += (lane & 7) == 0 ? 1u : 0u;
        }
        count -= k;
        wave_fence();
        for (int j = 0; j < nt && !hit; ++j) {
            const float4* tp = A.w.tris + (int64_t)(at + (uint32_t)j) * 3;
            const float4 a = tp[0], b = tp[1], c = tp[2];
            nfetch += (1ull << 32) + 1u;
            const int mesh = __float_as_int(b.w);
            float t, u, v;
            if (mesh != sm && mesh != dm && wide_tri_hit(a, b, c, o, d, t, u, v) && (!use || t < lim)) {
                bool touch;
                hit = leaf_entry(a, b, c, o, d, touch) >= 0.f;
                if (hit && touch) hit = reached(A.w, __float_as_int(a.w), o, d, bad);
            }
        }
        if (__ballot(hit)) {
            blocked = true;
            break;
        }
        const uint64_t im = __ballot(inner);
        const int ni = __popcll(im);
        if (count + ni > kPend) {
            failed = true;
            break;
        }
        if (inner) L.pend[count + __popcll(im & ((1ull << lane) - 1ull))] = at;
        count += ni;
        wave_fence();
    }
    wave_fence();
    if (!blocked && __ballot(bad)) failed = true;
    if (lane == 0) {
        if (failed) {
            uint32_t ovf = 0;
            blocked = reference_blocked(A.recs, o, d, lim, sm, dm, 2 * A.ntris - 1, L.stack, ovf);
            if (ovf) atomicAdd(A.overflow, ovf);
            atomicAdd(A.fails, 1u);
        }
        ovis[ri] = blocked ? 0 : 1;
    }
    wave_fence();
}

__global__ __launch_bounds__(64 * kFinishWaves) void k_wide_finish_closest(FinishArgs A, ClosestOut out) {
    union Lds {
        FinishLds wave[kFinishWaves];
        WholeLds whole;
    };
    __shared__ Lds lds;
    __shared__ uint32_t queue[64 * kFinishWaves];  // rays of this turn to take over their whole lines
    __shared__ uint32_t queued;
    const uint32_t all = *A.n;
    const uint32_t total = min(all, A.cap);
    if (blockIdx.x >= total) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint64_t nfetch = 0;  // triangles << 32 | records
    const auto leave = [&](uint32_t ri) {
        if (lane == 0) queue[atomicAdd(&queued, 1u)] = ri;
    };
    const auto take = [&](int64_t ri) {
        if (!finish_closest(A, ri, lds.wave[wave], out, nfetch)) leave((uint32_t)ri);
    };
    const auto wholes = [&]() {  // all threads
        __syncthreads();
        const uint32_t n = queued;
        for (uint32_t i = 0; i < n; ++i) finish_whole(A, queue[i], lds.whole, out, nfetch);
        __syncthreads();
        if (threadIdx.x == 0) queued = 0u;
        __syncthreads();
    };
    if (threadIdx.x == 0) queued = 0u;
    __syncthreads();
    // kFinishTurn rays a wave and turn; the first gridDim.x rays go to as many workgroups
    const int64_t lanes = (int64_t)gridDim.x * kFinishWaves;
    for (int64_t base = 0; base < (int64_t)total; base += lanes * kFinishTurn) {
        for (int j = 0; j < kFinishTurn; ++j) {
            const int64_t i = base + j * lanes + (int64_t)wave * gridDim.x + blockIdx.x;
            if (i >= (int64_t)total) break;
            const uint32_t id = A.ids[i];
            if (id & A.mark) leave(id & ~A.mark);
            else take(id);
        }
        wholes();
    }
    if (all > A.cap) {  // the list ran over: find the marked rays
        const int64_t nrays = A.nrays_dev ? (int64_t)*A.nrays_dev : A.nrays;
        for (int64_t b = (int64_t)blockIdx.x * 64 * kFinishWaves; b < nrays; b += lanes * 64) {
            const int64_t first = b + 64 * wave, i = first + lane;
            for (uint64_t m = __ballot(i < nrays && out.prim[i] == kUndecided); m; m &= m - 1ull)
                take(first + __ffsll((long long)m) - 1);
            wholes();
        }
    }
    add_fetches(A.fetched, nfetch);
}

__global__ __launch_bounds__(64) void k_wide_finish_any(FinishArgs A, const float* limit, const int32_t* src,
                                                        const int32_t* dst, uint8_t* ovis) {
    __shared__ FinishLds L;
    const uint32_t all = *A.n;
    const uint32_t total = min(all, A.cap);
    if (blockIdx.x >= total) return;
    uint64_t nfetch = 0;  // triangles << 32 | records
    for (uint32_t i = blockIdx.x; i < total; i += gridDim.x) finish_any(A, A.ids[i], L, limit, src, dst, ovis, nfetch);
    if (all > A.cap) {  // the list ran over: find the marked rays
        const int64_t nrays = A.nrays_dev ? (int64_t)*A.nrays_dev : A.nrays;
        for (int64_t b = (int64_t)blockIdx.x * 64; b < nrays; b += (int64_t)gridDim.x * 64) {
            const int64_t i = b + threadIdx.x;
            for (uint64_t m = __ballot(i < nrays && ovis[i] == 255); m; m &= m - 1ull)
                finish_any(A, b + __ffsll((long long)m) - 1, L, limit, src, dst, ovis, nfetch);
        }
    }
    add_fetches(A.fetched, nfetch);
}

constexpr int kFinishBlocks = 4096;

template <bool kAny, int B, typename... A>
void launch_wide(const TraceLaunch& L, int64_t nrays, LaunchSink& ls, A... args) {
    static const int per_cu = [] {
        int per = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, reinterpret_cast<const void*>(&k_wide_trace<kAny, B>), B,
                                                         0) != hipSuccess || per <= 0)
            per = 4 * 256 / B;
        return per;
    }();
    // the tree's nodes stay in the caches, so as many waves as fit: the
    // launch shape's workgroups per CU bound the reference's traversals only
    const int64_t need = (nrays + B - 1) / B;
    int64_t blocks = std::min<int64_t>((int64_t)device_cus() * per_cu, need);
    if (blocks < 1) blocks = 1;
    ls.launch(kAny ? "k_wide_trace<any>" : "k_wide_trace<closest>", &k_wide_trace<kAny, B>, dim3((unsigned)blocks),
              dim3(B), args..., L.chunk);
}
template <bool kAny, typename... A>
void launch_wide_block(const TraceLaunch& L, int64_t nrays, LaunchSink& ls, A... args) {
    if (L.block == 64) launch_wide<kAny, 64>(L, nrays, ls, args...);
    else if (L.block == 128) launch_wide<kAny, 128>(L, nrays, ls, args...);
    else launch_wide<kAny, 256>(L, nrays, ls, args...);
}

}  // namespace

// Words 26 (rays listed) and 30 (rays that took the reference's traversal) of
// the counters; the list is the cooperative pass's.
void wide_closest(const TraceBvh& bvh, const float* rays, int64_t nrays, const uint32_t* nrays_dev, int32_t* prim,
                  float* t, float* u, float* v, uint32_t* counters, const TraceLaunch& L, const TraceCoop& coop,
                  LaunchSink& ls) {
    const WideList wl{coop.longs, counters + 26, coop.long_cap, L.handoff, whole_mark(nrays)};
    launch_wide_block<false>(L, nrays, ls, bvh.wide.nodes, bvh.wide.tris, rays, nrays, nrays_dev, prim, t, u, v,
                             (const float*)nullptr, (const int32_t*)nullptr, (const int32_t*)nullptr,
                             (uint8_t*)nullptr, counters, reinterpret_cast<unsigned long long*>(counters + 2),
                             fetch_word(counters, true), wl, bvh.wide.far_origin, bvh.wide.rcp_max, bvh.wide.near_slack);
    const FinishArgs A{bvh.wide, bvh.rec, bvh.root, rays, nrays, nrays_dev, coop.longs, counters + 26,
                       coop.long_cap, counters + 30, counters, fetch_word(counters, true), bvh.ntris, wl.mark};
    const unsigned blocks = (unsigned)std::min<int64_t>(kFinishBlocks / kFinishWaves, nrays);
    ls.launch("k_wide_finish_closest", &k_wide_finish_closest, dim3(blocks), dim3(64 * kFinishWaves), A,
              ClosestOut{prim, t, u, v});
}

// Words 20 and 22 likewise; the list is the failure list behind the spill records.
void wide_occluded(const TraceBvh& bvh, const float* rays, int64_t nrays, const uint32_t* nrays_dev,
                   const float* limit, const int32_t* src, const int32_t* dst, uint8_t* visible, uint32_t* counters,
                   const TraceLaunch& L, const TraceCoop& coop, LaunchSink& ls) {
    uint32_t* ids = reinterpret_cast<uint32_t*>(coop.spill + coop.spill_cap);
    const WideList wl{ids, counters + 20, coop.spill_cap, L.handoff, 0u};
    launch_wide_block<true>(L, nrays, ls, bvh.wide.nodes, bvh.wide.tris, rays, nrays, nrays_dev, (int32_t*)nullptr,
                            (float*)nullptr, (float*)nullptr, (float*)nullptr, limit, src, dst, visible,
                            counters + 1, reinterpret_cast<unsigned long long*>(counters + 4),
                            fetch_word(counters, false), wl, bvh.wide.far_origin, bvh.wide.rcp_max, bvh.wide.near_slack);
    const FinishArgs A{bvh.wide, bvh.rec, bvh.root, rays, nrays, nrays_dev, ids, counters + 20,
                       coop.spill_cap, counters + 22, counters + 1, fetch_word(counters, false), bvh.ntris, 0u};
    const unsigned blocks = (unsigned)std::min<int64_t>(kFinishBlocks, nrays);
    ls.launch("k_wide_finish_any", &k_wide_finish_any, dim3(blocks), dim3(64), A, limit, src, dst, visible);
}

}  // namespace cav
