// The wide traversal tree: an 8-wide tree with 8-bit child boxes over the
// triangles, built beside the reference's BVH and walked by the closest-hit
// and any-hit traces in its place; see wide.hip and wide_trace.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dev_common.h"
#include "lbvh.h"

namespace cav {

// One node, 128 bytes (one L2 line), eight 16-byte words:
//   0: box origin xyz | scale exponents x, y, z (one byte each, biased by 127
//      and by kPlaneBits more) and the mask of slots holding an inner child
//   1: first inner child's node | first triangle | 8 slot bytes (WideSlot)
//   2, 3, 4: x, y, z: planes in units of 2^exponent from the origin, rounded
//      outwards; two slots to a word: low, low, high, high
//   5: build only: {binary node, first leaf, last leaf, 0}
// Inner children lie one after the other in slot order, and so do the
// triangles of the leaf slots.
// A slot's byte: 0 empty; inner 1 << 5 | (24 + slot); leaf of c triangles
// ((1 << c) - 1) << 5 | offset from the first triangle.
constexpr int kWideWords = 8;
constexpr int kPlaneBits = 24;  // a plane's byte as the bits of a half float is 2^-24 times its number
// byte of a slot's low plane of axis k (its high plane: two bytes on)
__host__ __device__ constexpr int wide_plane(int k, int slot) { return 32 + 16 * k + (slot >> 1) * 4 + (slot & 1); }
constexpr int kWideLeaf = 3;  // triangles per leaf slot at most
// nodes for n triangles: a node with inner children has all 8 slots filled,
// one without holds at least 4 triangles (or is the root)
inline int64_t wide_node_capacity(int64_t n) { return 2 * n / 7 + 16; }

// Limits that follow from the largest coordinate of a scene, 2^k at most
// (k from -20 to 40). A ray that hardly moves along an axis has a reciprocal
// there that is cut off at rcp_max, which brings the planes of that axis
// closer than they are. That must not end a box early: a ray that starts
// inside (or on the edge of) an exact box starts at least 2^-14 units inside
// the planes that hold it, or 2^(2k - 81), which rcp_max takes to 2^(k + 23);
// and a ray from within 2^(k + 20) has left the scene along its main axis
// before 2^(k + 21). Sums of two coordinates times rcp_max stay below 2^126.
struct WideScale {
    float far_origin;   // rays from beyond go to the reference's traversal
    float rcp_max;
    float near_slack;   // 2^(k - 16): how far beyond the nearest hit boxes are always visited (scaled directions)
    uint32_t min_unit;  // exponent (biased by 127) of the smallest unit, 2^(2k - 67)
};
__host__ __device__ inline WideScale wide_scale(const float* box6) {
    float m = 0.f;
    for (int i = 0; i < 6; ++i) m = __builtin_fmaxf(m, __builtin_fabsf(box6[i]));
    int k = (int)((__builtin_bit_cast(uint32_t, m) + 0x7fffffu) >> 23) - 127;
    k = k < -20 ? -20 : (k > 40 ? 40 : k);
    const auto pow2 = [](int e) { return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23); };
    const int e = 60 + 2 * k;
    return WideScale{pow2(k + 20), pow2(104 - k), pow2(k - 16), (uint32_t)(e < 40 ? 40 : e)};
}

// Where a build keeps its codes and its binary tree (112 bytes a triangle).
// Up to this many triangles in memory of their own: the traversal records are
// then written before the wide tree, which the first traces find in the
// caches (1M triangles, 131K rays: 1.36 ms a frame, 1.39 the other way
// round). Above, where neither stays cached, in the place of those records,
// which are written last.
constexpr int kWideApart = 1 << 21;

// The tree (library-owned, sized for n triangles): 89 bytes a triangle.
struct WideBuffers {
    void* base = nullptr;        // the one allocation that holds the rest
    void* scratch = nullptr;     // wide_scratch_bytes(n), part of it (null above kWideApart)
    uint32_t* ctr = nullptr;     // kWideCtrWords
    uint32_t* bounds = nullptr;  // 6 order-preserving ints: the triangles' box
    uint4* nodes = nullptr;
    float4* tris = nullptr;
    int32_t* leaf_of = nullptr;
};
constexpr int kWideCtrWords = 96;
size_t wide_bytes(int n);
void wide_carve(WideBuffers& w, void* base, int n);
// Builds the tree. bounds: the triangles' box (b.scene_ord when the caller
// gave none, else w.bounds). Uses b's sort work space, gates and level list
// and wide_scratch_bytes(n) at `scratch` on the same stream as b's own build
// and after it.
size_t wide_scratch_bytes(int n);
hipError_t wide_build(WideBuffers& w, LbvhBuffers& b, void* scratch, const float* tris, const int32_t* mesh, int n,
                      const uint32_t* bounds, hipStream_t s, Marker* mk);

}  // namespace cav
