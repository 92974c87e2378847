// Aila-Karras 7-leaf treelet restructuring, one treelet per 32-lane group.
//
// Reference: optimizeTreelet / optimizeBVHImpl / optimizeBVH
// (BVH/Optimization.cu:49-525). The reference runs one 32-lane warp per
// treelet; here each wave64 carries two independent 32-lane groups, and every
// cross-lane step uses 32-wide shuffles so the decisions follow the reference
// lane for lane: formation by largest surface area (lowest lane on ties), the
// scheduled partition enumeration for subsets of 2..5 leaves, the
// min(l+d,31) shuffle-reduction tree for 6 and 7 leaves, and reconstruction
// that hands the two halves of the first proposing lane to the next two lanes.
//
// Race-free by construction: a lane reads the treelet data it needs into
// registers before anything is written, and box/area/cost are recomputed
// bottom-up through shuffles instead of in-place sweeps over global memory.
#include "dev_common.h"
#include "lbvh.h"

namespace cav {
namespace {

constexpr int kBlock = 256;
constexpr int kGroups = kBlock / 32;
constexpr int kT = 13;  // 2*7-1 treelet nodes

// BVH/Optimization.cu:20-47
__constant__ uint8_t kSchedule[160] = {
    0b00011, 0b00110, 0b00101, 0b01001, 0b01010, 0b01100, 0b10001, 0b10010, 0b10100, 0b11000,
    0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
    0b00111, 0b01011, 0b01101, 0b01110, 0b10011, 0b10101, 0b10110, 0b11001, 0b11010, 0b11100,
    0b100001, 0b100010, 0b100100, 0b101000, 0b110000,
    0b1000001, 0b1000010, 0b1000100, 0b1001000, 0b1010000, 0b1100000,
    0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
    0b100011, 0b100101, 0b100110, 0b101001, 0b101010, 0b101100, 0b110001, 0b110010, 0b110100, 0b111000,
    0b1000011, 0b1000101, 0b1000110, 0b1001001, 0b1001010, 0b1001100, 0b1010001, 0b1010010,
    0b1010100, 0b1011000, 0b1100001, 0b1100010, 0b1100100, 0b1101000, 0b1110000,
    0b0001111, 0b0010111, 0b0011110,
    0, 0, 0, 0,
    0b1000111, 0b0011011, 0b0101011, 0b1001011, 0b0110011, 0b1010011, 0b1100011, 0b0011101,
    0b0101101, 0b1001101, 0b0110101, 0b1010101, 0b1100101, 0b0111001, 0b1011001, 0b1101001,
    0b1110001, 0b0100111, 0b0101110, 0b1001110, 0b0110110, 0b1010110, 0b1100110, 0b0111010,
    0b1011010, 0b1101010, 0b1110010, 0b0111100, 0b1011100, 0b1101100, 0b1110100, 0b1111000,
    0b0011111, 0b0101111, 0b1001111, 0b0110111, 0b1010111, 0b1100111, 0b0111011, 0b1011011,
    0b1101011, 0b1110011, 0b0111101, 0b1011101, 0b1101101, 0b1110101, 0b1111001, 0b0111110,
    0b1011110, 0b1101110, 0b1110110, 0b1111010, 0b1111100,
    0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

struct GroupLds {
    float area[128];
    float cost[128];
    float4 llo[7], lhi[7];  // the treelet leaves' boxes
    int leaf_lane[8];       // formation lane of each treelet leaf
    uint8_t part[128];
};

__device__ __forceinline__ int shi(int v, int src) { return __shfl(v, src, 32); }
__device__ __forceinline__ float shf(float v, int src) { return __shfl(v, src, 32); }
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Cross-lane moves inside rows of 16 lanes as VALU operands (DPP) instead of
// LDS permutes: the lane kShift above (row_shl), the row rotated (row_ror).
template <int kShift>
__device__ __forceinline__ int row_above(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x100 | kShift, 0xf, 0xf, true);
}
template <int kRot>
__device__ __forceinline__ uint32_t row_max_step(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 | kRot, 0xf, 0xf, true));
}
// the lane 16 away in the group's other row
__device__ __forceinline__ int other_row(int v) { return __builtin_amdgcn_ds_swizzle(v, 0x401f); }

// One step of the reference's min(l+d,31) reduction tree, as far as its lane 0
// depends on it: a lane keeps its own candidate unless the one kShift above is
// strictly smaller.
template <int kShift>
__device__ __forceinline__ void tree_step(float& c, int& who) {
    const float oc = __int_as_float(row_above<kShift>(__float_as_int(c)));
    const int ow = row_above<kShift>(who);
    const bool take = oc < c;
    c = take ? oc : c;
    who = take ? ow : who;
}
__device__ __forceinline__ void tree_row(float& c, int& who) {
    tree_step<8>(c, who);
    tree_step<4>(c, who);
    tree_step<2>(c, who);
    tree_step<1>(c, who);
}

struct LaneNode {
    int node;
    float lx, ly, lz, hx, hy, hz, sa, cost;
    int left, right, parent, prim;
    uint32_t height;  // of the subtree (0 for a triangle)
};

__device__ __forceinline__ void load_node(LaneNode& n, const NodeBox* nbox, const int4* topo, const uint32_t* hw,
                                          int id) {
    n.node = id;
    const NodeBox b = nbox[id];
    const int4 t = topo[id];
    const uint32_t h = hw[id];
    n.lx = b.a.x; n.ly = b.a.y; n.lz = b.a.z; n.sa = b.a.w;
    n.hx = b.b.x; n.hy = b.b.y; n.hz = b.b.z; n.cost = b.b.w;
    n.left = t.x; n.right = t.y; n.parent = t.z; n.prim = t.w;
    n.height = t.w >= 0 ? 0u : (h & 0xffffu);
}

// Subsets of kIters + 1 or fewer nontrivial partitions each (one lane per
// subset, 0 = idle): the partition costs are all read before any is compared,
// so that the LDS latency is paid once. The first smallest one wins, as in
// the reference's loop.
template <int kIters>
__device__ __forceinline__ void dp_round(GroupLds& L, int s) {
    const int delta = (s - 1) & s;
    float c[kIters];
    int p = (0 - delta) & s;
#pragma unroll
    for (int i = 0; i < kIters; ++i) {
        c[i] = L.cost[p] + L.cost[s ^ p];
        p = (p - delta) & s;
    }
    p = (0 - delta) & s;
    float best = c[0];
    int bestp = p;
#pragma unroll
    for (int i = 1; i < kIters; ++i) {
        p = p == 0 ? 0 : (p - delta) & s;  // 0 past the last partition
        if (p != 0 && c[i] < best) { best = c[i]; bestp = p; }
    }
    wave_sync();
    if (s != 0) {
        L.cost[s] = internal_cost2(L.area[s], best);
        L.part[s] = (uint8_t)bestp;
    }
    wave_sync();
}

// lane's partition of the 6-leaf subset without leaf e: the lane's bits
// spread over the subset's bits below its top one
__device__ __forceinline__ int part6(int lane, int e) {
    const int hm = 5 - e > 0 ? (((1 << (5 - e)) - 1) << (e + 1)) : 0;
    return (lane & ((1 << e) - 1)) | ((lane << 1) & hm);
}

// BVH/Optimization.cu:49-462 for the treelet rooted at `root` (an internal
// node). Every lane of the group calls it; control flow is group-uniform.
//
// Bound by instructions, not bytes (13 nodes of 52 B read and written): so
// the largest-area lane is found with a row maximum instead of a loop of
// permutes, the seven 6-leaf subsets are reduced two at a time (one per row)
// and independently of each other, boxes come from the subset's leaves
// instead of seven bottom-up sweeps, and a treelet leaf keeps the cost it has
// (its subtree did not change after it was computed). hw holds every internal
// node's height and is kept valid, so no round climbs the tree for it.
// 4M triangles, one round: 3.7 -> 3.3 ms in the wide levels, 0.49 -> 0.29 in
// the single-workgroup tail, 0.35 ms of climbing between rounds gone.
__device__ __forceinline__ void optimize_treelet(int root, NodeBox* nbox, int4* topo, uint32_t* hw, GroupLds& L) {
    const int lane = threadIdx.x & 31;
    const int half = threadIdx.x & 32;
    LaneNode me;
    me.node = -1;
    me.prim = -1;
    me.sa = 0.f;
    if (lane == 0) load_node(me, nbox, topo, hw, root);
    bool expanded = false;

    // formation: open the inner node of largest area (lowest lane on ties)
#pragma unroll
    for (int size = 1; size < kT; size += 2) {
        const bool open = me.node != -1 && !expanded && me.prim < 0 && me.sa >= 0.f;
        const uint32_t key = open ? (__float_as_uint(me.sa) | 0x80000000u) : 0u;
        uint32_t mx = row_max_step<8>(key);
        mx = row_max_step<4>(mx);
        mx = row_max_step<2>(mx);
        mx = row_max_step<1>(mx);
        const uint32_t at = (uint32_t)(__ballot(open && key == mx) >> half) & 0xffffu;
        if (at == 0u) return;  // fewer than 7 leaves below root
        const int ml = __ffs((int)at) - 1;
        if (lane == ml) expanded = true;
        const int cl = shi(me.left, ml), cr = shi(me.right, ml);
        if (lane == size) load_node(me, nbox, topo, hw, cl);
        if (lane == size + 1) load_node(me, nbox, topo, hw, cr);
    }
    // treelet leaves in lane order
    const uint32_t leaves = (uint32_t)(__ballot(lane < kT && !expanded) >> half);
    const bool tleaf = lane < kT && !expanded;
    const int tbit = __popc(leaves & ((1u << lane) - 1u));
    if (tleaf) {
        L.llo[tbit] = make_float4(me.lx, me.ly, me.lz, 0.f);
        L.lhi[tbit] = make_float4(me.hx, me.hy, me.hz, 0.f);
        L.leaf_lane[tbit] = lane;
    }
    wave_sync();

    // subset areas: lane l covers subsets (i << 5) | l. Unions start from
    // NaN, which min and max ignore.
    {
        const float nan = __builtin_nanf("");
        v3 lo = mk3(nan, nan, nan), hi = lo;
#pragma unroll
        for (int bit = 0; bit < 5; ++bit) {
            const float4 bl = L.llo[bit], bh = L.lhi[bit];
            if ((lane >> bit) & 1) {
                lo = mk3(fmn(lo.x, bl.x), fmn(lo.y, bl.y), fmn(lo.z, bl.z));
                hi = mk3(fmx(hi.x, bh.x), fmx(hi.y, bh.y), fmx(hi.z, bh.z));
            }
        }
        const float4 l5 = L.llo[5], h5 = L.lhi[5], l6 = L.llo[6], h6 = L.lhi[6];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v3 a = lo, b = hi;
            if (i & 1) {
                a = mk3(fmn(a.x, l5.x), fmn(a.y, l5.y), fmn(a.z, l5.z));
                b = mk3(fmx(b.x, h5.x), fmx(b.y, h5.y), fmx(b.z, h5.z));
            }
            if (i & 2) {
                a = mk3(fmn(a.x, l6.x), fmn(a.y, l6.y), fmn(a.z, l6.z));
                b = mk3(fmx(b.x, h6.x), fmx(b.y, h6.y), fmx(b.z, h6.z));
            }
            const int s = (i << 5) | lane;
            L.area[s] = s != 0 ? surface_area(a, b) : 0.f;
            L.cost[s] = -1.f;
        }
    }
    wave_sync();
    if (tleaf) L.cost[1 << tbit] = me.cost;
    wave_sync();

    // sizes 2..5 on the fixed schedule
    dp_round<1>(L, kSchedule[lane]);
    dp_round<3>(L, kSchedule[32 + lane]);
    dp_round<7>(L, kSchedule[64 + lane]);
    dp_round<7>(L, kSchedule[96 + lane]);
    dp_round<15>(L, kSchedule[128 + lane]);

    // sizes 6 and 7: one partition per lane (two for size 7), reduced over
    // the 32 lanes in the reference's tree order. Only lane 0's result of the
    // tree is used, and lane 0 has no partition of its own before the first
    // step (d = 16), which it takes from lane 16.
    {
        float tc[7];
#pragma unroll
        for (int e = 0; e < 7; ++e) {
            const int s = 0x7f ^ (1 << e), p = part6(lane, e);
            tc[e] = L.cost[p] + L.cost[s ^ p];
        }
        float rc[4];
        int rw[4];
        const bool up = lane >= 16;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // row 0 reduces subset 2k, row 1 subset 2k + 1 (after the step
            // over 16 lanes, whose lower lane keeps ties)
            const int e0 = 2 * k, e1 = 2 * k + 1 < 7 ? 2 * k + 1 : 2 * k;
            const float own = up ? tc[e1] : tc[e0];
            const float got = __int_as_float(other_row(__float_as_int(up ? tc[e0] : tc[e1])));
            const float lowc = up ? got : own, highc = up ? own : got;  // lane l & 15 and the one 16 above
            const bool take = (lane & 15) == 0 || highc < lowc;
            rc[k] = take ? highc : lowc;
            rw[k] = (lane & 15) | (take ? 16 : 0);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) tree_row(rc[k], rw[k]);
        wave_sync();
        if ((lane & 15) == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int e = up ? 2 * k + 1 : 2 * k;
                if (e < 7) {
                    const int s = 0x7f ^ (1 << e);
                    L.cost[s] = internal_cost2(L.area[s], rc[k]);
                    L.part[s] = (uint8_t)part6(rw[k], e);
                }
            }
        }
        wave_sync();
        const float c0 = L.cost[lane] + L.cost[0x7f ^ lane];
        const float c1 = L.cost[lane | 32] + L.cost[0x7f ^ (lane | 32)];
        const bool second = lane == 0 || c1 < c0;
        float c = second ? c1 : c0;
        int who = lane | (second ? 32 : 0);
        const float oc = __int_as_float(other_row(__float_as_int(c)));
        const int ow = other_row(who);
        if (oc < c) { c = oc; who = ow; }  // (row 1's copy is not used)
        tree_row(c, who);
        wave_sync();
        if (lane == 0) L.part[0x7f] = (uint8_t)who;
        wave_sync();
    }

    // reconstruction: the first lane holding a set of several leaves hands
    // its two halves to the next two lanes. packed = set | depth << 8.
    int packed = lane == 0 ? 0x7f : 0;
    bool rexp = false;
    int child_l = -1, parent_lane = 0;
    int depth = 0;
#pragma unroll
    for (int rsize = 1; rsize < kT; rsize += 2) {
        const int set = packed & 0xff;
        const bool propose = !rexp && (set & (set - 1)) != 0;
        const uint32_t gm = (uint32_t)(__ballot(propose) >> half);
        if (gm == 0u) return;  // unreachable for a valid partition table
        const int xl = __ffs((int)gm) - 1;
        const int ps = shi(packed, xl);
        const int s = ps & 0xff, p = L.part[s], d = (ps >> 8) + 1;
        if (lane == xl) {
            rexp = true;
            child_l = rsize;
        }
        if (lane == rsize || lane == rsize + 1) {
            packed = (lane == rsize ? p : s ^ p) | (d << 8);
            parent_lane = xl;
        }
        depth = max(depth, d);
    }
    const int set = packed & 0xff;

    // treelet leaves take over the content of the original leaf of their bit
    const int src = lane < kT && !rexp ? L.leaf_lane[__ffs(set) - 1] : lane;
    float cost = shf(me.cost, src);
    const int oleft = shi(me.left, src), oright = shi(me.right, src), oprim = shi(me.prim, src);
    int height = shi((int)me.height, src);
    const int new_left = shi(me.node, child_l & 31), new_right = shi(me.node, (child_l + 1) & 31);
    const int pnode = shi(me.node, parent_lane);
    v3 lo, hi;
    {
        const float nan = __builtin_nanf("");
        lo = mk3(nan, nan, nan);
        hi = lo;
#pragma unroll
        for (int bit = 0; bit < 7; ++bit) {
            const float4 bl = L.llo[bit], bh = L.lhi[bit];
            if ((set >> bit) & 1) {
                lo = mk3(fmn(lo.x, bl.x), fmn(lo.y, bl.y), fmn(lo.z, bl.z));
                hi = mk3(fmx(hi.x, bh.x), fmx(hi.y, bh.y), fmx(hi.z, bh.z));
            }
        }
    }
    const float sa = surface_area(lo, hi);
    // costs and heights of the new inner nodes, bottom-up (depth steps: a
    // node at depth d is final after step depth - d)
    const int cl = rexp ? child_l : lane, cr = rexp ? child_l + 1 : lane;
    for (int it = 0; it < depth; ++it) {
        const float ac = shf(cost, cl), bc = shf(cost, cr);
        const int ah = shi(height, cl), bh = shi(height, cr);
        if (rexp) {
            cost = internal_cost3(sa, ac, bc);
            height = min(max(ah, bh) + 1, 0xffff);
        }
    }
    if (lane < kT) {
        const int l = rexp ? new_left : oleft;
        const int r = rexp ? new_right : oright;
        const int pr = rexp ? -1 : oprim;
        nbox[me.node] = NodeBox{make_float4(lo.x, lo.y, lo.z, sa), make_float4(hi.x, hi.y, hi.z, cost)};
        topo[me.node] = make_int4(l, r, lane == 0 ? me.parent : pnode, pr);
        if (pr < 0) hw[me.node] = (2u << 16) | (uint32_t)height;
        if (!rexp && oprim < 0) {
            reinterpret_cast<int*>(&topo[oleft])[2] = me.node;
            reinterpret_cast<int*>(&topo[oright])[2] = me.node;
        }
    }
}

// BVH/Optimization.cu:467-507, scheduled by height: every internal node of
// height h is the root of one treelet; its 32-lane group runs once all nodes of
// lower height are done (kernel boundaries or, for the sparse top levels, the
// barriers of a single workgroup).
__global__ __launch_bounds__(kBlock) void k_treelet_level(NodeBox* nbox, int4* topo, uint32_t* hw,
                                                          const uint32_t* __restrict__ list,
                                                          int count) {
    __shared__ GroupLds lds[kGroups];
    const int group = (int)(((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 5);
    if (group >= count) return;
    optimize_treelet((int)list[group], nbox, topo, hw, lds[threadIdx.x >> 5]);
}

__global__ __launch_bounds__(1024) void k_treelet_tail(NodeBox* nbox, int4* topo, uint32_t* hw,
                                                       const uint32_t* __restrict__ list,
                                                       const uint32_t* __restrict__ off, int h0,
                                                       int h1) {
    __shared__ GroupLds lds[32];
    const int g = threadIdx.x >> 5;
    for (int h = h0; h <= h1; ++h) {
        const uint32_t b = off[h], e = off[h + 1];
        for (uint32_t i = b + g; i < e; i += 32) optimize_treelet((int)list[i], nbox, topo, hw, lds[g]);
        __syncthreads();
    }
}

}  // namespace

// One restructuring round over the nodes bucketed by height: the build's
// climb leaves every inner node's height, and each treelet keeps the heights
// of the nodes it rewrites (a tree of fewer than 7 leaves is never changed).
hipError_t treelet_round_impl(LbvhBuffers& b, int n, hipStream_t s, Marker* mk) {
    hipError_t e;
    if ((e = levels_bucket(b, n, s, nullptr)) != hipSuccess) return e;
    mark(mk, "treelet_setup");
    const int top = b.height;
    for (int h = 3; h <= top; ++h) {
        const uint32_t rest = b.h_off[top + 1] - b.h_off[h];
        if (rest <= (uint32_t)kTreeletTailNodes) {
            hipLaunchKernelGGL(k_treelet_tail, dim3(1), dim3(1024), 0, s, b.nbox, b.topo, b.visited,
                               b.lvl_list, b.lvl_off, h, top);
            break;
        }
        const int cnt = (int)b.h_lvl[h];
        if (cnt == 0) continue;
        const int64_t blocks = ((int64_t)cnt * 32 + kBlock - 1) / kBlock;
        hipLaunchKernelGGL(k_treelet_level, dim3((unsigned)blocks), dim3(kBlock), 0, s, b.nbox,
                           b.topo, b.visited, b.lvl_list + b.h_off[h], cnt);
    }
    mark(mk, "treelet");
    return hipGetLastError();
}

}  // namespace cav
