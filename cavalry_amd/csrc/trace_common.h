// Device code shared by the traversals: the reference's slab and triangle
// tests, evaluated operation by operation as it writes them, and ray loads.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dev_common.h"

namespace cav {

// Core/BoundingBox.h:55-74; returns the entry distance or -1.
__device__ __forceinline__ float slab(float lx, float ly, float lz, float hx, float hy, float hz,
                                      v3 o, v3 inv) {
    const float t0x = (lx - o.x) * inv.x, t0y = (ly - o.y) * inv.y, t0z = (lz - o.z) * inv.z;
    const float t1x = (hx - o.x) * inv.x, t1y = (hy - o.y) * inv.y, t1z = (hz - o.z) * inv.z;
    const float maxmin = fmin_fmax(t0x, t1x, fmin_fmax(t0y, t1y, fmn(t0z, t1z)));
    const float minmax = fmax_fmin(t0x, t1x, fmax_fmin(t0y, t1y, fmx(t0z, t1z)));
    if (maxmin <= minmax && minmax > 0) return fmx(0.f, maxmin);
    return -1.f;
}

// Core/Triangle.h:7-52
__device__ __forceinline__ bool tri_hit(const TTri& tr, v3 o, v3 d, float& t, float& u, float& v) {
    const v3 v0 = mk3(tr.a.x, tr.a.y, tr.a.z);
    const v3 e1 = mk3(tr.b.x, tr.b.y, tr.b.z);
    const v3 e2 = mk3(tr.c.x, tr.c.y, tr.c.z);
    const v3 tvec = sub3(o, v0);
    const v3 pvec = cross3(d, e2);
    float det = dot3(e1, pvec);
    if (det == 0) return false;
    det = 1.f / det;
    u = dot3(tvec, pvec) * det;
    if (u < 0.0f || u > 1.0f) return false;
    const v3 qvec = cross3(tvec, e1);
    v = dot3(d, qvec) * det;
    if (v < 0.0f || (u + v) > 1.0f) return false;
    t = dot3(e2, qvec) * det;
    return t > 0.f;
}

__device__ __forceinline__ void load_ray(const float* __restrict__ rays, int64_t i, v3& o, v3& d) {
    const float2* r = reinterpret_cast<const float2*>(rays + i * 6);
    const float2 a = r[0], b = r[1], c = r[2];
    o = mk3(a.x, a.y, b.x);
    d = mk3(b.y, c.x, c.y);
}

// 64-bit count of records fetched by closest-hit (words 16-17) or any-hit
// (words 18-19) launches; kFetchTris 64-bit words on, how many of them were
// triangles of the wide tree
constexpr int kFetchTris = 8;
__host__ __device__ inline unsigned long long* fetch_word(uint32_t* counters, bool closest) {
    return reinterpret_cast<unsigned long long*>(counters + (closest ? 16 : 18));
}

// compute units of the current device (asked for once)
inline int device_cus() {
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        return n;
    }();
    return cus;
}

}  // namespace cav
