// trace.hip - closest-hit ray traversal of a BVH8 (the compressed wide node
// of BVH.h:39-96, Ylitie, Karras and Laine, "Efficient Incoherent Ray
// Traversal on GPUs Through Compressed Wide BVHs", HPG 2017). The reference
// builds BVH8s but has no traversal; this is the consumer that checks the
// 80-byte format end to end and measures traced cost.
//
// A node's eight child boxes are decoded from the 8-bit grid (lo = p + qlo *
// 2^(e-127), hi = p + qhi * 2^(e-127)) and slab-tested; hit leaves (one
// triangle each) are intersected at once, and the hit inner children are
// pushed as one group entry (their parent's child base, inner mask and hit
// mask), so the stack holds at most one entry per level. Within a group the
// children go in the order slot ^ octant: the builder's greedy slot
// assignment puts the child on the -x side into slots with bit 2 clear
// (likewise y, bit 1, and z, bit 0), so this order is front to back along
// the ray's octant.
//
// Three kernels, of which each takes the smallest distance, then the smallest
// triangle index, of the triangles it tests. They visit nodes in different orders
// and skip those that start beyond the best distance so far, so their hits are the
// same as long as a triangle's computed distance lies within its box's widened
// interval. Rounding breaks that only for triangles that are lines at their
// coordinates' precision (6.6M rays into slivers and needles, many of them along a
// needle: no difference; 3 of 600,000 rays differ from k_trace's where needles 1e-7
// wide lie at coordinates of 50,000, whose floats are 4e-3 apart):
//   k_trace_group  eight lanes per node, one per child slot, and up to four
//                  nodes of a ray at once: few rays, where a ray's chain of
//                  dependent steps is what takes the time;
//   k_trace_lane   one lane per ray: many rays, where the instructions issued
//                  per ray count;
//   k_trace        one lane per ray, with the counts of nodes visited and
//                  triangles tested (d_stats): its slab test and its order of
//                  leaf tests define those counts.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "nxb_internal.h"

namespace nxb {

namespace {

constexpr int kTraceThreads = 128;
constexpr uint32_t kTraceStack = kBvh8LevelWords;  // deeper than any BVH8 the builder makes

struct Vec3 {
    float x, y, z;
};

__device__ __forceinline__ Vec3 sub3(Vec3 a, Vec3 b) { return Vec3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ Vec3 cross3(Vec3 a, Vec3 b) {
    return Vec3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float dot3(Vec3 a, Vec3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// Moller-Trumbore ("Fast, Minimum Storage Ray/Triangle Intersection", 1997)
// in FP32, evaluated in this exact order (no contraction). Updates the
// closest hit for tmin <= t <= best (equal t: smaller index).
// Triangle prim's corners: nine floats per triangle, or (indexed mesh) three
// vertex indices per triangle into vertices of three floats. A corner index
// past vertex_count drops the triangle.
struct TriSource {
    const float* __restrict__ v;
    const uint32_t* __restrict__ idx;  // null: triangle soup
    uint32_t vertex_count;
};

template <bool INDEXED>
__device__ __forceinline__ bool fetch_triangle(const TriSource& ts, uint32_t prim, Vec3& v0, Vec3& v1, Vec3& v2) {
    if constexpr (INDEXED) {
        const uint32_t a = ts.idx[(size_t)prim * 3], b = ts.idx[(size_t)prim * 3 + 1],
                       c = ts.idx[(size_t)prim * 3 + 2];
        if (a >= ts.vertex_count || b >= ts.vertex_count || c >= ts.vertex_count) return false;
        v0 = Vec3{ts.v[(size_t)a * 3], ts.v[(size_t)a * 3 + 1], ts.v[(size_t)a * 3 + 2]};
        v1 = Vec3{ts.v[(size_t)b * 3], ts.v[(size_t)b * 3 + 1], ts.v[(size_t)b * 3 + 2]};
        v2 = Vec3{ts.v[(size_t)c * 3], ts.v[(size_t)c * 3 + 1], ts.v[(size_t)c * 3 + 2]};
    } else {
        const float* v = ts.v + (size_t)prim * 9;
        v0 = Vec3{v[0], v[1], v[2]};
        v1 = Vec3{v[3], v[4], v[5]};
        v2 = Vec3{v[6], v[7], v[8]};
    }
    return true;
}

// The triangle's hit at t in [tmin, tmax] and its barycentrics, if any.
template <bool INDEXED>
__device__ __forceinline__ bool intersect(const TriSource& ts, uint32_t prim, Vec3 o, Vec3 d, float tmin, float tmax,
                                          float& t, float& u, float& w) {
    Vec3 v0, v1, v2;
    if (!fetch_triangle<INDEXED>(ts, prim, v0, v1, v2)) return false;
    const Vec3 e1 = sub3(v1, v0), e2 = sub3(v2, v0);
    const Vec3 pv = cross3(d, e2);
    const float det = dot3(e1, pv);
    if (det == 0.0f) return false;
    const float inv = 1.0f / det;
    const Vec3 tv = sub3(o, v0);
    u = dot3(tv, pv) * inv;
    if (!(u >= 0.0f && u <= 1.0f)) return false;
    const Vec3 qv = cross3(tv, e1);
    w = dot3(d, qv) * inv;
    if (!(w >= 0.0f && u + w <= 1.0f)) return false;
    t = dot3(e2, qv) * inv;
    return t >= tmin && t <= tmax;
}

template <bool INDEXED>
__device__ __forceinline__ void hit_triangle(const TriSource& ts, uint32_t prim, Vec3 o, Vec3 d, float tmin,
                                             float& best_t, uint32_t& best_prim, float& bu, float& bv) {
    float t, u, w;
    if (!intersect<INDEXED>(ts, prim, o, d, tmin, best_t, t, u, w)) return;
    if (t < best_t || prim < best_prim) {
        best_t = t;
        best_prim = prim;
        bu = u;
        bv = w;
    }
}

// Reciprocal of a direction component; a zero one becomes tiny, of the same sign.
__device__ __forceinline__ float safe_inv(float x) { return 1.0f / (fabsf(x) > 1e-30f ? x : copysignf(1e-30f, x)); }

__device__ __forceinline__ float exp_scale(uint32_t e) { return __uint_as_float(e << 23); }  // 2^(e-127)

// Slab test from the decoded child box, face by face: a node's origin p and
// scale s on an axis, the ray's origin o and reciprocal direction i.
struct FaceSlab {
    float p, s, o, i;
    // Distances t0, t1 of the faces at ql and qh, the box widened outward. The
    // grid bounds the child exactly, but two roundings move a decoded face
    // inward: the builder's difference fl(c - p), off by up to
    // |c - p| * 2^-24 <= (|c| + |p|) * 2^-24, which can land
    // exactly on a grid point, and the decode p + q * s, off by
    // |l| * 2^-24. (|l| + |p|) * 2^-21 covers both with margin.
    __device__ __forceinline__ void faces(uint32_t ql, uint32_t qh, float& t0, float& t1) const {
        float l = p + (float)ql * s, h = p + (float)qh * s;
        l -= (fabsf(l) + fabsf(p)) * 0x1p-21f;
        h += (fabsf(h) + fabsf(p)) * 0x1p-21f;
        t0 = (l - o) * i;
        t1 = (h - o) * i;
    }
};
__device__ __forceinline__ bool slab_hit_faces(const FaceSlab& x, const FaceSlab& y, const FaceSlab& z, uint32_t qlx,
                                               uint32_t qly, uint32_t qlz, uint32_t qhx, uint32_t qhy, uint32_t qhz,
                                               float tmin, float best_t) {
    float tx0, tx1, ty0, ty1, tz0, tz1;
    x.faces(qlx, qhx, tx0, tx1);
    y.faces(qly, qhy, ty0, ty1);
    z.faces(qlz, qhz, tz0, tz1);
    const float tn = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), tmin));
    // the far distance is widened by 2^-20 against the slab test's
    // own rounding (Ize, "Robust BVH Ray Traversal", 2013)
    const float tf = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fmaxf(tz0, tz1)) * (1.0f + 0x1p-20f);
    return tn <= tf && tn <= best_t;
}

template <bool INDEXED>
__global__ __launch_bounds__(kTraceThreads) void k_trace(const nxb_bvh8_node* __restrict__ nodes, uint32_t node_count,
                                                         const uint32_t* __restrict__ prim_idx, uint32_t prim_count,
                                                         TriSource tris,
                                                         const nxb_ray* __restrict__ rays, uint32_t ray_count,
                                                         nxb_hit* __restrict__ hits, uint32_t* __restrict__ stats) {
    const uint32_t r = blockIdx.x * kTraceThreads + threadIdx.x;
    if (r >= ray_count) return;
    const float4* rp = reinterpret_cast<const float4*>(rays + r);
    const float4 ra = rp[0], rb = rp[1];
    const Vec3 o{ra.x, ra.y, ra.z}, d{rb.x, rb.y, rb.z};
    const float tmin = ra.w;
    float best_t = rb.w, bu = 0.0f, bv = 0.0f;
    uint32_t best_prim = NXB_INVALID_IDX;
    const float ix = safe_inv(d.x), iy = safe_inv(d.y), iz = safe_inv(d.z);
    const uint32_t oct = (d.x < 0.0f ? 4u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 1u : 0u);

    uint2 stack[kTraceStack];
    uint32_t sp = 0, visited = 0, tested = 0;
    uint32_t node = 0;
    bool have = node_count > 0;
    for (;;) {
        if (have) {
            have = false;
            // a tree visits each node at most once: the bound only ends a
            // walk over a malformed node array
            if (node >= node_count || visited >= node_count) break;
            ++visited;
            const float4* np = reinterpret_cast<const float4*>(nodes + node);
            const float4 w0 = np[0], w1 = np[1], w2 = np[2], w3 = np[3], w4 = np[4];
            // p.xyz | e[3], imask | child_base | prim_base | meta[8] | q*[8] x 6
            const float px = w0.x, py = w0.y, pz = w0.z;
            const uint32_t em = __float_as_uint(w0.w);
            const float sx = exp_scale(em & 0xFFu), sy = exp_scale((em >> 8) & 0xFFu), sz = exp_scale((em >> 16) & 0xFFu);
            const uint32_t imask = em >> 24;
            const uint32_t child_base = __float_as_uint(w1.x), prim_base = __float_as_uint(w1.y);
            const uint32_t meta_lo = __float_as_uint(w1.z), meta_hi = __float_as_uint(w1.w);
            const uint32_t qlx[2] = {__float_as_uint(w2.x), __float_as_uint(w2.y)};
            const uint32_t qly[2] = {__float_as_uint(w2.z), __float_as_uint(w2.w)};
            const uint32_t qlz[2] = {__float_as_uint(w3.x), __float_as_uint(w3.y)};
            const uint32_t qhx[2] = {__float_as_uint(w3.z), __float_as_uint(w3.w)};
            const uint32_t qhy[2] = {__float_as_uint(w4.x), __float_as_uint(w4.y)};
            const uint32_t qhz[2] = {__float_as_uint(w4.z), __float_as_uint(w4.w)};
            uint32_t inner_hits = 0;
#pragma unroll
            for (uint32_t s = 0; s < 8; ++s) {
                const uint32_t h = s >> 2, sh = (s & 3) * 8;
                const uint32_t meta = ((s < 4 ? meta_lo : meta_hi) >> sh) & 0xFFu;
                if (meta == 0) continue;
                if (!slab_hit_faces(FaceSlab{px, sx, o.x, ix}, FaceSlab{py, sy, o.y, iy}, FaceSlab{pz, sz, o.z, iz},
                                    (qlx[h] >> sh) & 0xFFu, (qly[h] >> sh) & 0xFFu, (qlz[h] >> sh) & 0xFFu,
                                    (qhx[h] >> sh) & 0xFFu, (qhy[h] >> sh) & 0xFFu, (qhz[h] >> sh) & 0xFFu, tmin,
                                    best_t))
                    continue;
                if (imask & (1u << s)) {
                    inner_hits |= 1u << s;
                } else {
                    const uint32_t k = prim_base + (meta & 0x1Fu);
                    if (k < prim_count) {
                        ++tested;
                        const uint32_t prim = prim_idx[k];
                        if (prim < prim_count) hit_triangle<INDEXED>(tris, prim, o, d, tmin, best_t, best_prim, bu, bv);
                    }
                }
            }
            if (inner_hits && sp < kTraceStack) stack[sp++] = make_uint2(child_base, imask | (inner_hits << 8));
        }
        if (sp == 0) break;
        uint2& top = stack[sp - 1];
        const uint32_t im = top.y & 0xFFu;
        uint32_t hm = top.y >> 8;
        uint32_t s = 0;
#pragma unroll
        for (int k = 7; k >= 0; --k)  // the first slot in the order slot ^ oct
            if (hm & (1u << ((uint32_t)k ^ oct))) s = (uint32_t)k ^ oct;
        hm &= ~(1u << s);
        node = top.x + (uint32_t)__popc(im & ((1u << s) - 1u));
        if (hm) top.y = im | (hm << 8);
        else --sp;
        have = true;
    }
    hits[r] = nxb_hit{best_prim == NXB_INVALID_IDX ? rb.w : best_t, best_prim, bu, bv};
    if (stats) {
        stats[2 * (size_t)r] = visited;
        stats[2 * (size_t)r + 1] = tested;
    }
}

// Slab test of the uncounted kernels. Along one axis a decoded face p + q * s
// lies at t = (p - o) * i + q * (s * i) on the ray (i: reciprocal direction),
// one FMA per face once a node's `near`, `far` and `step` are known; the face
// that the ray meets first is the low one for i > 0, else the high one.
// With u = 2^-24, c = (p - o) * i and step = s * i, the roundings of p - o, c, i,
// the FMA and `near` or `far` move t by at most u * (5 |c| + 510 |step| + 2 e); the
// builder's rounding of the child face puts it up to (2 |p| + 256 s) * u off the
// grid point that stands for it. `near` and `far` are moved apart by
// e = 2^-21 * (|c| + 256 |step| + 2 |p i|), more than both together and not less
// than slab_hit_faces' widening of the faces.
// The low and the high face share c, so its overflow would put both on one side of
// the ray and lose the child (a zero direction component counts as 1e-30, so c
// overflows from |p - o| = 3.4e8). e, and so near, is infinite or NaN wherever c or
// step is: such a node is tested by slab_hit_faces, where each face overflows to its
// own side. Its exponents come through `again`, so that nothing of that test is
// computed early and kept in registers (one lane per ray: 77 of them instead of 71).
struct AxisSlab {
    float near, far, step;
};
__device__ __forceinline__ AxisSlab axis_slab(float p, float scale, float o, float i) {
    const float c = (p - o) * i, step = scale * i;
    const float e = __builtin_fmaf(fabsf(c), 0x1p-21f,
                                   __builtin_fmaf(fabsf(step), 0x1p-13f, fabsf(p) * (fabsf(i) * 0x1p-20f)));
    return AxisSlab{c - e, c + e, step};
}
__device__ __forceinline__ uint32_t again(uint32_t em) {
    asm("" : "+v"(em));
    return em;
}
__device__ __forceinline__ bool in_range(const AxisSlab& x, const AxisSlab& y, const AxisSlab& z) {
    return fabsf(x.near) + fabsf(y.near) + fabsf(z.near) < INFINITY;
}
// Whether (p - o) * i or s * i can overflow for a node below the root with first
// words w0: the nodes' origins lie in the root's grid, p to p + 255 s, and their
// scales are at most 2 s. Asked once per ray: in_range at every node took 3% of the
// traversal of 2^20 primary rays in 2M triangles (502 us; 517 with it, 506 so).
__device__ __forceinline__ bool may_overflow(float4 w0, Vec3 o, float ix, float iy, float iz) {
    const uint32_t em = __float_as_uint(w0.w);
    const float s = exp_scale(max(max(em & 0xFFu, (em >> 8) & 0xFFu), (em >> 16) & 0xFFu));
    const float d = fmaxf(fmaxf(fabsf(w0.x - o.x), fabsf(w0.y - o.y)), fabsf(w0.z - o.z));
    const float i = fmaxf(fmaxf(fabsf(ix), fabsf(iy)), fabsf(iz));
    return !((d + 512.0f * s) * i * 4.0f < INFINITY);
}
__device__ __forceinline__ bool slab_hit(const AxisSlab& x, const AxisSlab& y, const AxisSlab& z, float nx, float ny,
                                         float nz, float fx, float fy, float fz, float tmin, float best_t) {
    const float tn = fmaxf(fmaxf(__builtin_fmaf(nx, x.step, x.near), __builtin_fmaf(ny, y.step, y.near)),
                           fmaxf(__builtin_fmaf(nz, z.step, z.near), tmin));
    const float tf = fminf(fminf(__builtin_fmaf(fx, x.step, x.far), __builtin_fmaf(fy, y.step, y.far)),
                           __builtin_fmaf(fz, z.step, z.far));
    return tn <= tf && tn <= best_t;
}

// Takes the next child of the group (base; inner mask | remaining hits << 8):
// the first slot in the order slot ^ oct. hits & 0xFF must not be empty.
__device__ __forceinline__ uint32_t next_child(uint32_t base, uint32_t& group, uint32_t oct) {
    uint32_t f = group >> 8;  // bit k: slot k ^ oct, after exchanging halves, pairs and neighbours
    f = (oct & 4u) ? ((f >> 4) | (f << 4)) & 0xFFu : f;
    f = (oct & 2u) ? ((f >> 2) & 0x33u) | ((f << 2) & 0xCCu) : f;
    f = (oct & 1u) ? ((f >> 1) & 0x55u) | ((f << 1) & 0xAAu) : f;
    const uint32_t s = (uint32_t)__builtin_ctz(f) ^ oct;
    group &= ~(0x100u << s);
    return base + (uint32_t)__popc(group & ((1u << s) - 1u));
}

// One lane per ray. k_trace spent most of its instructions in the leaf tests:
// with 64 rays in a wave, nearly every slot of a node is a hit leaf for some
// ray, so a step ran the triangle test eight times. Here the slots are tested
// first, and the lanes then walk their own hit leaves together (as many
// triangle tests as the fullest lane has leaves); with the shorter slab test
// (20 instead of ~60 instructions a child) 2^20 rays against 2M triangles take
// 543 instead of 949 us (primary, surface) and 1031 instead of 1764 us
// (incoherent, uniform). The next node does not depend on the leaves, so its
// loads go out before their tests: 539 -> 501 and 1030 -> 962 us. Bound by the issue
// of vector instructions that few of a wave's rays still need: primary rays fill 71%
// of the issue slots with 27 of 64 lanes active, incoherent ones 99% with 6 (a wave
// runs until its longest ray ends); of their L2 requests 6 and 49% miss.
template <bool INDEXED>
__global__ __launch_bounds__(kTraceThreads) void k_trace_lane(const nxb_bvh8_node* __restrict__ nodes,
                                                              uint32_t node_count,
                                                              const uint32_t* __restrict__ prim_idx,
                                                              uint32_t prim_count, TriSource tris,
                                                              const nxb_ray* __restrict__ rays, uint32_t ray_count,
                                                              nxb_hit* __restrict__ hits) {
    const uint32_t r = blockIdx.x * kTraceThreads + threadIdx.x;
    if (r >= ray_count) return;
    const float4* rp = reinterpret_cast<const float4*>(rays + r);
    const float4 ra = rp[0], rb = rp[1];
    const Vec3 o{ra.x, ra.y, ra.z}, d{rb.x, rb.y, rb.z};
    const float tmin = ra.w;
    float best_t = rb.w, bu = 0.0f, bv = 0.0f;
    uint32_t best_prim = NXB_INVALID_IDX;
    const float ix = safe_inv(d.x), iy = safe_inv(d.y), iz = safe_inv(d.z);
    const bool negx = ix < 0.0f, negy = iy < 0.0f, negz = iz < 0.0f;
    const uint32_t oct = (d.x < 0.0f ? 4u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 1u : 0u);

    uint2 stack[kTraceStack];
    uint32_t sp = 0, visited = 0, base = 0, group = 0;
    bool more = node_count != 0;
    float4 w0{}, w1{}, w2{}, w3{}, w4{};
    auto load = [&](uint32_t node) {
        const float4* np = reinterpret_cast<const float4*>(nodes + node);
        w0 = np[0]; w1 = np[1]; w2 = np[2]; w3 = np[3]; w4 = np[4];
    };
    bool overflow = false;
    if (more) {
        load(0);
        overflow = may_overflow(w0, o, ix, iy, iz);
    }
    while (more) {
        ++visited;
        const uint32_t em = __float_as_uint(w0.w), imask = em >> 24;
        const uint32_t child_base = __float_as_uint(w1.x), prim_base = __float_as_uint(w1.y);
        const AxisSlab x = axis_slab(w0.x, exp_scale(em & 0xFFu), o.x, ix);
        const AxisSlab y = axis_slab(w0.y, exp_scale((em >> 8) & 0xFFu), o.y, iy);
        const AxisSlab z = axis_slab(w0.z, exp_scale((em >> 16) & 0xFFu), o.z, iz);
        uint32_t hit = 0;
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t lx = __float_as_uint(h ? w2.y : w2.x), ly = __float_as_uint(h ? w2.w : w2.z);
            const uint32_t lz = __float_as_uint(h ? w3.y : w3.x), hx = __float_as_uint(h ? w3.w : w3.z);
            const uint32_t hy = __float_as_uint(h ? w4.y : w4.x), hz = __float_as_uint(h ? w4.w : w4.z);
            const uint32_t nx = negx ? hx : lx, ny = negy ? hy : ly, nz = negz ? hz : lz;
            const uint32_t fx = negx ? lx : hx, fy = negy ? ly : hy, fz = negz ? lz : hz;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint32_t sh = 8 * k;
                auto at = [&](uint32_t q) { return (float)((q >> sh) & 0xFFu); };
                if (slab_hit(x, y, z, at(nx), at(ny), at(nz), at(fx), at(fy), at(fz), tmin, best_t))
                    hit |= 1u << (4 * h + k);
            }
        }
        if (overflow && !in_range(x, y, z)) {
            hit = 0;
            const uint32_t em2 = again(em);
#pragma unroll 1
            for (uint32_t s = 0; s < 8; ++s) {
                const uint32_t sh = 8 * (s & 3);
                auto at = [&](float lo, float hi) { return (__float_as_uint(s < 4 ? lo : hi) >> sh) & 0xFFu; };
                if (slab_hit_faces(FaceSlab{w0.x, exp_scale(em2 & 0xFFu), o.x, ix},
                                   FaceSlab{w0.y, exp_scale((em2 >> 8) & 0xFFu), o.y, iy},
                                   FaceSlab{w0.z, exp_scale((em2 >> 16) & 0xFFu), o.z, iz}, at(w2.x, w2.y),
                                   at(w2.z, w2.w), at(w3.x, w3.y), at(w3.z, w3.w), at(w4.x, w4.y), at(w4.z, w4.w),
                                   tmin, best_t))
                    hit |= 1u << s;
            }
        }
        // the next node, which the leaves do not change
        const uint32_t inner = hit & imask;
        if (inner) {
            if ((group >> 8) && sp < kTraceStack) stack[sp++] = make_uint2(base, group);
            base = child_base;
            group = imask | (inner << 8);
        }
        if ((group >> 8) == 0) {
            more = sp != 0;
            if (more) {
                const uint2 top = stack[--sp];
                base = top.x;
                group = top.y;
            }
        }
        const float m0 = w1.z, m1 = w1.w;  // metas of slots 0-3 and 4-7
        if (more) {
            const uint32_t node = next_child(base, group, oct);
            // a tree visits each node at most once: the bound only ends a walk
            // over a malformed node array
            more = node < node_count && visited < node_count;
            if (more) load(node);
        }
        // leaves: an empty slot (meta 0) is no leaf
        for (uint32_t leaf = hit & ~imask & 0xFFu; leaf; leaf &= leaf - 1u) {
            const uint32_t s = (uint32_t)__builtin_ctz(leaf);
            const uint32_t meta = (__float_as_uint(s < 4 ? m0 : m1) >> ((s & 3) * 8)) & 0xFFu;
            const uint32_t k = prim_base + (meta & 0x1Fu);
            if (meta == 0 || k >= prim_count) continue;
            const uint32_t prim = prim_idx[k];
            if (prim < prim_count) hit_triangle<INDEXED>(tris, prim, o, d, tmin, best_t, best_prim, bu, bv);
        }
    }
    hits[r] = nxb_hit{best_prim == NXB_INVALID_IDX ? rb.w : best_t, best_prim, bu, bv};
}

// A group of hit children still to visit: their parent's child base, and its
// inner mask | hits << 8 with the hit of slot s at bit s ^ oct, so that the
// lowest is the next.
__device__ __forceinline__ uint32_t in_octant_order(uint32_t f, uint32_t oct) {
    f = (oct & 4u) ? ((f >> 4) | (f << 4)) & 0xFFu : f;
    f = (oct & 2u) ? ((f >> 2) & 0x33u) | ((f << 2) & 0xCCu) : f;
    return (oct & 1u) ? ((f >> 1) & 0x55u) | ((f << 1) & 0xAAu) : f;
}
__device__ __forceinline__ uint32_t take_child(uint32_t base, uint32_t& group, uint32_t oct) {
    const uint32_t slot = (uint32_t)__builtin_ctz(group >> 8) ^ oct;
    group &= group - 0x100u;
    return base + (uint32_t)__popc(group & ((1u << slot) - 1u));
}

// Eight lanes per node, lane s of the eight for child slot s, and NODES nodes of
// a ray at a time: one slab test, and at most one triangle test, per lane and
// step, the hit masks from a ballot. The ray, the walk and the best hit are kept
// alike in all the ray's lanes; the stack is in LDS (one wave per block). The
// next nodes do not depend on the leaves: their loads are issued before the
// leaves' triangles are fetched and tested.
//
// Bound by the latency of a ray's steps (some 1.2 us each where nodes come from
// memory) with few waves to cover it: on the slivers below 57% of the waves' time is
// waiting, 2.8 waves per SIMD are in flight, 59% of the issue slots are filled, and
// 84% of the L2 requests miss (3.3 TB/s). Two nodes a step nearly halve the steps of
// the longest walk, for the same instructions per node. 16,384 rays took, with one
// node a step and the next node loaded after the leaves' tests; with it loaded
// before; with two nodes a step (us, rays a tenth of the scene long from near its
// surface):
//   2.9M slivers 955, 740, 490    28.1M blobs 493, 408, 309
//   1.1M surface  87,  75,  55    1.9M blobs  203, 169, 123
// and 4,096 rays in 48K slivers 45, 43 and with four nodes a step 27. Leaf tests
// spread over the next two steps, so that every load has a step to arrive, took
// as long or longer (738 and 481 us of the first two).
//
// Two or four nodes a step leave at most as many groups per level on the stack:
// nodes are taken in the stack's order, so a step that takes k nodes of a level
// has used up every deeper group, and leaves k groups one level down.
constexpr int kGroupThreads = 64;

template <bool INDEXED, uint32_t NODES>
__global__ __launch_bounds__(kGroupThreads) void k_trace_group(const nxb_bvh8_node* __restrict__ nodes,
                                                               uint32_t node_count,
                                                               const uint32_t* __restrict__ prim_idx,
                                                               uint32_t prim_count, TriSource tris,
                                                               const nxb_ray* __restrict__ rays, uint32_t ray_count,
                                                               nxb_hit* __restrict__ hits) {
    static_assert(NODES == 1 || NODES == 2 || NODES == 4, "one, two or four nodes a step");
    constexpr uint32_t kLanes = 8 * NODES, kRays = kGroupThreads / kLanes;
    constexpr uint32_t kStack = kTraceStack * NODES;
    __shared__ uint2 stack[kStack][kRays];
    const uint32_t lane = threadIdx.x, s = lane & 7u, h = lane / 8 % NODES, g = lane / kLanes;
    const uint32_t r = blockIdx.x * kRays + g;
    if (r >= ray_count) return;
    const float4* rp = reinterpret_cast<const float4*>(rays + r);
    const float4 ra = rp[0], rb = rp[1];
    const Vec3 o{ra.x, ra.y, ra.z}, d{rb.x, rb.y, rb.z};
    const float tmin = ra.w;
    float best_t = rb.w, bu = 0.0f, bv = 0.0f;
    uint32_t best_prim = NXB_INVALID_IDX;
    const float ix = safe_inv(d.x), iy = safe_inv(d.y), iz = safe_inv(d.z);
    const uint32_t oct = (d.x < 0.0f ? 4u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 1u : 0u);
    // byte offsets in a node of this slot's near and far faces: low faces of
    // x, y, z from byte 32, 40, 48, high faces 24 further
    const uint32_t nox = 32u + s + (ix < 0.0f ? 24u : 0u), fox = 32u + s + (ix < 0.0f ? 0u : 24u);
    const uint32_t noy = 40u + s + (iy < 0.0f ? 24u : 0u), foy = 40u + s + (iy < 0.0f ? 0u : 24u);
    const uint32_t noz = 48u + s + (iz < 0.0f ? 24u : 0u), foz = 48u + s + (iz < 0.0f ? 0u : 24u);
    // bit k: lane k of the ray
    auto ray_bits = [&](bool p) {
        return (uint32_t)((ballot(p) >> (lane & (64u - kLanes))) & ((1ull << kLanes) - 1u));
    };
    struct NodeSlot {  // this slot's part of a node
        float4 w0;
        uint2 w1;
        uint32_t meta, nx, ny, nz, fx, fy, fz;
    };
    auto load_slot = [&](uint32_t node) {
        const uint8_t* nb = reinterpret_cast<const uint8_t*>(nodes + node);
        return NodeSlot{reinterpret_cast<const float4*>(nb)[0], reinterpret_cast<const uint2*>(nb)[2], nb[24u + s],
                        nb[nox], nb[noy], nb[noz], nb[fox], nb[foy], nb[foz]};
    };

    uint32_t sp = 0, visited = 0, base = 0, group = 0;
    NodeSlot cur = {};
    bool more = node_count != 0, have = more && h == 0;  // the root
    if (have) cur = load_slot(0);
    const bool overflow = more && may_overflow(*reinterpret_cast<const float4*>(nodes), o, ix, iy, iz);
    while (more) {
        const uint32_t em = __float_as_uint(cur.w0.w), imask = em >> 24;
        const AxisSlab x = axis_slab(cur.w0.x, exp_scale(em & 0xFFu), o.x, ix);
        const AxisSlab y = axis_slab(cur.w0.y, exp_scale((em >> 8) & 0xFFu), o.y, iy);
        const AxisSlab z = axis_slab(cur.w0.z, exp_scale((em >> 16) & 0xFFu), o.z, iz);
        bool hit = slab_hit(x, y, z, (float)cur.nx, (float)cur.ny, (float)cur.nz, (float)cur.fx, (float)cur.fy,
                            (float)cur.fz, tmin, best_t);
        if (overflow && !in_range(x, y, z)) {
            const uint32_t em2 = again(em);
            const bool fx = ix < 0.0f, fy = iy < 0.0f, fz = iz < 0.0f;  // the far face is the low one
            hit = slab_hit_faces(FaceSlab{cur.w0.x, exp_scale(em2 & 0xFFu), o.x, ix},
                                 FaceSlab{cur.w0.y, exp_scale((em2 >> 8) & 0xFFu), o.y, iy},
                                 FaceSlab{cur.w0.z, exp_scale((em2 >> 16) & 0xFFu), o.z, iz}, fx ? cur.fx : cur.nx,
                                 fy ? cur.fy : cur.ny, fz ? cur.fz : cur.nz, fx ? cur.nx : cur.fx,
                                 fy ? cur.ny : cur.fy, fz ? cur.nz : cur.fz, tmin, best_t);
        }
        hit = hit && have && cur.meta != 0;
        const bool inner = (imask >> s) & 1u;
        const uint32_t inner_hits = ray_bits(hit && inner);
        uint32_t prim = NXB_INVALID_IDX;
        if (hit && !inner) {
            const uint32_t k = cur.w1.y + (cur.meta & 0x1Fu);
            if (k < prim_count) prim = prim_idx[k];
        }
        // the hit children of the step's nodes, in front of what is left
        if (inner_hits) {
            if ((group >> 8) && sp < kStack) stack[sp++][g] = make_uint2(base, group);
            uint32_t b0 = cur.w1.x, g0 = imask | (in_octant_order((inner_hits >> (8 * h)) & 0xFFu, oct) << 8);
            if constexpr (NODES == 2) {
                // the other node's, from the lane eight away
                const uint32_t b1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b0, 0x128, 0xF, 0xF, true);
                const uint32_t g1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)g0, 0x128, 0xF, 0xF, true);
                const bool swap = h ? (inner_hits & 0xFFu) != 0 : (inner_hits & 0xFFu) == 0;
                if ((inner_hits & 0xFFu) && (inner_hits >> 8) && sp < kStack)
                    stack[sp++][g] = h ? make_uint2(b0, g0) : make_uint2(b1, g1);
                b0 = swap ? b1 : b0;
                g0 = swap ? g1 : g0;
            }
            base = b0;
            group = g0;
            if constexpr (NODES == 4) {
                // all to the stack, the first node's on top
                uint32_t z = 0;
#pragma unroll
                for (uint32_t i = 0; i < NODES; ++i) z |= (inner_hits >> (8 * i)) & 0xFFu ? 1u << i : 0u;
                const uint32_t at = sp + (uint32_t)__popc(z >> (h + 1));
                if (s == 0 && ((z >> h) & 1u) && at < kStack) stack[at][g] = make_uint2(b0, g0);
                sp = min(sp + (uint32_t)__popc(z), kStack);
                group = 0;
                wave_lds_sync();
            }
        }
        // the next nodes
        uint32_t node = 0;
        have = false;
#pragma unroll
        for (uint32_t i = 0; i < NODES; ++i) {
            if ((group >> 8) == 0 && sp != 0) {
                const uint2 top = stack[--sp][g];
                base = top.x;
                group = top.y;
            }
            const bool any = (group >> 8) != 0;
            if (i == 0) more = any;
            if (any) {
                const uint32_t c = take_child(base, group, oct);
                // a tree visits each node at most once: the bound only ends a
                // walk over a malformed node array
                if (c >= node_count || ++visited >= node_count) more = false;
                else if (h == i) {
                    node = c;
                    have = true;
                }
            }
        }
        have = have && more;
        if (have) cur = load_slot(node);
        bool found = false;
        float t = INFINITY, u = 0.0f, w = 0.0f;
        if (prim < prim_count) found = intersect<INDEXED>(tris, prim, o, d, tmin, best_t, t, u, w);
        if (ray_bits(found)) {
            // the ray's nearest (then smallest index), taken by all its lanes
            float bt = found ? t : INFINITY;
            uint32_t bp = found ? prim : NXB_INVALID_IDX, from = lane;
#pragma unroll
            for (uint32_t x8 = 1; x8 < kLanes; x8 <<= 1) {
                const float ot = __shfl_xor(bt, (int)x8);
                const uint32_t op = (uint32_t)__shfl_xor((int)bp, (int)x8);
                const uint32_t of = (uint32_t)__shfl_xor((int)from, (int)x8);
                if (ot < bt || (ot == bt && op < bp)) {
                    bt = ot;
                    bp = op;
                    from = of;
                }
            }
            if (bt < best_t || bp < best_prim) {  // bt <= best_t
                best_t = bt;
                best_prim = bp;
                bu = __shfl(u, (int)from);
                bv = __shfl(w, (int)from);
            }
        }
    }
    if (s == 0 && h == 0) hits[r] = nxb_hit{best_prim == NXB_INVALID_IDX ? rb.w : best_t, best_prim, bu, bv};
}

// Rays up to which k_trace_group takes them, with four, two or one nodes a step
// (32, 16 or 8 lanes per ray). Over three scenes of 100K and 2M triangles,
// primary and incoherent (12 cases), times against the kernel for more rays:
//   four nodes against two    0.61-1.07 at 8,192 rays, 0.76-1.08 at 16,384 (but
//                             up to 1.17 for short rays near a surface)
//   two against one           0.69-0.98 at 32,768, 0.83-1.20 at 65,536
//   one against k_trace_lane  0.54-1.12 at 2^17, 0.69-1.50 at 2^18 (its wave's
//                             instructions per ray are about twice as many)
constexpr uint32_t kQuadMaxRays = 1u << 13;
constexpr uint32_t kPairMaxRays = 1u << 15;
constexpr uint32_t kGroupMaxRays = 1u << 17;

template <bool INDEXED, uint32_t NODES>
hipError_t launch_trace_group(const nxb_bvh8_node* nodes, uint32_t node_count, const uint32_t* prim_idx,
                              uint32_t prim_count, const TriSource& ts, const nxb_ray* rays, uint32_t ray_count,
                              nxb_hit* hits, hipStream_t s) {
    constexpr uint32_t per_block = kGroupThreads / (8 * NODES);
    hipLaunchKernelGGL((k_trace_group<INDEXED, NODES>), dim3((ray_count + per_block - 1) / per_block),
                       dim3(kGroupThreads), 0, s, nodes, node_count, prim_idx, prim_count, ts, rays, ray_count, hits);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_trace(const nxb_bvh8_node* nodes, uint32_t node_count, const uint32_t* prim_idx,
                        uint32_t prim_count, const float* tris, const nxb_ray* rays, uint32_t ray_count,
                        nxb_hit* hits, uint32_t* stats, hipStream_t s, const uint32_t* indices,
                        uint32_t vertex_count) {
    if (ray_count == 0) return hipSuccess;
    const TriSource ts{tris, indices, vertex_count};
    if (!stats && ray_count <= kGroupMaxRays) {
        auto launch = indices ? launch_trace_group<true, 1> : launch_trace_group<false, 1>;
        if (ray_count <= kPairMaxRays) launch = indices ? launch_trace_group<true, 2> : launch_trace_group<false, 2>;
        if (ray_count <= kQuadMaxRays) launch = indices ? launch_trace_group<true, 4> : launch_trace_group<false, 4>;
        return launch(nodes, node_count, prim_idx, prim_count, ts, rays, ray_count, hits, s);
    }
    const uint32_t grid = (ray_count + kTraceThreads - 1) / kTraceThreads;
    if (!stats)
        hipLaunchKernelGGL(indices ? k_trace_lane<true> : k_trace_lane<false>, dim3(grid), dim3(kTraceThreads), 0, s,
                           nodes, node_count, prim_idx, prim_count, ts, rays, ray_count, hits);
    else
        hipLaunchKernelGGL(indices ? k_trace<true> : k_trace<false>, dim3(grid), dim3(kTraceThreads), 0, s, nodes,
                           node_count, prim_idx, prim_count, ts, rays, ray_count, hits, stats);
    return hipGetLastError();
}

}  // namespace nxb
