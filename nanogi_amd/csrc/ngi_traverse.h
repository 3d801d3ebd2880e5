// FP32 closest-hit and any-hit BVH traversal (device).
//
// Replaces rtcIntersect inside Scene::Intersect / Scene::Visible
// (include/nanogi/rt.hpp:2162-2261): two-sided triangles, hit interval
// (tmin, tmax) exclusive, barycentrics (u, v) = weights of vertices 1 and 2.
//
// Triangle test: watertight ray/triangle intersection (Woop, Benthin, Wald,
// "Watertight Ray/Triangle Intersection", JCGT 2(1), 2013): shear to ray
// space, scaled edge functions with a double-precision recomputation when
// an edge function is exactly zero.  Box test: slabs with the far distance
// scaled up by 1 + 2*gamma(3) (Ize, "Robust BVH Ray Traversal", JCGT 2013)
// so traversal is conservative with respect to the triangle test.
#pragma once

#include "ngi_dev.h"
#include "ngi_quot.h"

namespace ngi {

struct TraceRay {
    float ox, oy, oz;
    float dx, dy, dz;
    float tmin, tmax;
};

struct TraceHit {
    float t, u, v;
    int32_t leaf;   // leaf-order triangle index, -1 = miss
};

struct TraceCounters {
    uint32_t nodes;
    uint32_t tris;
};

// Per-ray constants for the watertight test and the slab test.
struct RayPre {
    float ox, oy, oz;
    float ix, iy, iz;        // 1 / d (guarded against zero components)
    float sx, sy, sz;        // shear constants
    int kx, ky, kz;
    float dx, dy, dz;
    uint32_t octant;         // bit k set if d[k] < 0
};

__device__ __forceinline__ float guard_dir(float d) {
    return fabsf(d) < 1e-20f ? copysignf(1e-20f, d) : d;
}

__device__ __forceinline__ float pick(float a, float b, float c, int k) { return k == 0 ? a : (k == 1 ? b : c); }

// 1.0f / d, bit for bit, in quot_exact's range (ngi_quot.h).
__device__ __forceinline__ float rcp_ieee(float d) { return rcp_newton(d, __builtin_amdgcn_rcpf(d)); }

__device__ __forceinline__ RayPre make_pre(const TraceRay& r) {
    RayPre p;
    p.ox = r.ox, p.oy = r.oy, p.oz = r.oz;
    p.dx = r.dx, p.dy = r.dy, p.dz = r.dz;
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz + 1 == 3 ? 0 : kz + 1;
    int ky = kx + 1 == 3 ? 0 : kx + 1;
    // Component selection by value (no dynamically indexed private array).
    const float dz = pick(r.dx, r.dy, r.dz, kz);
    if (dz < 0.0f) {
        int t = kx;
        kx = ky;
        ky = t;
    }
    p.kx = kx, p.ky = ky, p.kz = kz;
    // The six quotients of a ray: bit for bit the divisions below, which only
    // rays along an axis and extreme lengths still need (three divisions of
    // 1 and two others were 55 VALU instructions of every ray set-up and
    // every resumed traversal, now 15; with the leaf and box tests' changes,
    // the nave's ptdirect 92.2 -> 89.4 ms for 67M paths, ltdirect 11.99 ->
    // 11.63 ms, bdpt on the Cornell box 10.94 -> 10.62 ms).
    const float dx = pick(r.dx, r.dy, r.dz, kx), dy = pick(r.dx, r.dy, r.dz, ky);
    p.ix = rcp_ieee(guard_dir(r.dx));
    p.iy = rcp_ieee(guard_dir(r.dy));
    p.iz = rcp_ieee(guard_dir(r.dz));
    p.sz = pick(p.ix, p.iy, p.iz, kz);
    p.sx = div_markstein(dx, dz, p.sz);
    p.sy = div_markstein(dy, dz, p.sz);
    if (!quot_exact(fminf(fabsf(dx), fabsf(dy)), dz)) {
        p.ix = 1.0f / guard_dir(r.dx);
        p.iy = 1.0f / guard_dir(r.dy);
        p.iz = 1.0f / guard_dir(r.dz);
        p.sx = dx / dz;
        p.sy = dy / dz;
        p.sz = 1.0f / dz;
    }
    p.octant = (r.dx < 0.0f ? 1u : 0u) | (r.dy < 0.0f ? 2u : 0u) | (r.dz < 0.0f ? 4u : 0u);
    return p;
}

// Watertight test; on a hit inside (tmin, tmax) writes t, u, v.
__device__ __forceinline__ bool tri_test(const RayPre& r, float4 a4, float4 b4, float4 c4, float tmin, float tmax, float& t,
                                         float& u, float& v) {
#pragma clang fp contract(off)
    const float Ax0 = a4.x - r.ox, Ay0 = a4.y - r.oy, Az0 = a4.z - r.oz;
    const float Bx0 = b4.x - r.ox, By0 = b4.y - r.oy, Bz0 = b4.z - r.oz;
    const float Cx0 = c4.x - r.ox, Cy0 = c4.y - r.oy, Cz0 = c4.z - r.oz;
    const float Akx = pick(Ax0, Ay0, Az0, r.kx), Aky = pick(Ax0, Ay0, Az0, r.ky), Akz = pick(Ax0, Ay0, Az0, r.kz);
    const float Bkx = pick(Bx0, By0, Bz0, r.kx), Bky = pick(Bx0, By0, Bz0, r.ky), Bkz = pick(Bx0, By0, Bz0, r.kz);
    const float Ckx = pick(Cx0, Cy0, Cz0, r.kx), Cky = pick(Cx0, Cy0, Cz0, r.ky), Ckz = pick(Cx0, Cy0, Cz0, r.kz);
    const float Ax = Akx - r.sx * Akz, Ay = Aky - r.sy * Akz;
    const float Bx = Bkx - r.sx * Bkz, By = Bky - r.sy * Bkz;
    const float Cx = Ckx - r.sx * Ckz, Cy = Cky - r.sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (fminf(fminf(fabsf(U), fabsf(V)), fabsf(W)) == 0.0f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if (fminf(fminf(U, V), W) < 0.0f && fmaxf(fmaxf(U, V), W) > 0.0f) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float Az = r.sz * Akz, Bz = r.sz * Bkz, Cz = r.sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    // Sign-corrected range test: tmin < T/det < tmax.
    const float sT = det < 0.0f ? -T : T;
    const float sd = fabsf(det);
    if (sT <= tmin * sd || sT >= tmax * sd) return false;
    const float rd = 1.0f / det;
    t = T * rd;
    if (!(t > tmin && t < tmax)) return false;
    u = V * rd;
    v = W * rd;
    return true;
}

#define NGI_SLAB_SCALE 1.00000036f   // 1 + 2*gamma(3), gamma(n) = n*eps/(1-n*eps), eps = 2^-24

// What a child reference of the wide BVH points at: the first 64 bytes of a
// node (origin, exponents and valid slots, quantised bounds), or a leaf's
// first two triangles (48 bytes each, contiguous; the fourth word of a
// single triangle is not its own, and the triangle array is one float4
// longer for it).  Inner and leaf lanes of a wavefront issue the same loads,
// so an iteration waits once for nodes and triangles instead of once for
// each: iterations spend about half their cycles waiting, and nearly all of
// them have lanes of both kinds (nave: 29 inner, 8 leaf).  Measured, ms
// before -> after: ptdirect on the nave 87.6 -> 84.9
// (67M paths), 16.8M paths on the sphere field 8.77 -> 8.43, 7.4M with FP64
// shading 5.12 -> 4.95, adjoint replay on the nave 16.7 -> 15.6, bdpt on the
// Cornell box 10.04 -> 9.77, 1.5M incoherent rays 0.367 -> 0.342.  (The
// pointer is made from an integer, so these are flat loads: they count as LDS
// accesses too, and the iteration's stack accesses wait for them.)
typedef uint32_t Word4 __attribute__((ext_vector_type(4)));
struct Fetch {
    Word4 w[6];
};
__device__ __forceinline__ Fetch fetch_child(const DevScene& sc, int32_t ref) {
    const bool leaf = ref < 0;
    const uint32_t v = (uint32_t)~ref;
    const uint64_t base = leaf ? (uint64_t)(v >> 4) * 48u + reinterpret_cast<uint64_t>(sc.tris)
                               : (uint64_t)(uint32_t)ref * 128u + reinterpret_cast<uint64_t>(sc.nodes);
    const Word4* p = reinterpret_cast<const Word4*>(base);
    Fetch f;
    f.w[0] = p[0], f.w[1] = p[1], f.w[2] = p[2], f.w[3] = p[3];
    if (leaf && (v & 15u)) f.w[4] = p[4], f.w[5] = p[5];
    return f;
}

// One triangle of a leaf against the ray; a hit shortens tmax.
__device__ __forceinline__ bool leaf_tri(const RayPre& r, uint32_t leaf, Word4 a, Word4 b, Word4 c, float tmin, float& tmax, TraceHit& h) {
    float t, u, v;
    if (!tri_test(r, __builtin_bit_cast(float4, a), __builtin_bit_cast(float4, b), __builtin_bit_cast(float4, c), tmin, tmax, t, u, v))
        return false;
    tmax = t;
    h.t = t, h.u = u, h.v = v, h.leaf = (int32_t)leaf;
    return true;
}

// The triangles of leaf `ref`, fetched into f, in their order.  ANY: true,
// and no further test, on the first hit.
template <bool ANY, bool COUNT>
__device__ __forceinline__ bool leaf_test(const DevScene& sc, const RayPre& r, int32_t ref, const Fetch& f, float tmin, float& tmax,
                                          TraceHit& h, TraceCounters& cnt) {
    const uint32_t v = (uint32_t)(~ref);
    const uint32_t first = v >> 4, count = (v & 15u) + 1u;
    if (COUNT) cnt.tris++;
    if (leaf_tri(r, first, f.w[0], f.w[1], f.w[2], tmin, tmax, h) && ANY) return true;
    if (count < 2u) return false;
    if (COUNT) cnt.tris++;
    if (leaf_tri(r, first + 1u, f.w[3], f.w[4], f.w[5], tmin, tmax, h) && ANY) return true;
    for (uint32_t k = 2; k < count; ++k) {
        const Word4* p = reinterpret_cast<const Word4*>(sc.tris + 3 * (size_t)(first + k));
        if (COUNT) cnt.tris++;
        if (leaf_tri(r, first + k, p[0], p[1], p[2], tmin, tmax, h) && ANY) return true;
    }
    return false;
}

// leaf_test for the binary BVH, whose lanes fetch leaves apart from nodes: two
// triangles at a time, so that their loads overlap.  Through fetch_child its
// kernels with two traversals spill more scalar registers and lose: ptdirect on
// the nave, 512x512 pixels at 32 spp, ms, fetch_child / this: FP64 persistent
// 31.2 / 28.1, megakernel 37.4 / 35.6 and FP64 57.8 / 55.0, FP32 persistent 27.6
// / 25.3; bdpt on the field 3.3 / 2.9.
// Sensitive to its form: with a returned bool in place of `done` and the hit
// stored by leaf_tri they are 35.6 -> 40.8 and 28.1 -> 31.7 again.
template <bool ANY, bool COUNT>
__device__ __forceinline__ void leaf_test_pairs(const DevScene& sc, const RayPre& r, int32_t ref, float tmin, float& tmax, TraceHit& h,
                                                TraceCounters& cnt, bool& done) {
    const uint32_t v = (uint32_t)(~ref);
    const uint32_t first = v >> 4, count = (v & 15u) + 1u;
    for (uint32_t k = 0; k < count; k += 2) {
        const uint32_t l0 = first + k;
        const bool two = k + 1 < count;
        const uint32_t l1 = two ? l0 + 1 : l0;
        const float4 a0 = sc.tris[3 * l0], b0 = sc.tris[3 * l0 + 1], c0 = sc.tris[3 * l0 + 2];
        const float4 a1 = sc.tris[3 * l1], b1 = sc.tris[3 * l1 + 1], c1 = sc.tris[3 * l1 + 2];
        if (COUNT) cnt.tris += two ? 2u : 1u;
        float t, u, w;
        if (tri_test(r, a0, b0, c0, tmin, tmax, t, u, w)) {
            tmax = t;
            h.t = t, h.u = u, h.v = w, h.leaf = (int32_t)l0;
            if (ANY) {
                done = true;
                return;
            }
        }
        if (two && tri_test(r, a1, b1, c1, tmin, tmax, t, u, w)) {
            tmax = t;
            h.t = t, h.u = u, h.v = w, h.leaf = (int32_t)l1;
            if (ANY) {
                done = true;
                return;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Binary BVH, private stack (depth is bounded by the builder).
// ---------------------------------------------------------------------------
#define NGI_BVH2_STACK 64

template <bool ANY, bool COUNT>
__device__ bool trace_bvh2(const DevScene& sc, const TraceRay& ray, TraceHit& h, TraceCounters& cnt) {
    const RayPre r = make_pre(ray);
    const float tmin = ray.tmin;
    float tmax = ray.tmax;
    h.leaf = -1;
    int32_t stack[NGI_BVH2_STACK];
    int sp = 0;
    int32_t node = 0;
    bool done = false;
    for (;;) {
        if (node >= 0) {
            const float4* n = sc.nodes + 4 * (size_t)node;
            const float4 n0 = n[0], n1 = n[1], n2 = n[2], n3 = n[3];
            if (COUNT) cnt.nodes++;
            float x0 = (n0.x - r.ox) * r.ix, x1 = (n0.y - r.ox) * r.ix;
            float y0 = (n0.z - r.oy) * r.iy, y1 = (n0.w - r.oy) * r.iy;
            float z0 = (n2.x - r.oz) * r.iz, z1 = (n2.y - r.oz) * r.iz;
            const float l0 = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
            const float f0 = fminf(fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1)) * NGI_SLAB_SCALE, tmax);
            x0 = (n1.x - r.ox) * r.ix, x1 = (n1.y - r.ox) * r.ix;
            y0 = (n1.z - r.oy) * r.iy, y1 = (n1.w - r.oy) * r.iy;
            z0 = (n2.z - r.oz) * r.iz, z1 = (n2.w - r.oz) * r.iz;
            const float l1 = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
            const float f1 = fminf(fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1)) * NGI_SLAB_SCALE, tmax);
            const bool hit0 = l0 <= f0;
            const bool hit1 = l1 <= f1;
            const int32_t ch0 = __float_as_int(n3.x), ch1 = __float_as_int(n3.y);
            if (hit0 && hit1) {
                int32_t near = ch0, far = ch1;
                if (l1 < l0) {
                    near = ch1;
                    far = ch0;
                }
                stack[sp++] = far;
                node = near;
            } else if (hit0) {
                node = ch0;
            } else if (hit1) {
                node = ch1;
            } else {
                if (sp == 0) break;
                node = stack[--sp];
            }
        } else {
            leaf_test_pairs<ANY, COUNT>(sc, r, node, tmin, tmax, h, cnt, done);
            if (ANY && done) return true;
            if (sp == 0) break;
            node = stack[--sp];
        }
    }
    return h.leaf >= 0;
}

// ---------------------------------------------------------------------------
// 8-wide BVH.  Child slots are assigned at build time by the octant of the
// child's centroid relative to the parent's; a ray visits hit children in
// slot order XOR its direction octant (near-to-far along each axis).
// The stack holds one entry per tree level: (node << 8) | pending mask.
// Stack entries live in LDS, one column per lane (conflict-free).
// ---------------------------------------------------------------------------
#define NGI_BVH8_STACK 32

__device__ __forceinline__ float exp2_bits(uint32_t biased) { return __uint_as_float(biased << 23); }

// Box test of the eight children of the node fetched into f: a mask of the hit children in
// processing order (bit i = slot i ^ octant).
//
// The near and far planes of every child are chosen once per node from the
// sign of the inverse direction (for 1/d >= 0 the low bound is near): with
// t(q) = fma(q, a, b) and a >= 0, q_lo <= q_hi gives t(q_lo) <= t(q_hi)
// because rounding is monotone, so this equals min/max of the two planes
// bit for bit.  Every child's sign bit of far - near is shifted into a miss
// mask, slot 7 first: a subtraction and a shift instead of a compare, a
// select and a share of the ors (208 -> 201 VALU instructions per visit).
// The far plane is scaled by a multiply-add of +0, which makes a far plane of
// -0 a +0: a ray that starts on a corner of the box (far -0 along one axis,
// near +0 along another) enters it, as 0 <= 0 says, although -0 - 0 is -0.
// The mask is inverted and limited to the valid slots once, and permuted to
// processing order at the end.  Which of two coincident surfaces is hit hangs
// on the rounding of near against tmax, so near and tmax stay as they are.
template <bool COUNT>
__device__ __forceinline__ uint32_t visit8(const Fetch& f, const RayPre& r, float tmin, float tmax, TraceCounters& cnt) {
    const float4 h0 = __builtin_bit_cast(float4, f.w[0]);
    const uint4 q0 = __builtin_bit_cast(uint4, f.w[1]);  // qlox[8], qloy[8]
    const uint4 q1 = __builtin_bit_cast(uint4, f.w[2]);  // qloz[8], qhix[8]
    const uint4 q2 = __builtin_bit_cast(uint4, f.w[3]);  // qhiy[8], qhiz[8]
    if (COUNT) cnt.nodes++;
    const uint32_t meta = __float_as_uint(h0.w);
    const float scx = exp2_bits(meta & 0xffu), scy = exp2_bits((meta >> 8) & 0xffu), scz = exp2_bits((meta >> 16) & 0xffu);
    // t(q) = (origin + q * scale - o) * invd = q * (scale * invd) + (origin - o) * invd
    const float ax = scx * r.ix, bx = (h0.x - r.ox) * r.ix;
    const float ay = scy * r.iy, by = (h0.y - r.oy) * r.iy;
    const float az = scz * r.iz, bz = (h0.z - r.oz) * r.iz;
    const bool fx = r.ix < 0.0f, fy = r.iy < 0.0f, fz = r.iz < 0.0f;
    // Near / far plane words for children 0-3 (.x) and 4-7 (.y).
    const uint2 nx = fx ? make_uint2(q1.z, q1.w) : make_uint2(q0.x, q0.y), ex = fx ? make_uint2(q0.x, q0.y) : make_uint2(q1.z, q1.w);
    const uint2 ny = fy ? make_uint2(q2.x, q2.y) : make_uint2(q0.z, q0.w), ey = fy ? make_uint2(q0.z, q0.w) : make_uint2(q2.x, q2.y);
    const uint2 nz = fz ? make_uint2(q2.z, q2.w) : make_uint2(q1.x, q1.y), ez = fz ? make_uint2(q1.x, q1.y) : make_uint2(q2.z, q2.w);
    uint32_t miss = 0;
#pragma unroll
    for (int k = 7; k >= 0; --k) {
        const int sh = (k & 3) * 8;
        const uint32_t wnx = k < 4 ? nx.x : nx.y, wny = k < 4 ? ny.x : ny.y, wnz = k < 4 ? nz.x : nz.y;
        const uint32_t wex = k < 4 ? ex.x : ex.y, wey = k < 4 ? ey.x : ey.y, wez = k < 4 ? ez.x : ez.y;
        const float tnx = fmaf((float)((wnx >> sh) & 0xffu), ax, bx), tfx = fmaf((float)((wex >> sh) & 0xffu), ax, bx);
        const float tny = fmaf((float)((wny >> sh) & 0xffu), ay, by), tfy = fmaf((float)((wey >> sh) & 0xffu), ay, by);
        const float tnz = fmaf((float)((wnz >> sh) & 0xffu), az, bz), tfz = fmaf((float)((wez >> sh) & 0xffu), az, bz);
        const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, tmin));
        const float tf = fminf(fmaf(fminf(fminf(tfx, tfy), tfz), NGI_SLAB_SCALE, 0.0f), tmax);
        miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(tf - tn), 31);
    }
    uint32_t hits = ~miss & (meta >> 24);   // valid slots
    // Slot order -> processing order: swap bit groups selected by the octant.
    const uint32_t o = r.octant;
    if (o & 1u) hits = ((hits & 0x55u) << 1) | ((hits >> 1) & 0x55u);
    if (o & 2u) hits = ((hits & 0x33u) << 2) | ((hits >> 2) & 0x33u);
    if (o & 4u) hits = ((hits & 0x0fu) << 4) | ((hits >> 4) & 0x0fu);
    return hits;
}

// The child of node `cur` that a ray visits next: the lowest bit of its mask
// of pending children.
__device__ __forceinline__ int32_t next_child(const DevScene& sc, const RayPre& r, uint32_t cur, uint32_t mask) {
    const uint32_t slot = (uint32_t)__builtin_ctz(mask) ^ r.octant;
    return reinterpret_cast<const int32_t*>(sc.nodes + 8 * (size_t)cur + 4)[slot];
}

template <bool ANY, bool COUNT>
__device__ bool trace_bvh8(const DevScene& sc, const TraceRay& ray, TraceHit& h, TraceCounters& cnt, uint32_t* lds_stack,
                           int lane_stride) {
    const RayPre r = make_pre(ray);
    const float tmin = ray.tmin;
    float tmax = ray.tmax;
    h.leaf = -1;
    int sp = 0;
    uint32_t cur = 0, mask = 0;
    int32_t ref = 0;   // the root
    for (;;) {
        const Fetch f = fetch_child(sc, ref);
        if (ref < 0) {
            if (leaf_test<ANY, COUNT>(sc, r, ref, f, tmin, tmax, h, cnt) && ANY) return true;
        } else {
            if (mask) lds_stack[(sp++) * lane_stride] = (cur << 8) | mask;
            cur = (uint32_t)ref;
            mask = visit8<COUNT>(f, r, tmin, tmax, cnt);
        }
        if (mask == 0) {
            if (sp == 0) break;
            const uint32_t e = lds_stack[(--sp) * lane_stride];
            cur = e >> 8;
            mask = e & 0xffu;
        }
        ref = next_child(sc, r, cur, mask);
        mask &= mask - 1u;
    }
    return h.leaf >= 0;
}

// Resumable closest-hit traversal of the wide BVH: the same visiting order
// and tests as trace_bvh8<false>, with the state kept by the caller so that a
// wavefront can stop traversing while some of its lanes are still inside the
// tree and resume them later (their stacks stay in LDS meanwhile).  The hit
// distance doubles as the interval's upper end: h.t starts at tmax.
struct Trav8 {
    uint32_t cur, mask;
    int sp;
    TraceHit h;
};

// Mask of a traversal about to visit the root (visited by the first
// iteration of trav8_run, with the other lanes' next nodes); clearing its
// lowest bit leaves the empty mask.
#define NGI_TRAV8_FRESH 0x100u
__device__ __forceinline__ void trav8_begin(float tmax, Trav8& t) {
    t.h.t = tmax;
    t.h.u = t.h.v = 0.0f;
    t.h.leaf = -1;
    t.sp = 0;
    t.cur = 0;
    t.mask = NGI_TRAV8_FRESH;
}

// Advances the traversals of the lanes with `busy` set, one node visit or
// leaf per lane and iteration, until at most `keep` lanes of the wavefront
// are still busy (at least one iteration; keep = 0 finishes them all).  A
// busy lane always has a pending child (the lowest bit of its mask, or the
// root); it clears `busy` when its traversal ends, and t.h then holds its
// closest hit or t.h.leaf = -1.
//
// An iteration visits the inner lanes' nodes, lets every lane choose its next
// child (a leaf's outcome does not change which comes next) and sends out the
// loads of the next references before it tests the leaf lanes' triangles, so
// that those tests hide them.  With forget_vertex, measured ms before ->
// after: ptdirect on the nave 84.9 -> 79.0, 16.8M paths on the sphere field
// 8.43 -> 7.96, 7.4M with FP64 shading 4.95 -> 4.39, ltdirect on the nave
// 10.20 -> 9.27, adjoint replay 15.6 -> 14.9.  (Fetching the next children
// too before a leaf's second triangle needs 24 registers more: 8.88.)
// With MIXED, the lanes with `any` set stop at their first hit (t.h.leaf tells
// whether there is one).
template <bool COUNT, bool MIXED = false>
__device__ __forceinline__ void trav8_run(const DevScene& sc, const RayPre& r, float tmin, Trav8& t, bool& busy, int keep,
                                          TraceCounters& cnt, uint32_t* lds_stack, int lane_stride, bool any = false) {
    int32_t ref = 0;
    if (busy && t.mask != NGI_TRAV8_FRESH) ref = next_child(sc, r, t.cur, t.mask);
    do {
        const bool leaf = busy && ref < 0;
        const int32_t lref = ref;
        bool more = busy;
        Fetch f;
        if (busy) {
            t.mask &= t.mask - 1u;   // a fresh traversal's mask: 0
            f = fetch_child(sc, ref);
            if (!leaf) {
                if (t.mask) lds_stack[(t.sp++) * lane_stride] = (t.cur << 8) | t.mask;
                t.cur = (uint32_t)ref;
                t.mask = visit8<COUNT>(f, r, tmin, t.h.t, cnt);
            }
            if (t.mask == 0) {
                if (t.sp == 0) {
                    more = false;
                } else {
                    const uint32_t e = lds_stack[(--t.sp) * lane_stride];
                    t.cur = e >> 8;
                    t.mask = e & 0xffu;
                }
            }
            if (more) ref = next_child(sc, r, t.cur, t.mask);
        }
        if (leaf) {
            (void)leaf_test<false, COUNT>(sc, r, lref, f, tmin, t.h.t, t.h, cnt);
            if (MIXED && any && t.h.leaf >= 0) more = false;
        }
        busy = more;
    } while (__popcll(__ballot(busy)) > (unsigned)keep);
}

}  // namespace ngi
