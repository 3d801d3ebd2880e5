// Device scene upload and the ray-query entry points (ngi_trace*).
//
// The upload replaces the Embree buffers of the reference (FP32 de-indexed
// triangle soup, include/nanogi/rt.hpp:2110-2135) with leaf-ordered FP32
// triangle records plus a parallel shading record per triangle (vertex
// normals and owning primitive, used to rebuild the FP64 surface of
// Scene::Intersect, rt.hpp:2197-2233, in the shade stage).
#include <cmath>
#include <cstring>

#include "ngi_dev.h"
#include "ngi_guide.h"
#include "ngi_mem.h"
#include "ngi_traverse.h"

namespace ngi {

// Fewest triangles for trace_refill_kernel.
#define NGI_TRACE_MIN_TRIS 256

static int device_ready() {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(NGI_ERR_DEVICE, "no HIP device available");
    NGI_HIP_CHECK(hipSetDevice(0));
    return NGI_OK;
}

template <typename T>
static int upload(DeviceScene& d, const T* host, size_t count, const T** out) {
    *out = nullptr;
    if (count == 0) return NGI_OK;
    void* p = nullptr;
    NGI_HIP_CHECK(device_malloc(&p, count * sizeof(T)));
    d.allocs.push_back(p);
    NGI_HIP_CHECK(hipMemcpy(p, host, count * sizeof(T), hipMemcpyHostToDevice));
    *out = reinterpret_cast<const T*>(p);
    return NGI_OK;
}

template <typename T>
static void fill_prim(const ngi_primitive& p, int light, DevPrim<T>& o) {
    memset(&o, 0, sizeof(o));
    o.type = p.type;
    o.light = light;
    o.spec_type = p.spec_type;
    for (int k = 0; k < 3; ++k) {
        o.R[k] = (T)((p.type & NGI_PRIM_D) ? p.D_R[k] : (p.type & NGI_PRIM_G) ? p.G_R[k] : p.S_R[k]);
        o.eta[k] = (T)p.G_eta[k];
        o.k[k] = (T)p.G_k[k];
        o.Le[k] = (T)p.Le[k];
    }
    o.roughness = (T)p.G_roughness;
    o.s_eta1 = (T)p.S_eta1;
    o.s_eta2 = (T)p.S_eta2;
}

// Guide bits of an area light's triangle CDF (FP64; its FP32 rounding is
// sorted and NaN-free whenever the FP64 CDF is).
static uint32_t light_guide_bits(const std::vector<double>& cdf) {
    const uint32_t m = (uint32_t)cdf.size();
    return m >= 2 && guide_sorted(cdf.data(), m) ? guide_bits(m - 1) : 0u;
}

// Wait for every kernel that may read the scene's device arrays: the
// scene's stream and the streams of the batches holding it.
static int wait_users(HostScene& s) {
    if (s.dev && s.dev->stream) NGI_HIP_CHECK(hipStreamSynchronize(s.dev->stream));
    for (void* u : s.user_streams) NGI_HIP_CHECK(hipStreamSynchronize(reinterpret_cast<hipStream_t>(u)));
    return NGI_OK;
}

// (Re)build the parameter-dependent tables: primitives and lights.
static int upload_params(HostScene& s, DeviceScene& d) {
    const size_t np = s.prims.size();
    std::vector<int> light_of(np, -1);
    for (size_t i = 0; i < s.light_prims.size(); ++i) light_of[s.light_prims[i]] = (int)i;
    std::vector<DevPrim<float>> pf(np);
    std::vector<DevPrim<double>> pd(np);
    for (size_t i = 0; i < np; ++i) {
        fill_prim(s.prims[i], light_of[i], pf[i]);
        fill_prim(s.prims[i], light_of[i], pd[i]);
    }
    std::vector<DevLight<float>> lf(s.light_prims.size());
    std::vector<DevLight<double>> ld(s.light_prims.size());
    uint32_t tri_row = 0, cdf_row = 0, guide_row = 0;
    for (size_t i = 0; i < s.light_prims.size(); ++i) {
        const int pi = s.light_prims[i];
        const ngi_primitive& p = s.prims[pi];
        DevLight<double> L;
        memset(&L, 0, sizeof(L));
        L.prim = pi;
        L.type = p.light_type;
        for (int k = 0; k < 3; ++k) L.Le[k] = p.Le[k], L.pos[k] = p.light_position[k];
        if (p.light_type == NGI_LIGHT_DIRECTIONAL) {
            for (int k = 0; k < 3; ++k) L.pos[k] = s.dir_center[3 * (size_t)pi + k], L.dir[k] = p.light_direction[k];
            L.radius = s.dir_radius[pi];
            L.inv_area = s.dir_inv_area[pi];
        }
        if (p.light_type == NGI_LIGHT_AREA) {
            L.tri_begin = tri_row;
            L.tri_count = p.tri_count;
            L.cdf_begin = cdf_row;
            L.guide_begin = guide_row;
            L.guide_bits = light_guide_bits(s.area_dist[pi].cdf);
            L.inv_area = s.area_dist[pi].inv_area;
            tri_row += p.tri_count;
            cdf_row += p.tri_count + 1;
            guide_row += (1u << L.guide_bits) + 1u;
        }
        ld[i] = L;
        DevLight<float>& F = lf[i];
        F.prim = L.prim, F.type = L.type, F.tri_begin = L.tri_begin, F.tri_count = L.tri_count, F.cdf_begin = L.cdf_begin;
        F.guide_begin = L.guide_begin, F.guide_bits = L.guide_bits, F.pad = 0;
        F.inv_area = (float)L.inv_area;
        for (int k = 0; k < 3; ++k) F.Le[k] = (float)L.Le[k], F.pos[k] = (float)L.pos[k], F.dir[k] = (float)L.dir[k];
        F.radius = (float)L.radius;
    }
    if (!d.prim_f_mem) {
        NGI_HIP_CHECK(device_malloc(&d.prim_f_mem, std::max<size_t>(np, 1) * sizeof(DevPrim<float>)));
        NGI_HIP_CHECK(device_malloc(&d.prim_d_mem, std::max<size_t>(np, 1) * sizeof(DevPrim<double>)));
        NGI_HIP_CHECK(device_malloc(&d.light_f_mem, std::max<size_t>(lf.size(), 1) * sizeof(DevLight<float>)));
        NGI_HIP_CHECK(device_malloc(&d.light_d_mem, std::max<size_t>(ld.size(), 1) * sizeof(DevLight<double>)));
        d.allocs.insert(d.allocs.end(), {d.prim_f_mem, d.prim_d_mem, d.light_f_mem, d.light_d_mem});
    }
    int st = wait_users(s);   // a running frame must not see a half-updated table
    if (st) return st;
    if (np) {
        NGI_HIP_CHECK(hipMemcpy(d.prim_f_mem, pf.data(), np * sizeof(pf[0]), hipMemcpyHostToDevice));
        NGI_HIP_CHECK(hipMemcpy(d.prim_d_mem, pd.data(), np * sizeof(pd[0]), hipMemcpyHostToDevice));
    }
    if (!lf.empty()) {
        NGI_HIP_CHECK(hipMemcpy(d.light_f_mem, lf.data(), lf.size() * sizeof(lf[0]), hipMemcpyHostToDevice));
        NGI_HIP_CHECK(hipMemcpy(d.light_d_mem, ld.data(), ld.size() * sizeof(ld[0]), hipMemcpyHostToDevice));
    }
    d.view.prims_f = reinterpret_cast<const DevPrim<float>*>(d.prim_f_mem);
    d.view.prims_d = reinterpret_cast<const DevPrim<double>*>(d.prim_d_mem);
    d.view.lights_f = reinterpret_cast<const DevLight<float>*>(d.light_f_mem);
    d.view.lights_d = reinterpret_cast<const DevLight<double>*>(d.light_d_mem);
    d.view.num_lights = (int)s.light_prims.size();
    d.view.any_glossy = 0;
    for (const ngi_primitive& p : s.prims)
        if (p.type & (NGI_PRIM_G | NGI_PRIM_S)) d.view.any_glossy = 1;
    d.params_version = s.params_version;
    return NGI_OK;
}

int device_prepare(HostScene& s) {
    int st = device_ready();
    if (st) return st;
    if (!s.built) {
        ngi_bvh_opts o;
        memset(&o, 0, sizeof(o));
        st = bvh_build(s, o, s.bvh);
        if (st) return st;
        s.built = true;
    }
    if (s.dev) {
        if (s.dev->params_version != s.params_version) return upload_params(s, *s.dev);
        return NGI_OK;
    }
    DeviceScene* d = new DeviceScene();
    s.dev = d;
    resident_scenes(+1);
    int dev = 0;
    NGI_HIP_CHECK(hipGetDevice(&dev));
    NGI_HIP_CHECK(hipDeviceGetAttribute(&d->cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
        d->stream = nullptr;
        return fail(NGI_ERR_DEVICE, "hipStreamCreate failed");
    }
    const size_t nt = s.faces.size() / 3;
    DevScene& v = d->view;
    v.bvh_width = s.bvh.width;
    v.stack_entries = s.bvh.width == 8 ? s.bvh.max_depth + 1 : 0;
    v.num_tris = (uint32_t)nt;
    v.sensor_prim = s.sensor_prim;
    // Geometry in leaf order.
    std::vector<float4> tris(3 * nt + (nt ? 1 : 0)), shade(3 * nt);   // fetch_child reads a float4 past the last triangle
    for (size_t j = 0; j < nt; ++j) {
        const uint32_t t = s.bvh.leaf_to_tri[j];
        for (int k = 0; k < 3; ++k) {
            const uint32_t vi = s.faces[3 * (size_t)t + k];
            float w = 0.0f, wn = 0.0f;
            if (k == 0) {
                uint32_t bits = t, pbits = s.tri_prim[t];
                memcpy(&w, &bits, 4);
                memcpy(&wn, &pbits, 4);
            } else if (k == 1) {
                const uint32_t tbits = (uint32_t)s.prims[s.tri_prim[t]].type;   // fixed by the scene (set_params keeps it)
                memcpy(&wn, &tbits, 4);
            }
            tris[3 * j + k] = make_float4((float)s.positions[3 * (size_t)vi], (float)s.positions[3 * (size_t)vi + 1],
                                          (float)s.positions[3 * (size_t)vi + 2], w);
            shade[3 * j + k] = make_float4((float)s.normals[3 * (size_t)vi], (float)s.normals[3 * (size_t)vi + 1],
                                           (float)s.normals[3 * (size_t)vi + 2], wn);
        }
    }
    if ((st = upload(*d, tris.data(), tris.size(), &v.tris))) return st;
    if ((st = upload(*d, shade.data(), shade.size(), &v.shade))) return st;
    const float4* nodes = nullptr;
    if ((st = upload(*d, reinterpret_cast<const float4*>(s.bvh.nodes.data()), s.bvh.nodes.size() / 16, &nodes))) return st;
    v.nodes = nodes;
    if (nt >= NGI_TRACE_MIN_TRIS) {
        NGI_HIP_CHECK(device_malloc(&d->scattered, sizeof(uint32_t)));
        d->allocs.push_back(d->scattered);
    }
    // Area-light triangles and CDFs, per light primitive.
    std::vector<float4> ltris;
    std::vector<float> cf;
    std::vector<double> cd;
    std::vector<uint32_t> gf, gd;
    for (int pi : s.light_prims) {
        const ngi_primitive& p = s.prims[pi];
        if (p.light_type != NGI_LIGHT_AREA) continue;
        for (uint32_t t = p.tri_begin; t < p.tri_begin + p.tri_count; ++t)
            for (int k = 0; k < 3; ++k) {
                const uint32_t vi = s.faces[3 * (size_t)t + k];
                ltris.push_back(make_float4((float)s.positions[3 * (size_t)vi], (float)s.positions[3 * (size_t)vi + 1],
                                            (float)s.positions[3 * (size_t)vi + 2], 0.0f));
            }
        const std::vector<double>& c = s.area_dist[pi].cdf;
        const size_t f0 = cf.size();
        for (double x : c) {
            cd.push_back(x);
            cf.push_back((float)x);
        }
        // The guides follow upload_params' order and light_guide_bits.
        const uint32_t bits = light_guide_bits(c), g0 = (uint32_t)gf.size();
        gf.resize(g0 + (1u << bits) + 1u);
        gd.resize(gf.size());
        guide_build(cf.data() + f0, (uint32_t)c.size(), bits, gf.data() + g0);
        guide_build(c.data(), (uint32_t)c.size(), bits, gd.data() + g0);
    }
    if ((st = upload(*d, ltris.data(), ltris.size(), &v.light_tris))) return st;
    if ((st = upload(*d, cf.data(), cf.size(), &v.cdf_f))) return st;
    if ((st = upload(*d, cd.data(), cd.size(), &v.cdf_d))) return st;
    if ((st = upload(*d, gf.data(), gf.size(), &v.guide_f))) return st;
    if ((st = upload(*d, gd.data(), gd.size(), &v.guide_d))) return st;
    // Pinhole camera (rt.hpp:1882-1902).
    memset(&v.cam, 0, sizeof(v.cam));
    if (s.sensor_prim >= 0 && s.prims[s.sensor_prim].sensor_type == NGI_SENSOR_PINHOLE) {
        const ngi_primitive& p = s.prims[s.sensor_prim];
        d3 eye(p.E_eye[0], p.E_eye[1], p.E_eye[2]), ctr(p.E_center[0], p.E_center[1], p.E_center[2]), up(p.E_up[0], p.E_up[1], p.E_up[2]);
        d3 vz = normalize(eye - ctr);
        d3 vx = normalize(cross(up, vz));
        d3 vy = cross(vz, vx);
        for (int k = 0; k < 3; ++k) v.cam.eye[k] = eye[k], v.cam.vx[k] = vx[k], v.cam.vy[k] = vy[k], v.cam.vz[k] = vz[k];
        v.cam.tan_fov = std::tan(p.E_fov_deg * M_PI / 180.0 * 0.5);
        v.cam.aspect = s.aspect;
    }
    return upload_params(s, *d);
}

void device_release(HostScene& s) {
    if (!s.dev) return;
    (void)wait_users(s);
    DeviceScene* d = s.dev;
    if (d->stream) {
        (void)hipStreamSynchronize(d->stream);
        (void)hipStreamDestroy(d->stream);
    }
    for (void* p : d->allocs) (void)hipFree(p);
    if (d->stage) (void)hipFree(d->stage);
    delete d;
    s.dev = nullptr;
    resident_scenes(-1);
}

int ensure_stage(DeviceScene& d, size_t bytes) {
    if (d.stage_bytes >= bytes) return NGI_OK;
    if (d.stage) {
        NGI_HIP_CHECK(hipStreamSynchronize(d.stream));
        NGI_HIP_CHECK(hipFree(d.stage));
        d.stage = nullptr;
        d.stage_bytes = 0;
    }
    NGI_HIP_CHECK(device_malloc(&d.stage, bytes));
    d.stage_bytes = bytes;
    return NGI_OK;
}

// ---------------------------------------------------------------------------
// Ray-query kernel: one lane per ray, rays and hits in the public layout.
// ---------------------------------------------------------------------------
#define NGI_TRACE_BLOCK 256
// Host queries whose rays and hits fit a pinned block (1,365 of them) are traced
// in mapped host memory; hits of at most NGI_TRACE_DIRECT_BYTES are copied back
// by the runtime, more through the pinned ring.
#define NGI_TRACE_DIRECT_BYTES ((size_t)3 << 19)

// LARGE: leaves the call to trace_refill_kernel where *scattered says so (a
// variant of its own: looking at a pointer cost a small call 0.3 of its 5.5 us).
template <int WIDTH, bool ANY, bool LARGE>
__global__ void __launch_bounds__(NGI_TRACE_BLOCK) trace_kernel(DevScene sc, const ngi_ray* __restrict__ rays, size_t n,
                                                                ngi_hit* __restrict__ hits, const uint32_t* __restrict__ scattered) {
    extern __shared__ uint32_t stk[];   // sc.stack_entries x block (wide BVH only)
    const size_t i = (size_t)blockIdx.x * NGI_TRACE_BLOCK + threadIdx.x;
    if (i >= n || (LARGE && *scattered)) return;
    const ngi_ray r = rays[i];
    TraceRay tr{r.o[0], r.o[1], r.o[2], r.d[0], r.d[1], r.d[2], r.tmin, r.tmax};
    TraceHit h;
    TraceCounters c{0, 0};
    bool hit;
    if (WIDTH == 8) hit = trace_bvh8<ANY, false>(sc, tr, h, c, stk + threadIdx.x, NGI_TRACE_BLOCK);
    else hit = trace_bvh2<ANY, false>(sc, tr, h, c);
    ngi_hit o;
    if (!hit) {
        o.t = r.tmax, o.u = 0.0f, o.v = 0.0f, o.tri = NGI_MISS;
    } else {
        o.t = h.t, o.u = h.u, o.v = h.v;
        o.tri = __float_as_uint(sc.tris[3 * (size_t)h.leaf].w);
    }
    hits[i] = o;
}

// Many scattered rays over the wide BVH (rays_scattered; the others are left to
// trace_kernel, launched behind it): every wavefront takes `per_wave`
// consecutive rays, and lanes whose rays have finished take the next ones as
// soon as NGI_TRACE_REFILL of them are idle, so a wavefront waits for its
// slowest ray once instead of after every 64 (one ray per lane left 11 of 64
// lanes active per VALU instruction).  Visits, tests and results are those of
// trace_bvh8; an iteration is as in trav8_run, but that the compiler waits for
// the next reference before the leaf tests, which do not hide it.  Bound by the
// latency of the traversal's loads and by instruction issue.  Measured, us, one
// ray per lane -> refills (1.5M / 6M random rays; closest hit): sphere field with
// 1.8M triangles 355 -> 314 / 1,070 -> 728, nave 296 -> 252 / 984 -> 809, a room
// of 4,000 triangles 215 -> 154 / 705 -> 432; any hit 1,064 -> 706 on 6M of the
// field's.  Refills of 8 or 24: the same within 3%.
#define NGI_TRACE_REFILL 16
// Blocks per CU: 2 / 3 / 4 / 5 / 6 took 1,068 / 888 / 787 / 728 / 740 us for
// the field's 6M rays and 409 / 337 / 342 / 314 / 325 for 1.5M.
#define NGI_TRACE_WAVES 5
// From four rays per lane and 256 triangles on.  With fewer rays a wavefront's
// last ones take as long as all of them do (660,000 scattered rays, one ray per
// lane / refills, us: nave 163 / 153, its any hit 132 / 125, field 225 / 228),
// and the rays of a wavefront hardly part among a few triangles (6M, Cornell
// box 293 / 290, its any hit 221 / 233; 1.4M, rooms of 40 / 100 / 300 triangles
// 56 / 59, 61 / 64, 130 / 101).
#define NGI_TRACE_RAYS_PER_LANE 4

// Whether the rays of a large call are scattered: at fewer than a quarter of 64
// places are a ray and those 1 and 8 places on neighbours (origins within a
// sixteenth of the scene's extent, directions within 25 degrees).  Rays in
// order, a camera's or the shadow rays of its hits, finish together and hold
// the same nodes; refills would mix them with new rays at the root and leave
// the device to a few long wavefronts at the end.  4.2M camera rays, one ray per
// lane / refills, us: field 470 / 740, nave 420 / 655, room of 4,000 triangles
// 163 / 270; refills only when a wavefront is empty, and ranges handed out
// round robin, in pieces of 256 rays by blocks or as the rays before turned
// out, kept at 0.5 to 1.0 of the former.  Deciding costs a call 3 us (this, and
// the blocks of the kernel that is not meant).  All lanes of a wavefront call
// this, and every wavefront finds the same.
__device__ __forceinline__ bool rays_scattered(const DevScene& sc, const ngi_ray* __restrict__ rays, size_t n) {
    // Places that follow no row length of an image (multiples of the golden ratio).
    const size_t i = (size_t)__umul64hi((uint64_t)__lane_id() * 0x9e3779b97f4a7c15ull, (uint64_t)(n - 8));
    const ngi_ray a = rays[i];
    const uint32_t meta = __float_as_uint(sc.nodes[0].w);
    const float ext = 255.0f * fmaxf(fmaxf(exp2_bits(meta & 0xffu), exp2_bits((meta >> 8) & 0xffu)), exp2_bits((meta >> 16) & 0xffu));
    bool near = true;
    for (int k = 1; k <= 8; k += 7) {
        const ngi_ray b = rays[i + k];
        const float o = fmaxf(fmaxf(fabsf(a.o[0] - b.o[0]), fabsf(a.o[1] - b.o[1])), fabsf(a.o[2] - b.o[2]));
        const float ab = a.d[0] * b.d[0] + a.d[1] * b.d[1] + a.d[2] * b.d[2];
        const float aa = a.d[0] * a.d[0] + a.d[1] * a.d[1] + a.d[2] * a.d[2], bb = b.d[0] * b.d[0] + b.d[1] * b.d[1] + b.d[2] * b.d[2];
        near = near && o <= ext * 0.0625f && ab > 0.0f && ab * ab > 0.82f * aa * bb;
    }
    return __popcll(__ballot(near)) < 16;
}

template <bool ANY>
__global__ void __launch_bounds__(NGI_TRACE_BLOCK, NGI_TRACE_WAVES) trace_refill_kernel(DevScene sc, const ngi_ray* __restrict__ rays, size_t n,
                                                                                        ngi_hit* __restrict__ hits, size_t per_wave,
                                                                                        uint32_t* __restrict__ scattered) {
    extern __shared__ uint32_t stk[];   // sc.stack_entries x block
    const bool mine = rays_scattered(sc, rays, n);
    if (blockIdx.x == 0 && threadIdx.x == 0) *scattered = mine ? 1u : 0u;
    if (!mine) return;
    uint32_t* lds_stack = stk + threadIdx.x;
    const uint32_t lane = __lane_id();
    const size_t wave = (size_t)blockIdx.x * (NGI_TRACE_BLOCK / 64) + (threadIdx.x >> 6);
    size_t next = wave * per_wave;   // wave-uniform; past n in the last wavefronts
    const size_t end = next + per_wave < n ? next + per_wave : n;
    bool busy = false;
    size_t id = 0;
    RayPre r;
    float tmin = 0.0f;
    Trav8 t;
    int32_t ref = 0;
    TraceCounters c{0, 0};
    for (;;) {
        const unsigned long long idle = __ballot(!busy);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (next < end && (nidle >= NGI_TRACE_REFILL || nidle == 64u)) {
            const size_t rank = (size_t)__popcll(idle & ((1ull << lane) - 1ull));
            if (!busy && next + rank < end) {
                id = next + rank;
                const ngi_ray q = rays[id];
                r = make_pre(TraceRay{q.o[0], q.o[1], q.o[2], q.d[0], q.d[1], q.d[2], q.tmin, q.tmax});
                tmin = q.tmin;
                trav8_begin(q.tmax, t);
                t.mask = 0;
                ref = 0;
                busy = true;
            }
            next += nidle;
        }
        if (__ballot(busy) == 0) break;
        const bool leaf = busy && ref < 0;
        const int32_t lref = ref;
        bool more = busy;
        Fetch f;
        if (busy) {
            f = fetch_child(sc, ref);
            if (!leaf) {
                if (t.mask) lds_stack[(t.sp++) * NGI_TRACE_BLOCK] = (t.cur << 8) | t.mask;
                t.cur = (uint32_t)ref;
                t.mask = visit8<false>(f, r, tmin, t.h.t, c);
            }
            if (t.mask == 0) {
                if (t.sp == 0) {
                    more = false;
                } else {
                    const uint32_t e = lds_stack[(--t.sp) * NGI_TRACE_BLOCK];
                    t.cur = e >> 8;
                    t.mask = e & 0xffu;
                }
            }
            if (more) {
                ref = next_child(sc, r, t.cur, t.mask);
                t.mask &= t.mask - 1u;
            }
        }
        if (leaf && leaf_test<ANY, false>(sc, r, lref, f, tmin, t.h.t, t.h, c) && ANY) more = false;
        if (busy && !more) {
            ngi_hit o;
            o.t = t.h.t, o.u = t.h.u, o.v = t.h.v;
            o.tri = t.h.leaf < 0 ? NGI_MISS : __float_as_uint(sc.tris[3 * (size_t)t.h.leaf].w);
            hits[id] = o;
        }
        busy = more;
    }
}

int launch_trace(HostScene& s, const ngi_ray* d_rays, size_t n, ngi_hit* d_hits, int any_hit) {
    DeviceScene& d = *s.dev;
    if (n == 0) return NGI_OK;
    if (d.view.num_tris == 0) {
        // No geometry: every query misses (fill on the device).
        std::vector<ngi_hit> miss(n);
        for (size_t i = 0; i < n; ++i) miss[i] = ngi_hit{0.0f, 0.0f, 0.0f, NGI_MISS};
        NGI_HIP_CHECK(hipMemcpyAsync(d_hits, miss.data(), n * sizeof(ngi_hit), hipMemcpyHostToDevice, d.stream));
        NGI_HIP_CHECK(hipStreamSynchronize(d.stream));
        return NGI_OK;
    }
    const unsigned grid = (unsigned)((n + NGI_TRACE_BLOCK - 1) / NGI_TRACE_BLOCK);
    if (d.view.bvh_width == 8) {
        const size_t lds = (size_t)d.view.stack_entries * NGI_TRACE_BLOCK * 4;
        const size_t lanes = (size_t)d.cus * NGI_TRACE_WAVES * NGI_TRACE_BLOCK;
        const bool many = n >= lanes * NGI_TRACE_RAYS_PER_LANE && d.view.num_tris >= NGI_TRACE_MIN_TRIS;
        if (many) {
            const unsigned blocks = (unsigned)d.cus * NGI_TRACE_WAVES;
            const size_t per = (n + (size_t)blocks * (NGI_TRACE_BLOCK / 64) - 1) / ((size_t)blocks * (NGI_TRACE_BLOCK / 64));
            if (any_hit) trace_refill_kernel<true><<<blocks, NGI_TRACE_BLOCK, lds, d.stream>>>(d.view, d_rays, n, d_hits, per, d.scattered);
            else trace_refill_kernel<false><<<blocks, NGI_TRACE_BLOCK, lds, d.stream>>>(d.view, d_rays, n, d_hits, per, d.scattered);
        }
        auto kern = many ? (any_hit ? trace_kernel<8, true, true> : trace_kernel<8, false, true>)
                         : (any_hit ? trace_kernel<8, true, false> : trace_kernel<8, false, false>);
        kern<<<grid, NGI_TRACE_BLOCK, lds, d.stream>>>(d.view, d_rays, n, d_hits, d.scattered);
    } else {
        auto kern = any_hit ? trace_kernel<2, true, false> : trace_kernel<2, false, false>;
        kern<<<grid, NGI_TRACE_BLOCK, 0, d.stream>>>(d.view, d_rays, n, d_hits, nullptr);
    }
    NGI_HIP_CHECK(hipGetLastError());
    return NGI_OK;
}

}  // namespace ngi

using namespace ngi;

extern "C" {

int ngi_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int ngi_trace(ngi_scene* s, const ngi_ray* rays, size_t n, ngi_hit* hits, int any_hit) {
    clear_error();
    if (!s || (n && (!rays || !hits))) return fail(NGI_ERR_INVALID_ARG, "null argument");
    int st = device_prepare(*s);
    if (st) return st;
    if (n == 0) return NGI_OK;
    DeviceScene& d = *s->dev;
    const size_t rb = n * sizeof(ngi_ray), hb = n * sizeof(ngi_hit);
    // A few rays: the kernel reads them from, and writes their hits to, mapped
    // host memory (two transfers less; 64 rays 59 -> 46 us per call).
    if (rb + hb <= NGI_PIN_BLOCK_BYTES && d.view.num_tris) {
        PinnedBlock buf(rb + hb);
        if (buf.get()) {
            ngi_ray* hr = reinterpret_cast<ngi_ray*>(buf.get());
            ngi_hit* hh = reinterpret_cast<ngi_hit*>(hr + n);
            memcpy(hr, rays, rb);
            if ((st = launch_trace(*s, hr, n, hh, any_hit))) return st;
            NGI_HIP_CHECK(hipStreamSynchronize(d.stream));
            memcpy(hits, hh, hb);
            return NGI_OK;
        }
    }
    if ((st = ensure_stage(d, rb + hb))) return st;
    ngi_ray* dr = reinterpret_cast<ngi_ray*>(d.stage);
    ngi_hit* dh = reinterpret_cast<ngi_hit*>(reinterpret_cast<char*>(d.stage) + rb);
    NGI_HIP_CHECK(hipMemcpyAsync(dr, rays, rb, hipMemcpyHostToDevice, d.stream));
    if ((st = launch_trace(*s, dr, n, dh, any_hit))) return st;
    // Small hits come back faster by the runtime's own copy, which is enqueued
    // behind the kernel (70,000 rays in a 2k-triangle room 214 us, through the ring
    // 217; 100,000: 259, 257; 200,000: 487, 438; 700,000: 1,527, 1,300).  So it is
    // enqueued at once, too, where the ring is not to be had (after waiting 2 to
    // 12% slower).
    if (hb > NGI_TRACE_DIRECT_BYTES && pinned_free()) {
        NGI_HIP_CHECK(hipStreamSynchronize(d.stream));   // before the ring is taken
        st = read_pinned(d.stream, hits, hb, [&](size_t at, size_t bytes, void* dst) {
            NGI_HIP_CHECK(hipMemcpyAsync(dst, reinterpret_cast<const char*>(dh) + at, bytes, hipMemcpyDeviceToHost, d.stream));
            return (int)NGI_OK;
        });
        if (st != NGI_NOT_PINNED) return st;
    }
    NGI_HIP_CHECK(hipMemcpyAsync(hits, dh, hb, hipMemcpyDeviceToHost, d.stream));
    NGI_HIP_CHECK(hipStreamSynchronize(d.stream));
    return NGI_OK;
}

int ngi_trace_device(ngi_scene* s, const ngi_ray* d_rays, size_t n, ngi_hit* d_hits, int any_hit) {
    clear_error();
    if (!s || (n && (!d_rays || !d_hits))) return fail(NGI_ERR_INVALID_ARG, "null argument");
    int st = device_prepare(*s);
    if (st) return st;
    return launch_trace(*s, d_rays, n, d_hits, any_hit);
}

}  // extern "C"
