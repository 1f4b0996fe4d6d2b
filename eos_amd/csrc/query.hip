// query.hip -- ray queries: the reference Scene's per-ray queries
// (src/Scene.h:69-71) answered for many caller-given rays at once.
//
//   EOS_QUERY_NEAREST         Scene::findMinDistanceIntersectionBVH
//   EOS_QUERY_OCCLUDED        Scene::shadowRayVisibilityBVH
//   EOS_QUERY_NEAREST_LINEAR  Scene::findMinDistanceIntersectionLinear
//
// The BVH queries run the render path's persistent traversal (k_trace in the
// MODE_RAYS / MODE_RAYS_ANY modes, rays read straight from the caller's
// arrays), then one thread per ray turns the hit record into the reference's
// RayIntersection fields with the same arithmetic the frame's set-up kernel
// uses.  The linear query tests every triangle, split into chunks whose results
// combine in index order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "eos_internal.h"
#include "trace.h"

namespace eos {
namespace {

// eos_ray_hit as three float4: (point, hit) (normal, material) (t, u, v, triangle)
static_assert(sizeof(eos_ray_hit) == 48, "ray hit record is three 16-byte words");

__device__ __forceinline__ void write_hit(float4* out, size_t i, bool found, F3 P, F3 N, int mat, float t, float u,
                                          float v, int tri) {
    out[3 * i] = make_float4(P.x, P.y, P.z, __int_as_float(found ? 1 : 0));
    out[3 * i + 1] = make_float4(N.x, N.y, N.z, __int_as_float(mat));
    out[3 * i + 2] = make_float4(t, u, v, __int_as_float(tri));
}

// Nearest-hit records (t, slot, u, v) of the traversal -> RayIntersection fields
// (src/BVH.cpp:342-383: point through M, normal through transpose(inverse) and
// normalised; material index of the triangle).  No hit: zero point and normal
// as RayIntersection's constructor leaves them (src/RayIntersection.h:34).
__global__ __launch_bounds__(256) void k_query_hits(int n, const float* ro, const float* rd, const float4* rec,
                                                     const float4* shade, const float4* geo, const float4* xf,
                                                     float4* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 h = rec[i];
    const int slot = __float_as_int(h.y);
    F3 P = {0, 0, 0}, N = {0, 0, 0};
    if (slot < 0) {
        write_hit(out, (size_t)i, false, P, N, -1, INFINITY, 0.0f, 0.0f, -1);
        return;
    }
    const F3 o = f3(ro[3 * (size_t)i], ro[3 * (size_t)i + 1], ro[3 * (size_t)i + 2]);
    const F3 d = f3(rd[3 * (size_t)i], rd[3 * (size_t)i + 1], rd[3 * (size_t)i + 2]);
    const float4 s0 = shade[3 * (size_t)slot], s1 = shade[3 * (size_t)slot + 1], s2 = shade[3 * (size_t)slot + 2];
    hit_surface(s0, s1, s2, xf, o, d, h.x, h.z, h.w, true, P, N);
    write_hit(out, (size_t)i, true, P, N, __float_as_int(s0.w), h.x, h.z, h.w,
              __float_as_int(geo[3 * (size_t)slot + 2].y));
}

// src/Scene.cpp:159-201 in parallel.  The reference walks the triangles in index
// order with two running bounds: Triangle::hit's `distance` (minTemp: a hit
// farther than the last accepted one is rejected; the first hit is always
// accepted, the reading of its uninitialised start value) and minDist (999999
// at first): an accepted hit is kept when 0 < t < minDist.  found: some triangle
// accepted a hit (the query's return value), even when none was kept.
//   Until an accepted hit has t = 0, a hit beyond minTemp is beyond minDist too, so
// a hit is kept when 0 < t < minDist; after a hit at t = 0 nothing is kept.  A
// hit whose t is not a number (a NaN passes Moller-Trumbore's comparisons) is
// accepted, lifts minTemp and leaves minDist, so hits are kept again.  A run of
// consecutive triangles is summed up by the first least t in (0, 999999) among the
// hits that it keeps: `head` those before its first NaN hit, which count only if
// no t = 0 is open before the run, and `best` those after it (without a NaN hit all
// are in `best`); and by whether a t = 0 is open at its end.  Neighbouring runs
// combine in order.
struct LinHit {
    float t = 999999.0f, u = 0.0f, v = 0.0f;
    int tri = -1;
    __device__ __forceinline__ void then(const LinHit& o) {
        if (o.t < t) *this = o;
    }
    __device__ __forceinline__ float4 pack() const {
        return make_float4(t, u, v, __uint_as_float((uint32_t)(tri + 1)));
    }
    __device__ __forceinline__ static LinHit unpack(float4 p) {
        LinHit h;
        h.t = p.x;
        h.u = p.y;
        h.v = p.z;
        h.tri = (int)(__float_as_uint(p.w) & 0x1FFFFFFFu) - 1;
        return h;
    }
};
struct LinRun {
    LinHit best;
    bool found = false, zero = false, nan = false;
    __device__ __forceinline__ void hit(float t, float u, float v, int tri) {
        found = true;
        if (!zero && t < best.t && t > 0.0f) {
            best.t = t;
            best.u = u;
            best.v = v;
            best.tri = tri;
        }
        zero |= t <= 0.0f;
    }
    // 16 bytes in memory: t, u, v, then the triangle + 1 (at most 2^28) and the flags
    __device__ __forceinline__ float4 pack() const {
        const uint32_t w = (uint32_t)(best.tri + 1) | (found ? 1u << 29 : 0u) | (zero ? 1u << 30 : 0u) | (nan ? 1u << 31 : 0u);
        return make_float4(best.t, best.u, best.v, __uint_as_float(w));
    }
};
struct LinSum : LinRun {
    LinHit head;
    __device__ __forceinline__ void lift() {
        if (!nan) {
            head = best;
            best = LinHit();
            nan = true;
        }
        zero = false;
    }
    __device__ __forceinline__ void hit(float t, float u, float v, int tri) {
        if (t == t) {
            LinRun::hit(t, u, v, tri);
        } else {
            found = true;
            lift();
        }
    }
    // this run, then the one of the triangles after it
    __device__ __forceinline__ void then(const LinSum& o) {
        const LinHit& first = o.nan ? o.head : o.best;
        if (!zero) best.then(first);
        if (o.nan) {
            lift();
            best.then(o.best);
        }
        found |= o.found;
        zero |= o.zero;
    }
    // the kept hit of the run over all triangles
    __device__ __forceinline__ LinHit kept() const {
        LinHit k = nan ? head : best;
        if (nan) k.then(best);
        return k;
    }
    __device__ __forceinline__ static bool has_head(float4 p) { return (__float_as_uint(p.w) >> 31) != 0; }
    __device__ __forceinline__ static LinSum unpack(float4 p, float4 head) {
        const uint32_t w = __float_as_uint(p.w);
        LinSum r;
        r.best = LinHit::unpack(p);
        r.found = (w >> 29) & 1u;
        r.zero = (w >> 30) & 1u;
        r.nan = (w >> 31) & 1u;
        if (r.nan) r.head = LinHit::unpack(head);
        return r;
    }
    // the wave's runs combined in lane order, `lanes` (a power of two) at a time:
    // right in the first lane of each
    __device__ __forceinline__ void reduce(int lanes) {
        for (int off = 1; off < lanes; off <<= 1) {
            const float4 p = shfl_down4(pack(), off);
            float4 h = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (__ballot(nan) != 0) h = shfl_down4(head.pack(), off);
            then(unpack(p, h));
        }
    }
    __device__ __forceinline__ static float4 shfl_down4(float4 p, int off) {
        return make_float4(__shfl_down(p.x, off), __shfl_down(p.y, off), __shfl_down(p.z, off), __shfl_down(p.w, off));
    }
};

// The ray as triangle xi meets it: in the triangle's local space, kept while the
// transformation stays the same.
struct LinRay {
    F3 o, d, lo, ld;
    int lxi = -1;
    __device__ __forceinline__ void load(const float* ro, const float* rd, size_t i) {
        lo = o = f3(ro[3 * i], ro[3 * i + 1], ro[3 * i + 2]);
        ld = d = f3(rd[3 * i], rd[3 * i + 1], rd[3 * i + 2]);
    }
    __device__ __forceinline__ bool test(const float4* xf, int xi, F3 v1, F3 e1, F3 e2, float& t, float& u, float& v) {
        F3 oo = o, dd = d;
        if (xi >= 0) {
            if (xi != lxi) {
                lo = o;
                ld = d;
                to_local<true>(xf, xi, lo, ld);
                lxi = xi;
            }
            oo = lo;
            dd = ld;
        }
        return moller_trumbore(oo, dd, v1, e1, e2, t, u, v);
    }
};

struct LinArgs {
    int n, n_tri, chunk, n_chunks;   // triangles per chunk, a multiple of kLinTile
    bool finish;                     // one chunk: the scanning kernel writes the answers
    const float *ro, *rd;
    const float *verts, *normals;    // the scene's triangles in their original order
    const int32_t *matidx, *xfi;
    const float4* xf;
    float4* part;                    // [n_chunks][n] runs, then their heads
    float4* out;
    __device__ __forceinline__ void keep(int chunk_no, int i, const LinRun& run) const {
        part[(size_t)chunk_no * n + i] = run.pack();
    }
    __device__ __forceinline__ void keep_head(int chunk_no, int i, const LinHit& head) const {
        part[(size_t)n_chunks * n + (size_t)chunk_no * n + i] = head.pack();
    }
    __device__ __forceinline__ LinSum kept(int chunk_no, int i) const {
        const size_t k = (size_t)chunk_no * n + i;
        const float4 p = part[k];
        return LinSum::unpack(p, LinSum::has_head(p) ? part[(size_t)n_chunks * n + k] : p);
    }
};

// A ray's answer from the hit its search kept.  The hit's point goes through M and
// its normal through transpose(inverse) without a second normalisation.
__device__ __forceinline__ void linear_answer(const LinArgs& a, int i, const LinRay& ray, bool found, const LinHit& k) {
    F3 P = {0, 0, 0}, N = {0, 0, 0};
    if (k.tri < 0) {
        write_hit(a.out, (size_t)i, found, P, N, -1, INFINITY, 0.0f, 0.0f, -1);
        return;
    }
    const float* nn = a.normals + 9 * (size_t)k.tri;
    const int xi = a.xfi ? a.xfi[k.tri] : -1;
    const float4 s0 = make_float4(nn[0], nn[1], nn[2], 0.0f);
    const float4 s1 = make_float4(nn[3], nn[4], nn[5], __int_as_float(xi));
    const float4 s2 = make_float4(nn[6], nn[7], nn[8], 0.0f);
    hit_surface(s0, s1, s2, a.xf, ray.o, ray.d, k.t, k.u, k.v, false, P, N);
    write_hit(a.out, (size_t)i, found, P, N, a.matidx[k.tri], k.t, k.u, k.v, k.tri);
}

// One run per ray and chunk of triangles, a workgroup per 256 rays and chunk:
// every lane tests every triangle of the chunk, staged in LDS as (v1, e1, e2,
// transformation) and read as broadcasts.  Bound by the tests' arithmetic (about
// 60 instructions each), so what counts is that every CU has rays: the
// triangles are split until the launch has kLinBlocks workgroups.  Where one chunk
// holds them all the answer is written here.
__global__ __launch_bounds__(kLinTile) void k_query_linear(LinArgs a) {
    __shared__ float4 tri[3 * kLinTile];
    const int i = blockIdx.x * kLinTile + (int)threadIdx.x;
    const bool act = i < a.n;
    LinRay ray;
    if (act) ray.load(a.ro, a.rd, (size_t)i);
    LinRun run;
    const int c0 = (int)blockIdx.y * a.chunk, c1 = min(a.n_tri, c0 + a.chunk);
    for (int base = c0; base < c1; base += kLinTile) {
        __syncthreads();
        const int k = base + (int)threadIdx.x;
        if (k < c1) {
            const float* w = a.verts + 9 * (size_t)k;
            const F3 v1 = f3(w[0], w[1], w[2]);
            const F3 e1 = sub(f3(w[3], w[4], w[5]), v1), e2 = sub(f3(w[6], w[7], w[8]), v1);
            tri[3 * threadIdx.x] = make_float4(v1.x, v1.y, v1.z, e1.x);
            tri[3 * threadIdx.x + 1] = make_float4(e1.y, e1.z, e2.x, e2.y);
            tri[3 * threadIdx.x + 2] = make_float4(e2.z, __int_as_float(a.xfi ? a.xfi[k] : -1), 0.0f, 0.0f);
        }
        __syncthreads();
        if (!act) continue;
        const int cnt = min(kLinTile, c1 - base);
        for (int j = 0; j < cnt; ++j) {
            const float4 p = tri[3 * j], q = tri[3 * j + 1], r = tri[3 * j + 2];
            float t, u, v;
            if (ray.test(a.xf, __float_as_int(r.y), f3(p.x, p.y, p.z), f3(p.w, q.x, q.y), f3(q.z, q.w, r.x), t, u, v)) {
                run.hit(t, u, v, base + j);
                if (__builtin_expect(!(t == t), 0)) {
                    // the head goes to memory at once (in registers it cost 100,000 rays
                    // against 4,000 triangles 583 -> 716 us); a run over every triangle
                    // has nothing before it, and goes on with what it holds
                    if (!run.nan && !a.finish) {
                        a.keep_head((int)blockIdx.y, i, run.best);
                        run.best = LinHit();
                    }
                    run.nan = true;
                    run.zero = false;
                }
            }
        }
    }
    if (!act) return;
    if (a.finish) linear_answer(a, i, ray, run.found, run.best);
    else a.keep((int)blockIdx.y, i, run);
}

// The same with few rays: P lanes (a power of two) share a ray, each a slice of
// consecutive triangles of the chunk, and combine their runs in order.
__global__ __launch_bounds__(kLinTile) void k_query_linear_few(LinArgs a, int P) {
    const int lane_p = (int)threadIdx.x & (P - 1);
    const int i = (int)(blockIdx.x * (kLinTile / P)) + (int)threadIdx.x / P;
    const bool act = i < a.n;
    const int c0 = (int)blockIdx.y * a.chunk, c1 = min(a.n_tri, c0 + a.chunk);
    const int len = a.chunk / P;
    LinSum run;
    if (act) {
        LinRay ray;
        ray.load(a.ro, a.rd, (size_t)i);
        const int k1 = min(c1, c0 + (lane_p + 1) * len);
        for (int k = c0 + lane_p * len; k < k1; ++k) {
            const float* w = a.verts + 9 * (size_t)k;
            const F3 v1 = f3(w[0], w[1], w[2]);
            const F3 e1 = sub(f3(w[3], w[4], w[5]), v1), e2 = sub(f3(w[6], w[7], w[8]), v1);
            float t, u, v;
            if (ray.test(a.xf, a.xfi ? a.xfi[k] : -1, v1, e1, e2, t, u, v)) run.hit(t, u, v, k);
        }
    }
    run.reduce(P);
    if (!act || lane_p != 0) return;
    a.keep((int)blockIdx.y, i, run);
    if (run.nan) a.keep_head((int)blockIdx.y, i, run.head);
}

// A wave per ray of a query of several chunks: its runs combined in order (each
// lane a stretch of chunks, then the lanes), then the answer.
__global__ __launch_bounds__(kLinMergeThreads) void k_linear_merge(LinArgs a) {
    const int i = blockIdx.x * (kLinMergeThreads / 64) + (int)(threadIdx.x >> 6);
    if (i >= a.n) return;
    const int lane = __lane_id();
    const int per = (a.n_chunks + 63) / 64;
    const int b1 = min(a.n_chunks, (lane + 1) * per);
    LinSum run;
    for (int b = lane * per; b < b1; ++b) run.then(a.kept(b, i));
    run.reduce(64);
    if (lane != 0) return;
    LinRay ray;
    ray.load(a.ro, a.rd, (size_t)i);
    linear_answer(a, i, ray, run.found, run.kept());
}

// A linear query of n rays (n >= 1); part: room for the split's runs.
LinArgs linear_args(const eos_scene* s, int n, const LinSplit& sp, const float* ro, const float* rd, float4* part,
                    float4* out) {
    LinArgs a{};
    a.n = n;
    a.n_tri = s->n_tri;
    a.chunk = sp.chunk;
    a.n_chunks = sp.n_chunks;
    a.finish = sp.runs == 0;
    a.verts = s->verts.as<const float>();
    a.normals = s->normals.as<const float>();
    a.matidx = s->matidx.as<const int32_t>();
    a.xfi = s->n_xf > 0 ? s->xf_index.as<const int32_t>() : nullptr;
    a.xf = s->n_xf > 0 ? s->xf.as<const float4>() : nullptr;
    a.ro = ro;
    a.rd = rd;
    a.part = part;
    a.out = out;
    return a;
}

void launch_linear(const LinArgs& a, const LinSplit& sp, hipStream_t S) {
    const dim3 grid(sp.scan_blocks, (unsigned)sp.n_chunks);
    if (sp.lanes_per_ray > 1)
        hipLaunchKernelGGL(k_query_linear_few, grid, dim3(kLinTile), 0, S, a, sp.lanes_per_ray);
    else
        hipLaunchKernelGGL(k_query_linear, grid, dim3(kLinTile), 0, S, a);
    if (sp.runs > 0) hipLaunchKernelGGL(k_linear_merge, dim3(sp.merge_blocks), dim3(kLinMergeThreads), 0, S, a);
}

// The BVH traversal for caller-given rays: the default launch shape (256
// threads, 16 LDS stack entries), the scene's tree width and transformations.
template <int MODE>
void launch_rays(int width, bool xf, bool big, int grid, hipStream_t s, const TraceArgs& a) {
    if (width == 4 && big) {
        hipLaunchKernelGGL((k_trace<MODE, 256, 16, false, false, 4, true, false, true>), dim3(grid), dim3(256), 0, s, a);
    } else if (width == 2) {
        if (xf) hipLaunchKernelGGL((k_trace<MODE, 256, 16, false, false, 2, true>), dim3(grid), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((k_trace<MODE, 256, 16, false, false, 2, false>), dim3(grid), dim3(256), 0, s, a);
    } else {
        if (xf) hipLaunchKernelGGL((k_trace<MODE, 256, 16, false, false, 4, true>), dim3(grid), dim3(256), 0, s, a);
        else hipLaunchKernelGGL((k_trace<MODE, 256, 16, false, false, 4, false>), dim3(grid), dim3(256), 0, s, a);
    }
}

// Fetch cursors of the query launch, then its error flag.
constexpr int kQueryCtrInts = kRanges * kCursorStride + 32;

__global__ void k_zero_i32_query(int* p, int n) {
    for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) p[i] = 0;
}

// ---- the allocation-free variant (eos_trace_rays_static) --------------------
// Its scratch is this fixed array (one copy per GPU, held until the process
// ends): the fetch cursors and the error flag in the first kStaticHeader bytes,
// then the nearest-hit records (16 bytes per ray) or a linear search's runs.  Host code reaches it only
// through the address hipGetSymbolAddress gives on each device.
constexpr size_t kStaticHeader = 4096;
static_assert(4 * (size_t)kQueryCtrInts <= kStaticHeader, "cursors and flag fit the header");
constexpr size_t kStaticBytes = kStaticHeader + 16 * (size_t)EOS_STATIC_MAX_RAYS;
static_assert(kLinRunBytes * kLinStaticRuns <= kStaticBytes - kStaticHeader, "a linear query's runs fit the records");
__device__ __align__(256) unsigned char scratch[kStaticBytes];

constexpr int kMaxDevices = 64;

// The device address of `scratch` on the current device, looked up once per
// device (null when the lookup fails).
void* static_scratch(int device) {
    static std::mutex mu;
    static void* ptr[kMaxDevices] = {};
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if (!ptr[device]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        ptr[device] = p;
    }
    return ptr[device];
}

}  // namespace

eos_status trace_rays_static(eos_scene* s, int n, const float* o, const float* d, const eos_trace_opts* opts,
                             eos_ray_hit* hits, uint8_t* occ) {
    const hipStream_t S = s->stream;
    void* base = static_scratch(s->device);
    if (!base) return fail(EOS_ERR_HIP, "eos_trace_rays_static: hipGetSymbolAddress of the scratch array failed");
    int* ctr = static_cast<int*>(base);
    float4* rec = reinterpret_cast<float4*>(static_cast<char*>(base) + kStaticHeader);
    float4* out = reinterpret_cast<float4*>(hits);
    const unsigned blocks = (unsigned)(((size_t)n + 255) / 256);
    if (opts->mode == EOS_QUERY_NEAREST_LINEAR) {
        const LinSplit sp = linear_split(n, s->n_tri, kLinStaticRuns);
        launch_linear(linear_args(s, n, sp, o, d, rec, out), sp, S);
        EOS_HIP(hipGetLastError());
        EOS_HIP(hipStreamSynchronize(S));
        return EOS_OK;
    }
    // every lane's stack lives in LDS: lane quads walk the 4-wide tree (96
    // entries per quad), single lanes walk the binary tree with all of its 64
    // entries in LDS, so no overflow stack is needed
    const int trace_grid = std::max(1, s->num_cu * std::min(s->cfg.waves_per_cu, 8) / 4);
    const int grid = (int)std::min<size_t>((size_t)trace_grid, std::max<size_t>(1, (4 * (size_t)n + 255) / 256));
    hipLaunchKernelGGL(k_zero_i32_query, dim3(1), dim3(256), 0, S, ctr, kQueryCtrInts);
    TraceArgs a{};
    a.sc = view_of(s);
    a.n_static = n;
    a.count_mul = 1;
    a.cursor = ctr;
    a.err = ctr + kRanges * kCursorStride;
    a.gstack = ctr;          // never dereferenced: no lane's stack leaves LDS
    a.refill = s->cfg.refill;
    a.batch = s->cfg.batch;
    a.coop = 4;
    a.ray_o = o;
    a.ray_d = d;
    const bool xf = s->n_xf > 0;
    if (opts->mode == EOS_QUERY_OCCLUDED) {
        a.vis_out = occ;
        if (s->width == 2) {
            if (xf) hipLaunchKernelGGL((k_trace<MODE_RAYS_ANY, 256, kMaxStack, false, false, 2, true>), dim3(grid), dim3(256), 0, S, a);
            else hipLaunchKernelGGL((k_trace<MODE_RAYS_ANY, 256, kMaxStack, false, false, 2, false>), dim3(grid), dim3(256), 0, S, a);
        } else {
            launch_rays<MODE_RAYS_ANY>(4, xf, s->tree_big(), grid, S, a);
        }
    } else {
        a.hit_out = rec;
        if (s->width == 2) {
            if (xf) hipLaunchKernelGGL((k_trace<MODE_RAYS, 256, kMaxStack, false, false, 2, true>), dim3(grid), dim3(256), 0, S, a);
            else hipLaunchKernelGGL((k_trace<MODE_RAYS, 256, kMaxStack, false, false, 2, false>), dim3(grid), dim3(256), 0, S, a);
        } else {
            launch_rays<MODE_RAYS>(4, xf, s->tree_big(), grid, S, a);
        }
        hipLaunchKernelGGL(k_query_hits, dim3(blocks), dim3(256), 0, S, n, o, d, rec, s->shade.as<const float4>(),
                           s->geo(), xf ? s->xf.as<const float4>() : nullptr, out);
    }
    EOS_HIP(hipGetLastError());
    int err = 0;
    EOS_HIP(hipMemcpyAsync(&err, a.err, sizeof err, hipMemcpyDeviceToHost, S));
    EOS_HIP(hipStreamSynchronize(S));
    if (err & 1) return fail(EOS_ERR_LIMIT, "eos_trace_rays_static: traversal stack overflow");
    if (err & 2) return fail(EOS_ERR_STATE, "eos_trace_rays_static: traversal exceeded its visit bound (corrupt BVH)");
    return EOS_OK;
}

eos_status trace_rays(eos_scene* s, int n, const float* o, const float* d, const eos_trace_opts* opts,
                      eos_ray_hit* hits, uint8_t* occ) {
    const bool dev = opts->memory == EOS_MEM_DEVICE;
    const int mode = opts->mode;
    const hipStream_t S = s->stream;
    const size_t nn = (size_t)n;
    const float* ro = o;
    const float* rd = d;
    if (!dev) {
        EOS_TRY(s->q_rays.ensure(24 * nn));
        EOS_HIP(hipMemcpyAsync(s->q_rays.ptr, o, 12 * nn, hipMemcpyHostToDevice, S));
        EOS_HIP(hipMemcpyAsync(s->q_rays.as<char>() + 12 * nn, d, 12 * nn, hipMemcpyHostToDevice, S));
        ro = s->q_rays.as<const float>();
        rd = reinterpret_cast<const float*>(s->q_rays.as<const char>() + 12 * nn);
    }
    float4* out = nullptr;
    uint8_t* occ_dev = nullptr;
    if (mode == EOS_QUERY_OCCLUDED) {
        if (dev) occ_dev = occ;
        else {
            EOS_TRY(s->q_out.ensure(nn));
            occ_dev = s->q_out.as<uint8_t>();
        }
    } else if (dev) {
        out = reinterpret_cast<float4*>(hits);
    } else {
        EOS_TRY(s->q_out.ensure(48 * nn));
        out = s->q_out.as<float4>();
    }
    const unsigned blocks = (unsigned)((nn + 255) / 256);
    int err = 0;
    if (mode == EOS_QUERY_NEAREST_LINEAR) {
        const LinSplit sp = linear_split(n, s->n_tri, kLinRuns);
        EOS_TRY(s->q_rec.ensure(kLinRunBytes * sp.runs));
        launch_linear(linear_args(s, n, sp, ro, rd, s->q_rec.as<float4>(), out), sp, S);
        EOS_HIP(hipGetLastError());
    } else {
        const LaunchCfg& cfg = s->cfg;
        const int trace_grid = std::max(1, s->num_cu * cfg.waves_per_cu / 4);
        const int grid = query_grid(nn, trace_grid);
        const int maxs = s->width == 4 ? kMaxStack4 : kMaxStack;
        EOS_TRY(s->q_ctr.ensure(4 * (size_t)kQueryCtrInts));
        EOS_TRY(s->q_gstack.ensure(4 * query_stack_lanes(nn, grid) * (size_t)(maxs - 16)));
        int* ctr = s->q_ctr.as<int>();
        hipLaunchKernelGGL(k_zero_i32_query, dim3(1), dim3(256), 0, S, ctr, kQueryCtrInts);
        TraceArgs a{};
        a.sc = view_of(s);
        a.n_static = n;
        a.count_mul = 1;
        a.cursor = ctr;
        a.err = ctr + kRanges * kCursorStride;
        a.gstack = s->q_gstack.as<int32_t>();
        a.refill = query_refill(cfg.refill);
        a.batch = cfg.batch;
        a.coop = cfg.coop;
        a.group = cfg.group;
        a.group_lanes = cfg.group_lanes;
        a.steal = cfg.steal;
        a.scatter = query_scatter(cfg.scatter);
        a.ray_o = ro;
        a.ray_d = rd;
        if (mode == EOS_QUERY_OCCLUDED) {
            a.vis_out = occ_dev;
            launch_rays<MODE_RAYS_ANY>(s->width, s->n_xf > 0, s->tree_big(), grid, S, a);
        } else {
            EOS_TRY(s->q_rec.ensure(16 * nn));
            a.hit_out = s->q_rec.as<float4>();
            launch_rays<MODE_RAYS>(s->width, s->n_xf > 0, s->tree_big(), grid, S, a);
            hipLaunchKernelGGL(k_query_hits, dim3(blocks), dim3(256), 0, S, n, ro, rd, s->q_rec.as<const float4>(),
                               s->shade.as<const float4>(), s->geo(),
                               s->n_xf > 0 ? s->xf.as<const float4>() : nullptr, out);
        }
        EOS_HIP(hipGetLastError());
        EOS_TRY(s->ensure_host_small());
        EOS_HIP(hipMemcpyAsync(s->host_small, a.err, sizeof err, hipMemcpyDeviceToHost, S));
    }
    if (!dev) {
        if (mode == EOS_QUERY_OCCLUDED) EOS_HIP(hipMemcpyAsync(occ, occ_dev, nn, hipMemcpyDeviceToHost, S));
        else EOS_HIP(hipMemcpyAsync(hits, out, 48 * nn, hipMemcpyDeviceToHost, S));
    }
    EOS_HIP(hipStreamSynchronize(S));
    if (mode != EOS_QUERY_NEAREST_LINEAR) err = s->host_small[0];
    if (err & 1) return fail(EOS_ERR_LIMIT, "eos_trace_rays: traversal stack overflow");
    if (err & 2) return fail(EOS_ERR_STATE, "eos_trace_rays: traversal exceeded its visit bound (corrupt BVH)");
    return EOS_OK;
}

}  // namespace eos
