// lbvh.hip -- GPU Morton-code LBVH build for gfx950.
//
// The reference builds its BVH on the CPU (src/BVH.cpp:97-111, hybrid
// median/SAH) and ships only a Morton bit-interleave it never calls
// (src/morton.h:30-48).  This file builds a Karras (2012) LBVH on the GPU:
//   1. centroid bounds (two-level reduction, deterministic)
//   2. 30-bit Morton codes (EncodeMorton3 bit layout: z above y above x)
//   3. stable LSD radix sort of (code, index), 3 passes of 10 bits
//   4. Karras hierarchy, one thread per internal node
//   5. boxes of aligned runs of 2^k leaves; a node covers consecutive leaves, so
//      its box is the union of a few such runs
//   6. 128-byte 4-wide nodes (64-byte binary nodes for width 2) and 48-byte
//      triangle records in leaf order
// Every step is integer or exact float min/max work, so the result is
// bit-identical to the CPU restatement of the same algorithm.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <string>
#include <vector>

#include "eos_internal.h"

namespace eos {
namespace {

constexpr int kDigitBits = 10, kDigits = 1 << kDigitBits;
constexpr int kSortWaves = 16, kSortThreads = 64 * kSortWaves;
constexpr int kSortBlocks = 256;                     // at most: a workgroup per CU

__device__ __forceinline__ uint32_t part1by2(uint32_t x) {
    x &= 0x000003ffu;
    x = (x ^ (x << 16)) & 0xff0000ffu;
    x = (x ^ (x << 8)) & 0x0300f00fu;
    x = (x ^ (x << 4)) & 0x030c30c3u;
    x = (x ^ (x << 2)) & 0x09249249u;
    return x;
}

// ((v1 + v2) + v3) / 3 per axis, the reference's centroid (src/Triangle.h:38).
__device__ __forceinline__ void centroid(const float* __restrict__ v, size_t i, float c[3]) {
    const float* t = v + 9 * i;
#pragma unroll
    for (int k = 0; k < 3; ++k) c[k] = ((t[k] + t[3 + k]) + t[6 + k]) / 3.0f;
}

// World-space vertices of a transformed triangle (M * (v, 1), glm's order of
// operations; the rows of M are kXfM..kXfM+2 of its record), the input vertices
// for the rest.  Keys and boxes of the build come from these; the triangle
// records keep the local vertices, as rays meet triangles in local space.
__device__ __forceinline__ void world_vertices(const float* __restrict__ t, int x, const float4* __restrict__ xf,
                                               int n_xf, float w[9]) {
    if (x < 0 || x >= n_xf) {
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = t[k];
        return;
    }
    const float4 r[3] = {xf[kXfRows * (size_t)x + kXfM], xf[kXfRows * (size_t)x + kXfM + 1],
                         xf[kXfRows * (size_t)x + kXfM + 2]};
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k)
            w[3 * c + k] = (r[k].x * t[3 * c] + r[k].y * t[3 * c + 1]) + (r[k].z * t[3 * c + 2] + r[k].w * 1.0f);
}

// Centroid bounds of each workgroup's triangles.  XF: also writes the world-space
// vertices of scenes with transformations.
template <bool XF>
__global__ __launch_bounds__(256) void k_cbounds_partial(const float* __restrict__ verts, int n,
                                                         const int32_t* __restrict__ xi, const float4* __restrict__ xf,
                                                         int n_xf, float* __restrict__ wverts,
                                                         float* __restrict__ part) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float c[3];
        if (XF) {
            float w[9];
            world_vertices(verts + 9 * (size_t)i, xi[i], xf, n_xf, w);
#pragma unroll
            for (int k = 0; k < 9; ++k) wverts[9 * (size_t)i + k] = w[k];
            centroid(w, 0, c);
        } else {
            centroid(verts, (size_t)i, c);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(lo[k], c[k]);
            hi[k] = fmaxf(hi[k], c[k]);
        }
    }
    __shared__ float s[6][256];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s[k][threadIdx.x] = lo[k];
        s[3 + k][threadIdx.x] = hi[k];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                s[k][threadIdx.x] = fminf(s[k][threadIdx.x], s[k][threadIdx.x + w]);
                s[3 + k][threadIdx.x] = fmaxf(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// One wave per component over all partials (min and max are exact, so the order
// does not matter; one lane per component walking them one after another took
// 98 us at 1M triangles), and the build's error counters set to zero.
__global__ __launch_bounds__(384) void k_cbounds_final(const float* __restrict__ part, int nparts,
                                                       float* __restrict__ cb, int32_t* __restrict__ err) {
    const int k = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float r = k < 3 ? INFINITY : -INFINITY;
    for (int b = lane; b < nparts; b += 64) r = k < 3 ? fminf(r, part[6 * b + k]) : fmaxf(r, part[6 * b + k]);
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(r, off);
        r = k < 3 ? fminf(r, o) : fmaxf(r, o);
    }
    if (lane == 0) cb[k] = r;
    if (threadIdx.x < 4) err[threadIdx.x] = 0;
}

__device__ __forceinline__ uint32_t quant10(float c, float lo, float hi) {
    float e = hi - lo;
    float s = e > 0.0f ? 1024.0f / e : 0.0f;
    float x = (c - lo) * s;
    x = fminf(fmaxf(x, 0.0f), 1023.0f);
    return (uint32_t)x;
}

__global__ __launch_bounds__(256) void k_morton(const float* __restrict__ verts, int n, const float* __restrict__ cb,
                                                uint32_t* __restrict__ codes) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float c[3];
    centroid(verts, (size_t)i, c);
    uint32_t x = quant10(c[0], cb[0], cb[3]);
    uint32_t y = quant10(c[1], cb[1], cb[4]);
    uint32_t z = quant10(c[2], cb[2], cb[5]);
    codes[i] = (part1by2(z) << 2) + (part1by2(y) << 1) + part1by2(x);
}

// ---- LSD radix sort, 10-bit digits: three launches per pass --------------------
// At most one workgroup of 16 waves per CU; each wave owns `seg` consecutive keys
// (a multiple of 64) and counts and ranks them in its own row of LDS counters, so
// the only barriers are around the counters, not between rounds of 256 keys.
// 1M keys: four 8-bit passes of five launches 156 us, three passes like this 92.
struct SortShape {
    int blocks, seg;
};
inline SortShape sort_shape(size_t n) {
    const size_t waves = (size_t)kSortBlocks * kSortWaves;
    const size_t seg = ((n + waves - 1) / waves + 63) / 64 * 64;
    return {(int)((n + seg * kSortWaves - 1) / (seg * kSortWaves)), (int)seg};
}
inline size_t sort_hist_bytes(const SortShape& sh) { return 4 * (size_t)kDigits * (size_t)(sh.blocks + 1); }

// Digit counts of each workgroup, digit-major.
__global__ __launch_bounds__(kSortThreads) void k_radix_hist(const uint32_t* __restrict__ keys, int n, int shift,
                                                             int seg, uint32_t* __restrict__ hist, int nblocks) {
    __shared__ uint32_t h[kDigits];
    h[threadIdx.x] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * seg * kSortWaves;
    const long long end = min((long long)n, base + (long long)seg * kSortWaves);
    for (long long i = base + threadIdx.x; i < end; i += kSortThreads)
        atomicAdd(&h[(keys[i] >> shift) & (kDigits - 1)], 1u);
    __syncthreads();
    hist[(size_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}
static_assert(kDigits == kSortThreads, "a thread per digit");

// A wave per digit: its counts become the exclusive prefix over the workgroups
// (at most 256, four per lane), and its total.
__global__ __launch_bounds__(256) void k_radix_scan(uint32_t* __restrict__ hist, int nblocks,
                                                    uint32_t* __restrict__ totals) {
    const int d = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    uint32_t* row = hist + (size_t)d * nblocks;
    uint32_t v[4], t = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = 4 * lane + k;
        v[k] = b < nblocks ? row[b] : 0u;
        t += v[k];
    }
    uint32_t x = t;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    uint32_t run = x - t;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = 4 * lane + k;
        if (b < nblocks) row[b] = run;
        run += v[k];
    }
    if (lane == 63) totals[d] = x;
}
static_assert(kSortBlocks <= 256, "four workgroups' counts per lane");

// Exclusive scan of one value per thread over a workgroup of 1024 threads.
__device__ __forceinline__ uint32_t block_scan_1024(uint32_t v, uint32_t* s_wave /* [16] */, uint32_t* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_wave[w] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int k = 0; k < 16; ++k) {
        before += k < w ? s_wave[k] : 0u;
        all += s_wave[k];
    }
    if (total) *total = all;
    return before + x - v;
}

// Stable scatter.  Each wave counts its keys' digits; a prefix over the digits,
// the workgroups and the waves turns the counters into destinations; then each
// wave walks its keys again in order, 64 at a time: lanes holding the same digit
// are matched with ten ballots and ranked by lane.  vin null: the values are the
// keys' indices.
__global__ __launch_bounds__(kSortThreads) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                                const int32_t* __restrict__ vin,
                                                                uint32_t* __restrict__ kout, int32_t* __restrict__ vout,
                                                                int n, int shift, int seg,
                                                                const uint32_t* __restrict__ hist, int nblocks,
                                                                const uint32_t* __restrict__ totals) {
    __shared__ uint32_t cnt[kSortWaves][kDigits];
    __shared__ uint32_t s_wave[16];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
#pragma unroll
    for (int k = 0; k < kSortWaves; ++k) cnt[k][tid] = 0;
    __syncthreads();
    const long long base = ((long long)blockIdx.x * kSortWaves + w) * seg;
    const long long end = min((long long)n, base + seg);
    for (long long i = base + lane; i < end; i += 64) atomicAdd(&cnt[w][(kin[i] >> shift) & (kDigits - 1)], 1u);
    uint32_t run = block_scan_1024(totals[tid], s_wave, nullptr);   // its barrier ends the counting too
    run += hist[(size_t)tid * nblocks + blockIdx.x];
#pragma unroll
    for (int k = 0; k < kSortWaves; ++k) {
        const uint32_t c = cnt[k][tid];
        cnt[k][tid] = run;
        run += c;
    }
    __syncthreads();
    volatile uint32_t* mine = cnt[w];
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t key = 0;
    int32_t val = 0;
    auto load = [&](long long i) {
        if (i < end) {
            key = kin[i];
            val = vin ? vin[i] : (int32_t)i;
        }
    };
    load(base + lane);
    for (long long i0 = base; i0 < end; i0 += 64) {
        const bool valid = i0 + lane < end;
        const uint32_t k = key;
        const int32_t v = val;
        load(i0 + 64 + lane);
        const uint32_t d = (k >> shift) & (kDigits - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < kDigitBits; ++bit) {
            const uint64_t b = __ballot((d >> bit) & 1u);
            peers &= ((d >> bit) & 1u) ? b : ~b;
        }
        const uint32_t rank = __popcll(peers & lt);
        const uint32_t off = mine[d];
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) mine[d] = off + __popcll(peers);
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            kout[off + rank] = k;
            vout[off + rank] = v;
        }
    }
}

// One pass over n keys (hist: sort_hist_bytes).
void radix_pass(hipStream_t S, const SortShape& sh, const uint32_t* kin, const int32_t* vin, uint32_t* kout,
                int32_t* vout, int n, int shift, uint32_t* hist) {
    uint32_t* totals = hist + (size_t)kDigits * sh.blocks;
    hipLaunchKernelGGL(k_radix_hist, dim3(sh.blocks), dim3(kSortThreads), 0, S, kin, n, shift, sh.seg, hist, sh.blocks);
    hipLaunchKernelGGL(k_radix_scan, dim3(kDigits / 4), dim3(256), 0, S, hist, sh.blocks, totals);
    hipLaunchKernelGGL(k_radix_scatter, dim3(sh.blocks), dim3(kSortThreads), 0, S, kin, vin, kout, vout, n, shift,
                       sh.seg, hist, sh.blocks, totals);
}

// ---- Karras hierarchy --------------------------------------------------------
__device__ __forceinline__ int delta(const uint32_t* __restrict__ k, int n, int i, int j) {
    if (j < 0 || j > n - 1) return -1;
    uint32_t a = k[i], b = k[j];
    if (a == b) return 32 + __clz((int)((uint32_t)i ^ (uint32_t)j));
    return __clz((int)(a ^ b));
}

__global__ __launch_bounds__(256) void k_karras(const uint32_t* __restrict__ k, int n, int2* __restrict__ kchild,
                                                int32_t* __restrict__ kparent, int2* __restrict__ fl) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) kparent[0] = -1;   // the root, or the only leaf
    if (i >= n - 1) return;
    const int d = (delta(k, n, i, i + 1) - delta(k, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(k, n, i, i - d);
    int lmax = 2;
    while (delta(k, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (delta(k, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(k, n, i, j);
    int s = 0;
    for (int div = 2;; div *= 2) {
        int t = (l + div - 1) / div;
        if (delta(k, n, i, i + (s + t) * d) > dnode) s += t;
        if (t <= 1) break;
    }
    const int g = i + s * d + min(d, 0);
    const int lo = min(i, j), hi = max(i, j);
    const int left = (lo == g) ? ~g : g;
    const int right = (hi == g + 1) ? ~(g + 1) : g + 1;
    kchild[i] = make_int2(left, right);
    fl[i] = make_int2(lo, hi);
    kparent[left >= 0 ? left : (n - 1 + ~left)] = i;
    kparent[right >= 0 ? right : (n - 1 + ~right)] = i;
}

// ---- boxes ------------------------------------------------------------------
// A box is six floats: lo.xyz, hi.xyz.  Level k >= 1 of the pyramid holds the
// boxes of the runs of 2^k leaves starting at multiples of 2^k, at entry
// top - (top >> (k - 1)) on, top = the leaf count rounded up to a power of two;
// level 0 is lbox.  (Boxing the tree level by level, each pass over every node
// still open, took 64 launches, 0.74 ms of a 1.4 ms build of 1M triangles.)
// An empty box is not a number, which fminf and fmaxf pass over: the union of
// boxes that hold no number at all (triangles of NaN corners) stays so, as it
// does where two children's boxes are joined.
struct Box6 {
    float v[6] = {NAN, NAN, NAN, NAN, NAN, NAN};
    __device__ __forceinline__ void add(const Box6& o) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            v[k] = fminf(v[k], o.v[k]);
            v[3 + k] = fmaxf(v[3 + k], o.v[3 + k]);
        }
    }
    __device__ __forceinline__ static Box6 load(const float* __restrict__ p, size_t i) {
        Box6 b;
#pragma unroll
        for (int k = 0; k < 6; ++k) b.v[k] = p[6 * i + k];
        return b;
    }
    __device__ __forceinline__ void store(float* __restrict__ p, size_t i) const {
#pragma unroll
        for (int k = 0; k < 6; ++k) p[6 * i + k] = v[k];
    }
};
inline size_t pyramid_top(size_t n) {
    size_t t = 1;
    while (t < n) t *= 2;
    return t;
}
__device__ __forceinline__ size_t pyramid_at(size_t top, int level, size_t i) { return top - (top >> (level - 1)) + i; }
constexpr int kBoxBlock = 1024;   // leaves per workgroup of k_leaf_boxes (levels 1..10)

// Leaf boxes (exact min/max of the three vertices of the sorted slots) and the
// first ten levels of the pyramid: four leaves per lane, then lane shuffles, then
// the four waves.
__global__ __launch_bounds__(256) void k_leaf_boxes(const float* __restrict__ verts, const int32_t* __restrict__ perm,
                                                    int n, float* __restrict__ lbox, float* __restrict__ pyr,
                                                    size_t top) {
    const size_t quad = (size_t)blockIdx.x * 256 + threadIdx.x;
    Box6 b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const size_t s = 4 * quad + q;
        if (s < (size_t)n) {
            const float* t = verts + 9 * (size_t)perm[s];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                b[q].v[k] = fminf(fminf(t[k], t[3 + k]), t[6 + k]);
                b[q].v[3 + k] = fmaxf(fmaxf(t[k], t[3 + k]), t[6 + k]);
            }
            b[q].store(lbox, s);
        }
    }
    b[0].add(b[1]);
    b[2].add(b[3]);
    if (4 * quad < (size_t)n) b[0].store(pyr, pyramid_at(top, 1, 2 * quad));
    if (4 * quad + 2 < (size_t)n) b[2].store(pyr, pyramid_at(top, 1, 2 * quad + 1));
    b[0].add(b[2]);
    if (n > 2 && 4 * quad < (size_t)n) b[0].store(pyr, pyramid_at(top, 2, quad));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int level = 3; level <= 8; ++level) {
        const int off = 1 << (level - 3);
        Box6 o;
#pragma unroll
        for (int k = 0; k < 6; ++k) o.v[k] = __shfl_down(b[0].v[k], off);
        b[0].add(o);   // right for the lanes that the next level reads
        if ((lane & (2 * off - 1)) == 0 && (size_t)n > ((size_t)1 << (level - 1)) && 4 * quad < (size_t)n)
            b[0].store(pyr, pyramid_at(top, level, quad >> (level - 2)));
    }
    __shared__ float s_box[6][4];
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 6; ++k) s_box[k][w] = b[0].v[k];
    __syncthreads();
    if (threadIdx.x < 2) {
        // level 9: one pair of waves per thread; level 10 by thread 0
        Box6 r[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            Box6 x, y;
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                x.v[k] = s_box[k][2 * q];
                y.v[k] = s_box[k][2 * q + 1];
            }
            x.add(y);
            r[q] = x;
        }
        const size_t first = (size_t)blockIdx.x * kBoxBlock + 512 * threadIdx.x;
        if (n > 256 && first < (size_t)n) (threadIdx.x == 0 ? r[0] : r[1]).store(pyr, pyramid_at(top, 9, first >> 9));
        r[0].add(r[1]);
        if (threadIdx.x == 0 && n > 512) r[0].store(pyr, pyramid_at(top, 10, blockIdx.x));
    }
}

// The levels above, in one workgroup (the eleventh has a box per 2,048 leaves).
__global__ __launch_bounds__(1024) void k_pyramid_top(int n, float* pyr, size_t top) {
    size_t below = ((size_t)n + 1023) / 1024;
    for (int level = 11; below > 1; ++level) {
        const size_t cnt = (below + 1) / 2;
        for (size_t j = threadIdx.x; j < cnt; j += 1024) {
            Box6 b = Box6::load(pyr, pyramid_at(top, level - 1, 2 * j));
            if (2 * j + 1 < below) b.add(Box6::load(pyr, pyramid_at(top, level - 1, 2 * j + 1)));
            b.store(pyr, pyramid_at(top, level, j));
        }
        __syncthreads();   // this workgroup's next level reads what it wrote
        below = cnt;
    }
}

// The box of leaves [l, r]: the fewest aligned runs that make it up.
__device__ __forceinline__ Box6 range_box(const float* __restrict__ lbox, const float* __restrict__ pyr, size_t top,
                                          int l, int r) {
    Box6 b;
    for (int i = l; i <= r;) {
        int k = 31 - __clz(r - i + 1);
        if (i != 0) k = min(k, __ffs(i) - 1);
        b.add(k == 0 ? Box6::load(lbox, (size_t)i) : Box6::load(pyr, pyramid_at(top, k, (size_t)(i >> k))));
        i += 1 << k;
    }
    return b;
}

__device__ __forceinline__ float inflate_pad(float lo, float hi, float eps) {
    float a = fabsf(lo), b = fabsf(hi);
    float m = a > b ? a : b;
    return m * 0x1p-16f + eps;
}

__device__ __forceinline__ int32_t leaf_ref(int32_t first, int32_t count) {
    return ~(first | ((count - 1) << kLeafShift));
}

__global__ __launch_bounds__(256) void k_nodes(const int2* __restrict__ kchild, const int2* __restrict__ fl,
                                               const float* __restrict__ ibox, const float* __restrict__ lbox,
                                               const float* __restrict__ cb, int n, int leaf_max, Node* __restrict__ nodes) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    float eps = 0.0f;
#pragma unroll
    for (int k = 0; k < 6; ++k) eps = fmaxf(eps, fabsf(cb[k]));
    eps = eps * 0x1p-22f;
    const int2 c = kchild[i];
    float lo[2][3], hi[2][3];
    int32_t ref[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int ch = j ? c.y : c.x;
        const float* b = ch >= 0 ? ibox + 6 * (size_t)ch : lbox + 6 * (size_t)~ch;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            float pad = inflate_pad(b[k], b[3 + k], eps);
            lo[j][k] = b[k] - pad;
            hi[j][k] = b[3 + k] + pad;
        }
        if (ch < 0) {
            ref[j] = leaf_ref(~ch, 1);
        } else {
            const int2 r = fl[ch];
            ref[j] = (r.y - r.x + 1 <= leaf_max) ? leaf_ref(r.x, r.y - r.x + 1) : ch;
        }
    }
    Node nd;
    nd.b0 = make_float4(lo[0][0], hi[0][0], lo[0][1], hi[0][1]);
    nd.b1 = make_float4(lo[1][0], hi[1][0], lo[1][1], hi[1][1]);
    nd.b2 = make_float4(lo[0][2], hi[0][2], lo[1][2], hi[1][2]);
    nd.c = make_int4(ref[0], ref[1], 0, 0);
    nodes[i] = nd;
}

// Triangle records in leaf order: geo = (v1, e1, e2, original index,
// transformation index), shade = (n1 material, n2 transformation index, n3).
__global__ __launch_bounds__(256) void k_tris(const float* __restrict__ verts, const float* __restrict__ normals,
                                              const int32_t* __restrict__ mat, const int32_t* __restrict__ perm, int n,
                                              int n_mat, const int32_t* __restrict__ xi, int n_xf,
                                              float4* __restrict__ geo, float4* __restrict__ shade,
                                              int32_t* __restrict__ err) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int o = perm[s];
    int x = xi ? xi[o] : -1;
    if (x < -1 || x >= n_xf) {
        atomicAdd(err + 2, 1);
        x = -1;
    }
    const float* t = verts + 9 * (size_t)o;
    const float* nn = normals + 9 * (size_t)o;
    const float v1x = t[0], v1y = t[1], v1z = t[2];
    const float e1x = t[3] - v1x, e1y = t[4] - v1y, e1z = t[5] - v1z;
    const float e2x = t[6] - v1x, e2y = t[7] - v1y, e2z = t[8] - v1z;
    geo[3 * (size_t)s + 0] = make_float4(v1x, v1y, v1z, e1x);
    geo[3 * (size_t)s + 1] = make_float4(e1y, e1z, e2x, e2y);
    geo[3 * (size_t)s + 2] = make_float4(e2z, __int_as_float(o), __int_as_float(x), 0.0f);
    int m = mat[o];
    if (m < 0 || m >= n_mat) {
        atomicAdd(err, 1);
        m = 0;
    }
    shade[3 * (size_t)s + 0] = make_float4(nn[0], nn[1], nn[2], __int_as_float(m));
    shade[3 * (size_t)s + 1] = make_float4(nn[3], nn[4], nn[5], __int_as_float(x));
    shade[3 * (size_t)s + 2] = make_float4(nn[6], nn[7], nn[8], 0.0f);
}

// ---- 4-wide collapse -----------------------------------------------------------
// A 4-wide node stands for every binary node that stays internal (range larger
// than leaf_max) at even depth; nodes are numbered in binary index order.  The
// nodes that stand are kept as one bit each, 64 per word, and a count per 256,
// which a scan turns into the first number of each 256.
constexpr int kNodeBlock = 256;
constexpr int kMaskWords = kNodeBlock / 64;

// Every lane of the workgroup calls it: node's bit and the workgroup's count.
__device__ __forceinline__ void keep_flags(bool stands, uint64_t* __restrict__ masks, int32_t* __restrict__ counts) {
    __shared__ int32_t s_n[kMaskWords];
    const uint64_t m = __ballot(stands);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        masks[(size_t)blockIdx.x * kMaskWords + w] = m;
        s_n[w] = __popcll(m);
    }
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}
static_assert(kMaskWords == 4, "four waves per workgroup");

// The number of the nodes that stand before node g.
__device__ __forceinline__ int number_of(const uint64_t* __restrict__ masks, const int32_t* __restrict__ first, int g) {
    const uint64_t* m = masks + (size_t)(g / kNodeBlock) * kMaskWords;
    const int w = (g / 64) % kMaskWords;
    int c = first[g / kNodeBlock] + __popcll(m[w] & ((1ull << (g & 63)) - 1));
    for (int k = 0; k < w; ++k) c += __popcll(m[k]);
    return c;
}
__device__ __forceinline__ bool stands(const uint64_t* __restrict__ masks, int g) {
    return (masks[(size_t)(g / kNodeBlock) * kMaskWords + (g / 64) % kMaskWords] >> (g & 63)) & 1ull;
}

// Exclusive scan of the counts in place (one workgroup, a stretch per thread) and
// their sum.
__global__ __launch_bounds__(1024) void k_scan_counts(int32_t* __restrict__ c, int nb, int32_t* __restrict__ total) {
    __shared__ uint32_t s_wave[16];
    const int per = (nb + 1023) / 1024;
    const int b0 = min(nb, (int)threadIdx.x * per), b1 = min(nb, b0 + per);
    uint32_t t = 0;
    for (int b = b0; b < b1; ++b) t += (uint32_t)c[b];
    uint32_t all = 0;
    uint32_t run = block_scan_1024(t, s_wave, &all);
    for (int b = b0; b < b1; ++b) {
        const uint32_t v = (uint32_t)c[b];
        c[b] = (int32_t)run;
        run += v;
    }
    if (threadIdx.x == 0) *total = (int32_t)all;
}

// Boxes of the internal nodes, and which of them stand as 4-wide nodes.
__global__ __launch_bounds__(kNodeBlock) void k_node_boxes(const int32_t* __restrict__ kparent,
                                                           const int2* __restrict__ fl, int n, int leaf_max,
                                                           const float* __restrict__ lbox,
                                                           const float* __restrict__ pyr, size_t top,
                                                           float* __restrict__ ibox, uint64_t* __restrict__ masks,
                                                           int32_t* __restrict__ counts) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool f = false;
    if (i < n - 1) {
        const int2 r = fl[i];
        range_box(lbox, pyr, top, r.x, r.y).store(ibox, (size_t)i);
        if (r.y - r.x + 1 > leaf_max) {
            int depth = 0;
            for (int p = kparent[i]; p >= 0 && depth < 128; p = kparent[p]) ++depth;
            f = (depth & 1) == 0;
        }
    }
    keep_flags(f, masks, counts);
}

__global__ __launch_bounds__(256) void k_nodes4(const int2* __restrict__ kchild, const int2* __restrict__ fl,
                                                const float* __restrict__ ibox, const float* __restrict__ lbox,
                                                const float* __restrict__ cb, const uint64_t* __restrict__ masks,
                                                const int32_t* __restrict__ first, int n, int leaf_max,
                                                Node4* __restrict__ nodes4) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1 || !stands(masks, i)) return;
    float eps = 0.0f;
#pragma unroll
    for (int k = 0; k < 6; ++k) eps = fmaxf(eps, fabsf(cb[k]));
    eps = eps * 0x1p-22f;
    int slots[4] = {0, 0, 0, 0};
    int ns = 0;
    const int2 c = kchild[i];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int ch = j ? c.y : c.x;
        bool internal = false;
        if (ch >= 0) {
            const int2 r = fl[ch];
            internal = r.y - r.x + 1 > leaf_max;
        }
        if (internal) {
            const int2 g = kchild[ch];
            slots[ns++] = g.x;
            slots[ns++] = g.y;
        } else {
            slots[ns++] = ch;
        }
    }
    float lo[3][4], hi[3][4];
    int32_t ref[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        ref[k] = kEmpty;
#pragma unroll
        for (int a = 0; a < 3; ++a) lo[a][k] = hi[a][k] = INFINITY;
        if (k < ns) {
            const int g = slots[k];
            const float* b = g >= 0 ? ibox + 6 * (size_t)g : lbox + 6 * (size_t)~g;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                float pad = inflate_pad(b[a], b[3 + a], eps);
                lo[a][k] = b[a] - pad;
                hi[a][k] = b[3 + a] + pad;
            }
            if (g < 0) {
                ref[k] = leaf_ref(~g, 1);
            } else {
                const int2 r = fl[g];
                ref[k] = (r.y - r.x + 1 <= leaf_max) ? leaf_ref(r.x, r.y - r.x + 1) : number_of(masks, first, g);
            }
        }
    }
    Node4 nd;
    nd.lox = make_float4(lo[0][0], lo[0][1], lo[0][2], lo[0][3]);
    nd.hix = make_float4(hi[0][0], hi[0][1], hi[0][2], hi[0][3]);
    nd.loy = make_float4(lo[1][0], lo[1][1], lo[1][2], lo[1][3]);
    nd.hiy = make_float4(hi[1][0], hi[1][1], hi[1][2], hi[1][3]);
    nd.loz = make_float4(lo[2][0], lo[2][1], lo[2][2], lo[2][3]);
    nd.hiz = make_float4(hi[2][0], hi[2][1], hi[2][2], hi[2][3]);
    nd.ref = make_int4(ref[0], ref[1], ref[2], ref[3]);
    nd.pad = make_int4(0, 0, 0, 0);
    nodes4[number_of(masks, first, i)] = nd;
}

inline unsigned blocks(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

eos_status build_lbvh(eos_scene* s, int leaf_max, int width, eos_build_stats* st) {
    const int n = s->n_tri;
    hipStream_t S = s->stream;
    s->built = false;
    s->batch_built = false;
    s->nodes_valid = false;
    s->fb.rec_valid = 0;
    s->leaf_max = leaf_max;
    s->width = width;
    s->n_nodes4 = 0;
    const size_t un = (size_t)n, m = n > 0 ? un - 1 : 0;
    const SortShape sh = sort_shape(std::max<size_t>(un, 1));
    const int nparts = n > 0 ? (int)std::min<size_t>(blocks(un, 256), 1024) : 1;
    const size_t nblk = blocks(std::max<size_t>(m, 1), kNodeBlock);
    const size_t top = pyramid_top(std::max<size_t>(un, 1));
    EOS_TRY(s->codes.ensure(4 * un));
    EOS_TRY(s->codes_sorted.ensure(4 * un));
    EOS_TRY(s->perm.ensure(4 * un));
    EOS_TRY(s->sort_tmp_k.ensure(4 * un));
    EOS_TRY(s->sort_tmp_v.ensure(4 * un));
    EOS_TRY(s->sort_hist.ensure(sort_hist_bytes(sh)));
    EOS_TRY(s->kchild.ensure(8 * m));
    EOS_TRY(s->kparent.ensure(4 * (2 * un)));
    EOS_TRY(s->first_last.ensure(8 * m));
    EOS_TRY(s->ibox.ensure(24 * m));
    EOS_TRY(s->lbox.ensure(24 * un));
    EOS_TRY(s->pyramid.ensure(24 * top));
    EOS_TRY(s->masks4.ensure(8 * kMaskWords * nblk + 4 * nblk));
    EOS_TRY(s->cbounds.ensure(64));
    EOS_TRY(s->bounds_part.ensure(24 * (size_t)nparts));
    EOS_TRY(s->shade.ensure(48 * un));
    // Room for the 4-wide nodes before their number is known: at most one per
    // internal node, and fewer than half a node per triangle when leaf_max >= 3.
    // (A standing node has k standing children among its two to four slots; with
    // none it holds at least four triangles, with one it has two other slots, with
    // two at least one unless it has four.  Counting nodes by their children,
    // S = 1 + S1 + 2 S2 + 3 S3 + 4 S4 and n >= 4 (1 + S2 + 2 S3 + 3 S4) + 2 S1.)
    const bool four = n > leaf_max;
    EOS_TRY(s->tree.ensure(s->tree_bytes(four ? (leaf_max >= 3 ? un / 2 : un) : 0)));
    EOS_HIP(hipEventRecord(s->ev[0], S));
    float* cb = s->cbounds.as<float>();
    int32_t* err = s->cbounds.as<int32_t>() + 8;   // [0] materials, [1] 4-wide nodes, [2] transformations out of range
    const bool xf = s->n_xf > 0;
    int32_t herr[4] = {0, 0, 0, 0};
    if (n > 0) {
        const float* V = s->verts.as<float>();   // keys and boxes: world space
        if (xf) {
            EOS_TRY(s->wverts.ensure(36 * un));
            hipLaunchKernelGGL(k_cbounds_partial<true>, dim3(nparts), dim3(256), 0, S, V, n,
                               s->xf_index.as<const int32_t>(), s->xf.as<const float4>(), s->n_xf,
                               s->wverts.as<float>(), s->bounds_part.as<float>());
            V = s->wverts.as<const float>();
        } else {
            hipLaunchKernelGGL(k_cbounds_partial<false>, dim3(nparts), dim3(256), 0, S, V, n, nullptr, nullptr, 0,
                               nullptr, s->bounds_part.as<float>());
        }
        hipLaunchKernelGGL(k_cbounds_final, dim3(1), dim3(384), 0, S, s->bounds_part.as<const float>(), nparts, cb, err);
        uint32_t* codes = s->codes.as<uint32_t>();
        hipLaunchKernelGGL(k_morton, dim3(blocks(un, 256)), dim3(256), 0, S, V, n, cb, codes);
        uint32_t *kA = s->codes_sorted.as<uint32_t>(), *kB = s->sort_tmp_k.as<uint32_t>();
        int32_t *vA = s->perm.as<int32_t>(), *vB = s->sort_tmp_v.as<int32_t>();
        uint32_t* H = s->sort_hist.as<uint32_t>();
        radix_pass(S, sh, codes, nullptr, kA, vA, n, 0, H);
        radix_pass(S, sh, kA, vA, kB, vB, n, kDigitBits, H);
        radix_pass(S, sh, kB, vB, kA, vA, n, 2 * kDigitBits, H);
        hipLaunchKernelGGL(k_karras, dim3(blocks(un, 256)), dim3(256), 0, S, kA, n, s->kchild.as<int2>(),
                           s->kparent.as<int32_t>(), s->first_last.as<int2>());
        hipLaunchKernelGGL(k_leaf_boxes, dim3(blocks(un, kBoxBlock)), dim3(256), 0, S, V, vA, n, s->lbox.as<float>(),
                           s->pyramid.as<float>(), top);
        if (n > kBoxBlock) hipLaunchKernelGGL(k_pyramid_top, dim3(1), dim3(1024), 0, S, n, s->pyramid.as<float>(), top);
        uint64_t* masks = s->masks4.as<uint64_t>();
        int32_t* counts = reinterpret_cast<int32_t*>(masks + kMaskWords * nblk);
        if (n > 1)
            hipLaunchKernelGGL(k_node_boxes, dim3((unsigned)nblk), dim3(kNodeBlock), 0, S,
                               s->kparent.as<const int32_t>(), s->first_last.as<const int2>(), n, leaf_max,
                               s->lbox.as<const float>(), s->pyramid.as<const float>(), top, s->ibox.as<float>(), masks,
                               counts);
        if (four) hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, S, counts, (int)nblk, err + 1);
        if (four)
            hipLaunchKernelGGL(k_nodes4, dim3(blocks(m, 256)), dim3(256), 0, S, s->kchild.as<const int2>(),
                               s->first_last.as<const int2>(), s->ibox.as<const float>(), s->lbox.as<const float>(),
                               cb, masks, counts, n, leaf_max, s->nodes4());
        hipLaunchKernelGGL(k_tris, dim3(blocks(un, 256)), dim3(256), 0, S, s->verts.as<const float>(),
                           s->normals.as<const float>(), s->matidx.as<const int32_t>(), vA, n, s->n_mat,
                           xf ? s->xf_index.as<const int32_t>() : nullptr, s->n_xf, s->geo(), s->shade.as<float4>(),
                           err);
        if (width == 2) EOS_TRY(make_binary_nodes(s));
        EOS_HIP(hipEventRecord(s->ev[1], S));
        EOS_TRY(s->ensure_host_small());
        EOS_HIP(hipMemcpyAsync(s->host_small, err, sizeof herr, hipMemcpyDeviceToHost, S));
        EOS_HIP(hipStreamSynchronize(S));
        std::copy(s->host_small, s->host_small + 4, herr);
        s->n_nodes4 = four ? herr[1] : 0;
    } else {
        EOS_HIP(hipEventRecord(s->ev[1], S));
        EOS_HIP(hipStreamSynchronize(S));
    }
    EOS_HIP(hipGetLastError());
    if (herr[0] != 0)
        return fail(EOS_ERR_INVALID, "eos_build_lbvh: " + std::to_string(herr[0]) + " material indices out of range");
    if (herr[2] != 0)
        return fail(EOS_ERR_INVALID,
                    "eos_build_lbvh: " + std::to_string(herr[2]) + " transformation indices out of range");
    float ms = 0.0f;
    EOS_HIP(hipEventElapsedTime(&ms, s->ev[0], s->ev[1]));
    if (n == 0) s->root = kDone;
    else if (n <= leaf_max) s->root = ~(0 | ((n - 1) << kLeafShift));
    else s->root = 0;
    s->root4 = s->root;
    s->built = true;
    if (st) {
        st->build_ms = ms;
        st->num_internal = n > 0 ? n - 1 : 0;
        st->root_ref = s->root;
        st->leaf_max = leaf_max;
        st->width = width;
        st->num_nodes4 = s->n_nodes4;
        st->root4 = s->root4;
    }
    return EOS_OK;
}

eos_status make_binary_nodes(eos_scene* s) {
    const size_t m = s->n_tri > 1 ? (size_t)s->n_tri - 1 : 0;
    if (s->nodes_valid || m == 0) return EOS_OK;
    EOS_TRY(s->nodes.ensure(64 * m));
    hipLaunchKernelGGL(k_nodes, dim3(blocks(m, 256)), dim3(256), 0, s->stream, s->kchild.as<const int2>(),
                       s->first_last.as<const int2>(), s->ibox.as<const float>(), s->lbox.as<const float>(),
                       s->cbounds.as<const float>(), s->n_tri, s->leaf_max, s->nodes.as<Node>());
    EOS_HIP(hipGetLastError());
    s->nodes_valid = true;
    return EOS_OK;
}

}  // namespace eos

// ---- many scenes in one launch sequence ---------------------------------------
// The scenes' triangles are concatenated (scene s at global slots
// [tri_off, tri_off + n)); every stage is one launch over all of them.  Each
// scene keeps its own centroid bounds, Morton codes and Karras tree: the sort
// orders (scene, code, index) -- three passes over the codes, then a stable pass
// over the scene index -- and the Karras kernel builds scene s's tree from the
// keys of its own segment with its own local indices, so every per-scene array
// is the one eos_build_lbvh_ex gives that scene alone, bit for bit.  Internal
// nodes of scene s sit at [node_off, node_off + n - 1) with node_off = tri_off - s,
// its parent links at [2 tri_off - s, 2 (tri_off + n) - s - 1); child references
// are local to the scene.
namespace eos {
namespace {

constexpr int kBoundsChunk = 4096;   // triangles per partial-bounds block

struct BuildSeg {
    int tri_off, n, node_off, blk_off;
    const float* verts;       // the scene's local vertices, original order
    const float* normals;
    const int32_t* mat;
    int n_mat;
    const int32_t* xi;        // transformation index per triangle (null: none)
    const float4* xf;
    int n_xf;
    Node* nodes;              // outputs: the scene's own buffers
    Node4* nodes4;
    float4* geo;
    float4* shade;
    int32_t* perm;
    uint32_t* codes_sorted;
    uint32_t* codes;
    int base4;                // global number of the scene's first 4-wide node
};

// The last segment whose offset is <= i (offsets ascending; a segment with no
// entries shares its offset with the next one, which is the one returned).
__device__ __forceinline__ int seg_of(const int* __restrict__ off, int nseg, int i) {
    int lo = 0, hi = nseg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// World-space vertices into one concatenated array.
__global__ __launch_bounds__(256) void k_bworld(const BuildSeg* __restrict__ seg, const int* __restrict__ seg_tri,
                                                int nseg, int N, float* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const BuildSeg& S = seg[seg_of(seg_tri, nseg, i)];
    const int li = i - S.tri_off;
    float w[9];
    world_vertices(S.verts + 9 * (size_t)li, S.xi ? S.xi[li] : -1, S.xf, S.n_xf, w);
#pragma unroll
    for (int k = 0; k < 9; ++k) out[9 * (size_t)i + k] = w[k];
}

// Partial centroid bounds: block b covers kBoundsChunk triangles of one scene.
__global__ __launch_bounds__(256) void k_bcb_partial(const float* __restrict__ W, const BuildSeg* __restrict__ seg,
                                                     const int* __restrict__ seg_blk, int nseg,
                                                     float* __restrict__ part) {
    const BuildSeg& S = seg[seg_of(seg_blk, nseg, (int)blockIdx.x)];
    const int lb = (int)blockIdx.x - S.blk_off;
    const int a = S.tri_off + lb * kBoundsChunk, b = min(S.tri_off + S.n, a + kBoundsChunk);
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = a + (int)threadIdx.x; i < b; i += blockDim.x) {
        float c[3];
        centroid(W, (size_t)i, c);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(lo[k], c[k]);
            hi[k] = fmaxf(hi[k], c[k]);
        }
    }
    __shared__ float s[6][256];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s[k][threadIdx.x] = lo[k];
        s[3 + k][threadIdx.x] = hi[k];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                s[k][threadIdx.x] = fminf(s[k][threadIdx.x], s[k][threadIdx.x + w]);
                s[3 + k][threadIdx.x] = fmaxf(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// One thread per (scene, component): min or max over the scene's partials.
__global__ void k_bcb_final(const float* __restrict__ part, const BuildSeg* __restrict__ seg, int nseg,
                            float* __restrict__ cb, int32_t* __restrict__ err) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 4) err[t] = 0;
    if (t >= 6 * nseg) return;
    const int sidx = t / 6, k = t - 6 * sidx;
    const BuildSeg& S = seg[sidx];
    const int nb = (S.n + kBoundsChunk - 1) / kBoundsChunk;
    float r = k < 3 ? INFINITY : -INFINITY;
    for (int b = 0; b < nb; ++b) {
        const float v = part[6 * (size_t)(S.blk_off + b) + k];
        r = k < 3 ? fminf(r, v) : fmaxf(r, v);
    }
    cb[t] = r;
}

__global__ __launch_bounds__(256) void k_bmorton(const float* __restrict__ W, const int* __restrict__ seg_tri, int nseg,
                                                 int N, const float* __restrict__ cb, uint32_t* __restrict__ codes) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float* c6 = cb + 6 * seg_of(seg_tri, nseg, i);
    float c[3];
    centroid(W, (size_t)i, c);
    const uint32_t x = quant10(c[0], c6[0], c6[3]);
    const uint32_t y = quant10(c[1], c6[1], c6[4]);
    const uint32_t z = quant10(c[2], c6[2], c6[5]);
    codes[i] = (part1by2(z) << 2) + (part1by2(y) << 1) + part1by2(x);
}

// Sort keys of the scene pass: the scene of each element.
__global__ __launch_bounds__(256) void k_bscene_keys(const int32_t* __restrict__ vals, const int* __restrict__ seg_tri,
                                                     int nseg, int N, uint32_t* __restrict__ keys) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) keys[i] = (uint32_t)seg_of(seg_tri, nseg, vals[i]);
}

// Sorted codes, and each scene's permutation and codes in its own buffers.
__global__ __launch_bounds__(256) void k_bgather(const int32_t* __restrict__ vals, const uint32_t* __restrict__ codes,
                                                 const BuildSeg* __restrict__ seg, const int* __restrict__ seg_tri,
                                                 int nseg, int N, uint32_t* __restrict__ sorted) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const BuildSeg& S = seg[seg_of(seg_tri, nseg, i)];
    const int g = vals[i], li = i - S.tri_off, o = g - S.tri_off;
    const uint32_t c = codes[g];
    sorted[i] = c;
    S.perm[li] = o;
    S.codes_sorted[li] = c;
    S.codes[o] = c;
}

// Karras over each scene's own segment: k_karras with the scene's keys, length
// and local indices; outputs at the scene's node and parent offsets.
__global__ __launch_bounds__(256) void k_bkarras(const uint32_t* __restrict__ sorted, const BuildSeg* __restrict__ seg,
                                                 const int* __restrict__ seg_tri, int nseg, int N,
                                                 int2* __restrict__ kchild, int32_t* __restrict__ kparent,
                                                 int2* __restrict__ fl) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= N) return;
    const int sidx = seg_of(seg_tri, nseg, gi);
    const BuildSeg& S = seg[sidx];
    const int n = S.n, i = gi - S.tri_off;
    if (i == 0) kparent[2 * (size_t)S.tri_off - sidx] = -1;
    if (i >= n - 1) return;
    const uint32_t* k = sorted + S.tri_off;
    const int d = (delta(k, n, i, i + 1) - delta(k, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(k, n, i, i - d);
    int lmax = 2;
    while (delta(k, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (delta(k, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(k, n, i, j);
    int s = 0;
    for (int div = 2;; div *= 2) {
        int t = (l + div - 1) / div;
        if (delta(k, n, i, i + (s + t) * d) > dnode) s += t;
        if (t <= 1) break;
    }
    const int g = i + s * d + min(d, 0);
    const int lo = min(i, j), hi = max(i, j);
    const int left = (lo == g) ? ~g : g;
    const int right = (hi == g + 1) ? ~(g + 1) : g + 1;
    kchild[S.node_off + i] = make_int2(left, right);
    fl[S.node_off + i] = make_int2(lo, hi);
    int32_t* kp = kparent + (2 * (size_t)S.tri_off - sidx);
    kp[left >= 0 ? left : (n - 1 + ~left)] = i;
    kp[right >= 0 ? right : (n - 1 + ~right)] = i;
}

// k_nodes per scene, into the scene's node array.
__global__ __launch_bounds__(256) void k_bnodes(const int2* __restrict__ kchild, const int2* __restrict__ fl,
                                                const float* __restrict__ ibox, const float* __restrict__ lbox,
                                                const float* __restrict__ cbs, const BuildSeg* __restrict__ seg,
                                                const int* __restrict__ seg_node, int nseg, int M, int leaf_max) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= M) return;
    const int sidx = seg_of(seg_node, nseg, gi);
    const BuildSeg& S = seg[sidx];
    const float* cb = cbs + 6 * sidx;
    float eps = 0.0f;
#pragma unroll
    for (int k = 0; k < 6; ++k) eps = fmaxf(eps, fabsf(cb[k]));
    eps = eps * 0x1p-22f;
    const int2 c = kchild[gi];
    float lo[2][3], hi[2][3];
    int32_t ref[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int ch = j ? c.y : c.x;
        const float* b = ch >= 0 ? ibox + 6 * (size_t)(S.node_off + ch) : lbox + 6 * (size_t)(S.tri_off + ~ch);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            float pad = inflate_pad(b[k], b[3 + k], eps);
            lo[j][k] = b[k] - pad;
            hi[j][k] = b[3 + k] + pad;
        }
        if (ch < 0) {
            ref[j] = leaf_ref(~ch, 1);
        } else {
            const int2 r = fl[S.node_off + ch];
            ref[j] = (r.y - r.x + 1 <= leaf_max) ? leaf_ref(r.x, r.y - r.x + 1) : ch;
        }
    }
    Node nd;
    nd.b0 = make_float4(lo[0][0], hi[0][0], lo[0][1], hi[0][1]);
    nd.b1 = make_float4(lo[1][0], hi[1][0], lo[1][1], hi[1][1]);
    nd.b2 = make_float4(lo[0][2], hi[0][2], lo[1][2], hi[1][2]);
    nd.c = make_int4(ref[0], ref[1], 0, 0);
    S.nodes[gi - S.node_off] = nd;
}

// k_tris per scene, into the scene's triangle records.
__global__ __launch_bounds__(256) void k_btris(const int32_t* __restrict__ vals, const BuildSeg* __restrict__ seg,
                                               const int* __restrict__ seg_tri, int nseg, int N,
                                               int32_t* __restrict__ err) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= N) return;
    const BuildSeg& S = seg[seg_of(seg_tri, nseg, gi)];
    const int s = gi - S.tri_off, o = vals[gi] - S.tri_off;
    int x = S.xi ? S.xi[o] : -1;
    if (x < -1 || x >= S.n_xf) {
        atomicAdd(err + 2, 1);
        x = -1;
    }
    const float* t = S.verts + 9 * (size_t)o;
    const float* nn = S.normals + 9 * (size_t)o;
    const float v1x = t[0], v1y = t[1], v1z = t[2];
    const float e1x = t[3] - v1x, e1y = t[4] - v1y, e1z = t[5] - v1z;
    const float e2x = t[6] - v1x, e2y = t[7] - v1y, e2z = t[8] - v1z;
    S.geo[3 * (size_t)s + 0] = make_float4(v1x, v1y, v1z, e1x);
    S.geo[3 * (size_t)s + 1] = make_float4(e1y, e1z, e2x, e2y);
    S.geo[3 * (size_t)s + 2] = make_float4(e2z, __int_as_float(o), __int_as_float(x), 0.0f);
    int m = S.mat[o];
    if (m < 0 || m >= S.n_mat) {
        atomicAdd(err, 1);
        m = 0;
    }
    S.shade[3 * (size_t)s + 0] = make_float4(nn[0], nn[1], nn[2], __int_as_float(m));
    S.shade[3 * (size_t)s + 1] = make_float4(nn[3], nn[4], nn[5], __int_as_float(x));
    S.shade[3 * (size_t)s + 2] = make_float4(nn[6], nn[7], nn[8], 0.0f);
}

// k_node_boxes over every scene's nodes (scenes of at most leaf_max triangles have
// no 4-wide nodes); the leaves are the concatenated sorted slots.
__global__ __launch_bounds__(kNodeBlock) void k_bnode_boxes(const int32_t* __restrict__ kparent,
                                                            const int2* __restrict__ fl,
                                                            const BuildSeg* __restrict__ seg,
                                                            const int* __restrict__ seg_node, int nseg, int M,
                                                            int leaf_max, const float* __restrict__ lbox,
                                                            const float* __restrict__ pyr, size_t top,
                                                            float* __restrict__ ibox, uint64_t* __restrict__ masks,
                                                            int32_t* __restrict__ counts) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    bool f = false;
    if (gi < M) {
        const int sidx = seg_of(seg_node, nseg, gi);
        const BuildSeg& S = seg[sidx];
        const int2 r = fl[gi];
        range_box(lbox, pyr, top, S.tri_off + r.x, S.tri_off + r.y).store(ibox, (size_t)gi);
        if (S.n > leaf_max && r.y - r.x + 1 > leaf_max) {
            const int32_t* kp = kparent + (2 * (size_t)S.tri_off - sidx);
            int depth = 0;
            for (int p = kp[gi - S.node_off]; p >= 0 && depth < 128; p = kp[p]) ++depth;
            f = (depth & 1) == 0;
        }
    }
    keep_flags(f, masks, counts);
}

// Per scene: 4-wide node count and global number of its first node.
__global__ void k_bcount4(const uint64_t* __restrict__ masks, const int32_t* __restrict__ first,
                          const BuildSeg* __restrict__ seg, int nseg, int32_t* __restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nseg) return;
    const BuildSeg& S = seg[t];
    int count = 0, base = 0;
    if (S.n > 1) {
        const int last = S.node_off + S.n - 2;
        base = number_of(masks, first, S.node_off);
        count = number_of(masks, first, last) + (stands(masks, last) ? 1 : 0) - base;
    }
    out[2 * t] = count;
    out[2 * t + 1] = base;
}

// k_nodes4 per scene, numbered within the scene.
__global__ __launch_bounds__(256) void k_bnodes4(const int2* __restrict__ kchild, const int2* __restrict__ fl,
                                                 const float* __restrict__ ibox, const float* __restrict__ lbox,
                                                 const float* __restrict__ cbs, const uint64_t* __restrict__ masks,
                                                 const int32_t* __restrict__ first, const BuildSeg* __restrict__ seg,
                                                 const int* __restrict__ seg_node, int nseg, int M, int leaf_max) {
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= M || !stands(masks, gi)) return;
    const int sidx = seg_of(seg_node, nseg, gi);
    const BuildSeg& S = seg[sidx];
    const float* cb = cbs + 6 * sidx;
    float eps = 0.0f;
#pragma unroll
    for (int k = 0; k < 6; ++k) eps = fmaxf(eps, fabsf(cb[k]));
    eps = eps * 0x1p-22f;
    int slots[4] = {0, 0, 0, 0};
    int ns = 0;
    const int2 c = kchild[gi];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int ch = j ? c.y : c.x;
        bool internal = false;
        if (ch >= 0) {
            const int2 r = fl[S.node_off + ch];
            internal = r.y - r.x + 1 > leaf_max;
        }
        if (internal) {
            const int2 g = kchild[S.node_off + ch];
            slots[ns++] = g.x;
            slots[ns++] = g.y;
        } else {
            slots[ns++] = ch;
        }
    }
    float lo[3][4], hi[3][4];
    int32_t ref[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        ref[k] = kEmpty;
#pragma unroll
        for (int a = 0; a < 3; ++a) lo[a][k] = hi[a][k] = INFINITY;
        if (k < ns) {
            const int g = slots[k];
            const float* b = g >= 0 ? ibox + 6 * (size_t)(S.node_off + g) : lbox + 6 * (size_t)(S.tri_off + ~g);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                float pad = inflate_pad(b[a], b[3 + a], eps);
                lo[a][k] = b[a] - pad;
                hi[a][k] = b[3 + a] + pad;
            }
            if (g < 0) {
                ref[k] = leaf_ref(~g, 1);
            } else {
                const int2 r = fl[S.node_off + g];
                ref[k] = (r.y - r.x + 1 <= leaf_max) ? leaf_ref(r.x, r.y - r.x + 1) : number_of(masks, first, S.node_off + g) - S.base4;
            }
        }
    }
    Node4 nd;
    nd.lox = make_float4(lo[0][0], lo[0][1], lo[0][2], lo[0][3]);
    nd.hix = make_float4(hi[0][0], hi[0][1], hi[0][2], hi[0][3]);
    nd.loy = make_float4(lo[1][0], lo[1][1], lo[1][2], lo[1][3]);
    nd.hiy = make_float4(hi[1][0], hi[1][1], hi[1][2], hi[1][3]);
    nd.loz = make_float4(lo[2][0], lo[2][1], lo[2][2], lo[2][3]);
    nd.hiz = make_float4(hi[2][0], hi[2][1], hi[2][2], hi[2][3]);
    nd.ref = make_int4(ref[0], ref[1], ref[2], ref[3]);
    nd.pad = make_int4(0, 0, 0, 0);
    S.nodes4[number_of(masks, first, gi) - S.base4] = nd;
}

// Scratch of the batched build (per process; calls must not overlap).
struct BatchBuild {
    DevBuf table, offs, W, part, cb, codes, kA, vA, kB, vB, sorted, hist, kchild, kparent, fl, lbox, ibox,
        pyramid, masks4, counts, misc;
    hipEvent_t ev[2] = {nullptr, nullptr};
};
BatchBuild g_bbuild;

}  // namespace

eos_status build_lbvh_batch(eos_scene* const* scenes, int n_scenes, int leaf_max, int width, eos_build_stats* st) {
    BatchBuild& B = g_bbuild;
    hipStream_t S = scenes[0]->stream;
    if (!B.ev[0]) {
        EOS_HIP(hipEventCreate(&B.ev[0]));
        EOS_HIP(hipEventCreate(&B.ev[1]));
    }
    // scenes with triangles form the segments; every scene's own buffers are sized here
    std::vector<BuildSeg> segs;
    std::vector<int> seg_scene, seg_tri, seg_node, seg_blk;
    size_t N = 0;
    int nblk = 0;
    for (int i = 0; i < n_scenes; ++i) {
        eos_scene* s = scenes[i];
        s->built = false;
        s->fb.rec_valid = 0;
        s->leaf_max = leaf_max;
        s->width = width;
        s->n_nodes4 = 0;
        s->batch_built = true;
        s->nodes_valid = true;
        const size_t un = (size_t)s->n_tri;
        if (un == 0) continue;
        if (N + un > (size_t)INT_MAX / 2)
            return fail(EOS_ERR_LIMIT, "eos_build_lbvh_batch: more than 2^30 triangles in one batch");
        EOS_TRY(s->nodes.ensure(64 * (un - 1)));
        EOS_TRY(s->shade.ensure(48 * un));
        EOS_TRY(s->perm.ensure(4 * un));
        EOS_TRY(s->codes_sorted.ensure(4 * un));
        EOS_TRY(s->codes.ensure(4 * un));
        BuildSeg g{};
        g.tri_off = (int)N;
        g.n = (int)un;
        g.node_off = (int)N - (int)segs.size();
        g.blk_off = nblk;
        g.verts = s->verts.as<const float>();
        g.normals = s->normals.as<const float>();
        g.mat = s->matidx.as<const int32_t>();
        g.n_mat = s->n_mat;
        g.xi = s->n_xf > 0 ? s->xf_index.as<const int32_t>() : nullptr;
        g.xf = s->n_xf > 0 ? s->xf.as<const float4>() : nullptr;
        g.n_xf = s->n_xf;
        g.nodes = s->nodes.as<Node>();
        g.shade = s->shade.as<float4>();
        g.perm = s->perm.as<int32_t>();
        g.codes_sorted = s->codes_sorted.as<uint32_t>();
        g.codes = s->codes.as<uint32_t>();
        segs.push_back(g);
        seg_scene.push_back(i);
        seg_tri.push_back(g.tri_off);
        seg_node.push_back(g.node_off);
        seg_blk.push_back(g.blk_off);
        nblk += (int)((un + kBoundsChunk - 1) / kBoundsChunk);
        N += un;
    }
    const int nseg = (int)segs.size();
    // wait for work already queued on the scenes' own streams (uploads, transformations)
    for (int i = 0; i < n_scenes; ++i)
        if (scenes[i]->stream != S) EOS_HIP(hipStreamSynchronize(scenes[i]->stream));
    EOS_HIP(hipEventRecord(B.ev[0], S));
    std::vector<int32_t> cnt4(2 * (size_t)std::max(nseg, 1), 0);
    int32_t herr[4] = {0, 0, 0, 0};
    if (nseg > 0) {
        const size_t M = N - (size_t)nseg;       // internal nodes of every scene
        const int Ni = (int)N, Mi = (int)M;
        const SortShape sh = sort_shape(N);
        const size_t top = pyramid_top(N), mblk = blocks(std::max<size_t>(M, 1), kNodeBlock);
        EOS_TRY(B.table.ensure(sizeof(BuildSeg) * nseg));
        EOS_TRY(B.offs.ensure(4 * 3 * (size_t)nseg));
        EOS_TRY(B.W.ensure(36 * N));
        EOS_TRY(B.part.ensure(24 * (size_t)nblk));
        EOS_TRY(B.cb.ensure(24 * (size_t)nseg));
        EOS_TRY(B.codes.ensure(4 * N));
        EOS_TRY(B.kA.ensure(4 * N));
        EOS_TRY(B.vA.ensure(4 * N));
        EOS_TRY(B.kB.ensure(4 * N));
        EOS_TRY(B.vB.ensure(4 * N));
        EOS_TRY(B.sorted.ensure(4 * N));
        EOS_TRY(B.hist.ensure(sort_hist_bytes(sh)));
        EOS_TRY(B.pyramid.ensure(24 * top));
        EOS_TRY(B.masks4.ensure(8 * kMaskWords * mblk + 4 * mblk));
        EOS_TRY(B.kchild.ensure(8 * M + 8));
        EOS_TRY(B.kparent.ensure(4 * (2 * N)));
        EOS_TRY(B.fl.ensure(8 * M + 8));
        EOS_TRY(B.lbox.ensure(24 * N));
        EOS_TRY(B.ibox.ensure(24 * M + 24));
        EOS_TRY(B.counts.ensure(8 * (size_t)nseg));
        EOS_TRY(B.misc.ensure(64));
        std::vector<int> offs;
        offs.insert(offs.end(), seg_tri.begin(), seg_tri.end());
        offs.insert(offs.end(), seg_node.begin(), seg_node.end());
        offs.insert(offs.end(), seg_blk.begin(), seg_blk.end());
        EOS_HIP(hipMemcpyAsync(B.table.ptr, segs.data(), sizeof(BuildSeg) * nseg, hipMemcpyHostToDevice, S));
        EOS_HIP(hipMemcpyAsync(B.offs.ptr, offs.data(), 4 * offs.size(), hipMemcpyHostToDevice, S));
        const BuildSeg* T = B.table.as<const BuildSeg>();
        const int* o_tri = B.offs.as<const int>();
        const int* o_node = o_tri + nseg;
        const int* o_blk = o_node + nseg;
        int32_t* err = B.misc.as<int32_t>();           // [0] materials, [1] 4-wide nodes, [2] transformations
        float* W = B.W.as<float>();
        hipLaunchKernelGGL(k_bworld, dim3(blocks(N, 256)), dim3(256), 0, S, T, o_tri, nseg, Ni, W);
        hipLaunchKernelGGL(k_bcb_partial, dim3(nblk), dim3(256), 0, S, W, T, o_blk, nseg, B.part.as<float>());
        hipLaunchKernelGGL(k_bcb_final, dim3(blocks(6 * (size_t)nseg, 64)), dim3(64), 0, S, B.part.as<const float>(),
                           T, nseg, B.cb.as<float>(), err);
        uint32_t* kA = B.kA.as<uint32_t>();
        int32_t* vA = B.vA.as<int32_t>();
        uint32_t* kB = B.kB.as<uint32_t>();
        int32_t* vB = B.vB.as<int32_t>();
        uint32_t* codes = B.codes.as<uint32_t>();
        hipLaunchKernelGGL(k_bmorton, dim3(blocks(N, 256)), dim3(256), 0, S, W, o_tri, nseg, Ni, B.cb.as<const float>(),
                           codes);
        // three passes over the codes, then one (two beyond 1,024 scenes) over the scene index
        uint32_t* H = B.hist.as<uint32_t>();
        radix_pass(S, sh, codes, nullptr, kA, vA, Ni, 0, H);
        radix_pass(S, sh, kA, vA, kB, vB, Ni, kDigitBits, H);
        radix_pass(S, sh, kB, vB, kA, vA, Ni, 2 * kDigitBits, H);
        hipLaunchKernelGGL(k_bscene_keys, dim3(blocks(N, 256)), dim3(256), 0, S, vA, o_tri, nseg, Ni, kA);
        radix_pass(S, sh, kA, vA, kB, vB, Ni, 0, H);
        const int32_t* vS = vB;
        if (nseg > kDigits) {
            radix_pass(S, sh, kB, vB, kA, vA, Ni, kDigitBits, H);
            vS = vA;
        }
        uint32_t* sorted = B.sorted.as<uint32_t>();
        hipLaunchKernelGGL(k_bgather, dim3(blocks(N, 256)), dim3(256), 0, S, vS, B.codes.as<const uint32_t>(), T, o_tri,
                           nseg, Ni, sorted);
        int32_t* kparent = B.kparent.as<int32_t>();
        int2* kchild = B.kchild.as<int2>();
        int2* fl = B.fl.as<int2>();
        hipLaunchKernelGGL(k_bkarras, dim3(blocks(N, 256)), dim3(256), 0, S, sorted, T, o_tri, nseg, Ni, kchild,
                           kparent, fl);
        hipLaunchKernelGGL(k_leaf_boxes, dim3(blocks(N, kBoxBlock)), dim3(256), 0, S, W, vS, Ni, B.lbox.as<float>(),
                           B.pyramid.as<float>(), top);
        if (Ni > kBoxBlock)
            hipLaunchKernelGGL(k_pyramid_top, dim3(1), dim3(1024), 0, S, Ni, B.pyramid.as<float>(), top);
        uint64_t* masks = B.masks4.as<uint64_t>();
        int32_t* first4 = reinterpret_cast<int32_t*>(masks + kMaskWords * mblk);
        if (M > 0) {
            hipLaunchKernelGGL(k_bnode_boxes, dim3((unsigned)mblk), dim3(kNodeBlock), 0, S, kparent, fl, T, o_node,
                               nseg, Mi, leaf_max, B.lbox.as<const float>(), B.pyramid.as<const float>(), top,
                               B.ibox.as<float>(), masks, first4);
            hipLaunchKernelGGL(k_bnodes, dim3(blocks(M, 256)), dim3(256), 0, S, kchild, fl, B.ibox.as<const float>(),
                               B.lbox.as<const float>(), B.cb.as<const float>(), T, o_node, nseg, Mi, leaf_max);
            // 4-wide collapse: one numbering over every scene's nodes, per-scene counts
            hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, S, first4, (int)mblk, err + 1);
            hipLaunchKernelGGL(k_bcount4, dim3(blocks((size_t)nseg, 64)), dim3(64), 0, S, masks, first4, T, nseg,
                               B.counts.as<int32_t>());
            EOS_HIP(hipMemcpyAsync(cnt4.data(), B.counts.ptr, 8 * (size_t)nseg, hipMemcpyDeviceToHost, S));
            EOS_HIP(hipStreamSynchronize(S));
        }
        for (int k = 0; k < nseg; ++k) {
            eos_scene* s = scenes[seg_scene[k]];
            s->n_nodes4 = cnt4[2 * k];
            EOS_TRY(s->tree.ensure(s->tree_bytes((size_t)s->n_nodes4)));
            segs[k].nodes4 = s->nodes4();
            segs[k].geo = s->geo();
            segs[k].base4 = cnt4[2 * k + 1];
        }
        EOS_HIP(hipMemcpyAsync(B.table.ptr, segs.data(), sizeof(BuildSeg) * nseg, hipMemcpyHostToDevice, S));
        if (M > 0)
            hipLaunchKernelGGL(k_bnodes4, dim3(blocks(M, 256)), dim3(256), 0, S, kchild, fl, B.ibox.as<const float>(),
                               B.lbox.as<const float>(), B.cb.as<const float>(), masks, first4, T, o_node, nseg, Mi,
                               leaf_max);
        hipLaunchKernelGGL(k_btris, dim3(blocks(N, 256)), dim3(256), 0, S, vS, T, o_tri, nseg, Ni, err);
        EOS_HIP(hipGetLastError());
        EOS_HIP(hipMemcpyAsync(herr, err, 12, hipMemcpyDeviceToHost, S));
    }
    EOS_HIP(hipEventRecord(B.ev[1], S));
    EOS_HIP(hipStreamSynchronize(S));
    if (herr[0] != 0)
        return fail(EOS_ERR_INVALID, "eos_build_lbvh_batch: " + std::to_string(herr[0]) + " material indices out of range");
    if (herr[2] != 0)
        return fail(EOS_ERR_INVALID,
                    "eos_build_lbvh_batch: " + std::to_string(herr[2]) + " transformation indices out of range");
    float ms = 0.0f;
    EOS_HIP(hipEventElapsedTime(&ms, B.ev[0], B.ev[1]));
    for (int i = 0; i < n_scenes; ++i) {
        eos_scene* s = scenes[i];
        const int n = s->n_tri;
        if (n == 0) s->root = kDone;
        else if (n <= leaf_max) s->root = ~(0 | ((n - 1) << kLeafShift));
        else s->root = 0;
        s->root4 = s->root;
        s->built = true;
        if (st) {
            st[i].build_ms = ms;
            st[i].num_internal = n > 0 ? n - 1 : 0;
            st[i].root_ref = s->root;
            st[i].leaf_max = leaf_max;
            st[i].width = width;
            st[i].num_nodes4 = s->n_nodes4;
            st[i].root4 = s->root4;
        }
    }
    return EOS_OK;
}

}  // namespace eos
