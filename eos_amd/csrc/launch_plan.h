// launch_plan.h -- how host code shapes launches and their scratch from sizes
// alone.  Plain C++ (no HIP), so that the shapes are checked without a GPU at sizes
// that no test renders.
#pragma once
#include <algorithm>
#include <cstddef>

#include "eos_c.h"

namespace eos {

// HIP refuses a launch dimension of 2^32 work items or more.
constexpr size_t kMaxLaunchItems = (size_t)1 << 32;

// ---- linear ray queries (every ray against every triangle) ---------------------
constexpr int kLinTile = 256;           // triangles staged at a time, and threads of the scanning kernels
constexpr int kLinMergeThreads = 256;   // four rays, a wave each
constexpr size_t kLinBlocks = 2048;     // scanning workgroups wanted
constexpr size_t kLinRunBytes = 32;     // one ray's run over one chunk of triangles, and its head
constexpr size_t kLinRuns = (size_t)1 << 20;   // kept at most
constexpr size_t kLinStaticRuns = (size_t)EOS_STATIC_MAX_RAYS / 2;   // by eos_trace_rays_static: 16 bytes per ray of scratch
constexpr int kLinFewRays = 128;        // up to here a ray's triangles are shared out over lanes as well

struct LinSplit {
    int lanes_per_ray = 1;      // a power of two up to 64
    int chunk = 0;              // triangles per chunk, a multiple of kLinTile
    int n_chunks = 1;
    size_t runs = 0;            // runs kept for the merge; 0: the scanning kernel writes the answers
    unsigned scan_blocks = 0;   // times n_chunks
    unsigned merge_blocks = 0;
};

// n rays (n >= 1) against n_tri triangles: as many chunks as give kLinBlocks
// workgroups, at most one per kLinTile triangles, and runs within max_runs.  One
// chunk needs no merge unless lanes share its rays: a merge there is a wave per
// ray for a single run, 64 n work items, which passes the launch limit from 2^26
// rays on.
inline LinSplit linear_split(int n, int n_tri, size_t max_runs) {
    LinSplit r;
    if (n <= kLinFewRays)
        while (r.lanes_per_ray < 64 && 2 * r.lanes_per_ray * n <= kLinTile) r.lanes_per_ray *= 2;
    const size_t blocks = ((size_t)n * r.lanes_per_ray + kLinTile - 1) / kLinTile;
    const size_t tiles = std::max<size_t>(1, ((size_t)n_tri + kLinTile - 1) / kLinTile);
    size_t c = std::min(tiles, (kLinBlocks + blocks - 1) / blocks);
    c = std::max<size_t>(1, std::min({c, max_runs / (size_t)n, (size_t)65535}));
    const size_t per = (tiles + c - 1) / c;
    r.chunk = (int)(per * kLinTile);
    r.n_chunks = (int)((tiles + per - 1) / per);
    r.scan_blocks = (unsigned)blocks;
    if (r.n_chunks > 1 || r.lanes_per_ray > 1) {
        r.runs = (size_t)n * (size_t)r.n_chunks;
        r.merge_blocks = (unsigned)(((size_t)n + kLinMergeThreads / 64 - 1) / (kLinMergeThreads / 64));
    }
    return r;
}

// ---- launch knobs ---------------------------------------------------------------
// The defaults of refill and scatter were measured on single frames of chains of
// reflections.  Where other launches measured better with another value, the
// default stands for that value there; a caller's own setting is taken as it is.
constexpr int kRefillDefault = 16, kScatterDefault = 4;

// Batched frames and ray trees scatter their claims up to two items per lane: beyond
// that the order's locality is worth more than the balance.  16 random scenes 4434 us
// with four, 3993 with two or none; eight of 30,000 triangles 2027 with five, 1916
// with two; three or sixteen small ones, whose launches have one item per lane, the
// same with one to five, 5-12% more with none.  Four glass samples in flight 2647 with
// four, 2497 with two, 2576 with none; single glass frames of 700 x 400 to 1920 x 1080
// within 4% with any.  A chain frame of 4.2M triangles 1729 with four, 1732 with two,
// 1904 with none.
inline int frame_scatter(int scatter, bool batch_or_tree) {
    return batch_or_tree && scatter == kScatterDefault ? 2 : scatter;
}

// A caller's rays diverge from the first node, so a refill that waits for twice as
// many idle lanes loses little and is paid half as often: 1M nearest rays 543 ->
// 521 us, 500,000 occlusion rays 408 -> 379; over four scenes, both modes and 3,000
// to 1M rays 32 idle lanes against 17 are 0-10% faster, but for 30,000 nearest rays
// among random triangles, 3% slower.
inline int query_refill(int refill) { return refill == kRefillDefault ? 2 * refill : refill; }

// Rays of a caller come in any order: claims are scattered only while a lane has
// one ray (1M rays 568 us with up to four per lane scattered, 555 without; 1M
// occlusion rays 3-5% slower scattered, fewer rays the same).
inline int query_scatter(int scatter) { return scatter == kScatterDefault ? 1 : scatter; }

// ---- tree queries (eos_trace_rays) ----------------------------------------------
constexpr int kQueryThreads = 256;

// Workgroups of a query's traversal launch: room for the walk of a whole wave per
// ray (two waves per ray; waves beyond the rays leave at once), never more than the
// persistent grid of `resident` workgroups.  With a quad per ray the launch was too
// small for any group walk: 1,000 host rays against 70k triangles 142 us, now 83.
inline int query_grid(size_t n, int resident) {
    return (int)std::min<size_t>((size_t)resident, std::max<size_t>(1, (128 * n + kQueryThreads - 1) / kQueryThreads));
}

// Lanes of that launch that can have a stack outgrow LDS: those of the walk with a
// ray per lane, whose waves beyond the ones that n rays fill leave before they touch
// it.  Group and wave walks keep their stacks in LDS.  (Sized for the whole grid, a
// scene's first query of 1,000 rays allocated 40 MiB.)
inline size_t query_stack_lanes(size_t n, int grid) {
    return std::min((size_t)grid * kQueryThreads, 64 * ((n + 63) / 64));
}

}  // namespace eos
