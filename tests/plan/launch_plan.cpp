// The launch shapes of eos_amd/csrc/launch_plan.h behind a C interface.
#include "launch_plan.h"

extern "C" {

// out: lanes per ray, chunk, chunks, runs, scan blocks, merge blocks, the scan
// launch's and the merge launch's work items in x, bytes of the runs
void plan_linear(int n, int n_tri, int fixed_scratch, long long* out) {
    const eos::LinSplit s = eos::linear_split(n, n_tri, fixed_scratch ? eos::kLinStaticRuns : eos::kLinRuns);
    out[0] = s.lanes_per_ray;
    out[1] = s.chunk;
    out[2] = s.n_chunks;
    out[3] = (long long)s.runs;
    out[4] = s.scan_blocks;
    out[5] = s.merge_blocks;
    out[6] = (long long)s.scan_blocks * eos::kLinTile;
    out[7] = (long long)s.merge_blocks * eos::kLinMergeThreads;
    out[8] = (long long)(s.runs * eos::kLinRunBytes);
}

// out: workgroups, lanes with an overflow stack
void plan_query(long long n, int resident, long long* out) {
    const int grid = eos::query_grid((size_t)n, resident);
    out[0] = grid;
    out[1] = (long long)eos::query_stack_lanes((size_t)n, grid);
}

// out: scatter of chain frames, of batches and ray trees, of queries; refill of queries
void plan_knobs(int refill, int scatter, int* out) {
    out[0] = eos::frame_scatter(scatter, false);
    out[1] = eos::frame_scatter(scatter, true);
    out[2] = eos::query_scatter(scatter);
    out[3] = eos::query_refill(refill);
}

long long plan_max_launch_items() { return (long long)eos::kMaxLaunchItems; }
}
