// hp_batch_kernels.hip -- persistent sweep kernels over a batch of boxes
// (throughput arithmetic of hp_fast.h, FP contraction on).  Each wave takes
// work units u = wave, wave + nwaves, ... of one plan table, finds the box by
// binary search over the table's unit prefix sums, and runs the same per-box
// sweep bodies as the single-box kernels (x_run / stream_run).  Every box
// uses the comoving form of the tracing (at = 1, dat = 0 for a static box);
// gravity is not supported in a batch.
#include "hp_batch.h"
#include "hp_sweep.h"

namespace hp {

__device__ __forceinline__ int table_find(const BatchTable& T, int u)
{
    int lo = 0, hi = T.n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (T.start[mid] <= u) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ void batch_view(const BatchBox& X, int slot, BoxView& V, Epilogue& E)
{
    int in, out, old;
    batch_sets(X.nsets, X.st->nstep_done, slot, in, out, old);
    in = __builtin_amdgcn_readfirstlane(in);
    out = __builtin_amdgcn_readfirstlane(out);
    old = __builtin_amdgcn_readfirstlane(old);
#pragma unroll
    for (int f = 0; f < 5; ++f) {
        V.in[f] = X.f[in][f];
        V.out[f] = X.f[out][f];
    }
    V.gforce = nullptr;
    V.prm = X.prm;
    V.st = X.st;
    V.nx = X.nx; V.ny = X.ny; V.nz = X.nz; V.nb = X.nb;
    const bool exp = slot == 2 && old >= 0;
    E.old[0] = exp ? X.f[old][0] : nullptr;
    E.old[1] = exp ? X.f[old][2] : nullptr;
    E.old[2] = exp ? X.f[old][3] : nullptr;
    E.old[3] = exp ? X.f[old][4] : nullptr;
    E.fac = X.st->fac;
    E.afact = E.afact1 = E.afact2 = 0.0;
    if (exp) {
        load_factors(E);
        E.afact = wave_uniform(E.afact);
        E.afact1 = wave_uniform(E.afact1);
        E.afact2 = wave_uniform(E.afact2);
    }
    E.ghost_mask = 7;
    E.do_speed = slot == 2;
}

template <class M, class R, bool EXP>
__global__ void __launch_bounds__(256) batch_x(const BatchBox* __restrict__ boxes, const BatchPlan* __restrict__ plan,
                                               int key, int slot)
{
    const BatchTable& T = plan->t[key];
    const int total = T.total;
    const int nwaves = (gridDim.x * blockDim.x) >> 6;
    // unit indices are wave-uniform; readfirstlane lets the table search and
    // the descriptor loads run on the scalar unit
    const int u0 = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    int cur = -1;                                    // box whose tallies t holds
    Tally t = tally0();
    for (int u = u0; u < total; u += nwaves) {
        const int i = __builtin_amdgcn_readfirstlane(table_find(T, u));
        const int b = __builtin_amdgcn_readfirstlane(T.box[i]);
        if (b != cur) {                              // one flush per box a wave visits
            if (cur >= 0) flush_counters(boxes[cur].st, t, slot == 2);
            t = tally0();
            cur = b;
        }
        const BatchBox& X = boxes[b];
        const int local = __builtin_amdgcn_readfirstlane(u - T.start[i]);
        BoxView V;
        Epilogue E;
        batch_view(X, slot, V, E);
        const unsigned nchunks = x_chunks(X.nx, X.ny, X.nz, X.nb);
        const unsigned c0 = (unsigned)local * (unsigned)X.xcpu;
        const unsigned c1 = min(c0 + (unsigned)X.xcpu, nchunks);
        const AllScalars<R> A = wave_uniform(load_scalars<M, R>(X.prm, X.st));
        x_run<M, R, false, true, EXP>(V, A, E, c0, c1, t);
    }
    if (cur >= 0) flush_counters(boxes[cur].st, t, slot == 2);
}

// Waves per SIMD as the single-box comoving sweeps (stream_waves): three for
// gamma = 5/3, two else; held there the bodies fit without a spill, left to
// itself the allocator takes a few registers more and a wave is lost.
template <class M, class R, int DIR, bool EXP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(stream_waves(M::G53, false))))
batch_stream(const BatchBox* __restrict__ boxes, const BatchPlan* __restrict__ plan, int key, int slot)
{
    __shared__ double window[stream_lds<false>() * 256];
    const BatchTable& T = plan->t[key];
    const int total = T.total;
    const int nwaves = (gridDim.x * blockDim.x) >> 6;
    // unit indices are wave-uniform; readfirstlane lets the table search and
    // the descriptor loads run on the scalar unit
    const int u0 = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    int cur = -1;
    Tally t = tally0();
    double* const column = stream_column<false>(window);
    reset_rare<false>(column);
    for (int u = u0; u < total; u += nwaves) {
        const int i = __builtin_amdgcn_readfirstlane(table_find(T, u));
        const int b = __builtin_amdgcn_readfirstlane(T.box[i]);
        if (b != cur) {
            if (cur >= 0) {
                take_rare<false>(column, t);
                flush_counters(boxes[cur].st, t, slot == 2);
            }
            t = tally0();
            reset_rare<false>(column);
            cur = b;
        }
        const BatchBox& X = boxes[b];
        const int local = __builtin_amdgcn_readfirstlane(u - T.start[i]);
        BoxView V;
        Epilogue E;
        batch_view(X, slot, V, E);
        const int Nbb = (DIR == 2) ? X.nz - 2 * X.nb : X.ny - 2 * X.nb;
        const StreamItem I = stream_item((unsigned)local, threadIdx.x & 63u, (unsigned)((X.nx - 2 * X.nb) * Nbb),
                                         (unsigned)X.nseg[DIR - 2]);
        const AllScalars<R> A = wave_uniform(load_scalars<M, R>(X.prm, X.st));
        stream_run<M, R, DIR, false, true, EXP>(V, A, E, I.pen, (int)I.seg, X.seglen[DIR - 2], I.active, t, column);
    }
    if (cur >= 0) {
        take_rare<false>(column, t);
        flush_counters(boxes[cur].st, t, slot == 2);
    }
}

template <class M, class R, bool EXP>
static void launch_dir(const BatchBox* boxes, const BatchPlan* plan, int key, int slot, int dir, int most,
                       int ncu, hipStream_t s)
{
    // blocks of four waves a CU holds: one for each wave of a SIMD
    constexpr int X = batch_x_waves(M::G53, sizeof(R) == 4), YZ = stream_waves(M::G53, false);
    const int grid = std::min(most, ncu * (dir == 1 ? X : YZ));
    if (dir == 1) hipLaunchKernelGGL((batch_x<M, R, EXP>), dim3(grid), dim3(256), 0, s, boxes, plan, key, slot);
    else if (dir == 2)
        hipLaunchKernelGGL((batch_stream<M, R, 2, EXP>), dim3(grid), dim3(256), 0, s, boxes, plan, key, slot);
    else hipLaunchKernelGGL((batch_stream<M, R, 3, EXP>), dim3(grid), dim3(256), 0, s, boxes, plan, key, slot);
}

template <class M>
static void launch_m(const BatchBox* boxes, const BatchPlan* plan, int key, int slot, int dir, int prec, int exp,
                     int grid, int ncu, hipStream_t s)
{
    if (prec == PREC_MIXED) {
        if (exp) launch_dir<M, float, true>(boxes, plan, key, slot, dir, grid, ncu, s);
        else launch_dir<M, float, false>(boxes, plan, key, slot, dir, grid, ncu, s);
    } else {
        if (exp) launch_dir<M, double, true>(boxes, plan, key, slot, dir, grid, ncu, s);
        else launch_dir<M, double, false>(boxes, plan, key, slot, dir, grid, ncu, s);
    }
}

hipError_t launch_batch_sweep(const BatchBox* boxes, const BatchPlan* plan, int slot, int dir, int prec, int exp,
                              int g53, int grid, int ncu, hipStream_t s)
{
    if (slot < 0 || slot > 2 || dir < 1 || dir > 3 || grid < 1) return hipErrorInvalidValue;
    const int key = table_key(slot, dir, prec, exp, g53);
    if (g53) launch_m<FastMath53>(boxes, plan, key, slot, dir, prec, exp, grid, ncu, s);
    else launch_m<FastMath>(boxes, plan, key, slot, dir, prec, exp, grid, ncu, s);
    return hipGetLastError();
}

}  // namespace hp
