// qk_readback.hip -- kernels that lay results out for the host: fields as
// the caller's interleaved (node, component) order, particle records as
// compact rows of the live slots.  They write into pinned host memory, in
// the region's precision; the host threads of qk_drain.h widen each block to
// FP64 in the caller's array while the next blocks are written.
//
// Bound by the host link: 55 GB/s for kernel stores to pinned memory,
// whatever the launch width (64 to 4096 workgroups, 4 or 16 bytes per lane).
// The records cross it in 4 or 8 bytes per number, not widened.
#include <algorithm>

#include "qk_kernels.h"

namespace qk {

namespace {

constexpr int kRBlock = 256;
constexpr int kPackBlocks = 128;   // workgroups of a pack kernel: the link is full from 64 on

// Every workgroup of a pack kernel ends here: the last one to arrive, with
// all stores of the launch visible to the host, writes the sequence number
// the host polls.  (With HIP events instead, the runtime's handler thread
// competed with the caller's own thread pool: one read of 128^3 cells in
// three was followed by 10 to 40 ms during which the caller's next parallel
// loop waited for a CPU.)
__device__ inline void signal_done(const ReadDone &d)
{
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x != 0) return;
    if (atomicAdd(d.arrived, 1u) != gridDim.x - 1) return;
    *d.arrived = 0;
    __threadfence_system();
    __hip_atomic_store(d.flag, d.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[3 m + c] = component c at node first + m: one number per thread, so a
// wavefront's stores are one contiguous run
template <typename real>
__global__ void __launch_bounds__(kRBlock) k_pack_fields(const real *__restrict__ a, const real *__restrict__ b,
                                                         const real *__restrict__ c, int64_t first, int n, real *out,
                                                         ReadDone done)
{
    for (int t = blockIdx.x * kRBlock + threadIdx.x; t < 3 * n; t += gridDim.x * kRBlock) {
        const int m = t / 3, comp = t - 3 * m;
        const real *src = comp == 0 ? a : (comp == 1 ? b : c);
        out[t] = src[first + m];
    }
    signal_done(done);
}

__global__ void __launch_bounds__(kRBlock) k_copy_out(const double *__restrict__ src, int n, double *out, ReadDone done)
{
    for (int t = blockIdx.x * kRBlock + threadIdx.x; t < n; t += gridDim.x * kRBlock) out[t] = src[t];
    signal_done(done);
}

// live particles per run of kLiveRun slots
__global__ void __launch_bounds__(kRBlock) k_count_live(const int *__restrict__ cell, int64_t n, int *__restrict__ counts)
{
    __shared__ int part[kRBlock / 64];
    const int64_t s = (int64_t)blockIdx.x * kLiveRun;
    int live = 0;
#pragma unroll
    for (int m = 0; m < kLiveRun / kRBlock; ++m) {
        const int64_t p = s + m * kRBlock + threadIdx.x;
        live += p < n && cell[p] >= 0;
    }
    for (int o = 32; o > 0; o >>= 1) live += __shfl_xor(live, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = live;
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
        for (int w = 0; w < kRBlock / 64; ++w) sum += part[w];
        counts[blockIdx.x] = sum;
    }
}

// rows of the live slots of [first, first + n), first a multiple of kLiveRun,
// in slot order: row r of the block is the r-th live slot.  A workgroup
// takes whole runs; a run's first row is its scanned count.  Each array of
// the block holds `stride` entries.
template <typename real>
__global__ void __launch_bounds__(kRBlock) k_pack_live(Species<real> s, int64_t first, int64_t end,
                                                       const int *__restrict__ offs, int stride, int *cell_out,
                                                       real *real_out, int *id_out, ReadDone done)
{
    __shared__ int part[kRBlock / 64];
    const int run0 = (int)(first / kLiveRun);
    const int turns = kLiveRun / kRBlock, runs = (int)((end - first + kLiveRun - 1) / kLiveRun);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int row = 0;
    for (int x = 0, run = blockIdx.x; run < runs; ++x, run += x % turns == 0 ? (int)gridDim.x : 0) {
        const int m = x % turns;
        if (m == 0) row = offs[run0 + run] - offs[run0];
        const int64_t p = first + (int64_t)run * kLiveRun + m * kRBlock + threadIdx.x;
        const int c = p < end ? s.cell[p] : -1;
        const unsigned long long mask = __ballot(c >= 0);
        if (lane == 0) part[w] = __popcll(mask);
        __syncthreads();
        int before = 0, total = 0;
        for (int k = 0; k < kRBlock / 64; ++k) {
            before += k < w ? part[k] : 0;
            total += part[k];
        }
        __syncthreads();   // part is rewritten in the next turn
        if (c >= 0) {
            const int r = row + before + __popcll(mask & ((1ull << lane) - 1ull));
            cell_out[r] = c;
            const real v[7] = {s.ox[p], s.oy[p], s.oz[p], s.ux[p], s.uy[p], s.uz[p], s.q[p]};
#pragma unroll
            for (int a = 0; a < 7; ++a) real_out[(int64_t)a * stride + r] = v[a];
            if (s.chi) real_out[(int64_t)7 * stride + r] = s.chi[p];
            if (s.id) id_out[r] = s.id[p];
        }
        row += total;
    }
    signal_done(done);
}

inline unsigned pack_blocks(int64_t n) { return (unsigned)std::min<int64_t>(kPackBlocks, (n + kRBlock - 1) / kRBlock); }

}  // namespace

template <typename real>
hipError_t launch_pack_fields(hipStream_t st, const real *a, const real *b, const real *c, int64_t first, int n, real *out,
                              const ReadDone &done)
{
    if (n <= 0) return hipErrorInvalidValue;   // nothing would set the flag
    k_pack_fields<real><<<pack_blocks(3 * (int64_t)n), kRBlock, 0, st>>>(a, b, c, first, n, out, done);
    return hipGetLastError();
}

hipError_t launch_copy_out(hipStream_t st, const double *src, int n, double *out, const ReadDone &done)
{
    if (n <= 0) return hipErrorInvalidValue;
    k_copy_out<<<pack_blocks(n), kRBlock, 0, st>>>(src, n, out, done);
    return hipGetLastError();
}

hipError_t launch_count_live(hipStream_t st, const int *cell, int64_t n, int *counts)
{
    if (n <= 0) return hipSuccess;
    k_count_live<<<(unsigned)((n + kLiveRun - 1) / kLiveRun), kRBlock, 0, st>>>(cell, n, counts);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_pack_live(hipStream_t st, const Species<real> &s, int64_t first, int64_t end, const int *offs,
                            int stride, int *cell_out, real *real_out, int *id_out, const ReadDone &done)
{
    if (end <= first) return hipErrorInvalidValue;
    k_pack_live<real><<<pack_blocks(end - first), kRBlock, 0, st>>>(s, first, end, offs, stride, cell_out, real_out,
                                                                   id_out, done);
    return hipGetLastError();
}

#define QK_INST(real)                                                                                            \
    template hipError_t launch_pack_fields<real>(hipStream_t, const real *, const real *, const real *, int64_t, int, \
                                                 real *, const ReadDone &);                                                        \
    template hipError_t launch_pack_live<real>(hipStream_t, const Species<real> &, int64_t, int64_t, const int *, int, \
                                               int *, real *, int *, const ReadDone &);
QK_INST(float)
QK_INST(double)
#undef QK_INST

}  // namespace qk
