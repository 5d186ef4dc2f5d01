// qk_fields.hip -- field kernels of the step on gfx950: the three Maxwell
// solvers (FDTD, NDFX, five-point) with the reference's boundary-plane sets,
// B interpolation to E positions, boundary zeroing, the laser initial
// condition and the FP64 field-energy reduction.
//
// Fields are structure-of-arrays, one array per component, [nx][ny][nz] with
// k fastest; a thread owns one cell and consecutive lanes walk k, so every
// stencil load of a wavefront is a coalesced run.
#include "qk_kernels.h"

namespace qk {

namespace {

constexpr int kBX = 64, kBY = 4;   // workgroup: 64 lanes along k, 4 rows along j

inline dim3 cell_grid(const Grid &g) { return dim3((g.nz + kBX - 1) / kBX, (g.ny + kBY - 1) / kBY, g.nx); }

// Block order of the field sweeps (grid x along k, y along j, z along the
// planes).  The hardware deals blocks to the 8 XCDs round-robin by linear
// index, which puts neighbouring rows of blocks on different XCDs (and
// L2s).  Here the planes still advance in lock-step over the XCDs, but each
// XCD takes one contiguous band of block rows in every plane, so a block
// finds the row above its own in its XCD's L2 (the neighbour plane is read
// by the same XCD a few blocks later, as before).  Field phase 1.18 -> 1.15
// ms at 512x256x256 and 0.145 -> 0.138 ms at 256x128x128; a contiguous
// range of whole planes per XCD was faster at the smaller grid only.
__device__ inline dim3 band_block()
{
    const int P = gridDim.x * gridDim.y;   // blocks per plane (run of planes)
    if (P % 8 != 0) return blockIdx;
    const int hb = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int x = hb % 8, l = hb / 8, q = P / 8;
    const int vin = x * q + l % q;
    return dim3((unsigned)(vin % gridDim.x), (unsigned)(vin / gridDim.x), (unsigned)(l / q));
}

// The Maxwell sweeps take a plane's cells as one run (j, k flattened), in
// blocks of kSweep, so that no lane is idle whatever nz is (64-column blocks
// left 22 % of them idle at nz = 199, 45 % at 71 and half at 32).  Planes of
// at least kBandMin blocks are dealt to the XCDs in bands as above, the
// blocks per plane rounded up to a multiple of 8 (under 12 % empty blocks);
// smaller ones in launch order.  Bound by HBM (3.0 -> 4.2 TB/s at 301x203x199,
// where a plain copy reaches 4.8): B 145 -> 102 us there, 13.4 -> 10.2 us at
// 135x75x71 (NDFX), 285 -> 277 us at 512x256x256, 35.6 -> 37.1 us at
// 256x128x128 (NDFX; the division per cell).
constexpr int kSweep = 256, kBandMin = 64;

struct SweepPlan {
    int per;      // blocks per plane, empty ones included
    bool banded;
};

inline SweepPlan sweep_plan(const Grid &g)
{
    const int P = (g.sx + kSweep - 1) / kSweep;
    return P >= kBandMin ? SweepPlan{(P + 7) / 8 * 8, true} : SweepPlan{P, false};
}

// this thread's cell; false past the plane's end
__device__ inline bool sweep_cell(const Grid &g, const SweepPlan &sw, int &i, int &j, int &k)
{
    int vin;
    if (sw.banded) {
        const int q = sw.per / 8, l = blockIdx.x / 8;
        i = l / q;
        vin = (int)(blockIdx.x % 8) * q + l % q;
    } else {
        i = blockIdx.x / sw.per;
        vin = blockIdx.x % sw.per;
    }
    const int t = vin * kSweep + (int)threadIdx.x;
    j = t / g.nz;
    k = t - j * g.nz;
    return t < g.sx;
}

__device__ inline bool in(int v, int lo, int hi) { return v >= lo && v <= hi; }

// which cells get component C of B updated
// (FDTD src/maxwell.cpp:445-484, NDFX :251-290, five-point :35-85)
template <int S, int C>
__device__ inline bool b_updates(const Grid &g, int i, int j, int k)
{
    const int c[3] = {i, j, k}, n[3] = {g.nx, g.ny, g.nz};
    if (S == 2) {   // each index in [1, n-3] or at n-1, at most one at n-1
        int top = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (c[a] == n[a] - 1) ++top;
            else if (!in(c[a], 1, n[a] - 3)) return false;
        }
        return top <= 1;
    }
    const int lo = (S == 0) ? 0 : 1;   // lowest plane updated
    int nlow = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (a == C) {
            if (!in(c[a], lo + 1, n[a] - 2)) return false;
        } else {
            if (!in(c[a], lo, n[a] - 2)) return false;
            nlow += (c[a] == lo);
        }
    }
    return nlow <= 1;
}

// which cells get component C of E updated
// (FDTD src/maxwell.cpp:486-522, NDFX :292-328, five-point :87-125)
template <int S, int C>
__device__ inline bool e_updates(const Grid &g, int i, int j, int k)
{
    const int c[3] = {i, j, k}, n[3] = {g.nx, g.ny, g.nz};
    const int lo = (S == 0) ? 0 : 1;
    const int top = (S == 2) ? 3 : 2;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int first = (a == C) ? lo : lo + 1;
        if (!in(c[a], first, n[a] - top)) return false;
    }
    return true;
}

template <typename real>
struct Coef {
    real a[3], b[3];
    real dtd[3];   // dt / d_alpha
    real d[3];     // d_alpha
};

template <int A>
__device__ inline int stride(const Grid &g)
{
    return A == 0 ? g.sx : (A == 1 ? g.sy : 1);
}

// F at offset `off` along axis A from the cell (index c of n along A, linear
// index id), zero outside the grid; used by the five-point planes at n-1
// (src/maxwell.cpp:52-84).  The load is unconditional, its index clamped, so
// that the loads of a cell are in flight together.
template <int A, typename real>
__device__ inline real rd0(const Grid &g, const real *__restrict__ F, int id, int c, int n, int off)
{
    const int at = min(max(c + off, 0), n - 1);
    const real v = F[id + (at - c) * (A == 0 ? g.sx : (A == 1 ? g.sy : 1))];
    return (unsigned)(c + off) < (unsigned)n ? v : real(0);
}

// Difference of component C (stored in F) along axis A at cell (i,j,k);
// FWD: F[+1] - F[0] (B update), else F[0] - F[-1] (E update).
//   FDTD:  plain difference
//   NDFX:  smoothed along the component's own axis C with (b_C, a_C)
//   five:  b_A (F[+1]-F[0]) + a_A (F[+2]-F[+1]+F[0]-F[-1]), zero outside
template <int S, int C, int A, bool FWD, typename real>
__device__ inline real diff(const Grid &g, const Coef<real> &cf, const real *__restrict__ F, int i, int j, int k)
{
    const int ua = (A == 0), va = (A == 1), wa = (A == 2);
    const int li = FWD ? i : i - ua, lj = FWD ? j : j - va, lk = FWD ? k : k - wa;
    const int lo = li * g.sx + lj * g.sy + lk;
    const int sA = stride<A>(g);
    const int hi = lo + sA;
    if (S == 0) {
        return F[hi] - F[lo];
    } else if (S == 1) {
        const int sC = stride<C>(g);
        return cf.b[C] * (F[hi] - F[lo]) + cf.a[C] * ((F[hi + sC] - F[lo + sC]) + (F[hi - sC] - F[lo - sC]));
    } else {
        const int id = i * g.sx + j * g.sy + k, c = A == 0 ? i : (A == 1 ? j : k);
        const int n = A == 0 ? g.nx : (A == 1 ? g.ny : g.nz), s = FWD ? 0 : -1;
        const real fm = rd0<A>(g, F, id, c, n, s - 1), f0 = rd0<A>(g, F, id, c, n, s);
        const real f1 = rd0<A>(g, F, id, c, n, s + 1), f2 = rd0<A>(g, F, id, c, n, s + 2);
        return cf.b[A] * (f1 - f0) + cf.a[A] * (f2 - f1 + f0 - fm);
    }
}

// rate of component C of B at cell (i,j,k); a half step adds half of it
template <int S, int C, typename real>
__device__ inline real b_rate(const Grid &g, const Coef<real> &cf, const real *__restrict__ ex, const real *__restrict__ ey,
                              const real *__restrict__ ez, int i, int j, int k)
{
    if (C == 0) return -cf.dtd[1] * diff<S, 2, 1, true>(g, cf, ez, i, j, k) + cf.dtd[2] * diff<S, 1, 2, true>(g, cf, ey, i, j, k);
    if (C == 1) return cf.dtd[0] * diff<S, 2, 0, true>(g, cf, ez, i, j, k) - cf.dtd[2] * diff<S, 0, 2, true>(g, cf, ex, i, j, k);
    return cf.dtd[1] * diff<S, 0, 1, true>(g, cf, ex, i, j, k) - cf.dtd[0] * diff<S, 1, 0, true>(g, cf, ey, i, j, k);
}

// B at the step's end, between two half steps taken together
template <typename real>
struct Mid {
    real *b[3];
};

// half step of B (maxwell_solver::advance_b, src/maxwell.cpp:10-22).  With
// energy != null the first half step also sums E^2 + B^2 of the fields it
// starts from, in FP64: compute_energy's field term, which the reference takes
// between padvance and fadvance (src/fout.cpp:102, src/main.cpp:2327-2331).
//
// TWICE: the second half step of one step and the first of the next, which
// use the same E when nothing reads B in between; the energy is that of the
// fields between the two.  36 instead of 72 B per cell: 104 us at 301x203x199,
// against 102 us for each half step.  HELD: the B between the two also goes
// to mid, for interpolate_be and the laser sources' corrections.
template <int S, bool TWICE, bool HELD, typename real>
__global__ void __launch_bounds__(kSweep) k_maxwell_b(Grid g, SweepPlan sw, Coef<real> cf, const real *__restrict__ ex,
                                                      const real *__restrict__ ey, const real *__restrict__ ez,
                                                      real *__restrict__ bx, real *__restrict__ by,
                                                      real *__restrict__ bz, double *energy, Mid<real> mid)
{
    __shared__ double part[kSweep / 64];
    int i, j, k;
    double en = 0;
    if (sweep_cell(g, sw, i, j, k)) {
        const int id = i * g.sx + j * g.sy + k;
        const real h = real(0.5);
        real b0 = bx[id], b1 = by[id], b2 = bz[id];
        auto add_energy = [&] {
            const double e0 = ex[id], e1 = ey[id], e2 = ez[id];
            en = e0 * e0 + e1 * e1 + e2 * e2 + (double)b0 * b0 + (double)b1 * b1 + (double)b2 * b2;
        };
        if (energy && !TWICE) add_energy();
        const bool u0 = b_updates<S, 0>(g, i, j, k), u1 = b_updates<S, 1>(g, i, j, k), u2 = b_updates<S, 2>(g, i, j, k);
        real d0 = real(0), d1 = real(0), d2 = real(0);
        if (u0) d0 = b_rate<S, 0>(g, cf, ex, ey, ez, i, j, k);
        if (u1) d1 = b_rate<S, 1>(g, cf, ex, ey, ez, i, j, k);
        if (u2) d2 = b_rate<S, 2>(g, cf, ex, ey, ez, i, j, k);
        if (u0) b0 += h * d0;
        if (u1) b1 += h * d1;
        if (u2) b2 += h * d2;
        if (TWICE) {
            if (energy) add_energy();
            if (HELD) {
                mid.b[0][id] = b0;
                mid.b[1][id] = b1;
                mid.b[2][id] = b2;
            }
            if (u0) b0 += h * d0;
            if (u1) b1 += h * d1;
            if (u2) b2 += h * d2;
        }
        if (u0) bx[id] = b0;
        if (u1) by[id] = b1;
        if (u2) bz[id] = b2;
    }
    if (energy) {   // uniform across the launch
        en = wave_sum(en);
        const int t = threadIdx.x;
        if ((t & 63) == 0) part[t >> 6] = en;
        __syncthreads();
        if (t == 0) {
            double s = 0;
            for (int w = 0; w < kSweep / 64; ++w) s += part[w];
            atomicAdd(energy + blockIdx.x % kEnergySlots, s);
        }
    }
}

// the current an E step takes: none, the FP32 or FP64 buffer, or that and the
// FP64 part next to it (k_push_tiled)
enum { kNoCurrent, kPlain, kWide };

// E step with the current of this step; also clears the other current
// buffer, which the next step deposits into (replaces the J reset of
// src/advance.cpp:112-123 without a separate pass).  kNoCurrent: both current
// buffers are known to be zero (no charged particles), 36 instead of 60 B per
// cell (92 us instead of 200 at 301x203x199, the sweep order included).  The last workgroup also hands the step's diagnostics over, complete
// by now: the accumulators go to pinned host memory and are cleared for the
// step after next.
template <int S, int CUR, typename real>
__global__ void __launch_bounds__(kSweep) k_maxwell_e(Grid g, SweepPlan sw, Coef<real> cf, real *__restrict__ ex,
                                                      real *__restrict__ ey, real *__restrict__ ez,
                                                      const real *__restrict__ bx, const real *__restrict__ by,
                                                      const real *__restrict__ bz, real *__restrict__ jx,
                                                      real *__restrict__ jy, real *__restrict__ jz,
                                                      real *__restrict__ njx, real *__restrict__ njy,
                                                      real *__restrict__ njz, DiagDrain dd, Current<double> wide)
{
    if (dd.n > 0 && blockIdx.x == gridDim.x - 1) {
        // eight threads per accumulator, each summing every eighth copy
        static_assert(kSweep == 8 * kDiagStride && kDiagSlots % 8 == 0, "a thread per accumulator and eighth of the copies");
        const int a = threadIdx.x / 8, p = threadIdx.x % 8;
        double v[kDiagSlots / 8], sum = 0;
#pragma unroll
        for (int m = 0; m < kDiagSlots / 8; ++m) {
            double *s = dd.acc + (p + 8 * m) * kDiagStride + a;
            v[m] = *s;
            *s = 0.0;
        }
#pragma unroll
        for (int m = 0; m < kDiagSlots / 8; ++m) sum += v[m];
        for (int o = 4; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (p == 0 && a < dd.nspread) dd.host[a] = sum;
        double *rest = dd.acc + kDiagSlots * kDiagStride;
        for (int t = threadIdx.x; t < dd.n; t += kSweep) {
            dd.host[dd.nspread + t] = rest[t];
            rest[t] = 0.0;
        }
    }
    int i, j, k;
    if (!sweep_cell(g, sw, i, j, k)) return;
    const int id = i * g.sx + j * g.sy + k;
    auto current = [&](real *j, double *w) -> real {
        if (CUR == kNoCurrent) return real(0);
        real v = j[id];
        if (CUR == kWide) {
            v = (real)((double)v + w[id]);
            w[id] = 0.0;
            j[id] = v;   // read back as the step's J
        }
        return v;
    };
    const real c0 = current(jx, wide.jx) * cf.d[0], c1 = current(jy, wide.jy) * cf.d[1], c2 = current(jz, wide.jz) * cf.d[2];
    if (e_updates<S, 0>(g, i, j, k))
        ex[id] += cf.dtd[1] * diff<S, 2, 1, false>(g, cf, bz, i, j, k) - cf.dtd[2] * diff<S, 1, 2, false>(g, cf, by, i, j, k) - c0;
    if (e_updates<S, 1>(g, i, j, k))
        ey[id] += -cf.dtd[0] * diff<S, 2, 0, false>(g, cf, bz, i, j, k) + cf.dtd[2] * diff<S, 0, 2, false>(g, cf, bx, i, j, k) - c1;
    if (e_updates<S, 2>(g, i, j, k))
        ez[id] += cf.dtd[0] * diff<S, 1, 0, false>(g, cf, by, i, j, k) - cf.dtd[1] * diff<S, 0, 1, false>(g, cf, bx, i, j, k) - c2;
    if (CUR != kNoCurrent) {
        njx[id] = real(0);
        njy[id] = real(0);
        njz[id] = real(0);
    }
}

// Be = B averaged to E positions (src/advance.cpp:20-83): each component is
// the mean over a 2x2x2 stencil (Bx over i..i+1, j-1..j, k-1..k; By over
// i-1..i, j..j+1, k-1..k; Bz over i-1..i, j-1..j, k..k+1); on a boundary plane
// the half that leaves the grid is dropped (4-point mean); cells on two or
// more boundary planes keep their value.
//
// Two forms with the same sums in the same order.  In FP32, and in FP64 up to
// kDirectBe cells, a thread of the flattened sweep takes its cell's squares
// from global memory.  Above that, FP64 stages B in LDS: field phase 126
// against 133 us at 128x128x128 and 321 against 334 us at 256x128x128
// (five-point; the direct form's eight cache lines per value).  The direct
// form is the faster one below (73.5 -> 69.3 us at 135x75x71 in FP64) and in
// FP32 (23.0 -> 17.8 us at 64x32x32, where the staged kernel has 64
// workgroups, 48.3 -> 41.3 at 135x75x71, 109.5 -> 101.2 at 251x97x89, 138.9 ->
// 131.6 at 256x128x128; equal at 512x256x256).
//
// Staged: a workgroup owns a kBeK x kBeJ block of (j, k) columns over a run
// of planes.  It loads B of its block plus the one-column rim each
// component's square reaches (Bx: rows j-1, columns k-1; By: rows j+1,
// columns k-1; Bz: rows j-1, columns k+1), on the run's planes plus one (Bx
// one plane ahead, By and Bz one behind), with every load issued before the
// first LDS write and unconditional (indices clamped into the grid, entries
// outside it set to zero), then takes each cell's sums from LDS.
constexpr int kDirectBe = 1 << 20;
constexpr int kBeK = 64, kBeJ = 8;
constexpr int kBeW = kBeK + 1, kBeH = kBeJ + 1;   // rim-extended block, per component
constexpr int kBeCols = kBeW * kBeH;
constexpr int kBeRun = 2;   // planes per run; the LDS holds the run plus one plane of three components

// 2x2 sum of the LDS plane P (kBeH rows of kBeW) at (r, c) with the
// neighbour row r + dr (when vj) and column c + dc (when vk)
__device__ inline double lds_sum(const double *P, int r, int c, int dr, int dc, bool vj, bool vk)
{
    double s = P[r * kBeW + c];
    if (vk) s += P[r * kBeW + c + dc];
    if (vj) s += P[(r + dr) * kBeW + c];
    if (vj && vk) s += P[(r + dr) * kBeW + c + dc];
    return s;
}

__global__ void __launch_bounds__(kBeK * kBeJ) k_interpolate_be(Grid g, const double *__restrict__ bx,
                                                                const double *__restrict__ by,
                                                                const double *__restrict__ bz, double *__restrict__ bex,
                                                                double *__restrict__ bey, double *__restrict__ bez)
{
    constexpr int R = kBeRun;
    constexpr int kN = (R + 1) * kBeCols;   // LDS entries per component
    constexpr int kIt = (kN + kBeK * kBeJ - 1) / (kBeK * kBeJ);
    // [plane][component][row][column]: plane m holds Bx at x = i0 + m and By,
    // Bz at x = i0 - 1 + m; component c's (row, column) is (j, k) =
    // (j0 - 1 + row, k0 - 1 + col) for Bx, (j0 + row, k0 - 1 + col) for By,
    // (j0 - 1 + row, k0 + col) for Bz
    __shared__ double L[R + 1][3][kBeCols];
    const dim3 vb = band_block();
    const int k0 = vb.x * kBeK, j0 = vb.y * kBeJ, i0 = vb.z * R;
    const int tid = threadIdx.y * kBeK + threadIdx.x;
    double v[3][kIt];
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
        const int w = tid + it * kBeK * kBeJ;
        const int m = w / kBeCols, e = w - m * kBeCols;
        const int r = e / kBeW, q = e - r * kBeW;
        const int px = i0 + m, pyz = i0 - 1 + m;
        const bool live = w < kN;
        const int jx = j0 - 1 + r, kx = k0 - 1 + q, jy = j0 + r, kz = k0 + q;
        const bool inx = live && px < g.nx && (unsigned)jx < (unsigned)g.ny && (unsigned)kx < (unsigned)g.nz;
        const bool iny = live && pyz >= 0 && pyz < g.nx && (unsigned)jy < (unsigned)g.ny && (unsigned)kx < (unsigned)g.nz;
        const bool inz = live && pyz >= 0 && pyz < g.nx && (unsigned)jx < (unsigned)g.ny && (unsigned)kz < (unsigned)g.nz;
        const int cpx = min(px, g.nx - 1), cpyz = max(min(pyz, g.nx - 1), 0);
        const int cjx = max(min(jx, g.ny - 1), 0), cjy = min(jy, g.ny - 1);
        const int ckx = max(min(kx, g.nz - 1), 0), ckz = min(kz, g.nz - 1);
        const double ax = bx[cpx * g.sx + cjx * g.sy + ckx];
        const double ay = by[cpyz * g.sx + cjy * g.sy + ckx];
        const double az = bz[cpyz * g.sx + cjx * g.sy + ckz];
        v[0][it] = inx ? ax : double(0);
        v[1][it] = iny ? ay : double(0);
        v[2][it] = inz ? az : double(0);
    }
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
        const int w = tid + it * kBeK * kBeJ;
        if (w < kN) {
            const int m = w / kBeCols, e = w - m * kBeCols;
            L[m][0][e] = v[0][it];
            L[m][1][e] = v[1][it];
            L[m][2][e] = v[2][it];
        }
    }
    __syncthreads();
    const int j = j0 + threadIdx.y, k = k0 + threadIdx.x;
    if (j >= g.ny || k >= g.nz) return;
    const int nbjk = (j == 0 || j == g.ny - 1) + (k == 0 || k == g.nz - 1);
    // entries of each component's 2x2 square inside the grid
    const bool xvj = j >= 1, xvk = k >= 1;           // Bx: rows j-1, j; columns k-1, k
    const bool yvj = j + 1 < g.ny, yvk = k >= 1;     // By: rows j, j+1; columns k-1, k
    const bool zvj = j >= 1, zvk = k + 1 < g.nz;     // Bz: rows j-1, j; columns k, k+1
    const int cx = (1 + xvj) * (1 + xvk), cy = (1 + yvj) * (1 + yvk), cz = (1 + zvj) * (1 + zvk);
    const int ty = threadIdx.y, tx = threadIdx.x;
#pragma unroll
    for (int m = 0; m < R; ++m) {
        // Be at x = i0 + m: Bx planes i, i + 1 (L[m], L[m + 1]), By and Bz
        // planes i - 1, i (L[m], L[m + 1])
        const int i = i0 + m;
        if (i < g.nx && nbjk + (i == 0 || i == g.nx - 1) < 2) {
            const bool up = i + 1 < g.nx;
            const double sx0 = lds_sum(L[m][0], ty + 1, tx + 1, -1, -1, xvj, xvk);
            const double px1 = up ? lds_sum(L[m + 1][0], ty + 1, tx + 1, -1, -1, xvj, xvk) : double(0);
            const double qy = i > 0 ? lds_sum(L[m][1], ty, tx + 1, 1, -1, yvj, yvk) : double(0);
            const double sy1 = lds_sum(L[m + 1][1], ty, tx + 1, 1, -1, yvj, yvk);
            const double rz = i > 0 ? lds_sum(L[m][2], ty + 1, tx, -1, 1, zvj, zvk) : double(0);
            const double sz1 = lds_sum(L[m + 1][2], ty + 1, tx, -1, 1, zvj, zvk);
            const int id = i * g.sx + j * g.sy + k;
            bex[id] = (sx0 + px1) * (cx * (1 + up) == 8 ? double(0.125) : double(0.25));
            bey[id] = (qy + sy1) * (cy * (1 + (i > 0)) == 8 ? double(0.125) : double(0.25));
            bez[id] = (rz + sz1) * (cz * (1 + (i > 0)) == 8 ? double(0.125) : double(0.25));
        }
    }
}

template <typename real>
__global__ void __launch_bounds__(kSweep) k_interpolate_be_direct(Grid g, SweepPlan sw, const real *__restrict__ bx,
                                                                  const real *__restrict__ by,
                                                                  const real *__restrict__ bz, real *__restrict__ bex,
                                                                  real *__restrict__ bey, real *__restrict__ bez)
{
    int i, j, k;
    if (!sweep_cell(g, sw, i, j, k)) return;
    if ((i == 0 || i == g.nx - 1) + (j == 0 || j == g.ny - 1) + (k == 0 || k == g.nz - 1) >= 2) return;
    const int id = i * g.sx + j * g.sy + k;
    // neighbours on each axis, clamped to the cell itself where they leave the grid
    const bool il = i > 0, iu = i + 1 < g.nx, jl = j > 0, ju = j + 1 < g.ny, kl = k > 0, ku = k + 1 < g.nz;
    const int ml = il ? -g.sx : 0, mu = iu ? g.sx : 0, nl = jl ? -g.sy : 0, nu = ju ? g.sy : 0, ol = kl ? -1 : 0,
              ou = ku ? 1 : 0;
    auto sum = [&](const real *__restrict__ F, int at, int dj, int dk, bool vj, bool vk) {
        const real a = F[at], b = F[at + dk], c = F[at + dj], d = F[at + dj + dk];
        real s = a;
        s += vk ? b : real(0);
        s += vj ? c : real(0);
        s += vj && vk ? d : real(0);
        return s;
    };
    const real x0 = sum(bx, id, nl, ol, jl, kl), x1 = sum(bx, id + mu, nl, ol, jl, kl);
    const real y0 = sum(by, id + ml, nu, ol, ju, kl), y1 = sum(by, id, nu, ol, ju, kl);
    const real z0 = sum(bz, id + ml, nl, ou, jl, ku), z1 = sum(bz, id, nl, ou, jl, ku);
    const int cx = (1 + jl) * (1 + kl) * (1 + iu), cy = (1 + ju) * (1 + kl) * (1 + il), cz = (1 + jl) * (1 + ku) * (1 + il);
    bex[id] = (x0 + (iu ? x1 : real(0))) * (cx == 8 ? real(0.125) : real(0.25));
    bey[id] = ((il ? y0 : real(0)) + y1) * (cy == 8 ? real(0.125) : real(0.25));
    bez[id] = ((il ? z0 : real(0)) + z1) * (cz == 8 ? real(0.125) : real(0.25));
}

// init_boundaries: zero components on boundary planes, transverse indices in
// [0, n-2] (FDTD src/maxwell.cpp:532-597, NDFX :338-438, five-point :135-236)
template <typename real>
__global__ void __launch_bounds__(kBX * kBY) k_init_boundaries(Grid g, int solver, Fields<real> f)
{
    const int k = blockIdx.x * kBX + threadIdx.x;
    const int j = blockIdx.y * kBY + threadIdx.y;
    const int i = blockIdx.z;
    if (k >= g.nz || j >= g.ny) return;
    const int c[3] = {i, j, k}, n[3] = {g.nx, g.ny, g.nz};
    int em = 0, bm = 0;
    for (int a = 0; a < 3; ++a) {
        const int b1 = (a + 1) % 3, b2 = (a + 2) % 3;
        if (c[b1] > n[b1] - 2 || c[b2] > n[b2] - 2) continue;
        const int normal = 1 << a, tang = 7 & ~normal;
        const int p = c[a];
        if (solver == 0) {          // FDTD
            if (p == 0) { em |= tang; bm |= normal; }
            if (p == n[a] - 1) { em |= 7; bm |= 7; }
        } else if (solver == 1) {   // NDFX
            if (p == 0 || p == n[a] - 1) { em |= 7; bm |= 7; }
            if (p == 1) { em |= tang; bm |= normal; }
        } else {                    // five-point
            if (p == 0 || p == n[a] - 1) { em |= 7; bm |= 7; }
            if (p == 1) em |= tang;
            if (p == n[a] - 2) bm |= tang;
        }
    }
    const int id = i * g.sx + j * g.sy + k;
    if (em & 1) f.ex[id] = real(0);
    if (em & 2) f.ey[id] = real(0);
    if (em & 4) f.ez[id] = real(0);
    if (bm & 1) f.bx[id] = real(0);
    if (bm & 2) f.by[id] = real(0);
    if (bm & 4) f.bz[id] = real(0);
}

// The pulse of f_init_cos with the cos envelope (src/init.cpp:6-210) at the
// point (px, py, pz) (c/omega units from the subdomain origin), after it has
// travelled `shift` along its direction of propagation (+r0 when b_sign, -r0
// otherwise: the direction of E x B); shift = 0 is f_init_cos itself.  FP64.
// Returns false outside the envelope (ev, bv untouched).
__device__ inline bool pulse_at(const LaserFrame &L, double px, double py, double pz, double shift, double ev[3],
                                double bv[3])
{
    const double PI = 3.141592653589793;
    const double X = px - L.x0 - L.xt, Y = py - L.y12 - L.y0 - L.yt, Z = pz - L.z12 - L.z0 - L.zt;
    double x = L.r0[0] * X + L.r0[1] * Y + L.r0[2] * Z;
    const double y = L.ey[0] * X + L.ey[1] * Y + L.ey[2] * Z;
    const double z = L.ez[0] * X + L.ez[1] * Y + L.ez[2] * Z;
    if (shift != 0) x -= L.b_sign ? shift : -shift;
    if (!(x < L.xs && x > -L.xs && y < L.ys && y > -L.ys && z < L.zs && z > -L.zs)) return false;
    const double xi = x + L.phase;
    double cx, sx, cy, sy, cz, sz, cxi, sxi;
    sincos(PI * x / 2 / L.xs, &sx, &cx);
    sincos(PI * y / 2 / L.ys, &sy, &cy);
    sincos(PI * z / 2 / L.zs, &sz, &cz);
    sincos(xi, &sxi, &cxi);
    const double tr = cy * cy * cz * cz;
    const double fy = L.a0y * tr * (cxi * cx * cx - PI / L.xs * sxi * cx * sx);
    const double fz = L.a0z * tr * (sxi * cx * cx + PI / L.xs * cxi * cx * sx);
    const double fx = L.a0y * sxi * cx * cx * cz * cz * PI / L.ys * cy * sy - L.a0z * cxi * cx * cx * cy * cy * PI / L.zs * cz * sz;
    double gx = L.a0z * cxi * cx * cx * PI / L.ys * cz * cz * cy * sy + L.a0y * sxi * cx * cx * cy * cy * PI / L.zs * cz * sz;
    double gy = -fz, gz = fy;
    if (!L.b_sign) { gx = -gx; gy = -gy; gz = -gz; }
    for (int m = 0; m < 3; ++m) {
        ev[m] = fx * L.r0[m] + fy * L.ey[m] + fz * L.ez[m];
        bv[m] = gx * L.r0[m] + gy * L.ey[m] + gz * L.ez[m];
    }
    return true;
}

// Laser initial condition f_init_cos (src/init.cpp:6-210), evaluated in FP64
// and stored in the field precision
template <typename real>
__global__ void __launch_bounds__(kBX * kBY) k_laser_cos(Grid g, Fields<real> f, LaserFrame L)
{
    const int k = blockIdx.x * kBX + threadIdx.x;
    const int j = blockIdx.y * kBY + threadIdx.y;
    const int i = blockIdx.z;
    if (k >= g.nz || j >= g.ny) return;
    const int id = i * g.sx + j * g.sy + k;
    real *E[3] = {f.ex, f.ey, f.ez}, *B[3] = {f.bx, f.by, f.bz};
    double ev[3], bv[3];
    if (pulse_at(L, i * g.dx, j * g.dy, k * g.dz, 0.0, ev, bv)) {
        for (int m = 0; m < 3; ++m) {
            if (L.append) {
                E[m][id] = (real)((double)E[m][id] + ev[m]);
                B[m][id] = (real)((double)B[m][id] + bv[m]);
            } else {
                E[m][id] = (real)ev[m];
                B[m][id] = (real)bv[m];
            }
        }
    } else if (!L.append) {
        for (int m = 0; m < 3; ++m) { E[m][id] = real(0); B[m][id] = real(0); }
    }
}

// Total-field / scattered-field laser source (qk_add_laser_source).  On the
// source's total side of its plane the grid holds the total field, on the
// other side the field scattered off the incident pulse; an update reading
// across the plane is corrected by the same update applied to the incident
// field on the far side: + L(inc on the scattered side) at total nodes,
// - L(inc on the total side) at scattered nodes, L being the solver's own
// update with its boundary-plane sets.  The incident field is sampled where
// each component lives on the staggered grid (E_a a half cell along a, B_a a
// half cell across a).
//
// The stencils reach kInjReach planes across, so only 2 kInjReach planes
// matter.  A workgroup evaluates the incident field of its rows of 64 columns
// (and, for NDFX, the rim its transverse smoothing reads) there into LDS, its
// threads sharing the points, and applies the masked update to the grid, a
// wavefront per plane and row: one launch per sub-step for both sides.  Only differences along x cross the plane, and NDFX's smoothing of
// the x component along x: component x is needed there only, and neither it
// nor its own update is ever corrected.
// Bound by the FP64 pulse (four sines and cosines per point, taken in pairs).
// Before, the pulse was evaluated on 18 planes of a stack
// that the solver then swept whole, three launches per side and sub-step: a
// sub-step took 66 us for two sides of 128 x 128 columns (five-point), now
// 7.3 us; 17.6 us for one of 32 x 32 (FDTD), now 4.7 us (9.3 and 5.4 us with
// sines and cosines apart).  With 64 x 4 columns per workgroup (six points in
// turn per thread instead of at most two) it was 21.7 us and 6.6 us.
template <int S>
constexpr int kInjReach = S == 2 ? 2 : 1;

// whether the corrections of a sub-step read component c of the incident
// field in plane m of the 2 kInjReach (m = kInjReach is the source plane);
// BF: B half step (forward differences of E), else E step (backward, of B)
template <int S, bool BF>
constexpr bool inj_reads(int c, int m)
{
    if (c == 0) return S == 1;
    if (S == 2) return BF ? m >= 1 : m <= 2;
    return BF ? m == 1 : m == 0;
}

struct InjectSides {
    InjectArgs s[2];
};

// TURN: the corrections of a half step of B and of the next step's first one
// (the same incident field) where both were taken together: mid takes them
// once, and the grid's B becomes mid after the second half step and its
// corrections, in the order of two half steps taken apart (corrected twice
// after both, FP32 runs came out 1 % further from FP64).  The energy of the
// fields between the two changes with mid.  9.4 us where a sub-step takes 7.7
// (two sides of 128 x 128 columns), 5.2 and 4.8 us (one of 32 x 32).
template <int S, bool BF, bool TURN, typename real>
__global__ void __launch_bounds__(kBX * kBY) k_inject(Grid g, Coef<real> cf, Fields<real> f, InjectSides sides,
                                                      Mid<real> mid, double *energy)
{
    constexpr int R = kInjReach<S>, M = S == 1 ? 1 : 0;   // planes per side, rim
    constexpr int kRows = kBY / (2 * R);                   // rows of columns: a thread owns one node of one plane
    constexpr int W = kBX + 2 * M, H = kRows + 2 * M;
    constexpr int kPairs = S == 0 ? 2 : (S == 1 ? 4 : 6);  // (component, plane) pairs read: see inj_reads
    __shared__ real inc[3][2 * R][H][W];
    const InjectArgs &a = sides.s[blockIdx.z];
    const int k0 = blockIdx.x * kBX, j0 = blockIdx.y * kRows, i0 = a.plane - R;
    for (int e = threadIdx.y * kBX + threadIdx.x; e < kPairs * H * W; e += kBX * kBY) {
        const int pair = e / (H * W), rq = e - pair * H * W, r = rq / W, q = rq - r * W;
        const int c = S == 0 ? 1 + pair : (S == 1 ? (pair < 2 ? 0 : pair - 1) : 1 + pair / 3);
        const int m = S == 2 ? pair % 3 + BF : (S == 1 && pair < 2 ? pair : (int)BF);
        const int i = i0 + m, j = j0 + r - M, k = k0 + q - M;
        // staggered position of component c of the input field
        const double hx = (BF ? c == 0 : c != 0) ? 0.5 : 0.0, hy = (BF ? c == 1 : c != 1) ? 0.5 : 0.0,
                     hz = (BF ? c == 2 : c != 2) ? 0.5 : 0.0;
        double v = 0;
        if ((unsigned)i < (unsigned)g.nx && (unsigned)j < (unsigned)g.ny && (unsigned)k < (unsigned)g.nz)
            for (int n = 0; n < a.nsrc; ++n) {
                double ev[3], bv[3];
                if (pulse_at(a.src[n], (i + a.ishift[n] + hx) * g.dx, (j + hy) * g.dy, (k + hz) * g.dz, a.shift[n], ev, bv)) {
                    const double *p = BF ? ev : bv;
                    v += c == 0 ? p[0] : (c == 1 ? p[1] : p[2]);
                }
            }
        inc[c][m][r][q] = (real)v;
    }
    __syncthreads();
    const int row = threadIdx.y / (2 * R), j = j0 + row, k = k0 + threadIdx.x;
    const int r = row + M, q = threadIdx.x + M;
    double en = 0;
#pragma unroll
    for (int m = 0; m < 2 * R; ++m) {
        if (m != (int)threadIdx.y % (2 * R) || j >= g.ny || k >= g.nz) continue;   // the plane is uniform over the wavefront
        const int i = i0 + m;
        if (i < 0 || i >= g.nx) continue;
        const bool low = m < R;
        // the incident field on the node's far side, zero on its own
        auto in = [&](int c, int mm, int dj, int dk) -> real {
            if (mm < 0 || mm >= 2 * R || (mm < R) == low || !inj_reads<S, BF>(c, mm)) return real(0);
            return inc[c][mm][r + dj][q + dk];
        };
        // difference along x of component c (1 or 2)
        auto dx = [&](int c) -> real {
            const int lo = BF ? m : m - 1;
            if (S == 0) return in(c, lo + 1, 0, 0) - in(c, lo, 0, 0);
            if (S == 1) {   // smoothed along the component's own axis
                const int uj = c == 1, uk = c == 2;
                return cf.b[c] * (in(c, lo + 1, 0, 0) - in(c, lo, 0, 0)) +
                       cf.a[c] * ((in(c, lo + 1, uj, uk) - in(c, lo, uj, uk)) +
                                  (in(c, lo + 1, -uj, -uk) - in(c, lo, -uj, -uk)));
            }
            const real fm = in(c, lo - 1, 0, 0), f0 = in(c, lo, 0, 0), f1 = in(c, lo + 1, 0, 0), f2 = in(c, lo + 2, 0, 0);
            return cf.b[0] * (f1 - f0) + cf.a[0] * (f2 - f1 + f0 - fm);
        };
        // difference along y or z of component x: NDFX's smoothing along x
        auto dt = [&](int axis) -> real {
            if (S != 1) return real(0);
            const int uj = axis == 1, uk = axis == 2, s = BF ? 0 : -1;
            auto d = [&](int mm) { return in(0, mm, (s + 1) * uj, (s + 1) * uk) - in(0, mm, s * uj, s * uk); };
            return cf.a[0] * (d(m + 1) + d(m - 1));
        };
        const bool tot = low == (a.side == 1);
        const int id = i * g.sx + j * g.sy + k;
        if (BF) {
            const real h = real(0.5);
            auto correct = [&](real *F, real *at_mid, real d, real rate) {
                if (!tot) d = -d;
                if (TURN) {
                    const real o = at_mid[id], w = o + d;
                    at_mid[id] = w;
                    en += (double)w * w - (double)o * o;
                    real v = w;
                    v += h * rate;
                    F[id] = v + d;
                } else {
                    F[id] += d;
                }
            };
            if (b_updates<S, 1>(g, i, j, k))
                correct(f.by, mid.b[1], h * (cf.dtd[0] * dx(2) - cf.dtd[2] * dt(2)),
                        TURN ? b_rate<S, 1>(g, cf, f.ex, f.ey, f.ez, i, j, k) : real(0));
            if (b_updates<S, 2>(g, i, j, k))
                correct(f.bz, mid.b[2], h * (cf.dtd[1] * dt(1) - cf.dtd[0] * dx(1)),
                        TURN ? b_rate<S, 2>(g, cf, f.ex, f.ey, f.ez, i, j, k) : real(0));
        } else {
            if (e_updates<S, 1>(g, i, j, k)) {
                const real d = -cf.dtd[0] * dx(2) + cf.dtd[2] * dt(2);
                f.ey[id] = tot ? f.ey[id] + d : f.ey[id] - d;
            }
            if (e_updates<S, 2>(g, i, j, k)) {
                const real d = cf.dtd[0] * dx(1) - cf.dtd[1] * dt(1);
                f.ez[id] = tot ? f.ez[id] + d : f.ez[id] - d;
            }
        }
    }
    if (TURN) {
        en = wave_sum(en);
        if (threadIdx.x == 0 && en != 0)
            atomicAdd(energy + (blockIdx.y * gridDim.x + blockIdx.x) % kEnergySlots, en);
    }
}

template <typename real>
Coef<real> make_coef(const Grid &g, const SolverCoef &c)
{
    Coef<real> r;
    const double d[3] = {g.dx, g.dy, g.dz};
    for (int a = 0; a < 3; ++a) {
        r.a[a] = (real)c.a[a];
        r.b[a] = (real)c.b[a];
        r.dtd[a] = (real)(g.dt / d[a]);
        r.d[a] = (real)d[a];
    }
    return r;
}

__global__ void k_zero(double *p, size_t n)
{
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = 0.0;
}

}  // namespace

hipError_t launch_zero(hipStream_t st, double *p, size_t n)
{
    if (n == 0) return hipSuccess;
    k_zero<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(p, n);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_maxwell_b(hipStream_t st, int solver, const Grid &g, const SolverCoef &c, const Fields<real> &f,
                            double *energy, bool twice, real *const *mid)
{
    const Coef<real> cf = make_coef<real>(g, c);
    const SweepPlan sw = sweep_plan(g);
    const dim3 grid((unsigned)(sw.per * g.nx));
    Mid<real> md{};
    for (int a = 0; a < 3 && mid; ++a) md.b[a] = mid[a];
#define QK_B(S, T, H) k_maxwell_b<S, T, H, real><<<grid, kSweep, 0, st>>>(g, sw, cf, f.ex, f.ey, f.ez, f.bx, f.by, f.bz, energy, md)
#define QK_BS(S)                              \
    if (twice && mid) QK_B(S, true, true);    \
    else if (twice) QK_B(S, true, false);     \
    else QK_B(S, false, false)
    if (solver == 0) { QK_BS(0); }
    else if (solver == 1) { QK_BS(1); }
    else { QK_BS(2); }
#undef QK_BS
#undef QK_B
    return hipGetLastError();
}

template <typename real>
hipError_t launch_maxwell_e(hipStream_t st, int solver, const Grid &g, const SolverCoef &c, const Fields<real> &f,
                            const Current<real> *j, const Current<real> *jn, const DiagDrain &dd,
                            const Current<double> *wide)
{
    const Coef<real> cf = make_coef<real>(g, c);
    const SweepPlan sw = sweep_plan(g);
    const dim3 grid((unsigned)(sw.per * g.nx));
    const Current<real> none{nullptr, nullptr, nullptr}, a = j ? *j : none, b = j ? *jn : none;
    const Current<double> w = wide ? *wide : Current<double>{};
    if (wide && (!j || sizeof(real) != 4)) return hipErrorInvalidValue;
    auto launch = [&](auto kernel) {
        kernel<<<grid, kSweep, 0, st>>>(g, sw, cf, f.ex, f.ey, f.ez, f.bx, f.by, f.bz, a.jx, a.jy, a.jz, b.jx, b.jy, b.jz,
                                        dd, w);
    };
#define QK_E(C)                                              \
    if (solver == 0) launch(k_maxwell_e<0, C, real>);        \
    else if (solver == 1) launch(k_maxwell_e<1, C, real>);   \
    else launch(k_maxwell_e<2, C, real>)
    if constexpr (sizeof(real) == 4) {
        if (wide) {
            QK_E(kWide);
            return hipGetLastError();
        }
    }
    if (j) { QK_E(kPlain); }
    else { QK_E(kNoCurrent); }
#undef QK_E
    return hipGetLastError();
}

template <typename real>
hipError_t launch_interpolate_be(hipStream_t st, const Grid &g, const Fields<real> &f, const real *const *b)
{
    const real *bx = b ? b[0] : f.bx, *by = b ? b[1] : f.by, *bz = b ? b[2] : f.bz;
    if (sizeof(real) == 4 || g.ncell <= kDirectBe) {
        const SweepPlan sw = sweep_plan(g);
        k_interpolate_be_direct<real><<<(unsigned)(sw.per * g.nx), kSweep, 0, st>>>(g, sw, bx, by, bz, f.bex, f.bey, f.bez);
    } else {
        const dim3 grid((g.nz + kBeK - 1) / kBeK, (g.ny + kBeJ - 1) / kBeJ, (g.nx + kBeRun - 1) / kBeRun);
        k_interpolate_be<<<grid, dim3(kBeK, kBeJ), 0, st>>>(g, (const double *)bx, (const double *)by, (const double *)bz,
                                                            (double *)f.bex, (double *)f.bey, (double *)f.bez);
    }
    return hipGetLastError();
}

template <typename real>
hipError_t launch_init_boundaries(hipStream_t st, int solver, const Grid &g, const Fields<real> &f)
{
    k_init_boundaries<real><<<cell_grid(g), dim3(kBX, kBY), 0, st>>>(g, solver, f);
    return hipGetLastError();
}

bool laser_frame(const Grid &g, const double *P, LaserFrame &L)
{
    // propagation frame (src/init.cpp:32-93)
    const double PI = 3.141592653589793;
    L.a0y = P[0];
    L.a0z = P[1];
    L.xs = P[2] * 2 * sqrt(2 * PI) / 3;
    L.ys = P[3] * 2 * sqrt(2 * PI) / 3;
    L.zs = P[4] * 2 * sqrt(2 * PI) / 3;
    L.x0 = P[5];
    L.b_sign = P[6] != 0;
    const double x1 = P[7];
    L.phase = P[8];
    L.y0 = P[9];
    L.z0 = P[10];
    L.append = P[11] != 0;
    const double phi = P[12];
    L.xt = P[13];
    L.yt = P[14];
    L.zt = P[15];
    L.y12 = 0.5 * g.ny * g.dy;
    L.z12 = 0.5 * g.nz * g.dz;
    const double rn = sqrt(x1 * x1 + L.y0 * L.y0 + L.z0 * L.z0);
    if (!(rn > 0)) return false;
    L.r0[0] = -x1 / rn;
    L.r0[1] = -L.y0 / rn;
    L.r0[2] = -L.z0 / rn;
    const double t = sqrt(L.r0[0] * L.r0[0] + L.r0[1] * L.r0[1]);
    if (t != 0) { L.ey[0] = -L.r0[1] / t; L.ey[1] = L.r0[0] / t; L.ey[2] = 0; }
    else { L.ey[0] = 0; L.ey[1] = 1; L.ey[2] = 0; }
    L.ez[0] = L.r0[1] * L.ey[2] - L.r0[2] * L.ey[1];
    L.ez[1] = L.r0[2] * L.ey[0] - L.r0[0] * L.ey[2];
    L.ez[2] = L.r0[0] * L.ey[1] - L.r0[1] * L.ey[0];
    if (phi != 0) {
        const double c = cos(phi), s = sin(phi);
        double y[3], z[3];
        for (int m = 0; m < 3; ++m) { y[m] = L.ey[m]; z[m] = L.ez[m]; }
        for (int m = 0; m < 3; ++m) { L.ey[m] = y[m] * c + z[m] * s; L.ez[m] = z[m] * c - y[m] * s; }
    }
    return true;
}

template <typename real>
hipError_t launch_laser_cos(hipStream_t st, const Grid &g, const Fields<real> &f, const double *P)
{
    LaserFrame L;
    if (!laser_frame(g, P, L)) return hipErrorInvalidValue;
    k_laser_cos<real><<<cell_grid(g), dim3(kBX, kBY), 0, st>>>(g, f, L);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_inject(hipStream_t st, int solver, const Grid &g, const SolverCoef &c, const Fields<real> &f,
                         int b_field, int nsides, const InjectArgs *a, real *const *mid, double *energy)
{
    if (nsides <= 0) return hipSuccess;
    const Coef<real> cf = make_coef<real>(g, c);
    Mid<real> md{};
    for (int x = 0; x < 3 && mid; ++x) md.b[x] = mid[x];
    const dim3 block(kBX, kBY);
    const int rows = solver == 2 ? 1 : 2;   // k_inject's kRows
    dim3 grid((g.nz + kBX - 1) / kBX, (g.ny + rows - 1) / rows, nsides);
    auto one = [&](const InjectArgs &a0, const InjectArgs &a1) {
        const InjectSides sides{{a0, a1}};
#define QK_INJ(S)                                                                                              \
    if (b_field && mid) k_inject<S, true, true, real><<<grid, block, 0, st>>>(g, cf, f, sides, md, energy);    \
    else if (b_field) k_inject<S, true, false, real><<<grid, block, 0, st>>>(g, cf, f, sides, md, nullptr);    \
    else k_inject<S, false, false, real><<<grid, block, 0, st>>>(g, cf, f, sides, md, nullptr)
        if (solver == 0) { QK_INJ(0); }
        else if (solver == 1) { QK_INJ(1); }
        else { QK_INJ(2); }
#undef QK_INJ
        return hipGetLastError();
    };
    // sides whose planes lie closer than the corrections reach follow each
    // other: in one launch they would update the same nodes
    if (nsides == 2 && !sides_apart(a[0].plane, a[1].plane)) {
        if (mid) return hipErrorInvalidValue;   // each would set B to its own corrections
        grid.z = 1;
        const hipError_t e = one(a[0], a[0]);
        return e != hipSuccess ? e : one(a[1], a[1]);
    }
    return one(a[0], a[nsides - 1]);
}

#define QK_INST(real)                                                                                            \
    template hipError_t launch_maxwell_b<real>(hipStream_t, int, const Grid &, const SolverCoef &, const Fields<real> &, \
                                               double *, bool, real *const *);                                  \
    template hipError_t launch_maxwell_e<real>(hipStream_t, int, const Grid &, const SolverCoef &, const Fields<real> &, \
                                               const Current<real> *, const Current<real> *, const DiagDrain &, \
                                               const Current<double> *);                                        \
    template hipError_t launch_interpolate_be<real>(hipStream_t, const Grid &, const Fields<real> &, const real *const *); \
    template hipError_t launch_init_boundaries<real>(hipStream_t, int, const Grid &, const Fields<real> &);     \
    template hipError_t launch_laser_cos<real>(hipStream_t, const Grid &, const Fields<real> &, const double *); \
    template hipError_t launch_inject<real>(hipStream_t, int, const Grid &, const SolverCoef &, const Fields<real> &, \
                                            int, int, const InjectArgs *, real *const *, double *);
QK_INST(float)
QK_INST(double)
#undef QK_INST

}  // namespace qk
