// qk_particles.hip -- particle kernels of the step on gfx950: the fused
// gather + push + charge-conserving deposit + re-binning kernels (the particle
// loop of src/advance.cpp:90-387) in two forms, photon transport, the device
// plasma loader and the node-charge deposit used for the Gauss-law check.
//
//   k_push_global  one thread per particle, each current contribution a global
//                  atomic (the plain method, used for the FP64 comparison)
//   k_push_tiled   one workgroup per chunk of an 8x8x8 cell tile; particles are
//                  sorted by tile, so the workgroup stages the tile's E and Be
//                  nodes in LDS once, gathers from there, and deposits into an
//                  LDS window of the tile plus a halo, flushed once with one
//                  global atomic per nonzero window entry.  Inside a tile the
//                  storage order puts particles of distinct cells in
//                  consecutive slots, so a wavefront's LDS atomics do not
//                  collide.  A particle that drifted out of the window since
//                  the last sort gathers and deposits through global memory.
#include <algorithm>

#include "qk_push.h"

namespace qk {

namespace {

// A workgroup of the tiled kernel serves particles whose start cell lies
// within kHalo cells of its tile ("in the window").  Relative to the tile's
// lower corner such a cell has r in [-kHalo, kT + kHalo) on each axis.
#ifndef QK_HALO
#define QK_HALO 1
#endif
constexpr int kHalo = QK_HALO;
constexpr int kT[3] = {kTx, kTy, kTz};
// threads per workgroup of the tiled kernel: the LDS window and field stage
// (78 KB) admit two workgroups per CU, so the workgroup is made large enough
// to keep four wavefronts per SIMD in flight
#ifndef QK_TBLOCK
#define QK_TBLOCK 512
#endif
constexpr int kTBlock = QK_TBLOCK;
// out-of-window particles listed per workgroup and pushed after its rounds:
// at most this many per chunk, the rest inline
constexpr int kDefer = 512;

// Current window, FP64, one block per component.  A deposit from start cell
// r touches cells r-1 .. r+1 (one face crossing per axis at most) and, for
// the two axes transverse to the component, the node above as well: the
// window spans r - 1 .. r + 1 along the component's axis and r - 1 .. r + 2
// across it, i.e. window index = r + kHalo + 1.
__host__ __device__ constexpr int jdim(int c, int a) { return kT[a] + 2 * kHalo + (a == c ? 2 : 3); }
__host__ __device__ constexpr int jsize(int c) { return jdim(c, 0) * jdim(c, 1) * jdim(c, 2); }
__host__ __device__ constexpr int joff(int c) { return c == 0 ? 0 : (c == 1 ? jsize(0) : jsize(0) + jsize(1)); }
constexpr int kJWin = jsize(0) + jsize(1) + jsize(2);

// Field stage: E and Be nodes a window particle interpolates from.  Each
// component needs its own axis at the start cell only and the node above
// across it (gather at the lower node, src/deposition.cpp:431-471): index =
// r + kHalo, extent kT + 2 kHalo along the component, one more across.
__host__ __device__ constexpr int fdim(int c, int a) { return kT[a] + 2 * kHalo + (a == c ? 0 : 1); }
__host__ __device__ constexpr int fsize(int c) { return fdim(c, 0) * fdim(c, 1) * fdim(c, 2); }
__host__ __device__ constexpr int foff(int c) { return c == 0 ? 0 : (c == 1 ? fsize(0) : fsize(0) + fsize(1)); }
constexpr int kFStage = fsize(0) + fsize(1) + fsize(2);

// contributions go to the workgroup's LDS current window (one block per
// component, dims jdim).  The window is FP64 for both particle precisions:
// on gfx950 an FP64 LDS atomic add sustains about twenty times the rate of
// an FP32 one, and the tile's partial sums keep more bits before the single
// FP32/FP64 flush.
template <typename real>
struct LdsAcc {
    double *win;
    int base[3];   // window index of the particle's start cell, per component
    int cur[3];    // ... of the current piece's cell
    __device__ inline LdsAcc(double *w, int ri, int rj, int rk) : win(w)
    {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            base[c] = ((ri + kHalo + 1) * jdim(c, 1) + (rj + kHalo + 1)) * jdim(c, 2) + (rk + kHalo + 1);
    }
    __device__ inline void set_cell(int wi, int wj, int wk)
    {
#pragma unroll
        for (int c = 0; c < 3; ++c) cur[c] = base[c] + (wi * jdim(c, 1) + wj) * jdim(c, 2) + wk;
    }
    __device__ inline void operator()(int comp, int di, int dj, int dk, real v)
    {
        const int d1 = jdim(comp, 1), d2 = jdim(comp, 2);
        atomicAdd(win + joff(comp) + cur[comp] + (di * d1 + dj) * d2 + dk, (double)v);
    }
};

// The second piece of a path that crossed one face, kept by its lane until
// another one comes to the same lane or the rounds end; then every lane of
// the wavefront deposits its own.  Some 1 % of the particles of a thermal
// plasma cross per step, so that every other wavefront would run the second
// piece for a lane or two in each round.  FP32 push 592 -> 578 us at 256x128x128
// (NDFX, Vay), 4.91 -> 4.84 ms at 512x256x256; in FP64, where the registers do
// not limit it but the second piece is a smaller share, 150 -> 152 us at
// 97x61x53, so there it is deposited at once.
template <typename real>
struct Pending {
    real q, p[3], s[3];
    int cell = -1;   // window index of its cell, a byte per axis; negative: none
};

template <typename real>
__device__ inline void deposit_pending(double *win, Pending<real> &pd)
{
    LdsAcc<real> acc(win, (pd.cell >> 16) - kHalo - 1, (pd.cell >> 8 & 255) - kHalo - 1, (pd.cell & 255) - kHalo - 1);
    acc.set_cell(0, 0, 0);
    deposit_segment<real>(acc, pd.q, pd.p[0], pd.p[1], pd.p[2], pd.s[0], pd.s[1], pd.s[2]);
    pd.cell = -1;
}

// E and Be of one node and component side by side in the field stage: one
// 8-byte LDS read takes 5.6 clocks per wavefront and CU at random cells, two
// 4-byte reads 10.4.  With the integer counters of DiagAcc and the crossing
// fractions taken only where a lane crosses (deposit_path): push 95.1 -> 92.5
// us at 128x64x64, 4.48 -> 4.38 ms at 512x256x256
template <typename real>
struct alignas(2 * sizeof(real)) EB {
    real e, b;
};

// Corner nodes of a window particle from the field stage (one block per
// component, dims fdim); the same squares as load_corners.
template <typename real>
__device__ inline void load_corners_stage(const EB<real> *st, int ri, int rj, int rk, Corners<real> &c)
{
    int b[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
        b[a] = foff(a) + ((ri + kHalo) * fdim(a, 1) + (rj + kHalo)) * fdim(a, 2) + (rk + kHalo);
    const int sx0 = fdim(0, 2), sx1 = fdim(1, 1) * fdim(1, 2), sy2 = fdim(2, 1) * fdim(2, 2), sz2 = fdim(2, 2);
    const int o[3][4] = {{0, sx0, 1, sx0 + 1},          // x components: (j, k) square
                         {0, sx1, 1, sx1 + 1},          // y components: (i, k) square
                         {0, sy2, sz2, sy2 + sz2}};     // z components: (i, j) square
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const EB<real> v = st[b[a] + o[a][m]];
            c.e[a][m] = v.e;
            c.b[a][m] = v.b;
        }
}

// w / D for 0 <= w < kMost (entries of a window or stage block) with a 24-bit
// multiplication: the general division's high multiplication takes four
// times as long
template <int D, int kMost>
__device__ inline int small_div(int w)
{
    constexpr int M = (65536 + D - 1) / D;
    static_assert((int64_t)kMost * (M * D - 65536) < 65536 && (int64_t)kMost * M < (1ll << 32), "w * M >> 16 is w / D");
    return (int)(__umul24((unsigned)w, (unsigned)M) >> 16);
}

// the node `rel` nodes after the one that first points to (which may lie before
// the array, as a window's first node may); rel * sizeof(real) fits 32 bits
// inside a window or stage, so the address is a scalar base and one register
template <typename real>
__device__ inline real &node_after(real *first, int rel)
{
    return at32(first, (uint32_t)rel * (uint32_t)sizeof(real));
}

// Component C of E and of Be into the stage, in two passes over a thread's
// share of the block: the loads (load_component), then the LDS writes
// (store_component).  Indices are clamped into the grid (no particle reads the
// nodes outside it), so that no load waits for a branch.  With the loads of
// all three components issued before the first write, a thread waits for
// memory once while staging, not once per block and share (the push measured
// 5 % faster at 256x128x128).  With the branches and the general divisions
// the push took 22.5 us at 64x32x32 and 98.6 us at 128x64x64, now 21.4 and 97.
constexpr int kStageIt = (fsize(0) + kTBlock - 1) / kTBlock;   // every block has fsize(0) nodes

template <int C, typename real>
__device__ inline void load_component(real (&e)[kStageIt], real (&b)[kStageIt], const real *__restrict__ E,
                                      const real *__restrict__ B, const Grid &g, int gi0, int gj0, int gk0)
{
    static_assert(fsize(C) == fsize(0), "stage blocks of equal size");
    constexpr int d1 = fdim(C, 1), d2 = fdim(C, 2);
    // the block's first node inside the grid, and each node relative to it
    const int ib = min(max(gi0, 0), g.nx - 1), jb = min(max(gj0, 0), g.ny - 1), kb = min(max(gk0, 0), g.nz - 1);
    const int64_t first = (int64_t)ib * g.sx + (int64_t)jb * g.sy + kb;
#pragma unroll
    for (int m = 0; m < kStageIt; ++m) {
        const int w = min((int)threadIdx.x + m * kTBlock, fsize(C) - 1);
        const int t = small_div<d2, fsize(C)>(w), li = small_div<d1, fsize(C)>(t);
        const int lk = w - t * d2, lj = t - li * d1;
        const int i = min(max(li + (gi0 - ib), -ib), g.nx - 1 - ib), j = min(max(lj + (gj0 - jb), -jb), g.ny - 1 - jb),
                  k = min(max(lk + (gk0 - kb), -kb), g.nz - 1 - kb);
        const int rel = (int)(__umul24((unsigned)i, (unsigned)g.sx) + __umul24((unsigned)j, (unsigned)g.sy)) + k;
        e[m] = node_after(E + first, rel);
        b[m] = node_after(B + first, rel);
    }
}

template <int C, typename real>
__device__ inline void store_component(EB<real> *dst, const real (&e)[kStageIt], const real (&b)[kStageIt])
{
#pragma unroll
    for (int m = 0; m < kStageIt; ++m) {
        const int w = threadIdx.x + m * kTBlock;
        if (w < fsize(C)) dst[foff(C) + w] = EB<real>{e[m], b[m]};
    }
}

// add component C of the current window to the grid: one global atomic per
// nonzero entry.  v holds the thread's share of the window block (entry
// threadIdx.x + m kTBlock), read from LDS for all three components before the
// first atomic; first is the window's first node.  A particle that deposits is
// is_inside (1 .. n - 3) and crosses one face per axis at most, so the nodes it
// reaches lie in the grid (0 .. n - 1) and entries outside it hold zero.  T:
// the precision of the sums over the workgroups.
constexpr int kFlushIt = (jsize(0) + kTBlock - 1) / kTBlock;

template <int C, typename T>
__device__ inline void flush_component(T *__restrict__ dst, const double (&v)[kFlushIt], const Grid &g, int64_t first)
{
    static_assert(jsize(C) <= kFlushIt * kTBlock, "window block larger than the thread shares");
    constexpr int d1 = jdim(C, 1), d2 = jdim(C, 2), most = kFlushIt * kTBlock;
#pragma unroll
    for (int m = 0; m < kFlushIt; ++m) {
        const int w = threadIdx.x + m * kTBlock;
        const int t = small_div<d2, most>(w), wi = small_div<d1, most>(t);
        const int wk = w - t * d2, wj = t - wi * d1;
        if (v[m] != 0.0) {   // zero past the block's end
            const int rel = (int)(__umul24((unsigned)wi, (unsigned)g.sx) + __umul24((unsigned)wj, (unsigned)g.sy)) + wk;
            unsafeAtomicAdd(&node_after(dst + first, rel), (T)v[m]);
        }
    }
}

template <typename real, int PUSHER>
__global__ void __launch_bounds__(kBlock) k_push_global(Grid g, Fields<real> f, Current<real> cur, Species<real> s,
                                                        int64_t first, int64_t n, StepConst<real> sc, double *diag)
{
    const int64_t p = first + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    DiagAcc da;
    if (p < first + n) {
        auto dep = [&](int, int, int, int base, real q, real pos[3], const real d[3], DiagAcc &) {
            GlobalAcc<real> acc{cur.jx, cur.jy, cur.jz, g.sx, g.sy, base, base};
            deposit_path<real>(acc, q, pos, d);
        };
        PRec<real> r;
        load_rec(s, p, r);
        if (r.cell >= 0) {
            Corners<real> nodes;
            load_corners(f, cell_base(g, r.cell), g.sx, g.sy, nodes);
            advance_particle<real, PUSHER>(g, nodes, r, sc, dep, da);
            store_rec(s, p, r);
        }
    }
    diag_accumulate(diag, da.q, da.e, da.n, da.fallback);
}


// A particle that starts outside the window is not pushed in its round but
// listed (its slot) in LDS, and the workgroup pushes the listed particles
// after its rounds, one per thread, through global memory.  Inline, every
// wavefront with one such lane would run the global gather and deposit for
// it; listed, they run densely (the push measured 3.8 % faster at
// 512x256x256, where they gather in the laser's wake, and 1.5 % slower at
// 256x128x128, where a few per chunk make a short serial tail).
//
// The chunks of all species follow each other in one launch: a launch takes
// some 20 us to fill the chip and to drain it, with every workgroup staging
// and flushing at once in between.  Particle phase 303 -> 252 us for three
// species at 135x75x71 (3 per cell), 54 -> 39 us for two at 64x32x32, FP64 175
// -> 152 us for two at 97x61x53; one species as before.
template <typename real>
struct TiledSpecies {
    Species<real> s;
    StepConst<real> sc;
    const int4 *chunks;
    double *diag;
    int first;     // workgroup of the species' first chunk
    int ishift;    // a tile's cells now start at i = 8 ti - ishift
};

template <typename real>
struct TiledArgs {
    TiledSpecies<real> sp[kMaxTiled];
    int ns;
};

//
// WIDE: the windows are added to FP64 arrays, which the E step takes along.
// Where tiles are cut into several chunks (chunk_size), a node's current would
// otherwise be the FP32 sum of so many more parts: its error against FP64 (rms
// of one step's J at 56x32x32 with 8 per cell) was 7.86e-8, with whole tiles
// 7.49e-8, and two runs differed by 2.3e-8 and 4.5e-9; now 7.33e-8, and two
// runs give the same bits.  The push takes 22.1 us instead of 21.6
// at 64x32x32, the E step 4.7 instead of 4.4 (a step 40.5 instead of 39.8 us, at
// 96x48x48 76.2 instead of 74.2).
template <typename real, int PUSHER, bool WIDE>
__global__ void __launch_bounds__(kTBlock) k_push_tiled(Grid g, Fields<real> f, Current<real> cur, Current<double> wide,
                                                        TileGeom tg, TiledArgs<real> args)
{
    __shared__ alignas(16) double win[kJWin];
    __shared__ EB<real> stage[kFStage];
    __shared__ uint32_t listed[kDefer];
    __shared__ int nlisted;
    // Chunks in groups of kXcdGroup per XCD.  Workgroups are dealt to the
    // XCDs round-robin; a line of the field arrays spans four tiles along k,
    // and neighbouring tiles share their halos, so with neighbours on
    // different XCDs each L2 fetches (and, for the current's flush, merges)
    // its own copy.  The groups leave the set of chunks in flight as it is.
    // Push 4.72 -> 4.40 ms at 512x256x256 and 0.615 -> 0.60 ms at 256x128x128;
    // groups of 2, 4, 8: 4.64, 4.59, 4.53 ms; 32 to 512: 4.37-4.45 ms but
    // 95-97 us at 128x64x64, against 93; one range per XCD: 4.48 ms.
    constexpr int kXcdGroup = 16;
    int vb = (int)blockIdx.x;
    if (vb < (int)gridDim.x / (8 * kXcdGroup) * (8 * kXcdGroup)) {
        const int xcd = vb % 8, l = vb / 8;
        vb = (l / kXcdGroup * 8 + xcd) * kXcdGroup + l % kXcdGroup;
    }
    int m = 0;
    while (m + 1 < args.ns && vb >= args.sp[m + 1].first) ++m;
    const TiledSpecies<real> &sp = args.sp[m];
    const Species<real> s = sp.s;
    const StepConst<real> sc = sp.sc;
    const int4 ch = sp.chunks[vb - sp.first];
    const int tile = ch.x;
    const int tk = tile % tg.ntz, t2 = tile / tg.ntz;
    const int tj = t2 % tg.nty, ti = t2 / tg.nty;
    const int i0 = ti * kTx - sp.ishift, j0 = tj * kTy, k0 = tk * kTz;
    // Slots as 32-bit indices: the record arrays are addressed as scalar
    // base + one shared 32-bit byte offset (capacity keeps slot * size below
    // 2^32).  The first two rounds' records load while the tile is staged.
    //
    // The rounds start at the chunk's first whole 128-byte line and the up to
    // 31 particles before it come last, so that a wavefront's accesses are
    // whole lines.  A tile starts anywhere, and the non-temporal stores write
    // a line that two wavefronts share twice, each time in part: the record
    // stream alone takes 3.79 ms for 260 M particles from an odd slot and
    // 2.67 ms from an aligned one (5.8 TB/s; 2.90 and 2.78 ms with cached
    // accesses, which cost the field sweeps 20 % at 256x128x128).  Push 5.36 ->
    // 4.73 ms at 512x256x256, 0.675 -> 0.62 ms at 256x128x128.
    const uint32_t count = (uint32_t)ch.z, end32 = (uint32_t)ch.y + count;
    const uint32_t aligned = min(((uint32_t)ch.y + 31u) & ~31u, end32);
    auto slot_of = [&](uint32_t n) {   // the n-th particle in the order of the rounds
        const uint32_t q = aligned + n;
        return q < end32 ? q : q - count;
    };
    uint32_t n = threadIdx.x;
    PRec<real> r1, r2;   // the records one and two rounds ahead
    if (n < count) load_rec32(s, slot_of(n), r1);
    if (n + kTBlock < count) load_rec32(s, slot_of(n + kTBlock), r2);
    static_assert(kJWin % 2 == 0, "cleared in pairs");
#pragma unroll
    for (int m = 0; m < (kJWin / 2 + kTBlock - 1) / kTBlock; ++m) {
        const int w = threadIdx.x + m * kTBlock;
        if (w < kJWin / 2) ((double2 *)win)[w] = make_double2(0.0, 0.0);
    }
    if (threadIdx.x == 0) nlisted = 0;
    {
        const int si = i0 - kHalo, sj = j0 - kHalo, sk = k0 - kHalo;
        real e[3][kStageIt], b[3][kStageIt];
        load_component<0>(e[0], b[0], f.ex, f.bex, g, si, sj, sk);
        load_component<1>(e[1], b[1], f.ey, f.bey, g, si, sj, sk);
        load_component<2>(e[2], b[2], f.ez, f.bez, g, si, sj, sk);
        store_component<0>(stage, e[0], b[0]);
        store_component<1>(stage, e[1], b[1]);
        store_component<2>(stage, e[2], b[2]);
    }
    __syncthreads();

    DiagAcc da;
    Pending<real> pd;
    // start cell relative to the tile, and whether it lies in the window
    int ri = 0, rj = 0, rk = 0;
    bool in_win = false;
    auto dep = [&](int, int, int, int base, real q, real pos[3], const real d[3], DiagAcc &acc_d) {
        // one accumulator per branch: a shared one with per-lane atomics
        // (path split once, two masked atomics per term) measured 2.5 % slower
        if (in_win) {
            LdsAcc<real> acc(win, ri, rj, rk);
            if (sizeof(real) == 8) {
                deposit_path<real>(acc, q, pos, d);
                return;
            }
            auto before = [&](bool crosses) {
                if (__any(crosses && pd.cell >= 0) && pd.cell >= 0) deposit_pending(win, pd);
            };
            auto pend = [&](real pq, const real pp[3], const real ps[3], const int w[3]) {
                pd.q = pq;
                for (int m = 0; m < 3; ++m) {
                    pd.p[m] = pp[m];
                    pd.s[m] = ps[m];
                }
                pd.cell = (ri + w[0] + kHalo + 1) << 16 | (rj + w[1] + kHalo + 1) << 8 | (rk + w[2] + kHalo + 1);
            };
            deposit_path_pending<real>(acc, q, pos, d, before, pend);
        } else {
            GlobalAcc<real> acc{cur.jx, cur.jy, cur.jz, g.sx, g.sy, base, base};
            deposit_path<real>(acc, q, pos, d);
            acc_d.fallback += 1;
        }
    };
    // software pipeline over the rounds of kTBlock particles: while one
    // particle is pushed, the next round's record has its field nodes
    // gathered and the record two rounds ahead is loading (the first two
    // rounds' records were issued before the staging).  listed_q: the
    // particle was listed for the pass after the rounds.
    auto gather = [&](const PRec<real> &q, uint32_t slot, int &a, int &b, int &cc, bool &w, bool &listed_q,
                      Corners<real> &nd) {
        listed_q = false;
        if (q.cell < 0) return;
        a = cell_i(q.cell) - i0;
        b = cell_j(q.cell) - j0;
        cc = cell_k(q.cell) - k0;
        w = (unsigned)(a + kHalo) < (unsigned)(kTx + 2 * kHalo) && (unsigned)(b + kHalo) < (unsigned)(kTy + 2 * kHalo) &&
            (unsigned)(cc + kHalo) < (unsigned)(kTz + 2 * kHalo);
        if (w) {
            load_corners_stage(stage, a, b, cc, nd);
            return;
        }
        const int at = atomicAdd(&nlisted, 1);
        if (at < kDefer) {
            listed[at] = slot;
            listed_q = true;
            return;
        }
        load_corners(f, cell_base(g, q.cell), g.sx, g.sy, nd);
    };
    int ri1 = 0, rj1 = 0, rk1 = 0;
    bool w1 = false, l1 = false;
    // The pipeline carries the next particle's E and Be (six values), not
    // its 24 field nodes: the nodes' LDS reads are issued before the push of
    // the current particle and interpolated after it, so the nodes are dead
    // at the loop's end and only six values are copied there (about a
    // hundred fewer register moves per round; push 0.5 % faster).
    real e1[3] = {}, b1[3] = {};
    if (n < count) {
        Corners<real> nd;
        gather(r1, slot_of(n), ri1, rj1, rk1, w1, l1, nd);
        if (r1.cell >= 0 && !l1) interp_corners(nd, r1.o[0], r1.o[1], r1.o[2], e1, b1);
    }
    // Each round stores the record of the round before it, right after
    // issuing its own loads: gfx9 counts loads and stores in one vmcnt, so
    // the loop's wait for those loads (one round later) then waits for
    // stores that have had a whole push to complete, not for stores just
    // issued.  The first round rewrites its own record unchanged, and free
    // and listed slots are rewritten unchanged, which keeps the stores
    // unconditional.
    PRec<real> rs = r1;
    uint32_t ps = slot_of(n);
    const bool started = n < count;
    for (; n < count; n += kTBlock) {
        PRec<real> r = r1;
        const real e[3] = {e1[0], e1[1], e1[2]}, b[3] = {b1[0], b1[1], b1[2]};
        ri = ri1;
        rj = rj1;
        rk = rk1;
        in_win = w1;
        const bool is_listed = l1;
        r1 = r2;
        const bool more = n + kTBlock < count;
        Corners<real> nd;
        // The round's memory operations (the next particle's LDS reads, the
        // record two rounds ahead, the previous record's store) are issued
        // at a raised wavefront priority, so that they reach the memory
        // system ahead of the other wavefronts' arithmetic: push 1.3 %
        // faster at both 512x256x256 and 256x128x128 (priority 1 or 3, or
        // raised also for the staging or the flush, measured less).
        __builtin_amdgcn_s_setprio(2);
        if (more) gather(r1, slot_of(n + kTBlock), ri1, rj1, rk1, w1, l1, nd);
        if (n + 2 * kTBlock < count) load_rec32(s, slot_of(n + 2 * kTBlock), r2);
        store_rec32(s, ps, rs);
        __builtin_amdgcn_s_setprio(0);
        if (r.cell >= 0 && !is_listed) advance_particle_eb<real, PUSHER>(g, e, b, r, sc, dep, da);
        if (more && r1.cell >= 0 && !l1) interp_corners(nd, r1.o[0], r1.o[1], r1.o[2], e1, b1);
        rs = r;
        ps = slot_of(n);
    }
    if (started) store_rec32(s, ps, rs);
    if (sizeof(real) == 4 && pd.cell >= 0) deposit_pending(win, pd);
    // the listed slots' rewrites complete before the pass below stores them
    // again (vmcnt 0; expcnt and lgkmcnt left at their maxima)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    {
        auto gdep = [&](int, int, int, int base, real q, real pos[3], const real d[3], DiagAcc &acc_d) {
            GlobalAcc<real> acc{cur.jx, cur.jy, cur.jz, g.sx, g.sy, base, base};
            deposit_path<real>(acc, q, pos, d);
            acc_d.fallback += 1;
        };
        const int nl = min(nlisted, kDefer);
        for (int e = threadIdx.x; e < nl; e += kTBlock) {
            const uint32_t q = listed[e];
            PRec<real> rr;
            load_rec32(s, q, rr);
            Corners<real> nn;
            load_corners(f, cell_base(g, rr.cell), g.sx, g.sy, nn);
            advance_particle<real, PUSHER>(g, nn, rr, sc, gdep, da);
            store_rec32(s, q, rr);
        }
    }

    {
        const int64_t first = (int64_t)(i0 - kHalo - 1) * g.sx + (j0 - kHalo - 1) * g.sy + k0 - kHalo - 1;
        double v[3][kFlushIt];
#pragma unroll
        for (int m = 0; m < kFlushIt; ++m) {
            const int w = threadIdx.x + m * kTBlock;
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c][m] = w < jsize(c) ? win[joff(c) + w] : 0.0;
        }
        if (WIDE) {
            flush_component<0>(wide.jx, v[0], g, first);
            flush_component<1>(wide.jy, v[1], g, first);
            flush_component<2>(wide.jz, v[2], g, first);
        } else {
            flush_component<0>(cur.jx, v[0], g, first);
            flush_component<1>(cur.jy, v[1], g, first);
            flush_component<2>(cur.jz, v[2], g, first);
        }
    }
    diag_accumulate(sp.diag, da.q, da.e, da.n, da.fallback);
}

// Photons with QED off move on straight lines (src/advance.cpp:173-183) and
// carry no current.
template <typename real>
__global__ void __launch_bounds__(kBlock) k_photon_move(Grid g, Species<real> s, int64_t first, int64_t n,
                                                        StepConst<real> sc, double *diag)
{
    const int64_t p = first + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    DiagAcc da;
    if (p < first + n) {
        const int c = s.cell[p];
        if (c >= 0 && !is_inside(g, cell_i(c), cell_j(c), cell_k(c))) {
            s.cell[p] = -1;   // p_boundary (src/plist.cpp:73-102)
        } else if (c >= 0) {
            const real u[3] = {s.ux[p], s.uy[p], s.uz[p]};
            const real gam = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
            const real a = sc.dt / gam;
            real pos[3] = {s.ox[p] + u[0] * a * sc.inv_d[0], s.oy[p] + u[1] * a * sc.inv_d[1],
                           s.oz[p] + u[2] * a * sc.inv_d[2]};
            int ci[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                const real fl = floor(pos[m]);
                ci[m] = (int)fl;
                pos[m] -= fl;
                if (pos[m] >= real(1)) {
                    pos[m] = real(0);
                    ci[m] += 1;
                }
            }
            const int ni = cell_i(c) + ci[0], nj = cell_j(c) + ci[1], nk = cell_k(c) + ci[2];
            const bool finite = fabs(u[0] * a) < real(1e30) && fabs(u[1] * a) < real(1e30) && fabs(u[2] * a) < real(1e30);
            if (!finite) count_nonfinite(sc.nonfinite);
            if (finite && is_inside(g, ni, nj, nk)) {
                s.cell[p] = pack_cell(ni, nj, nk);
                s.ox[p] = pos[0];
                s.oy[p] = pos[1];
                s.oz[p] = pos[2];
                const double q = s.q[p];
                da.q = q;
                da.n = 1;
                da.e = (double)gam * q;
            } else {
                s.cell[p] = -1;
            }
        }
    }
    diag_accumulate(diag, da.q, da.e, da.n, 0.0);
}

// Uniform thermal plasma: ppc particles per is_inside cell with ilo <= i < ihi,
// Philox keyed by (seed, cell * ppc + slot), 24-bit uniform offsets and
// Box-Muller normal momenta; written in cell order after slot `first`.
template <typename real>
__global__ void __launch_bounds__(kBlock) k_load_uniform(Grid g, Species<real> s, int64_t first, int ppc, double q,
                                                         double sigma, uint64_t seed, int ilo, int ihi, int64_t total)
{
    const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= total) return;
    const int slot = (int)(t % ppc);
    int64_t c = t / ppc;
    const int nk = g.nz - 3, nj = g.ny - 3;
    const int k = 1 + (int)(c % nk);
    c /= nk;
    const int j = 1 + (int)(c % nj);
    const int i = ilo + (int)(c / nj);
    const uint64_t cell = ((uint64_t)i * g.ny + j) * g.nz + k;
    const uint64_t gid = cell * (uint64_t)ppc + slot;
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    const u32x4 a = philox(u32x4{{(uint32_t)gid, (uint32_t)(gid >> 32), 0u, 0x51ADu}}, k0, k1);
    const u32x4 b = philox(u32x4{{(uint32_t)gid, (uint32_t)(gid >> 32), 1u, 0x51ADu}}, k0, k1);
    const double two_pi = 6.283185307179586;
    const double r1 = sqrt(-2.0 * log(u24_open0(a.v[3])));
    const double t1 = two_pi * u24(b.v[0]);
    const double r2 = sqrt(-2.0 * log(u24_open0(b.v[1])));
    const double t2 = two_pi * u24(b.v[2]);
    const int64_t o = first + t;
    s.cell[o] = pack_cell(i, j, k);
    s.ox[o] = (real)u24(a.v[0]);
    s.oy[o] = (real)u24(a.v[1]);
    s.oz[o] = (real)u24(a.v[2]);
    s.ux[o] = (real)(sigma * r1 * cos(t1));
    s.uy[o] = (real)(sigma * r1 * sin(t1));
    s.uz[o] = (real)(sigma * r2 * cos(t2));
    s.q[o] = (real)q;
    if (s.chi) s.chi[o] = real(0);
    if (s.id) s.id[o] = (int)gid;
}

// pmerging (src/mc.cpp:202-462), per species: total charge and count, the
// random deletion, the rescale of the survivors
template <typename real>
__global__ void __launch_bounds__(kBlock) k_charge_sum(Species<real> s, int64_t n, double *acc)
{
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double q = 0, c = 0;
    if (p < n && s.cell[p] >= 0) {
        q = fabs((double)s.q[p]);
        c = 1;
    }
    block_accumulate(acc, q, 0.0, c, 0.0);
}

template <typename real>
__global__ void __launch_bounds__(kBlock) k_merge_delete(Species<real> s, int64_t n, int mode, double pd, double av_q,
                                                         uint64_t seed, uint32_t step, uint32_t tag, double *acc)
{
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double sum = 0, c = 0;
    if (p < n && s.cell[p] >= 0) {
        const double q = (double)s.q[p], aq = fabs(q);
        const u32x4 v = philox(u32x4{{(uint32_t)p, step, tag, 0x3E76Eu}}, (uint32_t)seed, (uint32_t)(seed >> 32));
        const double r = ((double)(v.v[0] >> 11) * 4294967296.0 + (double)v.v[1]) * (1.0 / 9007199254740992.0);
        if (mode == 1) {
            if (r < pd) {
                s.cell[p] = -1;
                sum = aq;
                c = 1;
            }
        } else {
            const double x = 2 * aq / av_q, pp = pd / (1 + x * x * x * x);   // _ppd, src/mc.cpp:198-200
            if (r < pp) {
                s.cell[p] = -1;
                c = 1;
            } else {
                const real qn = (real)(q / (1 - pp));
                s.q[p] = qn;
                sum = fabs((double)qn);
            }
        }
    }
    block_accumulate(acc, sum, 0.0, c, 0.0);
}

template <typename real>
__global__ void __launch_bounds__(kBlock) k_scale_charge(Species<real> s, int64_t n, double a)
{
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p < n && s.cell[p] >= 0) s.q[p] = (real)((double)s.q[p] * a);
}

// node charge with trilinear weights (rhodeposition, src/deposition.cpp:358-429):
// add(node, value) with the node's offsets (0 or 1 per axis)
template <typename real, class Add>
__device__ inline void deposit_rho(const Species<real> &s, int64_t p, Add &&add)
{
    const double xa = s.ox[p], ya = s.oy[p], za = s.oz[p];
    const double xb = 1 - xa, yb = 1 - ya, zb = 1 - za;
    const double q = s.q[p];
    add(0, 0, 0, q * xb * yb * zb);
    add(1, 0, 0, q * xa * yb * zb);
    add(0, 1, 0, q * xb * ya * zb);
    add(0, 0, 1, q * xb * yb * za);
    add(1, 1, 0, q * xa * ya * zb);
    add(1, 0, 1, q * xa * yb * za);
    add(0, 1, 1, q * xb * ya * za);
    add(1, 1, 1, q * xa * ya * za);
}

template <typename real>
__device__ inline void deposit_rho_global(const Grid &g, const Species<real> &s, int64_t p, int c, double *rho)
{
    double *r = rho + 3 * (int64_t)(cell_i(c) * g.sx + cell_j(c) * g.sy + cell_k(c));
    deposit_rho(s, p, [&](int di, int dj, int dk, double v) {
        unsafeAtomicAdd(r + 3 * ((int64_t)di * g.sx + dj * g.sy + dk), v);
    });
}

template <typename real>
__global__ void __launch_bounds__(kBlock) k_compute_rho(Grid g, Species<real> s, int64_t first, int64_t n, double *rho)
{
    const int64_t p = first + (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    const int c = s.cell[p];
    if (c >= 0) deposit_rho_global(g, s, p, c, rho);
}

// The same for the sorted slots: a workgroup sums one chunk in an LDS window
// of its tile's nodes and one cell around them, and adds each nonzero node
// once.  Bound by the FP64 atomics: with eight global ones per particle
// qk_compute_rho took 972 us at 70x60x60 cells, 4 per cell, and 217 us at
// 50x36x34, now 661 and 141 us (the read-back included).
constexpr int kRho[3] = {kTx + 2 * kHalo + 1, kTy + 2 * kHalo + 1, kTz + 2 * kHalo + 1};   // nodes of the window

template <typename real>
__global__ void __launch_bounds__(kBlock) k_rho_tiled(Grid g, Species<real> s, const int4 *chunks, TileGeom tg,
                                                      int ishift, double *rho)
{
    constexpr int kNodes = kRho[0] * kRho[1] * kRho[2], kRow = kRho[2], kPlane = kRho[1] * kRho[2];
    __shared__ double win[kNodes];
    for (int w = threadIdx.x; w < kNodes; w += kBlock) win[w] = 0.0;
    const int4 ch = chunks[blockIdx.x];
    const int tk = ch.x % tg.ntz, t2 = ch.x / tg.ntz, tj = t2 % tg.nty, ti = t2 / tg.nty;
    const int i0 = ti * kTx - ishift - kHalo, j0 = tj * kTy - kHalo, k0 = tk * kTz - kHalo;
    __syncthreads();
    for (int m = threadIdx.x; m < ch.z; m += kBlock) {
        const int64_t p = (int64_t)ch.y + m;
        const int c = s.cell[p];
        if (c < 0) continue;
        const int ri = cell_i(c) - i0, rj = cell_j(c) - j0, rk = cell_k(c) - k0;
        if ((unsigned)ri < (unsigned)(kRho[0] - 1) && (unsigned)rj < (unsigned)(kRho[1] - 1) &&
            (unsigned)rk < (unsigned)(kRho[2] - 1)) {
            double *w = win + ri * kPlane + rj * kRow + rk;
            deposit_rho(s, p, [&](int di, int dj, int dk, double v) { atomicAdd(w + di * kPlane + dj * kRow + dk, v); });
        } else {
            deposit_rho_global(g, s, p, c, rho);
        }
    }
    __syncthreads();
    for (int w = threadIdx.x; w < kNodes; w += kBlock) {
        const double v = win[w];
        if (v == 0.0) continue;   // nodes outside the grid are no particle's
        const int wi = w / kPlane, wr = w - wi * kPlane, wj = wr / kRow, wk = wr - wj * kRow;
        unsafeAtomicAdd(rho + 3 * ((int64_t)(i0 + wi) * g.sx + (j0 + wj) * g.sy + (k0 + wk)), v);
    }
}

}  // namespace

template <typename real>
hipError_t launch_push_global(hipStream_t st, const Grid &g, const Fields<real> &f, const Current<real> &j,
                              const Species<real> &s, const PushArgs &a)
{
    if (a.n <= 0) return hipSuccess;
    const StepConst<real> sc = step_const<real>(g, a);
    if (a.kind == 1)
        k_photon_move<real><<<blocks_for(a.n), kBlock, 0, st>>>(g, s, a.first, a.n, sc, a.diag);
    else if (a.pusher == 1)
        k_push_global<real, 1><<<blocks_for(a.n), kBlock, 0, st>>>(g, f, j, s, a.first, a.n, sc, a.diag);
    else
        k_push_global<real, 0><<<blocks_for(a.n), kBlock, 0, st>>>(g, f, j, s, a.first, a.n, sc, a.diag);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_push_tiled(hipStream_t st, const Grid &g, const Fields<real> &f, const Current<real> &j,
                             const TileGeom &tg, int ns, const Species<real> *s, const PushArgs *a,
                             const Current<double> *wide)
{
    TiledArgs<real> args{};
    int total = 0;
    for (int m = 0; m < ns; ++m) {
        if (a[m].nchunks <= 0) continue;
        TiledSpecies<real> &t = args.sp[args.ns++];
        t.s = s[m];
        t.sc = step_const<real>(g, a[m]);
        t.chunks = a[m].chunks;
        t.diag = a[m].diag;
        t.first = total;
        t.ishift = a[m].ishift;
        total += a[m].nchunks;
    }
    if (total == 0) return hipSuccess;
    const Current<double> w = wide ? *wide : Current<double>{};
    auto launch = [&](auto kernel) { kernel<<<total, kTBlock, 0, st>>>(g, f, j, w, tg, args); };
    if constexpr (sizeof(real) == 4) {
        if (wide) {
            if (a[0].pusher == 1) launch(k_push_tiled<real, 1, true>);
            else launch(k_push_tiled<real, 0, true>);
            return hipGetLastError();
        }
    }
    if (a[0].pusher == 1) launch(k_push_tiled<real, 1, false>);
    else launch(k_push_tiled<real, 0, false>);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_load_uniform(hipStream_t st, const Grid &g, const Species<real> &s, int64_t first, int ppc,
                               double q, double sigma, uint64_t seed, int ilo, int ihi)
{
    const int64_t total = (int64_t)(ihi - ilo) * (g.ny - 3) * (g.nz - 3) * ppc;
    if (total <= 0) return hipSuccess;
    k_load_uniform<real><<<blocks_for(total), kBlock, 0, st>>>(g, s, first, ppc, q, sigma, seed, ilo, ihi, total);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_compute_rho(hipStream_t st, const Grid &g, const Species<real> &s, int64_t n, double *rho, int slot,
                              const TileGeom &tg, const int4 *chunks, int nchunks, int ishift, int64_t n_sorted)
{
    rho += slot;
    const int64_t first = nchunks > 0 ? std::min(n_sorted, n) : 0;
    if (first > 0) {
        k_rho_tiled<real><<<nchunks, kBlock, 0, st>>>(g, s, chunks, tg, ishift, rho);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (n <= first) return hipSuccess;
    k_compute_rho<real><<<blocks_for(n - first), kBlock, 0, st>>>(g, s, first, n, rho);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_charge_sum(hipStream_t st, const Species<real> &s, int64_t n, double *acc)
{
    if (n <= 0) return hipSuccess;
    k_charge_sum<real><<<blocks_for(n), kBlock, 0, st>>>(s, n, acc);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_merge_delete(hipStream_t st, const Species<real> &s, int64_t n, int mode, double p, double av_q,
                               uint64_t seed, uint32_t step, uint32_t tag, double *acc)
{
    if (n <= 0) return hipSuccess;
    k_merge_delete<real><<<blocks_for(n), kBlock, 0, st>>>(s, n, mode, p, av_q, seed, step, tag, acc);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_scale_charge(hipStream_t st, const Species<real> &s, int64_t n, double a)
{
    if (n <= 0) return hipSuccess;
    k_scale_charge<real><<<blocks_for(n), kBlock, 0, st>>>(s, n, a);
    return hipGetLastError();
}

#define QK_INST(real)                                                                                            \
    template hipError_t launch_push_global<real>(hipStream_t, const Grid &, const Fields<real> &,               \
                                                 const Current<real> &, const Species<real> &, const PushArgs &); \
    template hipError_t launch_push_tiled<real>(hipStream_t, const Grid &, const Fields<real> &,                \
                                                const Current<real> &, const TileGeom &, int,                   \
                                                const Species<real> *, const PushArgs *, const Current<double> *); \
    template hipError_t launch_load_uniform<real>(hipStream_t, const Grid &, const Species<real> &, int64_t, int, \
                                                  double, double, uint64_t, int, int);                           \
    template hipError_t launch_compute_rho<real>(hipStream_t, const Grid &, const Species<real> &, int64_t,       \
                                                 double *, int, const TileGeom &, const int4 *, int, int, int64_t); \
    template hipError_t launch_charge_sum<real>(hipStream_t, const Species<real> &, int64_t, double *);           \
    template hipError_t launch_merge_delete<real>(hipStream_t, const Species<real> &, int64_t, int, double, double, \
                                                  uint64_t, uint32_t, uint32_t, double *);                        \
    template hipError_t launch_scale_charge<real>(hipStream_t, const Species<real> &, int64_t, double);
QK_INST(float)
QK_INST(double)
#undef QK_INST

}  // namespace qk
