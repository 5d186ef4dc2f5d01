// qk_api.hip -- the C ABI of include/quillk.h: context (the reference's
// spatial_region at n_sr = 1, include/main.h:17-170), device buffers, the
// step driver in the order of src/main.cpp:2319-2332, and copies in and out.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "quillk.h"
#include "qk_drain.h"
#include "qk_kernels.h"

using namespace qk;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg)
{
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                                                    \
    do {                                                                                                 \
        hipError_t e_ = (expr);                                                                          \
        if (e_ != hipSuccess) return fail(QK_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

#define QK_TRY(expr)              \
    do {                          \
        int rc_ = (expr);         \
        if (rc_ != QK_OK) return rc_; \
    } while (0)

// Device scratch of qk_compute_rho_noalloc: the three FP64 node-charge
// arrays of a grid of up to kNoallocCells cells (48 MiB, held on each GPU the
// library runs on until the process ends).  In host code `scratch` is a
// host-side stand-in, not a device address: each device's copy is resolved
// once, by qk_create with that device current, into g_scratch_ptr[device],
// and only that pointer reaches kernels and copies.
constexpr int64_t kNoallocCells = int64_t(1) << 21;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) double scratch[3 * kNoallocCells];

std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

// this device's copy of `scratch`; the device must be current
int resolve_scratch(int dev)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev]) return QK_OK;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return fail(QK_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = (double *)ptr;
    return QK_OK;
}

double *scratch_ptr(int dev)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_ptr[dev];
}

// the arrays of one particle buffer (structure of arrays)
struct SoA {
    void *mem = nullptr;   // one allocation holding every array
    int *cell = nullptr;
    void *a[8] = {};       // ox oy oz ux uy uz q chi (chi only with QED)
    int *id = nullptr;     // only with track_ids
};

struct SpeciesBuf {
    bool active = false;
    double cmr = 0;
    int kind = 0;           // 0 charged, 1 photon
    int energy_mode = 0;    // 0 (g-1) q, 1 g q, 2 (g-1) q / cmr
    int64_t cap = 0;
    int64_t n = 0;          // slots in use (live or free)
    int64_t n_sorted = 0;   // slots [0, n_sorted) are in tile order with a valid work list
    SoA buf[2];             // current and sort target
    int cur = 0;
    int4 *chunks = nullptr; // tiled-kernel work list
    int max_chunks = 0;     // capacity of chunks
    int nchunks = 0;        // host copy after the last sort
    bool cut = false;       // tiles were cut into smaller chunks than kChunk (chunk_size)
    int steps_since_sort = 0;
    double fb_last = -1;    // window-fallback fraction of the last finished step (-1: unknown or re-sorted since)
    int ishift = 0;         // moving-window shifts since the last sort
    int *tile_start = nullptr;   // ntiles + 1: the tiles of slots [0, n_sorted) (the next sort's source)
};

// The recorded trajectory of qk_tape_begin: snapshots of the whole device
// state (the 15 field arrays and each species' record arrays) at steps 0,
// every, 2 every, ...  The adjoint recomputes one segment at a time from its
// snapshot, keeping that segment's per-step states, and runs the step
// adjoints backwards over them.
struct Tape {
    bool active = false;
    bool replay = false;          // recomputing a segment: no snapshots
    bool dirty = false;           // the state was changed outside qk_step
    int every = 0;
    int steps = 0;                // steps since qk_tape_begin
    int64_t n[QK_MAX_SPECIES] = {};
    size_t field_bytes = 0, bytes = 0;
    std::vector<void *> ckpt;     // snapshots at steps 0, every, ...
    std::vector<int> ckpt_jcur;
    std::vector<uint32_t> ckpt_step;   // step index at each snapshot (laser sources depend on it)
    void *seg = nullptr;          // every per-step states of one segment
    void *fin = nullptr;          // the end state, restored after the adjoint
    double *lam = nullptr;        // 12 field adjoints: E, B, Be, J
    double *lpart = nullptr;      // 7 record adjoints per species
    // tangent-linear run along the recorded steps (qk_tangent_begin)
    bool tangent = false;
    double *tfield = nullptr;     // 15 FP64 arrays: E, B, Be, J (two buffers)
    int tjcur = 0;
    double *tpart = nullptr;      // 7 record tangents per species (x y z ux uy uz q)
};

// the laser sources of one side of the box (qk_add_laser_source)
struct InjSide {
    int nsrc = 0;
    int plane = 0;
    LaserFrame src[kMaxSources];
    uint32_t t0[kMaxSources] = {};   // step index at which each source was added
    int shifts0[kMaxSources] = {};   // window shifts at that time
};

}  // namespace

struct qk_ctx {
    qk_params p;
    Grid g;
    TileGeom tg;
    SolverCoef coef;
    hipStream_t stream = nullptr;
    size_t rsize = 4;               // bytes per real
    void *fmem = nullptr;           // all field arrays
    void *mid = nullptr;            // B at the step's end while the grid's B is half a step ahead (three arrays)
    bool no_mid = false;            // the memory for it is not there
    void *wide = nullptr;           // FP32: FP64 part of the current where tiles are cut (three arrays)
    bool wide_clear = false;        // whether it is zero
    bool b_ahead = false, b_held = false;   // the grid's B is half a step ahead; and mid holds the step's
    void *F[15] = {};               // ex ey ez bx by bz bex bey bez j0x j0y j0z j1x j1y j1z
    int jcur = 0;                   // current buffer deposited this step
    bool j_zero[2] = {true, true};  // which current buffers are known to be zero
    bool have_step = false;
    SpeciesBuf sp[QK_MAX_SPECIES];
    // shared sort buffers (allocated at the first sort)
    int *s_counts = nullptr, *s_imm = nullptr, *s_offsets = nullptr, *s_tile_start = nullptr, *s_tile_mult = nullptr,
        *s_chunk_n = nullptr, *s_chunk_off = nullptr, *s_scratch = nullptr;
    int *h_sortinfo = nullptr;      // pinned: [live count, chunk count]
    double *d_diag = nullptr;       // two rows (steps alternate) of kDiagRow
    double *diag_row = nullptr;     // the current step's
    bool diag_clear = false;        // whether both rows are zero
    double *h_diag = nullptr;       // pinned per-step copies of the accumulators
    size_t h_diag_cap = 0;          // steps that fit in h_diag
    std::vector<hipEvent_t> ev;     // timing events
    double ms_total = 0, ms_part = 0, ms_field = 0, fallback_frac = 0;
    // QED: device slot counters of every species plus an overflow flag and the
    // word that lets the push go ahead, and their pinned host mirror; the global step index keys the random streams
    int *d_count = nullptr;
    int *h_count = nullptr;         // pinned: values on their way to d_count
    int dev_n[QK_MAX_SPECIES];      // what d_count holds as far as the host knows (-1: unknown)
    QedCounts *h_qed = nullptr;     // pinned: [0] after the pairs from vacuum, [1] at the step's end
    unsigned qed_seq = 0, qed_end = 0;   // last one launched; the step's end
    uint32_t step_index = 0;
    // merging: device accumulators, their pinned mirror, and the deletion
    // fractions of a merge due at the start of the next step
    double *d_merge = nullptr;
    double *h_merge = nullptr;
    bool merge_due = false;
    double merge_ppd[QK_MAX_SPECIES] = {};
    // moving window: get_max_w result (device, pinned mirror) and the staging
    // buffer of qk_fill_cells' cell lists
    unsigned long long *d_maxw = nullptr, *h_maxw = nullptr;   // the value, then the workgroups done / the flag
    unsigned maxw_seq = 0;
    void *d_fill = nullptr;
    size_t fill_cap = 0;
    void *h_fill = nullptr;         // pinned, and the event after its last copy
    hipEvent_t fill_read = nullptr;
    Tape tape;
    // read-backs: pinned slots on the way to the caller's arrays, and the
    // scanned live counts of the species being read
    Drain drain;
    int *d_live = nullptr;
    size_t live_cap = 0;            // runs that fit
    // rows of particles on their way from and to the caller's arrays
    double *rows = nullptr;
    size_t rows_cap = 0;            // bytes
    // laser sources at an x plane, per side (0: x-min, 1: x-max)
    InjSide inj[2];
    int window_shifts = 0;          // qk_moving_window calls so far
};

namespace {

// a step's results: per-species accumulators, then the field-energy slots and
// the count of particles dropped for a non-finite momentum
constexpr size_t kSpeciesLen = QK_MAX_SPECIES * kDiagPerSpecies;
constexpr size_t kDiagLen = kSpeciesLen + kEnergySlots + 1;
constexpr size_t kNonfiniteSlot = kDiagLen - 1;
// and where they are accumulated: the copies of the species' accumulators first
constexpr size_t kRowEnergy = (size_t)kDiagSlots * kDiagStride;
constexpr size_t kRowNonfinite = kRowEnergy + kEnergySlots;
constexpr size_t kDiagRow = kRowNonfinite + 1;
static_assert(kSpeciesLen <= (size_t)kDiagStride, "one copy holds every species");

template <typename real>
Fields<real> fields_of(qk_ctx *c)
{
    Fields<real> f;
    f.ex = (real *)c->F[0]; f.ey = (real *)c->F[1]; f.ez = (real *)c->F[2];
    f.bx = (real *)c->F[3]; f.by = (real *)c->F[4]; f.bz = (real *)c->F[5];
    f.bex = (real *)c->F[6]; f.bey = (real *)c->F[7]; f.bez = (real *)c->F[8];
    return f;
}

template <typename real>
Current<real> current_of(qk_ctx *c, int which)
{
    Current<real> j;
    j.jx = (real *)c->F[9 + 3 * which];
    j.jy = (real *)c->F[10 + 3 * which];
    j.jz = (real *)c->F[11 + 3 * which];
    return j;
}

template <typename real>
Species<real> view(const SoA &b)
{
    Species<real> s;
    s.cell = b.cell;
    s.ox = (real *)b.a[0]; s.oy = (real *)b.a[1]; s.oz = (real *)b.a[2];
    s.ux = (real *)b.a[3]; s.uy = (real *)b.a[4]; s.uz = (real *)b.a[5];
    s.q = (real *)b.a[6];
    s.chi = (real *)b.a[7];
    s.id = b.id;
    return s;
}

double species_cmr(const qk_params &p, int s)
{
    if (s == QK_ELECTRON) return -1;
    if (s == QK_POSITRON) return 1;
    if (s == QK_PHOTON) return 0;
    return p.ion_cmr[s - QK_ION0];
}

bool species_valid(const qk_ctx *c, int s)
{
    if (s < 0 || s >= QK_MAX_SPECIES) return false;
    if (s >= QK_ION0 && s - QK_ION0 >= c->p.n_ion) return false;
    return true;
}

int alloc_soa(qk_ctx *c, SoA &b, int64_t cap)
{
    const size_t r = c->rsize;
    const bool chi = c->p.qed != 0, ids = c->p.track_ids != 0;
    auto align = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t a_int = align((size_t)cap * 4), a_real = align((size_t)cap * r);
    const size_t bytes = a_int + 7 * a_real + (chi ? a_real : 0) + (ids ? a_int : 0);
    void *mem = nullptr;
    HIP_TRY(hipMalloc(&mem, bytes));
    char *m = (char *)mem;
    b.mem = mem;
    b.cell = (int *)m;
    m += a_int;
    for (int a = 0; a < 7; ++a, m += a_real) b.a[a] = m;
    b.a[7] = chi ? (void *)m : nullptr;
    m += chi ? a_real : 0;
    b.id = ids ? (int *)m : nullptr;
    return QK_OK;
}

// (re)allocate both buffers of one species to cap slots, keeping slots [0, n)
int reserve(qk_ctx *c, int s, int64_t cap)
{
    SpeciesBuf &b = c->sp[s];
    if (cap <= b.cap) return QK_OK;
    SoA nb[2];
    for (int k = 0; k < 2; ++k) {
        int rc = alloc_soa(c, nb[k], cap);
        if (rc) {
            for (int m = 0; m < k; ++m) (void)hipFree(nb[m].mem);
            return rc;
        }
    }
    const size_t r = c->rsize;
    SoA &old = b.buf[b.cur];
    if (old.mem && b.n > 0) {
        HIP_TRY(hipMemcpyAsync(nb[0].cell, old.cell, (size_t)b.n * 4, hipMemcpyDeviceToDevice, c->stream));
        for (int a = 0; a < 8; ++a)
            if (old.a[a] && nb[0].a[a])
                HIP_TRY(hipMemcpyAsync(nb[0].a[a], old.a[a], (size_t)b.n * r, hipMemcpyDeviceToDevice, c->stream));
        if (old.id && nb[0].id) HIP_TRY(hipMemcpyAsync(nb[0].id, old.id, (size_t)b.n * 4, hipMemcpyDeviceToDevice, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
    }
    for (int k = 0; k < 2; ++k)
        if (b.buf[k].mem) HIP_TRY(hipFree(b.buf[k].mem));
    b.buf[0] = nb[0];
    b.buf[1] = nb[1];
    b.cur = 0;
    b.cap = cap;
    // work list capacity: every tile may end in a partial chunk
    const int64_t mc = (int64_t)c->tg.ntiles + cap / kMinChunk + 1;
    if (b.chunks) HIP_TRY(hipFree(b.chunks));
    b.chunks = nullptr;
    HIP_TRY(hipMalloc(&b.chunks, (size_t)mc * sizeof(int4)));
    b.max_chunks = (int)mc;
    b.n_sorted = 0;   // the work list refers to the old buffers
    b.nchunks = 0;
    return QK_OK;
}

int ensure_species(qk_ctx *c, int s, int64_t extra)
{
    SpeciesBuf &b = c->sp[s];
    if (!b.active) {
        b.active = true;
        b.cmr = species_cmr(c->p, s);
        b.kind = (s == QK_PHOTON) ? 1 : 0;
        b.energy_mode = (s == QK_PHOTON) ? 1 : (s >= QK_ION0 ? 2 : 0);
    }
    const int64_t need = b.n + extra;
    if (need <= b.cap) return QK_OK;
    // the push kernels address records with 32-bit byte offsets
    const int64_t limit = ((int64_t)1 << 32) / (int64_t)c->rsize;
    if (need >= limit)
        return fail(QK_ERR_CAPACITY, "more than " + std::to_string(limit - 1) + " particles in one species");
    int64_t cap = c->p.capacity > 0 ? c->p.capacity : std::min(std::max<int64_t>(need + need / 4, 1024), limit - 1);
    if (cap >= limit) return fail(QK_ERR_CAPACITY, "capacity " + std::to_string(cap) + " exceeds the 32-bit record offsets");
    if (cap < need) {
        if (c->p.capacity > 0)
            return fail(QK_ERR_CAPACITY, "particle capacity " + std::to_string(c->p.capacity) + " exceeded (need " +
                                             std::to_string(need) + ")");
        cap = need;
    }
    return reserve(c, s, cap);
}

int ensure_sort_buffers(qk_ctx *c)
{
    if (c->s_counts) return QK_OK;
    const size_t nk = (size_t)c->tg.nkeys + 1, nt = (size_t)c->tg.ntiles + 1;
    HIP_TRY(hipMalloc(&c->s_counts, nk * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_imm, nk * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_offsets, nk * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_tile_start, nt * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_tile_mult, nt * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_chunk_n, nt * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_chunk_off, nt * sizeof(int)));
    HIP_TRY(hipMalloc(&c->s_scratch, scan_scratch_ints(std::max(nk, nt)) * sizeof(int)));
    HIP_TRY(hipHostMalloc((void **)&c->h_sortinfo, 2 * sizeof(int)));
    return QK_OK;
}

// Most particles per workgroup of the tiled push.  With more than twice as
// many tiles as the chip has CUs a tile is one chunk (kChunk).  Fewer tiles
// leave CUs idle, or with one tile while others have two, and run their
// particles in long serial rounds.
//
// Up to half as many tiles as CUs: cut into as many parts as give one workgroup
// per CU; 1.3 covers the tiles at the box's faces, which hold less than the inner
// ones.  A second workgroup per CU (FP32 only: two fit) pays for its own staging
// and flush only where the parts stay above half of kChunk.  Particle phase at
// 128 tiles, 8 per cell: 35.3 -> 22.6 us (with other kernels of the time 36.8 ->
// 26.5, 33.9 with four parts per tile, 31.9 with 4096 per part; FP64 45.6 -> 30.3);
// 27 per cell: 57.0 -> 38.7 us (57.0 -> 47.1, 51.9 at three parts, 62.5 at six);
// 27 tiles: 31.4 -> 15.1 us.
//
// From there to twice as many tiles as CUs: halves, where they fill the CUs
// better and hold enough for their staging and flush: with 150 tiles 39.9 ->
// 26.3 us, 250 43.6 -> 32.2, 432 57.8 -> 50.3, FP64 77.9 -> 75.1 (8 per cell);
// but 27.3 -> 31.8 with 432 tiles and 2 per cell (20.5 us either way with 250).  FP64 has one
// workgroup per CU and gains only beyond one tile per CU.  With 576 tiles
// halves take 65 us against 71 at 8 per cell and 40 against 34 at 2, with 750
// tiles 78 against 76.
//
// Where FP32 tiles are cut, their currents are summed in FP64 (see k_push_tiled).
int chunk_size(const qk_ctx *c, int64_t n)
{
    constexpr int kCU = 256, kHalfMean = 2048;
    const int tiles = c->tg.ntiles;
    if (tiles > 2 * kCU) return kChunk;
    int64_t chunk;
    if (tiles > kCU / 2) {
        const bool halves = tiles > kCU ? n >= (int64_t)kHalfMean * tiles : c->rsize == 4;
        if (!halves) return kChunk;
        chunk = (13 * n / 10 / tiles + 1) / 2;
    } else {
        chunk = (13 * n / 10 + kCU - 1) / kCU;
        if (c->rsize == 4 && chunk > kChunk / 2) chunk = (chunk + 1) / 2;
    }
    return (int)std::min<int64_t>(std::max<int64_t>(chunk, kMinChunk), kChunk);
}

// the FP64 part of an FP32 region's current
Current<double> wide_of(const qk_ctx *c)
{
    const size_t n = c->g.ncell;
    double *w = (double *)c->wide;
    return w ? Current<double>{w, w + n, w + 2 * n} : Current<double>{};
}

// sort species s by (tile, cell), compacting free slots; builds its work list
template <typename real>
int sort_species(qk_ctx *c, int s)
{
    QK_TRY(ensure_sort_buffers(c));
    SpeciesBuf &b = c->sp[s];
    if (!b.tile_start) HIP_TRY(hipMalloc(&b.tile_start, ((size_t)c->tg.ntiles + 1) * sizeof(int)));
    SortBuffers sb;
    sb.counts = c->s_counts;
    sb.imm = c->s_imm;
    sb.old_start = b.n_sorted > 0 ? b.tile_start : nullptr;
    sb.n_sorted = b.n_sorted;
    sb.offsets = c->s_offsets;
    sb.tile_start = c->s_tile_start;
    sb.tile_mult = c->s_tile_mult;
    sb.chunk_n = c->s_chunk_n;
    sb.chunk_off = c->s_chunk_off;
    sb.chunks = b.chunks;
    sb.scratch = c->s_scratch;
    sb.max_chunks = b.max_chunks;
    sb.chunk = chunk_size(c, b.n);
    if (c->rsize == 4 && sb.chunk < kChunk && !c->wide &&
        hipMalloc(&c->wide, 3 * (size_t)c->g.ncell * sizeof(double)) != hipSuccess) {
        (void)hipGetLastError();   // the tiles stay whole
        c->wide = nullptr;
        sb.chunk = kChunk;
    }
    sb.info = c->h_sortinfo;
    HIP_TRY(launch_sort<real>(c->stream, c->tg, view<real>(b.buf[b.cur]), view<real>(b.buf[b.cur ^ 1]), b.n, sb));
    HIP_TRY(hipStreamSynchronize(c->stream));
    std::swap(b.tile_start, c->s_tile_start);   // the next sort's source
    b.cur ^= 1;
    b.cut = sb.chunk < kChunk;
    b.n = c->h_sortinfo[0];
    b.n_sorted = b.n;
    b.nchunks = c->h_sortinfo[1];
    b.steps_since_sort = 0;
    b.fb_last = -1;
    b.ishift = 0;
    if (b.nchunks > b.max_chunks) return fail(QK_ERR_STATE, "tile work list overflow");
    return QK_OK;
}

void unpack_diag(const qk_ctx *c, const double *h, qk_diag &d)
{
    std::memset(&d, 0, sizeof d);
    const double nn = c->p.norm_n, ef = c->p.norm_ef, ep = c->p.norm_ep;
    const double *e = h + QK_ELECTRON * kDiagPerSpecies, *po = h + QK_POSITRON * kDiagPerSpecies,
                 *ph = h + QK_PHOTON * kDiagPerSpecies;
    d.N_e = -e[0] * nn;   // electrons count with the opposite sign (fout.cpp:62)
    d.n_e = (int64_t)e[2];
    d.energy_e = -e[1] * ep;
    d.N_p = po[0] * nn;
    d.n_p = (int64_t)po[2];
    d.energy_p = po[1] * ep;
    d.N_ph = ph[0] * nn;
    d.n_ph = (int64_t)ph[2];
    d.energy_ph = ph[1] * ep;
    for (int s = QK_ION0; s < QK_MAX_SPECIES; ++s) {
        d.n_ion += (int64_t)h[s * kDiagPerSpecies + 2];
        d.energy_ions[s - QK_ION0] = h[s * kDiagPerSpecies + 1] * ep;
        d.energy_ion += d.energy_ions[s - QK_ION0];
    }
    double ef_sum = 0;
    for (int m = 0; m < kEnergySlots; ++m) ef_sum += h[kSpeciesLen + m];
    d.energy_f = ef_sum * ef;
    d.n_nonfinite = (int64_t)h[kNonfiniteSlot];
}

int ensure_events(qk_ctx *c, size_t n)
{
    while (c->ev.size() < n) {
        hipEvent_t e;
        HIP_TRY(hipEventCreate(&e));
        c->ev.push_back(e);
    }
    return QK_OK;
}

// pmerging (src/mc.cpp:202-462) on every species; see qk_pmerging
template <typename real>
int merge_impl(qk_ctx *c, int mode, const double *ppd)
{
    if (!c->d_merge) {
        HIP_TRY(hipMalloc(&c->d_merge, 4 * sizeof(double)));
        HIP_TRY(hipHostMalloc((void **)&c->h_merge, 4 * sizeof(double)));
    }
    auto reduce = [&](auto &&launch, double out[4]) -> int {
        HIP_TRY(launch_zero(c->stream, c->d_merge, 4));
        HIP_TRY(launch());
        HIP_TRY(hipMemcpyAsync(c->h_merge, c->d_merge, 4 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        for (int a = 0; a < 4; ++a) out[a] = c->h_merge[a];
        return QK_OK;
    };
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        SpeciesBuf &b = c->sp[s];
        if (!b.active || b.n == 0) continue;
        const double pd = mode == 1 ? ppd[0] : ppd[s];
        if (!(pd > 0)) continue;
        const Species<real> v = view<real>(b.buf[b.cur]);
        double tot[4], got[4];
        QK_TRY(reduce([&] { return launch_charge_sum<real>(c->stream, v, b.n, c->d_merge); }, tot));
        if (tot[2] == 0) continue;
        const double av_q = tot[0] / tot[2];
        QK_TRY(reduce([&] {
            return launch_merge_delete<real>(c->stream, v, b.n, mode, pd, av_q, c->p.seed, c->step_index,
                                             0x400u + (uint32_t)s, c->d_merge);
        }, got));
        // "ti": Q / (Q - deleted); "nl": Q / (sum of the raised survivors)
        double a;
        if (mode == 1) a = tot[0] - got[0] != 0 ? tot[0] / (tot[0] - got[0]) : 1;
        else a = got[0] != 0 ? tot[0] / got[0] : 0;
        HIP_TRY(launch_scale_charge<real>(c->stream, v, b.n, a));
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

// evaluate_merging_condition (src/main.cpp:1691-1748) on the live
// counts after the step just finished
void merge_condition(qk_ctx *c, const double (&live)[QK_MAX_SPECIES])
{
    const double crnp = c->p.crnp;
    const int nsp = QK_ION0 + c->p.n_ion;
    double cnt[QK_MAX_SPECIES] = {}, total = 0;
    for (int s = 0; s < nsp; ++s) {
        cnt[s] = live[s];
        total += cnt[s];
    }
    c->merge_due = false;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) c->merge_ppd[s] = 0;
    if (c->p.merging == 1) {
        if (total > nsp * crnp) {
            c->merge_due = true;
            c->merge_ppd[0] = (total - nsp * crnp) / total;
        }
    } else if (c->p.merging == 2) {
        for (int s = 0; s < nsp; ++s)
            if (cnt[s] > crnp) {
                c->merge_due = true;
                c->merge_ppd[s] = (cnt[s] - crnp) / cnt[s];
            }
    }
}

// QED slot counters to the device where the host has changed them since
int qed_upload_counts(qk_ctx *c)
{
    bool same = true;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) same = same && c->dev_n[s] == (int)c->sp[s].n;
    if (same) return QK_OK;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) c->dev_n[s] = c->h_count[s] = (int)c->sp[s].n;
    c->h_count[QK_MAX_SPECIES] = 0;
    HIP_TRY(hipMemcpyAsync(c->d_count, c->h_count, (QK_MAX_SPECIES + 1) * sizeof(int), hipMemcpyHostToDevice,
                           c->stream));
    return QK_OK;
}

// The counters (and, with diag, the live counts) to h_qed[which], and the wait
// for them.  The GPU stores them and the host polls: the host has the counts
// while the GPU works on what was enqueued behind them, where a copy and a
// stream synchronization emptied the queue twice per step.
int qed_publish(qk_ctx *c, int which, const double *diag, const BornLimit &lim = BornLimit())
{
    HIP_TRY(launch_publish_counts(c->stream, c->d_count, QK_MAX_SPECIES + 1, diag, QK_MAX_SPECIES, c->h_qed + which,
                                  ++c->qed_seq, lim));
    return QK_OK;
}

int qed_wait(qk_ctx *c, int which, unsigned seq)
{
    const QedCounts &h = c->h_qed[which];
    HIP_TRY(wait_flag(c->stream, &h.flag, seq));
    if (h.n[QK_MAX_SPECIES]) {
        c->dev_n[0] = -1;   // the next upload clears the overflow flag
        return fail(QK_ERR_CAPACITY, "QED appends exceeded the reserved capacity");
    }
    for (int s = 0; s < QK_MAX_SPECIES; ++s)
        if (c->sp[s].active) c->dev_n[s] = (int)(c->sp[s].n = h.n[s]);
    return QK_OK;
}

// whether species s can take `extra` more slots (see ensure_species)
bool fits(const qk_ctx *c, int s, int64_t extra)
{
    const int64_t need = c->sp[s].n + extra;
    if (need <= c->sp[s].cap) return true;
    return c->p.capacity > 0 ? need <= c->p.capacity : need < ((int64_t)1 << 32) / (int64_t)c->rsize;
}

// The particle phase with QED on (src/main.cpp:2323-2324): birth_from_vacuum,
// then padvance with photon emission for leptons and pair creation for
// photons.  Capacity is reserved for the worst case (every cell bears a pair,
// every lepton emits, every photon converts) before the first push, so that no
// append can fail and a step that finds no room has moved nothing.  The
// particles that were there are pushed while the host waits for the number of
// pairs born from vacuum, which follow in a launch of their own (mostly none
// are).  Where there is no room for both worst cases at once, or more are born
// than the free photon slots can take the photons of (the kernel then returns
// at once), the host waits first and reserves for what was born.
template <typename real>
int qed_particle_phase(qk_ctx *c, const Fields<real> &f, const Current<real> &jc)
{
    SpeciesBuf &be = c->sp[QK_ELECTRON], &bp = c->sp[QK_POSITRON], &bph = c->sp[QK_PHOTON];
    const QedArgs qa{c->p.e_s, c->p.seed, c->step_index};
    auto target = [&](int s) {
        SpeciesBuf &b = c->sp[s];
        AppendTarget<real> t;
        t.s = view<real>(b.buf[b.cur]);
        t.count = c->d_count + s;
        t.cap = (int)b.cap;
        t.overflow = c->d_count + QK_MAX_SPECIES;
        t.diag = c->diag_row + s * kDiagPerSpecies;
        return t;
    };
    auto push_args = [&](int s, int64_t first, int64_t n) {
        const SpeciesBuf &b = c->sp[s];
        PushArgs a{};
        a.pusher = c->p.pusher;
        a.kind = b.kind;
        a.cmr = b.cmr;
        a.external_bz = c->p.external_bz;
        a.diag = c->diag_row + s * kDiagPerSpecies;
        a.energy_mode = b.energy_mode;
        a.nonfinite = c->diag_row + kRowNonfinite;
        a.first = first;
        a.n = n;
        return a;
    };
    // electrons, positrons and photons from their slot `first` on
    auto push = [&](const int64_t (&first)[3], const int64_t (&n)[3], const int *go = nullptr) -> int {
        const int sp[3] = {QK_ELECTRON, QK_POSITRON, QK_PHOTON};
        Species<real> s[3];
        PushArgs a[3];
        for (int m = 0; m < 3; ++m) {
            s[m] = view<real>(c->sp[sp[m]].buf[c->sp[sp[m]].cur]);
            a[m] = push_args(sp[m], first[m], n[m]);
        }
        HIP_TRY(launch_qed_particles<real>(c->stream, c->g, f, jc, s, a, qa, target(QK_ELECTRON), target(QK_POSITRON),
                                           target(QK_PHOTON), go));
        return QK_OK;
    };
    const int64_t ninner = std::max<int64_t>(0, (int64_t)(c->p.nx - 4) * (c->p.ny - 4) * (c->p.nz - 4));
    const int64_t ne = be.n, np = bp.n, nph = bph.n;   // photons emitted in this step are not visited
    bool ahead = ninner > 0 && fits(c, QK_ELECTRON, ninner + nph) && fits(c, QK_POSITRON, ninner + nph) &&
                 fits(c, QK_PHOTON, ne + np) && ensure_species(c, QK_ELECTRON, ninner + nph) == QK_OK &&
                 ensure_species(c, QK_POSITRON, ninner + nph) == QK_OK &&
                 ensure_species(c, QK_PHOTON, ne + np) == QK_OK;
    if (!ahead) (void)hipGetLastError();
    if (ninner > 0) {
        QK_TRY(ensure_species(c, QK_ELECTRON, ninner));
        QK_TRY(ensure_species(c, QK_POSITRON, ninner));
        QK_TRY(qed_upload_counts(c));
        HIP_TRY(launch_vacuum_pairs<real>(c->stream, c->g, f, c->p.pusher, c->p.q_vac, qa, target(QK_ELECTRON),
                                          target(QK_POSITRON)));
        const int64_t room = bph.cap - nph;   // leptons that may emit
        int *go = ahead ? c->d_count + QK_MAX_SPECIES + 1 : nullptr;
        QK_TRY(qed_publish(c, 0, nullptr, {go, QK_ELECTRON, QK_POSITRON, room}));
        if (ahead) QK_TRY(push({0, 0, 0}, {ne, np, nph}, go));
        QK_TRY(qed_wait(c, 0, c->qed_seq));
        ahead = ahead && be.n + bp.n <= room;
    }
    const int64_t born_e = be.n - ne, born_p = bp.n - np;
    if (!ahead) {
        QK_TRY(ensure_species(c, QK_PHOTON, be.n + bp.n));
        QK_TRY(ensure_species(c, QK_ELECTRON, nph));
        QK_TRY(ensure_species(c, QK_POSITRON, nph));
        QK_TRY(qed_upload_counts(c));
        QK_TRY(push({0, 0, 0}, {be.n, bp.n, nph}));
    } else if (born_e > 0 || born_p > 0) {
        QK_TRY(push({ne, np, 0}, {born_e, born_p, 0}));
    }
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        SpeciesBuf &b = c->sp[s];
        const int64_t n = s == QK_ELECTRON ? ne + born_e : (s == QK_POSITRON ? np + born_p : (s == QK_PHOTON ? nph : b.n));
        if (!b.active || n == 0) continue;
        if (s >= QK_ION0)
            HIP_TRY(launch_push_global<real>(c->stream, c->g, f, jc, view<real>(b.buf[b.cur]), push_args(s, 0, n)));
        ++b.steps_since_sort;
    }
    QK_TRY(qed_publish(c, 1, c->diag_row));
    c->qed_end = c->qed_seq;
    return QK_OK;
}

// ---- adjoint tape -----------------------------------------------------------

// the record arrays a snapshot keeps per species: cell, ox oy oz ux uy uz q
size_t species_state_bytes(const qk_ctx *c, int64_t n) { return (size_t)n * (4 + 7 * c->rsize); }

// the whole state to (save) or from a snapshot
int tape_copy(qk_ctx *c, void *snap, bool save)
{
    WordCopies w{};
    char *d = (char *)snap;
    auto add = [&](void *state, size_t bytes) {
        w.src[w.count] = (const uint32_t *)(save ? state : d);
        w.dst[w.count] = (uint32_t *)(save ? d : state);
        w.n[w.count++] = (int64_t)(bytes / 4);
        d += bytes;
    };
    static_assert(1 + 8 * QK_MAX_SPECIES <= WordCopies::kMost, "an entry per array");
    add(c->fmem, c->tape.field_bytes);
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        const int64_t n = c->tape.n[s];
        if (n == 0) continue;
        const SoA &b = c->sp[s].buf[c->sp[s].cur];
        add(b.cell, (size_t)n * 4);
        for (int a = 0; a < 7; ++a) add(b.a[a], (size_t)n * c->rsize);
    }
    HIP_TRY(launch_copy_words(c->stream, w));
    return QK_OK;
}

int tape_save(qk_ctx *c, void *dst) { return tape_copy(c, dst, true); }
int tape_load(qk_ctx *c, const void *src) { return tape_copy(c, const_cast<void *>(src), false); }

// views of a saved state: the fields (E, Be) and one species' records
template <typename real>
Fields<real> saved_fields(const qk_ctx *c, const void *state)
{
    const size_t fb = c->tape.field_bytes / 15;
    const char *m = (const char *)state;
    Fields<real> f;
    real *F[9];
    for (int a = 0; a < 9; ++a) F[a] = (real *)(m + a * fb);
    f.ex = F[0]; f.ey = F[1]; f.ez = F[2];
    f.bx = F[3]; f.by = F[4]; f.bz = F[5];
    f.bex = F[6]; f.bey = F[7]; f.bez = F[8];
    return f;
}

template <typename real>
Species<real> saved_species(const qk_ctx *c, const void *state, int s)
{
    const char *d = (const char *)state + c->tape.field_bytes;
    for (int t = 0; t < s; ++t) d += species_state_bytes(c, c->tape.n[t]);
    const int64_t n = c->tape.n[s];
    Species<real> v;
    v.cell = (int *)d;
    d += (size_t)n * 4;
    real *a[7];
    for (int k = 0; k < 7; ++k) {
        a[k] = (real *)d;
        d += (size_t)n * c->rsize;
    }
    v.ox = a[0]; v.oy = a[1]; v.oz = a[2];
    v.ux = a[3]; v.uy = a[4]; v.uz = a[5];
    v.q = a[6];
    v.chi = nullptr;
    v.id = nullptr;
    return v;
}

int tape_snapshot(qk_ctx *c)
{
    void *m = nullptr;
    HIP_TRY(hipMalloc(&m, c->tape.bytes));
    c->tape.ckpt.push_back(m);
    c->tape.ckpt_jcur.push_back(c->jcur);
    c->tape.ckpt_step.push_back(c->step_index);
    return tape_save(c, m);
}

void tape_free(qk_ctx *c)
{
    Tape &t = c->tape;
    for (void *m : t.ckpt) (void)hipFree(m);
    t.ckpt.clear();
    t.ckpt_jcur.clear();
    t.ckpt_step.clear();
    if (t.seg) (void)hipFree(t.seg);
    if (t.fin) (void)hipFree(t.fin);
    if (t.lam) (void)hipFree(t.lam);
    if (t.lpart) (void)hipFree(t.lpart);
    if (t.tfield) (void)hipFree(t.tfield);
    if (t.tpart) (void)hipFree(t.tpart);
    t.seg = t.fin = nullptr;
    t.lam = t.lpart = nullptr;
    t.tfield = t.tpart = nullptr;
    t.tangent = false;
    t.active = t.replay = t.dirty = false;
    t.steps = 0;
}

template <typename real>
int step_impl(qk_ctx *c, int nsteps, qk_diag *diag);
int download_fields(qk_ctx *c, int nf, double *const *aos, void *const (*comp)[3], size_t rsize);
int download_doubles(qk_ctx *c, double *dst, const double *src, int64_t n, int64_t of = 0);

// at least `bytes` at c->rows; callers move their rows in blocks of at most kRowBytes
constexpr size_t kRowBytes = (size_t)64 << 20, kRow = 7 * sizeof(double);

int ensure_rows(qk_ctx *c, size_t bytes)
{
    if (bytes <= c->rows_cap) return QK_OK;
    if (c->rows) HIP_TRY(hipFree(c->rows));
    c->rows = nullptr;
    c->rows_cap = 0;
    HIP_TRY(hipMalloc(&c->rows, bytes));
    c->rows_cap = bytes;
    return QK_OK;
}

// whether the ids of slots [0, n) name each row 0 .. n - 1 once
int check_row_ids(qk_ctx *c, const int *id, int64_t n)
{
    if (!id) return fail(QK_ERR_STATE, "rows by id need track_ids");
    int *seen = nullptr, bad = 0;
    HIP_TRY(hipMalloc(&seen, ((size_t)n + 1) * sizeof(int)));
    hipError_t e = launch_fill_int(c->stream, seen, (size_t)n + 1, 0);
    if (e == hipSuccess) e = launch_check_ids(c->stream, id, n, seen, seen + n);
    if (e == hipSuccess) e = hipMemcpyAsync(&bad, seen + n, sizeof(int), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    const hipError_t e2 = hipFree(seen);
    HIP_TRY(e);
    HIP_TRY(e2);
    return bad ? fail(QK_ERR_INVALID, "rows by id: the ids are not 0 .. n - 1") : QK_OK;
}

// the adjoint sweep of qk_adjoint (see there)
template <typename real>
int adjoint_impl(qk_ctx *c, const double *lam_E, const double *lam_B, const double *const *lam_part, double *grad_E,
                 double *grad_B, double *const *grad_part, bool by_id)
{
    Tape &t = c->tape;
    const int64_t nc = c->g.ncell;
    const int T = t.steps;
    // adjoint buffers
    int64_t np_total = 0;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) np_total += t.n[s];
    if (!t.lam) HIP_TRY(hipMalloc(&t.lam, (size_t)nc * 12 * sizeof(double)));
    if (!t.lpart && np_total > 0) HIP_TRY(hipMalloc(&t.lpart, (size_t)np_total * 7 * sizeof(double)));
    if (!t.fin) HIP_TRY(hipMalloc(&t.fin, t.bytes));
    if (!t.seg) HIP_TRY(hipMalloc(&t.seg, t.bytes * (size_t)t.every));
    double *lam[12];
    for (int a = 0; a < 12; ++a) lam[a] = t.lam + (size_t)a * nc;
    double *lpart[QK_MAX_SPECIES][7] = {};
    {
        double *m = t.lpart;
        for (int s = 0; s < QK_MAX_SPECIES; ++s)
            for (int a = 0; a < 7; ++a) {
                lpart[s][a] = m;
                m += t.n[s];
            }
    }
    // the end state, and its bookkeeping, to come back to
    const int jcur_end = c->jcur;
    const uint32_t step_end = c->step_index;
    QK_TRY(tape_save(c, t.fin));
    // seeds: interleaved fields and rows go up in blocks of at most
    // kRowBytes and are laid out by kernels
    constexpr size_t kNode = 3 * sizeof(double);
    int64_t n_most = 0;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) n_most = std::max(n_most, t.n[s]);
    const size_t row_bytes = std::min(kRowBytes, std::max((size_t)n_most * kRow, (size_t)nc * kNode));
    const int64_t row_per = (int64_t)(row_bytes / kRow), node_per = (int64_t)(row_bytes / kNode);
    QK_TRY(ensure_rows(c, row_bytes));
    const int *row_id[QK_MAX_SPECIES] = {};
    for (int s = 0; s < QK_MAX_SPECIES && by_id; ++s)
        if (t.n[s] > 0) {
            row_id[s] = c->sp[s].buf[c->sp[s].cur].id;
            QK_TRY(check_row_ids(c, row_id[s], t.n[s]));
        }
    HIP_TRY(launch_zero(c->stream, t.lam, (size_t)nc * 12));
    for (int f = 0; f < 2; ++f) {
        const double *src = f == 0 ? lam_E : lam_B;
        for (int64_t m = 0; src && m < nc; m += node_per) {
            const int64_t k = std::min(node_per, nc - m);
            HIP_TRY(hipMemcpyAsync(c->rows, src + 3 * m, (size_t)k * kNode, hipMemcpyHostToDevice, c->stream));
            HIP_TRY(launch_split_fields(c->stream, c->rows, lam + 3 * f, m, k));
        }
    }
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        const int64_t n = t.n[s];
        if (n == 0) continue;
        if (!lam_part || !lam_part[s]) {
            HIP_TRY(launch_zero(c->stream, lpart[s][0], (size_t)n * 7));
            continue;
        }
        for (int64_t r = 0; r < n; r += row_per) {
            const int64_t k = std::min(row_per, n - r);
            HIP_TRY(hipMemcpyAsync(c->rows, lam_part[s] + 7 * r, (size_t)k * kRow, hipMemcpyHostToDevice, c->stream));
            HIP_TRY(launch_rows_in(c->stream, lpart[s], c->rows, row_id[s], c->sp[s].buf[c->sp[s].cur].cell, n, r, r + k));
        }
    }
    // the caller's arrays are free again (and a failed copy is reported here)
    HIP_TRY(hipStreamSynchronize(c->stream));
    // segments, last first
    t.replay = true;
    const int nseg = (T + t.every - 1) / t.every;
    for (int seg = nseg - 1; seg >= 0; --seg) {
        const int first = seg * t.every, last = std::min(T, first + t.every);
        QK_TRY(tape_load(c, t.ckpt[seg]));
        c->jcur = t.ckpt_jcur[seg];
        c->step_index = t.ckpt_step[seg];
        for (int n = first; n < last; ++n) {
            QK_TRY(tape_save(c, (char *)t.seg + (size_t)(n - first) * t.bytes));
            if (n + 1 < last) QK_TRY(step_impl<real>(c, 1, nullptr));
        }
        for (int n = last - 1; n >= first; --n) {
            const void *st = (const char *)t.seg + (size_t)(n - first) * t.bytes;
            HIP_TRY(launch_adj_fields(c->stream, c->p.solver, c->g, c->coef, lam));
            const Fields<real> f = saved_fields<real>(c, st);
            for (int s = 0; s < QK_MAX_SPECIES; ++s) {
                if (t.n[s] == 0) continue;
                PushArgs a{};
                a.pusher = c->p.pusher;
                a.kind = 0;
                a.cmr = c->sp[s].cmr;
                a.external_bz = c->p.external_bz;
                // the sort of qk_tape_begin, where there was one
                const SpeciesBuf &b = c->sp[s];
                a.chunks = b.chunks;
                a.nchunks = b.nchunks;
                a.ishift = b.ishift;
                a.first = b.n_sorted;
                HIP_TRY(launch_adj_particles<real>(c->stream, c->g, f, saved_species<real>(c, st, s), t.n[s], a, lam,
                                                   lpart[s], c->tg));
            }
        }
    }
    t.replay = false;
    // Be of step 0 came from interpolate_be, and init_boundaries zeroed the
    // boundary planes of the fields set before it: their adjoints are zero
    HIP_TRY(launch_adj_interp_be(c->stream, c->g, lam));
    {
        Fields<double> lf;
        lf.ex = lam[0]; lf.ey = lam[1]; lf.ez = lam[2];
        lf.bx = lam[3]; lf.by = lam[4]; lf.bz = lam[5];
        lf.bex = lam[6]; lf.bey = lam[7]; lf.bez = lam[8];
        HIP_TRY(launch_init_boundaries<double>(c->stream, c->p.solver, c->g, lf));
    }
    // results
    for (int f = 0; f < 2; ++f) {
        double *dst = f == 0 ? grad_E : grad_B;
        void *const comp[1][3] = {{lam[3 * f], lam[3 * f + 1], lam[3 * f + 2]}};
        if (dst) QK_TRY(download_fields(c, 1, &dst, comp, sizeof(double)));
    }
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        const int64_t n = t.n[s];
        if (n == 0 || !grad_part || !grad_part[s]) continue;
        for (int64_t r = 0; r < n; r += row_per) {
            const int64_t k = std::min(row_per, n - r);
            HIP_TRY(launch_rows_out(c->stream, lpart[s], c->rows, row_id[s], n, r, r + k));
            QK_TRY(download_doubles(c, grad_part[s] + 7 * r, c->rows, 7 * k, 7 * n));
        }
    }
    QK_TRY(tape_load(c, t.fin));
    c->jcur = jcur_end;
    c->step_index = step_end;
    c->j_zero[0] = c->j_zero[1] = false;   // the replayed steps' bookkeeping
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

// the tangent state: FP64 fields (E, B, Be) and the current buffer `which`
Fields<double> tangent_fields(const qk_ctx *c)
{
    const size_t n = (size_t)c->g.ncell;
    double *m = c->tape.tfield;
    Fields<double> f;
    f.ex = m; f.ey = m + n; f.ez = m + 2 * n;
    f.bx = m + 3 * n; f.by = m + 4 * n; f.bz = m + 5 * n;
    f.bex = m + 6 * n; f.bey = m + 7 * n; f.bez = m + 8 * n;
    return f;
}

Current<double> tangent_current(const qk_ctx *c, int which)
{
    const size_t n = (size_t)c->g.ncell;
    double *m = c->tape.tfield + (9 + 3 * which) * n;
    return Current<double>{m, m + n, m + 2 * n};
}

// the 7 record tangents of species s (slots of the tape)
void tangent_records(const qk_ctx *c, int s, double *out[7])
{
    double *m = c->tape.tpart;
    for (int t = 0; t < s; ++t) m += 7 * c->tape.n[t];
    for (int a = 0; a < 7; ++a) out[a] = m + (size_t)a * c->tape.n[s];
}

// Whether any pulse of the side can be nonzero near its plane after
// travelling shift[n]: the envelope is |x| < xs along the propagation axis,
// and x is linear in position, so the slab's corner points bound it.
bool side_active(const qk_ctx *c, const InjSide &side, const InjectArgs &a)
{
    const int lo = side.plane - 6 > 0 ? side.plane - 6 : 0;
    const int hi = side.plane + 6 < c->g.nx ? side.plane + 6 : c->g.nx;
    for (int n = 0; n < side.nsrc; ++n) {
        const LaserFrame &L = side.src[n];
        double xmin = 1e300, xmax = -1e300;
        for (int corner = 0; corner < 8; ++corner) {
            const double px = ((corner & 1) ? hi : lo) * c->g.dx + a.ishift[n] * c->g.dx;
            const double py = ((corner & 2) ? c->g.ny : 0) * c->g.dy, pz = ((corner & 4) ? c->g.nz : 0) * c->g.dz;
            double x = L.r0[0] * (px - L.x0 - L.xt) + L.r0[1] * (py - L.y12 - L.y0 - L.yt) +
                       L.r0[2] * (pz - L.z12 - L.z0 - L.zt);
            x -= L.b_sign ? a.shift[n] : -a.shift[n];
            xmin = std::min(xmin, x);
            xmax = std::max(xmax, x);
        }
        if (xmax > -L.xs && xmin < L.xs) return true;
    }
    return false;
}

// the laser sources' corrections of one sub-step of fadvance: b_field = 1
// after a B half step at time (step + frac) dt, 0 after the E step
template <typename real>
int inject_impl(qk_ctx *c, int b_field, double frac, real *const *mid = nullptr, double *energy = nullptr)
{
    InjectArgs a[2];
    int n = 0;
    for (int sd = 0; sd < 2; ++sd) {
        const InjSide &side = c->inj[sd];
        if (side.nsrc == 0) continue;
        InjectArgs &s = a[n];
        s = InjectArgs{};
        s.nsrc = side.nsrc;
        for (int m = 0; m < side.nsrc; ++m) {
            s.src[m] = side.src[m];
            s.shift[m] = ((double)(c->step_index - side.t0[m]) + frac) * c->g.dt;
            s.ishift[m] = c->window_shifts - side.shifts0[m];
        }
        s.side = sd;
        s.plane = side.plane;
        n += side_active(c, side, s);
    }
    HIP_TRY(launch_inject<real>(c->stream, c->p.solver, c->g, c->coef, fields_of<real>(c), b_field, n, a, mid, energy));
    return QK_OK;
}

// The fields at the end of the last finished step, where a call failed with B
// half a step ahead (step_all): B from mid, Be from that B.  Errors are not
// reported, the caller has one.
template <typename real>
void settle_b(qk_ctx *c)
{
    c->b_ahead = false;
    if (!c->b_held) return;   // neither particles nor sources: only the GPU itself can have failed
    const size_t fb = ((size_t)c->g.ncell * sizeof(real) + 255) & ~(size_t)255;
    WordCopies w{};
    for (; w.count < 3; ++w.count) {
        w.src[w.count] = (const uint32_t *)((char *)c->mid + w.count * fb);
        w.dst[w.count] = (uint32_t *)c->F[3 + w.count];
        w.n[w.count] = (int64_t)((size_t)c->g.ncell * sizeof(real) / 4);
    }
    (void)launch_copy_words(c->stream, w);
    (void)launch_interpolate_be<real>(c->stream, c->g, fields_of<real>(c));
    (void)hipStreamSynchronize(c->stream);
}

template <typename real>
int step_all(qk_ctx *c, int nsteps, qk_diag *diag)
{
    const Fields<real> f = fields_of<real>(c);
    // three events per step: before the particle phase (see `start`), between phases, after the field phase
    QK_TRY(ensure_events(c, 3 * (size_t)nsteps));
    if (c->h_diag_cap < (size_t)nsteps) {
        if (c->h_diag) HIP_TRY(hipHostFree(c->h_diag));
        c->h_diag = nullptr;
        HIP_TRY(hipHostMalloc((void **)&c->h_diag, (size_t)nsteps * kDiagLen * sizeof(double)));
        c->h_diag_cap = (size_t)nsteps;
    }
    double *hd = c->h_diag;
    const bool qed = c->p.qed != 0;
    // the QED kernels deposit through global atomics
    const bool tiled = c->p.deposit == QK_DEPOSIT_TILED && !qed;
    Tape &tp = c->tape;
    // Within a call the second half step of B runs together with the next
    // step's first one, which uses the same E: 72 instead of 96 B per cell for
    // B and Be (field phase 1.11 -> 0.99 ms per step at 512x256x256, 130 -> 117
    // us at 256x128x128 and 29.6 -> 22.5 us at 128x64x64 in calls of four
    // steps; 64x32x32 with a laser source, 73 -> 60 us per step).  The B
    // between the two, at the step's end, is what Be, the laser sources'
    // corrections and the field energy want: it is kept in `mid`.  A call that
    // fails on its way gets it back from there (settle_b): with particles a
    // later step may find no room for its appends or its sort.  Without
    // charged particles nothing reads Be between two steps, and without any
    // particles and laser sources nothing needs mid either.  The tape keeps the
    // state of every step, so there each half step runs by itself, and so it
    // does where the sources of both sides correct the same nodes.
    bool charged = qed || tp.active, any = charged;
    for (const SpeciesBuf &b : c->sp) {
        any = any || (b.active && b.n > 0);
        charged = charged || (b.active && b.n > 0 && b.kind == 0);
    }
    const bool need_mid = any || c->inj[0].nsrc > 0 || c->inj[1].nsrc > 0;
    bool fuse_b = !tp.active && (c->inj[0].nsrc == 0 || c->inj[1].nsrc == 0 ||
                                 sides_apart(c->inj[0].plane, c->inj[1].plane));
    real *mid_b[3] = {};
    if (fuse_b && need_mid && nsteps > 1) {
        const size_t fb = ((size_t)c->g.ncell * sizeof(real) + 255) & ~(size_t)255;
        if (!c->mid && !c->no_mid && hipMalloc(&c->mid, 3 * fb) != hipSuccess) {
            (void)hipGetLastError();   // the steps run without it
            c->mid = nullptr;
            c->no_mid = true;
        }
        fuse_b = c->mid != nullptr;
        for (int a = 0; a < 3; ++a) mid_b[a] = (real *)((char *)c->mid + a * fb);
    }
    real *const *mid = need_mid ? mid_b : nullptr;
    // the event that marks the start of each step's particle phase: the end
    // of the step before unless something ran in between
    std::vector<int> start((size_t)nsteps);
    // The E step clears what it hands over, so that a call that ended well
    // leaves both rows at zero (a launch less: 33.4 -> 30.3 us per call of one
    // step at 64x32x32 without particles).
    if (!c->diag_clear) HIP_TRY(launch_zero(c->stream, c->d_diag, 2 * kDiagRow));
    c->diag_clear = false;
    for (int l = 0; l < nsteps; ++l) {
        bool between = l == 0;
        c->diag_row = c->d_diag + (l & 1) * kDiagRow;
        if (tp.active && !tp.replay) {
            if (tp.steps > 0 && tp.steps % tp.every == 0) {
                QK_TRY(tape_snapshot(c));
                between = true;
            }
            ++tp.steps;
        }
        // The window fallback of step l - 2: once that step has ended, its
        // diagnostics are here, and the GPU still has step l - 1 queued while
        // the host decides.  The
        // first two steps of a call use the last step of the previous call
        // (kept per species), so the rule holds for callers that step one
        // step per call.
        bool fb_high[QK_MAX_SPECIES] = {};
        if (tiled && c->p.sort_fallback > 0 && l >= 2) {
            HIP_TRY(hipEventSynchronize(c->ev[3 * (l - 2) + 2]));
            const double *h = hd + (size_t)(l - 2) * kDiagLen;
            for (int s = 0; s < QK_MAX_SPECIES; ++s) {
                const double live = h[s * kDiagPerSpecies + 2], fb = h[s * kDiagPerSpecies + 3];
                fb_high[s] = live > 0 && fb > c->p.sort_fallback * live;
            }
        } else if (tiled && c->p.sort_fallback > 0) {
            for (int s = 0; s < QK_MAX_SPECIES; ++s) fb_high[s] = c->sp[s].fb_last > c->p.sort_fallback;
        }
        // cell-tile sort: the cadence, a fallback above sort_fallback (seen
        // on a layout at least two steps old), or an unsorted tail (appended
        // particles, pushed by the global kernel meanwhile) above 1/16 of the
        // sorted part (photons only with QED, where pair creation leaves free
        // slots)
        for (int s = 0; s < QK_MAX_SPECIES; ++s) {
            SpeciesBuf &b = c->sp[s];
            if (!b.active || b.n == 0 || (b.kind == 1 && !qed)) continue;
            const bool due = (c->p.sort_every > 0 && b.steps_since_sort >= c->p.sort_every) ||
                             (fb_high[s] && b.steps_since_sort >= 2);
            const bool tail = tiled && (b.n_sorted == 0 || (b.n - b.n_sorted) * 16 > b.n_sorted);
            if (tail || due) {
                QK_TRY(sort_species<real>(c, s));
                between = true;
            }
        }
        // a merge decided after the previous step runs first (pmerging before
        // birth_from_vacuum, src/main.cpp:2321-2322)
        if (c->merge_due) {
            QK_TRY(merge_impl<real>(c, c->p.merging, c->merge_ppd));
            c->merge_due = false;
            between = true;
        }
        const Current<real> jc = current_of<real>(c, c->jcur), jn = current_of<real>(c, c->jcur ^ 1);
        // padvance (src/advance.cpp:90-387); the push kernels erase the
        // particles p_boundary (src/plist.cpp:73-102) would: those outside
        // is_inside, which only a moving-window shift leaves behind
        if (between) HIP_TRY(hipEventRecord(c->ev[3 * l], c->stream));
        start[l] = between ? 3 * l : 3 * (l - 1) + 2;
        if (qed) QK_TRY(qed_particle_phase<real>(c, f, jc));
        // the sorted slots of every charged species go in one tiled launch, the
        // rest (photons, unsorted tails, the global deposit) one by one
        Species<real> ts[kMaxTiled];
        PushArgs ta[kMaxTiled];
        int nt = 0;
        bool cut = false;
        for (int s = 0; s < QK_MAX_SPECIES && !qed; ++s) {
            SpeciesBuf &b = c->sp[s];
            if (!b.active || b.n == 0) continue;
            PushArgs a{};
            a.pusher = c->p.pusher;
            a.kind = b.kind;
            a.cmr = b.cmr;
            a.external_bz = c->p.external_bz;
            a.diag = c->diag_row + s * kDiagPerSpecies;
            a.energy_mode = b.energy_mode;
            a.nonfinite = c->diag_row + kRowNonfinite;
            const Species<real> v = view<real>(b.buf[b.cur]);
            if (tp.tangent && !tp.replay && b.kind == 0 && tp.n[s] > 0) {
                // the tangent of this push, from the state before it
                double *tr[7];
                tangent_records(c, s, tr);
                const Current<double> tj = tangent_current(c, tp.tjcur);
                double *dj[3] = {tj.jx, tj.jy, tj.jz};
                HIP_TRY(launch_tlm_particles<real>(c->stream, c->g, f, tangent_fields(c), v, tp.n[s], a, dj, tr));
            }
            if (tiled && b.kind == 0) {
                a.chunks = b.chunks;
                a.nchunks = b.nchunks;
                a.ishift = b.ishift;
                ts[nt] = v;
                ta[nt++] = a;
                cut = cut || b.cut;
                a.first = b.n_sorted;   // the unsorted tail, if any
                a.n = b.n - b.n_sorted;
            } else {
                a.first = 0;
                a.n = b.n;
            }
            HIP_TRY(launch_push_global<real>(c->stream, c->g, f, jc, v, a));
            ++b.steps_since_sort;
        }
        const Current<double> wide = wide_of(c), *const w = cut && sizeof(real) == 4 ? &wide : nullptr;
        if (w && !c->wide_clear) HIP_TRY(launch_zero(c->stream, (double *)c->wide, 3 * (size_t)c->g.ncell));
        if (w) c->wide_clear = false;
        if (nt > 0) HIP_TRY(launch_push_tiled<real>(c->stream, c->g, f, jc, c->tg, nt, ts, ta, w));
        HIP_TRY(hipEventRecord(c->ev[3 * l + 1], c->stream));
        // fadvance (src/advance.cpp:13-18): B half, E, B half, interpolate_be.  The
        // first half step also sums compute_energy's field term, which sees the
        // fields before fadvance (src/main.cpp:2327)
        if (charged) c->j_zero[c->jcur] = false;
        const bool no_j = !charged && c->j_zero[0] && c->j_zero[1], last = l + 1 == nsteps;
        if (!c->b_ahead) {
            HIP_TRY(launch_maxwell_b<real>(c->stream, c->p.solver, c->g, c->coef, f, c->diag_row + kRowEnergy));
            QK_TRY(inject_impl<real>(c, 1, 0.0));
        }
        const DiagDrain dd{c->diag_row, hd + (size_t)l * kDiagLen, (int)kSpeciesLen, (int)(kDiagLen - kSpeciesLen)};
        HIP_TRY(launch_maxwell_e<real>(c->stream, c->p.solver, c->g, c->coef, f, no_j ? nullptr : &jc,
                                       no_j ? nullptr : &jn, dd, w));
        if (w) c->wide_clear = true;
        c->b_ahead = false;   // E has caught up
        c->j_zero[c->jcur ^ 1] = true;
        QK_TRY(inject_impl<real>(c, 0, 0.5));
        if (fuse_b && !last) {
            double *next_en = c->d_diag + ((l + 1) & 1) * kDiagRow + kRowEnergy;
            HIP_TRY(launch_maxwell_b<real>(c->stream, c->p.solver, c->g, c->coef, f, next_en, true, mid));
            c->b_ahead = true;
            c->b_held = mid != nullptr;
            if (mid) QK_TRY(inject_impl<real>(c, 1, 1.0, mid, next_en));
        } else {
            HIP_TRY(launch_maxwell_b<real>(c->stream, c->p.solver, c->g, c->coef, f, nullptr));
            QK_TRY(inject_impl<real>(c, 1, 1.0));
        }
        if (charged || last)
            HIP_TRY(launch_interpolate_be<real>(c->stream, c->g, f, fuse_b && !last ? mid_b : nullptr));
        if (tp.tangent && !tp.replay) {
            // the tangent fields advance with the same (linear) field step
            const Fields<double> tf = tangent_fields(c);
            const Current<double> tjc = tangent_current(c, tp.tjcur), tjn = tangent_current(c, tp.tjcur ^ 1);
            HIP_TRY(launch_maxwell_b<double>(c->stream, c->p.solver, c->g, c->coef, tf, nullptr));
            HIP_TRY(launch_maxwell_e<double>(c->stream, c->p.solver, c->g, c->coef, tf, &tjc, &tjn));
            HIP_TRY(launch_maxwell_b<double>(c->stream, c->p.solver, c->g, c->coef, tf, nullptr));
            HIP_TRY(launch_interpolate_be<double>(c->stream, c->g, tf));
            tp.tjcur ^= 1;
        }
        HIP_TRY(hipEventRecord(c->ev[3 * l + 2], c->stream));
        c->jcur ^= 1;
        if (qed) QK_TRY(qed_wait(c, 1, c->qed_end));
        if (c->p.merging) {
            double live[QK_MAX_SPECIES];
            if (!qed) HIP_TRY(hipStreamSynchronize(c->stream));
            for (int s = 0; s < QK_MAX_SPECIES; ++s)
                live[s] = qed ? c->h_qed[1].live[s] : hd[(size_t)l * kDiagLen + s * kDiagPerSpecies + 2];
            merge_condition(c, live);
        }
        ++c->step_index;
    }
    HIP_TRY(wait_event(c->ev[3 * (size_t)(nsteps - 1) + 2]));   // the last thing enqueued
    float t_part = 0, t_field = 0, t_tot = 0;
    for (int l = 0; l < nsteps; ++l) {
        float a = 0, b = 0;
        HIP_TRY(hipEventElapsedTime(&a, c->ev[start[l]], c->ev[3 * l + 1]));
        HIP_TRY(hipEventElapsedTime(&b, c->ev[3 * l + 1], c->ev[3 * l + 2]));
        t_part += a;
        t_field += b;
    }
    HIP_TRY(hipEventElapsedTime(&t_tot, c->ev[0], c->ev[3 * (nsteps - 1) + 2]));
    double fb = 0, live = 0;
    for (int l = 0; l < nsteps; ++l) {
        const double *h = hd + (size_t)l * kDiagLen;
        for (int s = 0; s < QK_MAX_SPECIES; ++s) {
            live += h[s * kDiagPerSpecies + 2];
            fb += h[s * kDiagPerSpecies + 3];
        }
        if (diag) unpack_diag(c, h, diag[l]);
    }
    c->fallback_frac = live > 0 ? fb / live : 0;
    {
        const double *h = hd + (size_t)(nsteps - 1) * kDiagLen;
        for (int s = 0; s < QK_MAX_SPECIES; ++s) {
            SpeciesBuf &b = c->sp[s];
            const double n_s = h[s * kDiagPerSpecies + 2];
            // a sort after the last push leaves the measurement stale
            b.fb_last = (n_s > 0 && b.steps_since_sort > 0) ? h[s * kDiagPerSpecies + 3] / n_s : -1;
        }
    }
    c->ms_total = t_tot;
    c->ms_part = t_part;
    c->ms_field = t_field;
    c->have_step = true;
    c->diag_clear = true;
    return QK_OK;
}

template <typename real>
int step_impl(qk_ctx *c, int nsteps, qk_diag *diag)
{
    const int rc = step_all<real>(c, nsteps, diag);
    if (c->b_ahead) settle_b<real>(c);
    return rc;
}

template <typename T>
void aos_to_soa(const double *aos, int64_t n, T *a, T *b, T *c)
{
    for (int64_t m = 0; m < n; ++m) {
        a[m] = (T)aos[3 * m];
        b[m] = (T)aos[3 * m + 1];
        c[m] = (T)aos[3 * m + 2];
    }
}

int upload3(qk_ctx *c, const double *aos, void *d0, void *d1, void *d2)
{
    const int64_t n = c->g.ncell;
    std::vector<char> buf((size_t)n * c->rsize * 3);
    if (c->rsize == 4) {
        float *h = (float *)buf.data();
        aos_to_soa<float>(aos, n, h, h + n, h + 2 * n);
    } else {
        double *h = (double *)buf.data();
        aos_to_soa<double>(aos, n, h, h + n, h + 2 * n);
    }
    const size_t bytes = (size_t)n * c->rsize;
    HIP_TRY(hipMemcpy(d0, buf.data(), bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(d1, buf.data() + bytes, bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(d2, buf.data() + 2 * bytes, bytes, hipMemcpyHostToDevice));
    return QK_OK;
}

// widen n numbers of rsize bytes to FP64
void widen(size_t rsize, const void *src, int64_t n, double *dst)
{
    if (rsize == 8) {
        std::memcpy(dst, src, (size_t)n * sizeof(double));
        return;
    }
    const float *f = (const float *)src;
    for (int64_t m = 0; m < n; ++m) dst[m] = f[m];
}

// up to four fields (three component arrays each) into interleaved FP64 arrays
int download_fields(qk_ctx *c, int nf, double *const *aos, void *const (*comp)[3], size_t rsize)
{
    const int64_t n = c->g.ncell;
    const size_t node = 3 * rsize;
    const bool shared = c->drain.shares((size_t)nf * n * node, Drain::kFields);
    const int64_t per = (int64_t)(Drain::slot_bytes(shared) / node);   // nodes per block
    const int64_t nb = (n + per - 1) / per;                            // blocks per field
    auto launch = [&](int64_t b, void *slot, const ReadDone &done) {
        void *const *s = comp[b / nb];
        const int64_t first = b % nb * per;
        const int m = (int)std::min(per, n - first);
        return rsize == 4 ? launch_pack_fields<float>(c->stream, (const float *)s[0], (const float *)s[1],
                                                         (const float *)s[2], first, m, (float *)slot, done)
                             : launch_pack_fields<double>(c->stream, (const double *)s[0], (const double *)s[1],
                                                          (const double *)s[2], first, m, (double *)slot, done);
    };
    auto take = [&](int64_t b, const void *slot) {
        const int64_t first = b % nb * per;
        widen(rsize, slot, 3 * std::min(per, n - first), aos[b / nb] + 3 * first);
    };
    HIP_TRY(c->drain.run(c->p.device, c->stream, shared, nf * nb, launch, take));
    return QK_OK;
}

// the live count of each run of slots of species b, scanned, in d_live:
// entry r is the row of run r's first live slot; `live` the total
int scan_live(qk_ctx *c, const SpeciesBuf &b, int64_t &live, std::vector<int> *offs)
{
    const int64_t runs = (b.n + kLiveRun - 1) / kLiveRun;
    const size_t row = ((size_t)runs + 64) & ~(size_t)63;   // counts, then offsets, then scan scratch
    if (c->live_cap < (size_t)runs) {
        if (c->d_live) HIP_TRY(hipFree(c->d_live));
        c->d_live = nullptr;
        c->live_cap = 0;
        HIP_TRY(hipMalloc(&c->d_live, (2 * row + scan_scratch_ints(row)) * sizeof(int)));
        c->live_cap = (size_t)runs;
    }
    int *counts = c->d_live + row;
    HIP_TRY(launch_count_live(c->stream, b.buf[b.cur].cell, b.n, counts));
    HIP_TRY(launch_fill_int(c->stream, counts + runs, 1, 0));
    HIP_TRY(launch_exclusive_scan(c->stream, counts, c->d_live, (int)runs, c->d_live + 2 * row));
    int total = 0;
    if (offs) {
        offs->resize((size_t)runs + 1);
        HIP_TRY(hipMemcpyAsync(offs->data(), c->d_live, ((size_t)runs + 1) * sizeof(int), hipMemcpyDeviceToHost, c->stream));
    } else {
        HIP_TRY(hipMemcpyAsync(&total, c->d_live + runs, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    live = offs ? offs->back() : total;
    return QK_OK;
}

// the records of species b's live slots, in slot order, as qk_get_particles
// gives them
template <typename real>
int download_particles(qk_ctx *c, const SpeciesBuf &b, const std::vector<int> &offs, double *rec, int32_t *ids)
{
    const SoA &src = b.buf[b.cur];
    const Species<real> v = view<real>(src);
    const int nreal = src.a[7] ? 8 : 7;
    const bool has_id = src.id != nullptr;
    const size_t row = 4 + (size_t)nreal * sizeof(real) + (has_id ? 4 : 0);
    const bool shared = c->drain.shares((size_t)offs.back() * row, Drain::kRecords);
    const int64_t per = (int64_t)(Drain::slot_bytes(shared) / row) / kLiveRun * kLiveRun;   // slots per block
    const int64_t nb = (b.n + per - 1) / per;
    // a slot holds `per` rows: the reals first (aligned), then cells and ids
    auto reals = [&](void *slot) { return (real *)slot; };
    auto cells = [&](void *slot) { return (int *)((char *)slot + (size_t)per * nreal * sizeof(real)); };
    auto launch = [&](int64_t k, void *slot, const ReadDone &done) {
        return launch_pack_live<real>(c->stream, v, k * per, std::min(b.n, (k + 1) * per), c->d_live, (int)per,
                                      cells(slot), reals(slot), cells(slot) + per, done);
    };
    const double cmr = b.cmr;
    const bool photon = b.kind == 1;
    auto take = [&](int64_t k, void *slot) {
        const size_t run0 = (size_t)(k * per / kLiveRun), run1 = std::min((size_t)((k + 1) * per / kLiveRun), offs.size() - 1);
        const int64_t at = offs[run0], m1 = offs[run1] - at;
        const real *x = reals(slot);
        const int *cc = cells(slot), *id = cc + per;
        for (int64_t m = 0; m < m1; ++m) {
            double *w = rec + 10 * (at + m);
            w[0] = cell_i(cc[m]) + (double)x[m];
            w[1] = cell_j(cc[m]) + (double)x[per + m];
            w[2] = cell_k(cc[m]) + (double)x[2 * per + m];
            w[3] = (double)x[3 * per + m];
            w[4] = (double)x[4 * per + m];
            w[5] = (double)x[5 * per + m];
            const double u2 = w[3] * w[3] + w[4] * w[4] + w[5] * w[5];
            w[6] = photon ? std::sqrt(u2) : std::sqrt(1 + u2);
            w[7] = (double)x[6 * per + m];
            w[8] = cmr;
            w[9] = nreal == 8 ? (double)x[7 * per + m] : 0.0;
        }
        if (ids) {
            if (has_id) std::memcpy(ids + at, id, (size_t)m1 * sizeof(int));
            else std::fill(ids + at, ids + at + m1, 0);
        }
    };
    HIP_TRY(c->drain.run(c->p.device, c->stream, shared, nb, launch, take));
    return QK_OK;
}

// node charge of species b into rho[3 node + slot]
template <typename real>
hipError_t rho_species(qk_ctx *c, const SpeciesBuf &b, double *rho, int slot)
{
    return launch_compute_rho<real>(c->stream, c->g, view<real>(b.buf[b.cur]), b.n, rho, slot, c->tg, b.chunks, b.nchunks,
                                    b.ishift, b.n_sorted);
}

// n doubles from device memory, a part of a result of `of` (0: all of it)
int download_doubles(qk_ctx *c, double *dst, const double *src, int64_t n, int64_t of)
{
    const bool shared = (size_t)std::max(n, of) * sizeof(double) > Drain::kNumbers;
    const int64_t per = (int64_t)(Drain::slot_bytes(shared) / sizeof(double));
    auto count = [&](int64_t b) { return (size_t)std::min(per, n - b * per); };
    auto launch = [&](int64_t b, void *slot, const ReadDone &done) {
        return launch_copy_out(c->stream, src + b * per, (int)count(b), (double *)slot, done);
    };
    auto take = [&](int64_t b, const void *slot) { std::memcpy(dst + b * per, slot, count(b) * sizeof(double)); };
    HIP_TRY(c->drain.run(c->p.device, c->stream, shared, (n + per - 1) / per, launch, take));
    return QK_OK;
}

}  // namespace

extern "C" {

const char *qk_last_error(void) { return g_err.c_str(); }

int qk_create(const qk_params *params, qk_ctx **out)
{
    if (!params || !out) return fail(QK_ERR_INVALID, "null argument");
    *out = nullptr;
    const qk_params &p = *params;
    if (p.nx < 5 || p.ny < 5 || p.nz < 5) return fail(QK_ERR_INVALID, "grid must be at least 5 cells per axis");
    if (p.nx > 2048 || p.ny > 1024 || p.nz > 1024)
        return fail(QK_ERR_INVALID, "grid exceeds 2048 x 1024 x 1024 (packed cell index)");
    {
        // cell and sort-key indices are 32-bit: the cell count and the tile
        // keys (whole 8x8x8 tiles) must stay below 2^31
        const int64_t ncell = (int64_t)p.nx * p.ny * p.nz;
        const int64_t nkeys = (int64_t)((p.nx + kTx - 1) / kTx) * ((p.ny + kTy - 1) / kTy) *
                              ((p.nz + kTz - 1) / kTz) * kTileCells;
        if (ncell >= ((int64_t)1 << 31) || nkeys >= ((int64_t)1 << 31))
            return fail(QK_ERR_INVALID, "grid too large: cell and tile-key indices must stay below 2^31");
    }
    if (!(p.dx > 0 && p.dy > 0 && p.dz > 0 && p.dt > 0)) return fail(QK_ERR_INVALID, "dx, dy, dz, dt must be > 0");
    if (p.solver < 0 || p.solver > 2) return fail(QK_ERR_INVALID, "unknown solver");
    if (p.pusher < 0 || p.pusher > 1) return fail(QK_ERR_INVALID, "unknown pusher");
    if (p.precision != QK_FP32 && p.precision != QK_FP64) return fail(QK_ERR_INVALID, "unknown precision");
    if (p.deposit != QK_DEPOSIT_TILED && p.deposit != QK_DEPOSIT_GLOBAL) return fail(QK_ERR_INVALID, "unknown deposit");
    if (p.n_ion < 0 || p.n_ion > QK_MAX_ION) return fail(QK_ERR_INVALID, "n_ion out of range");
    if (p.sort_every < 0) return fail(QK_ERR_INVALID, "sort_every must be >= 0");
    if (!(p.sort_fallback >= 0 && p.sort_fallback <= 1)) return fail(QK_ERR_INVALID, "sort_fallback must be in [0, 1]");
    if (p.qed && !(p.e_s > 0)) return fail(QK_ERR_INVALID, "QED needs e_s > 0");
    if (p.merging < 0 || p.merging > 2) return fail(QK_ERR_INVALID, "merging must be 0, 1 (ti) or 2 (nl)");
    if (p.merging && !(p.crnp > 0)) return fail(QK_ERR_INVALID, "merging needs crnp > 0");
    // the reference's deposit splits a path at no more than one face per axis
    if (p.dt >= p.dx || p.dt >= p.dy || p.dt >= p.dz)
        return fail(QK_ERR_INVALID, "dt must be below dx, dy and dz (one face crossing per axis and step)");

    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev == 0) return fail(QK_ERR_HIP, "no HIP device available");
    if (p.device < 0 || p.device >= ndev || p.device >= kMaxDevices)
        return fail(QK_ERR_INVALID, "device ordinal out of range");
    e = hipSetDevice(p.device);
    if (e != hipSuccess) return fail(QK_ERR_HIP, hipGetErrorString(e));
    if (int rc = resolve_scratch(p.device)) return rc;

    qk_ctx *c = new qk_ctx;
    c->p = p;
    if (c->p.norm_n == 0) c->p.norm_n = 1;
    if (c->p.norm_ef == 0) c->p.norm_ef = 1;
    if (c->p.norm_ep == 0) c->p.norm_ep = 1;
    c->g.nx = p.nx;
    c->g.ny = p.ny;
    c->g.nz = p.nz;
    c->g.sy = p.nz;
    c->g.sx = p.ny * p.nz;
    c->g.ncell = p.nx * p.ny * p.nz;
    c->g.dx = p.dx;
    c->g.dy = p.dy;
    c->g.dz = p.dz;
    c->g.dt = p.dt;
    c->tg.ntx = (p.nx + kTx - 1) / kTx;
    c->tg.nty = (p.ny + kTy - 1) / kTy;
    c->tg.ntz = (p.nz + kTz - 1) / kTz;
    c->tg.ntiles = c->tg.ntx * c->tg.nty * c->tg.ntz;
    c->tg.nkeys = c->tg.ntiles * kTileCells;
    c->rsize = p.precision == QK_FP64 ? 8 : 4;
    // solver coefficients (src/maxwell.cpp:24-33, 238-249)
    for (int a = 0; a < 3; ++a) {
        c->coef.a[a] = 0;
        c->coef.b[a] = 1;
    }
    const double d[3] = {p.dx, p.dy, p.dz};
    if (p.solver == QK_SOLVER_NDFX) {
        const double kappa = 1.25 * (std::sqrt(3.0) - 1) * 0.5 / std::sqrt(3.0);
        for (int a = 0; a < 3; ++a) {
            c->coef.b[a] = 1 - kappa * p.dx * p.dx / (d[a] * d[a]);
            c->coef.a[a] = 0.5 * (1 - c->coef.b[a]);
        }
        c->coef.b[0] = 1 - kappa;
        c->coef.a[0] = 0.5 * (1 - c->coef.b[0]);
    } else if (p.solver == QK_SOLVER_FIVE_POINT) {
        const double PI = 3.141592653589793;
        for (int a = 0; a < 3; ++a) {
            c->coef.a[a] = 0.25 * (1 - d[a] / p.dt * std::sin(0.5 * PI * std::fmin(1.0, p.dt / d[a])));
            c->coef.b[a] = 1 - 2 * c->coef.a[a];
        }
    }
    auto bail = [&](int code) {
        qk_destroy(c);
        return code;
    };
    if ((e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess)
        return bail(fail(QK_ERR_HIP, hipGetErrorString(e)));
    const size_t fbytes = ((size_t)c->g.ncell * c->rsize + 255) & ~(size_t)255;
    if ((e = hipMalloc(&c->fmem, fbytes * 15)) != hipSuccess)
        return bail(fail(QK_ERR_HIP, std::string("field allocation: ") + hipGetErrorString(e)));
    if ((e = hipMemset(c->fmem, 0, fbytes * 15)) != hipSuccess) return bail(fail(QK_ERR_HIP, hipGetErrorString(e)));
    for (int a = 0; a < 15; ++a) c->F[a] = (char *)c->fmem + a * fbytes;
    if ((e = hipMalloc(&c->d_diag, 2 * kDiagRow * sizeof(double))) != hipSuccess)
        return bail(fail(QK_ERR_HIP, hipGetErrorString(e)));
    if (p.qed) {
        if ((e = hipMalloc(&c->d_count, (QK_MAX_SPECIES + 2) * sizeof(int))) != hipSuccess ||
            (e = hipHostMalloc((void **)&c->h_count, (QK_MAX_SPECIES + 1) * sizeof(int))) != hipSuccess ||
            (e = hipHostMalloc((void **)&c->h_qed, 2 * sizeof(QedCounts))) != hipSuccess)
            return bail(fail(QK_ERR_HIP, hipGetErrorString(e)));
        c->h_qed[0].flag = c->h_qed[1].flag = 0;
        std::fill(c->dev_n, c->dev_n + QK_MAX_SPECIES, -1);
        // the species that QED appends to exist from the start
        for (int s : {QK_ELECTRON, QK_POSITRON, QK_PHOTON})
            if (int rc = ensure_species(c, s, 0)) return bail(rc);
    }
    *out = c;
    return QK_OK;
}

int qk_destroy(qk_ctx *c)
{
    if (!c) return QK_OK;
    // release everything even if one call fails; report the first failure
    hipError_t first = hipSuccess;
    auto note = [&](hipError_t e) {
        if (first == hipSuccess && e != hipSuccess) first = e;
    };
    if (c->stream) note(hipStreamSynchronize(c->stream));
    for (auto &b : c->sp) {
        for (auto &k : b.buf)
            if (k.mem) note(hipFree(k.mem));
        if (b.chunks) note(hipFree(b.chunks));
        if (b.tile_start) note(hipFree(b.tile_start));
    }
    int *sb[8] = {c->s_counts, c->s_imm, c->s_offsets, c->s_tile_start, c->s_tile_mult, c->s_chunk_n, c->s_chunk_off,
                  c->s_scratch};
    for (int *p : sb)
        if (p) note(hipFree(p));
    if (c->h_sortinfo) note(hipHostFree(c->h_sortinfo));
    if (c->rows) note(hipFree(c->rows));
    if (c->fmem) note(hipFree(c->fmem));
    if (c->mid) note(hipFree(c->mid));
    if (c->wide) note(hipFree(c->wide));
    if (c->d_diag) note(hipFree(c->d_diag));
    if (c->h_diag) note(hipHostFree(c->h_diag));
    if (c->d_count) note(hipFree(c->d_count));
    if (c->h_count) note(hipHostFree(c->h_count));
    if (c->h_qed) note(hipHostFree(c->h_qed));
    if (c->d_merge) note(hipFree(c->d_merge));
    if (c->h_merge) note(hipHostFree(c->h_merge));
    for (void *m : c->tape.ckpt) note(hipFree(m));
    if (c->tape.seg) note(hipFree(c->tape.seg));
    if (c->tape.fin) note(hipFree(c->tape.fin));
    if (c->tape.lam) note(hipFree(c->tape.lam));
    if (c->tape.lpart) note(hipFree(c->tape.lpart));
    if (c->d_maxw) note(hipFree(c->d_maxw));
    if (c->h_maxw) note(hipHostFree(c->h_maxw));
    if (c->h_fill) note(hipHostFree(c->h_fill));
    if (c->fill_read) note(hipEventDestroy(c->fill_read));
    if (c->d_fill) note(hipFree(c->d_fill));
    if (c->d_live) note(hipFree(c->d_live));
    note(c->drain.release());
    for (auto e : c->ev) note(hipEventDestroy(e));
    if (c->stream) note(hipStreamDestroy(c->stream));
    delete c;
    if (first != hipSuccess) return fail(QK_ERR_HIP, std::string("qk_destroy: ") + hipGetErrorString(first));
    return QK_OK;
}

int qk_set_fields(qk_ctx *c, const double *E, const double *B)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    c->tape.dirty = c->tape.active;
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (E) QK_TRY(upload3(c, E, c->F[0], c->F[1], c->F[2]));
    if (B) QK_TRY(upload3(c, B, c->F[3], c->F[4], c->F[5]));
    return QK_OK;
}

int qk_get_fields(qk_ctx *c, double *E, double *B, double *J, double *Be)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    const int w = c->have_step ? (c->jcur ^ 1) : c->jcur;   // current buffer of the last step
    double *const out[4] = {E, B, J, Be};
    const int at[4] = {0, 3, 9 + 3 * w, 6};
    double *aos[4];
    void *comp[4][3];
    int nf = 0;
    for (int k = 0; k < 4; ++k) {
        if (!out[k]) continue;
        aos[nf] = out[k];
        for (int a = 0; a < 3; ++a) comp[nf][a] = c->F[at[k] + a];
        ++nf;
    }
    const DeviceScope on(c->p.device);
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (nf > 0) QK_TRY(download_fields(c, nf, aos, comp, c->rsize));
    return QK_OK;
}

int qk_add_particles(qk_ctx *c, int s, int64_t n, const double *x, const double *y, const double *z, const double *ux,
                     const double *uy, const double *uz, const double *q, const int32_t *ids, int64_t *kept)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    if (!species_valid(c, s)) return fail(QK_ERR_INVALID, "invalid species");
    if (n < 0 || (n > 0 && (!x || !y || !z || !ux || !uy || !uz || !q))) return fail(QK_ERR_INVALID, "bad particle arrays");
    c->tape.dirty = c->tape.active;
    // place(): keep particles in is_inside cells (src/plist.cpp:22-31)
    std::vector<int64_t> keep;
    keep.reserve((size_t)n);
    for (int64_t m = 0; m < n; ++m) {
        if (!(x[m] >= 0 && y[m] >= 0 && z[m] >= 0 && x[m] < c->p.nx && y[m] < c->p.ny && z[m] < c->p.nz)) continue;
        const int i = (int)x[m], j = (int)y[m], k = (int)z[m];
        if (i > 0 && i < c->p.nx - 2 && j > 0 && j < c->p.ny - 2 && k > 0 && k < c->p.nz - 2) keep.push_back(m);
    }
    const int64_t nk = (int64_t)keep.size();
    QK_TRY(ensure_species(c, s, nk));
    SpeciesBuf &b = c->sp[s];
    SoA &dst = b.buf[b.cur];
    const size_t r = c->rsize;
    std::vector<int> cell((size_t)nk), id((size_t)nk);
    std::vector<char> buf((size_t)nk * r * 8);
    for (int64_t t = 0; t < nk; ++t) {
        const int64_t m = keep[(size_t)t];
        const int i = (int)x[m], j = (int)y[m], k = (int)z[m];
        cell[(size_t)t] = pack_cell(i, j, k);
        id[(size_t)t] = ids ? ids[m] : 0;
        const double v[8] = {x[m] - i, y[m] - j, z[m] - k, ux[m], uy[m], uz[m], q[m], 0.0};
        for (int a = 0; a < 8; ++a) {
            if (r == 4) {
                float fv = (float)v[a];
                if (a < 3 && fv >= 1.0f) fv = 0.99999994f;   // offsets stay below 1
                ((float *)buf.data())[(size_t)a * nk + t] = fv;
            } else {
                ((double *)buf.data())[(size_t)a * nk + t] = v[a];
            }
        }
    }
    if (nk > 0) {
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(dst.cell + b.n, cell.data(), (size_t)nk * 4, hipMemcpyHostToDevice));
        for (int a = 0; a < 8; ++a)
            if (dst.a[a])
                HIP_TRY(hipMemcpy((char *)dst.a[a] + (size_t)b.n * r, buf.data() + (size_t)a * nk * r, (size_t)nk * r,
                                  hipMemcpyHostToDevice));
        if (dst.id) HIP_TRY(hipMemcpy(dst.id + b.n, id.data(), (size_t)nk * 4, hipMemcpyHostToDevice));
        b.n += nk;
    }
    if (kept) *kept = nk;
    return QK_OK;
}

int qk_load_uniform_plasma(qk_ctx *c, int s, int ppc, double density, double sigma, uint64_t seed, int ilo, int ihi,
                           int64_t *added)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    c->tape.dirty = c->tape.active;
    if (!species_valid(c, s) || s == QK_PHOTON) return fail(QK_ERR_INVALID, "invalid species for a plasma");
    if (ppc <= 0) return fail(QK_ERR_INVALID, "ppc must be positive");
    if (ilo < 1) ilo = 1;
    if (ihi > c->p.nx - 2) ihi = c->p.nx - 2;
    const int64_t total = ihi > ilo ? (int64_t)(ihi - ilo) * (c->p.ny - 3) * (c->p.nz - 3) * ppc : 0;
    QK_TRY(ensure_species(c, s, total));
    SpeciesBuf &b = c->sp[s];
    const double q = (b.cmr < 0 ? -1.0 : 1.0) * density / ppc;   // init.cpp:413-414
    if (total > 0) {
        if (c->rsize == 4)
            HIP_TRY(launch_load_uniform<float>(c->stream, c->g, view<float>(b.buf[b.cur]), b.n, ppc, q, sigma, seed, ilo, ihi));
        else
            HIP_TRY(launch_load_uniform<double>(c->stream, c->g, view<double>(b.buf[b.cur]), b.n, ppc, q, sigma, seed, ilo, ihi));
        HIP_TRY(hipStreamSynchronize(c->stream));
        b.n += total;
    }
    if (added) *added = total;
    return QK_OK;
}

int qk_init_laser_cos(qk_ctx *c, const double L[16])
{
    if (!c || !L) return fail(QK_ERR_INVALID, "null argument");
    c->tape.dirty = c->tape.active;
    hipError_t e = c->rsize == 4 ? launch_laser_cos<float>(c->stream, c->g, fields_of<float>(c), L)
                                 : launch_laser_cos<double>(c->stream, c->g, fields_of<double>(c), L);
    if (e == hipErrorInvalidValue) return fail(QK_ERR_INVALID, "laser direction undefined (x1 = y0 = z0 = 0)");
    HIP_TRY(e);
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

int qk_init_boundaries(qk_ctx *c)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    c->tape.dirty = c->tape.active;
    if (c->rsize == 4) {
        HIP_TRY(launch_init_boundaries<float>(c->stream, c->p.solver, c->g, fields_of<float>(c)));
        HIP_TRY(launch_interpolate_be<float>(c->stream, c->g, fields_of<float>(c)));
    } else {
        HIP_TRY(launch_init_boundaries<double>(c->stream, c->p.solver, c->g, fields_of<double>(c)));
        HIP_TRY(launch_interpolate_be<double>(c->stream, c->g, fields_of<double>(c)));
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

int qk_step(qk_ctx *c, int nsteps, qk_diag *diag)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    if (nsteps < 0) return fail(QK_ERR_INVALID, "negative step count");
    if (nsteps == 0) return QK_OK;
    return c->rsize == 4 ? step_impl<float>(c, nsteps, diag) : step_impl<double>(c, nsteps, diag);
}

int qk_sync(qk_ctx *c)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

int qk_particle_count(qk_ctx *c, int s, int64_t *n)
{
    if (!c || !n) return fail(QK_ERR_INVALID, "null argument");
    if (!species_valid(c, s)) return fail(QK_ERR_INVALID, "invalid species");
    SpeciesBuf &b = c->sp[s];
    *n = 0;
    if (b.n == 0) return QK_OK;
    const DeviceScope on(c->p.device);
    QK_TRY(scan_live(c, b, *n, nullptr));
    return QK_OK;
}

int qk_get_rows_by_id(qk_ctx *c, int s, int64_t n, double *rows, int32_t *live)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    if (!species_valid(c, s)) return fail(QK_ERR_INVALID, "invalid species");
    if (n < 0 || (n > 0 && (!rows || !live))) return fail(QK_ERR_INVALID, "bad output buffers");
    if (!c->p.track_ids) return fail(QK_ERR_STATE, "rows by id need track_ids");
    if (n == 0) return QK_OK;
    const DeviceScope on(c->p.device);
    const SpeciesBuf &b = c->sp[s];
    const int64_t per = std::min(n, (int64_t)(kRowBytes / (kRow + sizeof(int))));
    QK_TRY(ensure_rows(c, (size_t)per * (kRow + sizeof(int)) + sizeof(int)));
    int *const l = (int *)(c->rows + 7 * per);
    int bad = 0;
    for (int64_t r = 0; r < n; r += per) {
        const int64_t k = std::min(per, n - r);
        HIP_TRY(launch_zero(c->stream, c->rows, (size_t)per * 7));
        HIP_TRY(launch_fill_int(c->stream, l, (size_t)per + 1, 0));
        if (b.n > 0)
            HIP_TRY(c->rsize == 4 ? launch_state_rows<float>(c->stream, view<float>(b.buf[b.cur]), b.n, n, r, r + k,
                                                             c->rows, l, l + per)
                                  : launch_state_rows<double>(c->stream, view<double>(b.buf[b.cur]), b.n, n, r, r + k,
                                                              c->rows, l, l + per));
        HIP_TRY(hipMemcpyAsync(live + r, l, (size_t)k * sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipMemcpyAsync(&bad, l + per, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        QK_TRY(download_doubles(c, rows + 7 * r, c->rows, 7 * k, 7 * n));
        if (bad) return fail(QK_ERR_INVALID, "rows by id: an id lies outside 0 .. n - 1, or two particles share it");
    }
    return QK_OK;
}

int qk_get_particles(qk_ctx *c, int s, int64_t cap, double *rec, int32_t *ids, int64_t *n_out)
{
    if (!c || !n_out) return fail(QK_ERR_INVALID, "null argument");
    if (!species_valid(c, s)) return fail(QK_ERR_INVALID, "invalid species");
    SpeciesBuf &b = c->sp[s];
    *n_out = 0;
    if (b.n == 0) return QK_OK;
    if (!rec) return fail(QK_ERR_INVALID, "null output buffer");
    const DeviceScope on(c->p.device);
    std::vector<int> offs;
    int64_t live = 0;
    QK_TRY(scan_live(c, b, live, &offs));
    if (live > cap) return fail(QK_ERR_CAPACITY, "output buffer too small");
    if (live > 0)
        QK_TRY(c->rsize == 4 ? download_particles<float>(c, b, offs, rec, ids)
                             : download_particles<double>(c, b, offs, rec, ids));
    *n_out = live;
    return QK_OK;
}

int qk_compute_rho(qk_ctx *c, double *rho)
{
    if (!c || !rho) return fail(QK_ERR_INVALID, "null argument");
    const DeviceScope on(c->p.device);
    const size_t bytes = (size_t)c->g.ncell * 3 * sizeof(double);
    double *d = nullptr;
    HIP_TRY(hipMalloc(&d, bytes));
    hipError_t e = launch_zero(c->stream, d, (size_t)c->g.ncell * 3);
    const int slots[3] = {QK_ELECTRON, QK_POSITRON, QK_PHOTON};
    for (int t = 0; t < 3 && e == hipSuccess; ++t) {
        SpeciesBuf &b = c->sp[slots[t]];
        if (!b.active || b.n == 0) continue;
        e = c->rsize == 4 ? rho_species<float>(c, b, d, t)
                          : rho_species<double>(c, b, d, t);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    const int rc = e == hipSuccess ? download_doubles(c, rho, d, 3 * (int64_t)c->g.ncell) : QK_OK;
    const hipError_t ef = hipFree(d);
    HIP_TRY(e);
    QK_TRY(rc);
    HIP_TRY(ef);
    return QK_OK;
}

// qk_compute_rho without allocating: the node charges accumulate in this
// device's `scratch` (resolved by qk_create), cleared by a fill kernel first.
// Calls that overlap on one GPU (two contexts on two threads) share it and race.
int qk_compute_rho_noalloc(qk_ctx *c, double *rho)
{
    if (!c || !rho) return fail(QK_ERR_INVALID, "null argument");
    if ((int64_t)c->g.ncell > kNoallocCells)
        return fail(QK_ERR_CAPACITY, "qk_compute_rho_noalloc: the grid has " + std::to_string(c->g.ncell) +
                                         " cells, above its limit of " + std::to_string(kNoallocCells) +
                                         " (qk_compute_rho has none)");
    double *d = scratch_ptr(c->p.device);
    if (!d) return fail(QK_ERR_STATE, "qk_compute_rho_noalloc: no scratch resolved for this device");
    const size_t n = (size_t)c->g.ncell * 3;
    HIP_TRY(launch_zero(c->stream, d, n));
    const int slots[3] = {QK_ELECTRON, QK_POSITRON, QK_PHOTON};
    for (int t = 0; t < 3; ++t) {
        SpeciesBuf &b = c->sp[slots[t]];
        if (!b.active || b.n == 0) continue;
        HIP_TRY(c->rsize == 4 ? rho_species<float>(c, b, d, t)
                              : rho_species<double>(c, b, d, t));
    }
    HIP_TRY(hipMemcpyAsync(rho, d, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

int qk_add_laser_source(qk_ctx *c, const double L[16], int side, int plane)
{
    if (!c || !L) return fail(QK_ERR_INVALID, "null argument");
    const int nx = c->p.nx;
    if (side == 0 ? !(plane >= 2 && plane <= nx - 6) : !(side == 1 && plane >= 6 && plane <= nx - 2))
        return fail(QK_ERR_INVALID, "laser source: side 0 needs 2 <= plane <= nx - 6, side 1 6 <= plane <= nx - 2");
    InjSide &sd = c->inj[side];
    if (sd.nsrc == kMaxSources) return fail(QK_ERR_CAPACITY, "at most 4 laser sources per side");
    if (sd.nsrc > 0 && sd.plane != plane) return fail(QK_ERR_INVALID, "the sources of one side share one plane");
    LaserFrame F;
    if (!laser_frame(c->g, L, F)) return fail(QK_ERR_INVALID, "laser source: x1, y0, z0 all zero");
    sd.plane = plane;
    sd.src[sd.nsrc] = F;
    sd.t0[sd.nsrc] = c->step_index;
    sd.shifts0[sd.nsrc] = c->window_shifts;
    ++sd.nsrc;
    return QK_OK;
}

int qk_pmerging(qk_ctx *c, int mode, const double *ppd)
{
    if (!c || !ppd) return fail(QK_ERR_INVALID, "null argument");
    c->tape.dirty = c->tape.active;
    if (mode != 1 && mode != 2) return fail(QK_ERR_INVALID, "merging mode must be 1 (ti) or 2 (nl)");
    for (int s = 0; s < QK_ION0 + c->p.n_ion; ++s)
        if (!(ppd[s] >= 0 && ppd[s] < 1)) return fail(QK_ERR_INVALID, "ppd must lie in [0, 1)");
    return c->rsize == 4 ? merge_impl<float>(c, mode, ppd) : merge_impl<double>(c, mode, ppd);
}

int qk_moving_window(qk_ctx *c)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    c->tape.dirty = c->tape.active;
    if (c->rsize == 4) HIP_TRY(launch_shift_fields<float>(c->stream, c->g, fields_of<float>(c)));
    else HIP_TRY(launch_shift_fields<double>(c->stream, c->g, fields_of<double>(c)));
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        SpeciesBuf &b = c->sp[s];
        if (!b.active) continue;
        HIP_TRY(launch_shift_particles(c->stream, b.buf[b.cur].cell, b.n));
        ++b.ishift;   // the tiles of the last sort moved with their particles
    }
    ++c->window_shifts;   // grid plane i now lies at (i + shifts) dx in the frame of the laser sources
    return QK_OK;
}

int qk_max_w(qk_ctx *c, int ilo, int ihi, double *max_w)
{
    if (!c || !max_w) return fail(QK_ERR_INVALID, "null argument");
    if (ilo < 0 || ihi > c->p.nx) return fail(QK_ERR_INVALID, "planes outside [0, nx)");
    if (ilo >= ihi) {
        *max_w = 0;
        return QK_OK;
    }
    if (!c->d_maxw) {
        HIP_TRY(hipMalloc(&c->d_maxw, 2 * sizeof(unsigned long long)));
        HIP_TRY(launch_fill_int(c->stream, (int *)c->d_maxw, 4, 0));
    }
    if (!c->h_maxw) {
        HIP_TRY(hipHostMalloc((void **)&c->h_maxw, 2 * sizeof(unsigned long long)));
        *(unsigned *)(c->h_maxw + 1) = 0;
    }
    const ReadDone done{(unsigned *)(c->d_maxw + 1), (unsigned *)(c->h_maxw + 1), ++c->maxw_seq};
    if (c->rsize == 4)
        HIP_TRY(launch_max_w<float>(c->stream, c->g, fields_of<float>(c), ilo, ihi, c->d_maxw, c->h_maxw, done));
    else
        HIP_TRY(launch_max_w<double>(c->stream, c->g, fields_of<double>(c), ilo, ihi, c->d_maxw, c->h_maxw, done));
    HIP_TRY(wait_flag(c->stream, done.flag, done.seq));
    std::memcpy(max_w, c->h_maxw, sizeof(double));
    return QK_OK;
}

int qk_fill_cells(qk_ctx *c, int s, int64_t ncells, const int32_t *cells, const double *density,
                  const int32_t npic[3], double ux0, int32_t first_id, int64_t *added)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    c->tape.dirty = c->tape.active;
    if (!species_valid(c, s)) return fail(QK_ERR_INVALID, "invalid species");
    if (ncells < 0 || (ncells > 0 && (!cells || !density)) || !npic) return fail(QK_ERR_INVALID, "bad cell list");
    if (npic[0] <= 0 || npic[1] <= 0 || npic[2] <= 0 || (int64_t)npic[0] * npic[1] * npic[2] > 4096)
        return fail(QK_ERR_INVALID, "npic must be positive with at most 4096 particles per cell");
    if (added) *added = 0;
    // place() keeps the cells inside is_inside (src/plist.cpp:22-31); the ids
    // of a listed cell are fixed by its index in the list
    const int npt = npic[0] * npic[1] * npic[2];
    std::vector<int> kc, kid;
    std::vector<double> kd;
    kc.reserve(3 * (size_t)ncells);
    kid.reserve((size_t)ncells);
    kd.reserve((size_t)ncells);
    for (int64_t m = 0; m < ncells; ++m) {
        const int i = cells[3 * m], j = cells[3 * m + 1], k = cells[3 * m + 2];
        if (!(i > 0 && i < c->p.nx - 2 && j > 0 && j < c->p.ny - 2 && k > 0 && k < c->p.nz - 2)) continue;
        kc.insert(kc.end(), {i, j, k});
        kd.push_back(density[m]);
        kid.push_back(first_id + (int32_t)(m * npt));
    }
    const int64_t nk = (int64_t)kd.size();
    if (nk == 0) return QK_OK;
    const int64_t total = nk * npt;
    QK_TRY(ensure_species(c, s, total));
    const size_t need = (size_t)nk * (3 * sizeof(int) + sizeof(double) + sizeof(int));
    if (need > c->fill_cap) {
        HIP_TRY(hipStreamSynchronize(c->stream));
        if (c->d_fill) HIP_TRY(hipFree(c->d_fill));
        c->d_fill = nullptr;
        c->fill_cap = 0;
        HIP_TRY(hipMalloc(&c->d_fill, need));
        c->fill_cap = need;
    }
    double *dd = (double *)c->d_fill;
    int *dc = (int *)(dd + nk), *di = dc + 3 * nk;
    auto lay_out = [&](void *at) {   // densities, cells, ids
        char *w = (char *)at;
        std::memcpy(w, kd.data(), (size_t)nk * sizeof(double));
        std::memcpy(w += (size_t)nk * sizeof(double), kc.data(), (size_t)nk * 3 * sizeof(int));
        std::memcpy(w + (size_t)nk * 3 * sizeof(int), kid.data(), (size_t)nk * sizeof(int));
    };
    // A list of up to kFillPinned bytes goes through a pinned buffer in one
    // copy, and the call returns with the work enqueued; the buffer is
    // written again only after that copy (fill_read).  Three copies from
    // pageable memory, each waited for, and a wait before and after them took
    // 71 us per call at 64x32x32, now 15 us.
    constexpr size_t kFillPinned = (size_t)512 << 10;
    const bool pinned = need <= kFillPinned;
    std::vector<char> pageable;
    if (pinned) {
        if (!c->h_fill) HIP_TRY(hipHostMalloc(&c->h_fill, kFillPinned));
        if (!c->fill_read) HIP_TRY(hipEventCreateWithFlags(&c->fill_read, hipEventDisableTiming));
        HIP_TRY(hipEventSynchronize(c->fill_read));
        lay_out(c->h_fill);
        HIP_TRY(hipMemcpyAsync(dd, c->h_fill, need, hipMemcpyHostToDevice, c->stream));
        HIP_TRY(hipEventRecord(c->fill_read, c->stream));
    } else {
        pageable.resize(need);
        lay_out(pageable.data());
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(dd, pageable.data(), need, hipMemcpyHostToDevice));
    }
    SpeciesBuf &b = c->sp[s];
    const double sign = b.cmr < 0 ? -1.0 : 1.0;
    if (c->rsize == 4)
        HIP_TRY(launch_fill_cells<float>(c->stream, view<float>(b.buf[b.cur]), b.n, nk, dc, dd, di, npic, sign, ux0));
    else
        HIP_TRY(launch_fill_cells<double>(c->stream, view<double>(b.buf[b.cur]), b.n, nk, dc, dd, di, npic, sign, ux0));
    if (!pinned) HIP_TRY(hipStreamSynchronize(c->stream));
    b.n += total;
    if (added) *added = total;
    return QK_OK;
}

int qk_tape_begin(qk_ctx *c, int every)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    if (every <= 0) return fail(QK_ERR_INVALID, "checkpoint interval must be positive");
    const qk_params &p = c->p;
    if (p.qed || p.merging || p.sort_every != 0 || p.sort_fallback != 0)
        return fail(QK_ERR_INVALID, "the adjoint needs qed = 0, merging = 0, sort_every = 0, sort_fallback = 0");
    if (c->sp[QK_PHOTON].active && c->sp[QK_PHOTON].n > 0) return fail(QK_ERR_INVALID, "the adjoint covers charged species only");
    // With the tiled deposit the particles are sorted into tiles once, here;
    // no later sort runs (sort_every = 0, nothing is appended), so every
    // particle keeps its slot from snapshot to snapshot.  The tiles' windows
    // then age, and particles that leave them go through the kernel's global
    // fallback.
    if (p.deposit == QK_DEPOSIT_TILED)
        for (int s = 0; s < QK_MAX_SPECIES; ++s)
            if (c->sp[s].active && c->sp[s].n > 0 && c->sp[s].kind == 0)
                QK_TRY(c->rsize == 4 ? sort_species<float>(c, s) : sort_species<double>(c, s));
    tape_free(c);
    Tape &t = c->tape;
    t.every = every;
    t.field_bytes = (((size_t)c->g.ncell * c->rsize + 255) & ~(size_t)255) * 15;
    t.bytes = t.field_bytes;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        t.n[s] = c->sp[s].active ? c->sp[s].n : 0;
        t.bytes += species_state_bytes(c, t.n[s]);
    }
    t.active = true;
    QK_TRY(tape_snapshot(c));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return QK_OK;
}

int qk_tangent_begin(qk_ctx *c, const double *dE, const double *dB, const double *const *dpart)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    Tape &t = c->tape;
    if (!t.active || t.steps != 0) return fail(QK_ERR_STATE, "qk_tangent_begin goes right after qk_tape_begin");
    const int64_t nc = c->g.ncell;
    int64_t np_total = 0;
    for (int s = 0; s < QK_MAX_SPECIES; ++s) np_total += t.n[s];
    if (!t.tfield) HIP_TRY(hipMalloc(&t.tfield, (size_t)nc * 15 * sizeof(double)));
    if (!t.tpart && np_total > 0) HIP_TRY(hipMalloc(&t.tpart, (size_t)np_total * 7 * sizeof(double)));
    // seeds: fields AoS -> SoA (then the boundary zeroing and interpolate_be
    // the set-up applied to the fields), records AoS (x y z ux uy uz q) -> SoA
    {
        std::vector<double> h((size_t)nc * 15, 0.0);
        for (int64_t m = 0; m < nc; ++m)
            for (int a = 0; a < 3; ++a) {
                if (dE) h[(size_t)a * nc + m] = dE[3 * m + a];
                if (dB) h[(size_t)(3 + a) * nc + m] = dB[3 * m + a];
            }
        HIP_TRY(hipMemcpy(t.tfield, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
        for (int s = 0; s < QK_MAX_SPECIES; ++s) {
            const int64_t n = t.n[s];
            if (n == 0) continue;
            std::vector<double> hp((size_t)n * 7, 0.0);
            if (dpart && dpart[s])
                for (int64_t p = 0; p < n; ++p)
                    for (int a = 0; a < 7; ++a) hp[(size_t)a * n + p] = dpart[s][7 * p + a];
            double *tr[7];
            tangent_records(c, s, tr);
            HIP_TRY(hipMemcpy(tr[0], hp.data(), hp.size() * sizeof(double), hipMemcpyHostToDevice));
        }
    }
    const Fields<double> tf = tangent_fields(c);
    HIP_TRY(launch_init_boundaries<double>(c->stream, c->p.solver, c->g, tf));
    HIP_TRY(launch_interpolate_be<double>(c->stream, c->g, tf));
    HIP_TRY(hipStreamSynchronize(c->stream));
    t.tjcur = 0;
    t.tangent = true;
    return QK_OK;
}

int qk_tangent_get(qk_ctx *c, double *dE, double *dB, double *const *dpart)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    Tape &t = c->tape;
    if (!t.tangent) return fail(QK_ERR_STATE, "no tangent: call qk_tangent_begin after qk_tape_begin");
    HIP_TRY(hipStreamSynchronize(c->stream));
    const int64_t nc = c->g.ncell;
    std::vector<double> h((size_t)nc * 6);
    HIP_TRY(hipMemcpy(h.data(), t.tfield, h.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int64_t m = 0; m < nc; ++m)
        for (int a = 0; a < 3; ++a) {
            if (dE) dE[3 * m + a] = h[(size_t)a * nc + m];
            if (dB) dB[3 * m + a] = h[(size_t)(3 + a) * nc + m];
        }
    for (int s = 0; s < QK_MAX_SPECIES; ++s) {
        const int64_t n = t.n[s];
        if (n == 0 || !dpart || !dpart[s]) continue;
        std::vector<double> hp((size_t)n * 7);
        double *tr[7];
        tangent_records(c, s, tr);
        HIP_TRY(hipMemcpy(hp.data(), tr[0], hp.size() * sizeof(double), hipMemcpyDeviceToHost));
        for (int64_t p = 0; p < n; ++p)
            for (int a = 0; a < 7; ++a) dpart[s][7 * p + a] = hp[(size_t)a * n + p];
    }
    return QK_OK;
}

static int adjoint_call(qk_ctx *c, const double *lam_E, const double *lam_B, const double *const *lam_part, double *grad_E,
                        double *grad_B, double *const *grad_part, bool by_id)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    if (!c->tape.active) return fail(QK_ERR_STATE, "no tape: call qk_tape_begin before the steps");
    if (c->tape.dirty) return fail(QK_ERR_STATE, "fields or particles changed outside qk_step since qk_tape_begin");
    return c->rsize == 4 ? adjoint_impl<float>(c, lam_E, lam_B, lam_part, grad_E, grad_B, grad_part, by_id)
                         : adjoint_impl<double>(c, lam_E, lam_B, lam_part, grad_E, grad_B, grad_part, by_id);
}

int qk_adjoint(qk_ctx *c, const double *lam_E, const double *lam_B, const double *const *lam_part, double *grad_E,
               double *grad_B, double *const *grad_part)
{
    return adjoint_call(c, lam_E, lam_B, lam_part, grad_E, grad_B, grad_part, false);
}

int qk_adjoint_by_id(qk_ctx *c, const double *lam_E, const double *lam_B, const double *const *lam_part, double *grad_E,
                     double *grad_B, double *const *grad_part)
{
    return adjoint_call(c, lam_E, lam_B, lam_part, grad_E, grad_B, grad_part, true);
}

int qk_last_timing(qk_ctx *c, double *ms_total, double *ms_particles, double *ms_fields)
{
    if (!c) return fail(QK_ERR_INVALID, "null context");
    if (ms_total) *ms_total = c->ms_total;
    if (ms_particles) *ms_particles = c->ms_part;
    if (ms_fields) *ms_fields = c->ms_field;
    return QK_OK;
}

int qk_last_fallback(qk_ctx *c, double *fraction)
{
    if (!c || !fraction) return fail(QK_ERR_INVALID, "null argument");
    *fraction = c->fallback_frac;
    return QK_OK;
}

int qk_get_stream(qk_ctx *c, void **stream)
{
    if (!c || !stream) return fail(QK_ERR_INVALID, "null argument");
    *stream = (void *)c->stream;
    return QK_OK;
}

}  // extern "C"
