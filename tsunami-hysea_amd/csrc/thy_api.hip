// thy_api.hip -- C-ABI of libthysea.so (declared in include/thysea.h).
//
// Host side of the MI355X time-stepping library: device memory layout, launch
// dispatch, graph-captured step batches and the driver loop with the semantics of
// the reference's shallowWater (src/GPU/ShallowWater.cu:182-500).
//
// Device layout (structure of arrays, row pitch a multiple of 64 elements):
//   e[2], qx[2], qy[2]   ping-pong state (eta relative to sea level, discharges)
//   D                    still-water depth (changes only at Okada time)
//   emax, arr            metrics (arr, when arrival times are tracked: eta_ini until a
//                        cell arrives, then its arrival time; see Arrival<T>)
//   row[ny], fy[ny+1]    per-row / per-face-row geometry constants
//   ctrl[3], dtmin       device control blocks and dt minima (3 launch slots of
//                        kDtParts partials, dt_at)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include "../../include/thysea.h"
#include "thy_aux.hpp"
#include "thy_pool.hpp"
#include "thy_sweep.hpp"

using namespace thy;

// the device array behind thy_mass_noalloc's partial sums (see kScratchPartials)
static __device__ __align__(256) double scratch[1024];

// Work lists of a step, on the device: deep-water strips, and the items (one per
// workgroup: four strips, or a general tile; item_origin)
struct WorkLists {
    int2 *deep = nullptr, *items = nullptr;
    int n_deep = 0, n_items = 0, deep_cap = 0, items_cap = 0;
    std::vector<int2> tile_h;    // the general tiles, costliest first, and their costs
    std::vector<int> tcost_h;
};

struct thy_ctx {
    int nx = 0, ny = 0, pitch = 0;
    int device = -1;    // the device the context lives on
    thy_params prm{};
    int prec = 0;       // 0 float, 1 double
    size_t esz = 4;
    std::vector<double> lon, lat, area, cosphi, ancho, alto;
    void *e[2] = {nullptr, nullptr}, *qx[2] = {nullptr, nullptr}, *qy[2] = {nullptr, nullptr};
    void *D = nullptr, *emax = nullptr, *arr = nullptr;
    void *state = nullptr;   // one allocation holding e, qx, qy (x2), D, emax and arr
    size_t state_bytes = 0;
    void *row = nullptr, *fy = nullptr, *deep_row = nullptr;
    double *area_d = nullptr;
    Ctrl *ctrl = nullptr;
    unsigned int *dtmin = nullptr;
    unsigned int *scratch_u = nullptr;  // [0]: initial dt, [1]: okada max
    double *ftime = nullptr;
    int nf_cap = 0;
    int *gpos = nullptr;
    float *gbuf = nullptr, *gtime = nullptr;
    int ng = 0, gcap = 0;
    double *okada_def = nullptr;
    OkadaRow *okada_row = nullptr;     // per row of the grid
    OkadaPlane *okada_plane = nullptr; // of the fault in hand
    double *mass_partial = nullptr;
    float *outbuf = nullptr;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // two replays in flight: start / end / control-copied events, pinned copies of the
    // control block, the last launch's dt partials and the health flag after each replay
    hipEvent_t rev[2][3] = {{nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr}};
    Ctrl *h_snap = nullptr;
    unsigned int *h_aux = nullptr;     // [2]: health flag
    unsigned int *h_dt = nullptr;      // [2][kDtSlot]: dt partials of one launch slot
    int slot = 0;
    bool back = false;  // the next launch takes the strips in reverse order
    int cur = 0;                 // host mirror of ctrl.cur after a sync
    int tx = 64, ty = 16;
    int chunk_rows = 1;          // tile (strip) rows per XCD chunk of the step kernel's order
    int kernel = 0;              // 0 row sweep (deep-water strips and general tiles), 1 2D tiles, 2 general tiles only
    int srows = 24;              // row sweep: rows per deep-water strip
    int trows = kTileRows;       //   rows per general tile
    int tuned_srows = 0, tuned_trows = 0;  // the heights thy_autotune chose (0: it has not run)
    int tuning = 0;              // launches recorded for timing replays publish no control block
    int ncu = 256;               // compute units of the device
    bool uploaded = false;       // row sweep: the lists describe an uploaded state
    std::vector<int> coastal, cost;  // [s * (ny + 1) + j]: coastal rows, and cost, of segment s before row j
    WorkLists alone, batched;    // the lists of a run alone and of a batch (built when first prepared)
    unsigned int *health = nullptr;    // non-finite flag raised by the step kernels
    // captured sequences of gk steps, one per launch slot a replay starts at
    hipGraphExec_t gexec[3] = {nullptr, nullptr, nullptr};
    int gk = 0;
    double last_ms = 0.0;
    std::vector<float> g_time, g_eta, g_u, g_v;
    int nsamples = 0;
    bool gauges_stale = false;   // the device holds samples not yet copied to g_*
    // host copy of the control block in launch slot `slot`, when the host knows it
    // (written by the host, or collected after a replay); saves a synchronous read
    Ctrl ctrl_h{};
    bool ctrl_h_valid = false;
    // schedule of the current run (kept so that thy_run_more can continue it)
    std::vector<thy_fault> faults;
    std::vector<double> ftimes;
    int crop_flag = 0;
    double crop_value = 0.0, save_interval = -1.0, next_save = INFINITY;
    int K = 24, nsnap = 0;
    thy_snapshot_fn on_snapshot = nullptr;
    thy_okada_fn on_okada = nullptr;
    thy_step_fn on_step = nullptr;
    void *user = nullptr;
    bool run_active = false;
    bool batch_ready = false;    // prepared by thy_batch_prepare, not yet admitted
    thy_run_result prep_res{};   // its run result so far (initial dt)
    double *steplog = nullptr;
    int logcap = 4096;
    int64_t logged = 0;  // iterations already delivered to on_step
    std::string err;
};

namespace {

constexpr int kMassBlocks = 1024;

// Scratch of thy_mass_noalloc: the kMassBlocks workgroup partial sums of the mass kernel
// (8 KiB, whatever the grid size: the mass kernel always runs kMassBlocks workgroups).
// Each device holds its own copy until the process ends.  Its device address is taken
// once per device, with that device current, when thy_create first runs there; host code
// uses only that address (the array's name is a host-side stand-in, not a device address).
constexpr int kScratchPartials = 1024;
static_assert(kMassBlocks <= kScratchPartials, "the mass partials must fit the scratch");
static_assert(sizeof(scratch) == kScratchPartials * sizeof(double), "scratch size");
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
double *g_scratch_ptr[kScratchDevices] = {};

int fail(thy_ctx *c, int code, const std::string &msg) {
    if (c) c->err = msg;
    return code;
}

// captured step sequences hold the dispatch tables, grid sizes and launch slots of the
// time they were recorded
void drop_graphs(thy_ctx *c) {
    for (hipGraphExec_t &g : c->gexec)
        if (g) {
            (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
    c->gk = 0;
}

// A context's copies and fills go through its own stream and are complete on return.
// The null stream would order them against every blocking stream, one that another
// thread is capturing into a graph included, and so invalidate that capture.
hipError_t ctx_copy(thy_ctx *c, void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
    hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, c->stream);
    return e == hipSuccess ? hipStreamSynchronize(c->stream) : e;
}

hipError_t ctx_fill(thy_ctx *c, void *dst, size_t bytes) {
    hipError_t e = hipMemsetAsync(dst, 0, bytes, c->stream);
    return e == hipSuccess ? hipStreamSynchronize(c->stream) : e;
}

// Entry points run with the calling thread's stream-capture mode relaxed.  Their
// allocations and synchronous copies touch only their own context's or batch's
// streams, none of which another thread can be capturing; under the default (global)
// mode the runtime would invalidate any capture in progress on another thread, such as
// a batch's step sequence being recorded while a worker thread sets up the next context.
struct RelaxedCapture {
    hipStreamCaptureMode m = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&m); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&m); }
    RelaxedCapture(const RelaxedCapture &) = delete;
    RelaxedCapture &operator=(const RelaxedCapture &) = delete;
};

#define HIPCHK(call)                                                                   \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess)                                                          \
            return fail(ctx, e_ == hipErrorOutOfMemory ? THY_ERR_DEVICE_MEMORY : THY_ERR_HIP, \
                        std::string(#call) + ": " + hipGetErrorString(e_));            \
    } while (0)

struct TileShape { int tx, ty; };

// tile shapes compiled into the library (the autotuner chooses among these)
template <typename T> bool tile_supported(int tx, int ty);
template <> bool tile_supported<float>(int tx, int ty) {
    return (tx == 64 && ty == 16) || (tx == 64 && ty == 8) || (tx == 32 && ty == 16) || (tx == 128 && ty == 8) ||
           (tx == 64 && ty == 12) || (tx == 32 && ty == 8) || (tx == 32 && ty == 24);
}
template <> bool tile_supported<double>(int tx, int ty) { return (tx == 32 && ty == 8) || (tx == 64 && ty == 4); }

template <typename T>
StepArgs<T> make_args(thy_ctx *c, const bool batch = false) {
    StepArgs<T> a;
    memset(&a, 0, sizeof(a));
    const thy_params &p = c->prm;
    a.nx = c->nx; a.ny = c->ny; a.pitch = c->pitch;
    a.periodic = (std::fabs(p.borde_izq - 2.0) < 2.220446049250313e-16 && std::fabs(p.borde_der - 2.0) < 2.220446049250313e-16) ? 1 : 0;
    if (c->kernel == 0 || c->kernel == 2) {
        const WorkLists &w = batch ? c->batched : c->alone;
        a.items = w.items;
        a.n_items = w.n_items;
        a.deep = w.deep;
    } else {
        a.tiles_x = (c->nx + c->tx - 1) / c->tx;
        a.tiles_y = (c->ny + c->ty - 1) / c->ty;
    }
    a.n_tiles = a.tiles_x * a.tiles_y;
    a.chunk = a.tiles_x * c->chunk_rows;
    a.sp_sup = p.sponge_sup; a.sp_inf = p.sponge_inf; a.sp_izq = p.sponge_izq; a.sp_der = p.sponge_der;
    a.track_arrival = p.track_arrival;
    a.n_gauges = c->ng;
    a.bsup = (T)p.borde_sup; a.binf = (T)p.borde_inf; a.bizq = (T)p.borde_izq; a.bder = (T)p.borde_der;
    a.cfl = (T)p.cfl; a.mf0 = (T)p.mf0; a.vmax = (T)p.vmax;
    // an infinite hpos as a large one: no depth reaches either and the exponentials of its
    // quotients saturate alike, but a quotient without special cases takes finite numbers
    a.hpos = (T)std::max(std::min(p.hpos, 1e30), -1e30);
    // (the same for an eps_h whose fourth power overflows: every cell is dry with either)
    a.eps_h = sizeof(T) == 8 ? (T)std::min(p.eps_h, 1e70) : (T)p.eps_h;
    a.cvis = (T)p.cvis; a.dif_at = (T)p.dif_at; a.sea_level = (T)p.sea_level;
    a.Href = (T)p.H; a.Q_over_H = (T)(p.Q / p.H);
    for (int b = 0; b < 2; b++) {
        a.e[b] = (T *)c->e[b]; a.qx[b] = (T *)c->qx[b]; a.qy[b] = (T *)c->qy[b];
    }
    a.D = (const T *)c->D;
    a.emax = (T *)c->emax;
    a.arr = (T *)c->arr;
    a.block = (const char *)c->state;
    a.block_bytes = (int)std::min(c->state_bytes, (size_t)INT32_MAX);  // kernel 0 only when it fits
    a.row = (const RowGeo<T> *)c->row;
    a.fy = (const FaceGeoY<T> *)c->fy;
    a.deep_row = (const DeepRow<T> *)c->deep_row;
    a.ctrl = c->ctrl;
    a.dtmin = c->dtmin;
    a.ftime = c->ftime;
    a.gpos = c->gpos;
    a.gbuf = c->gbuf;
    a.gtime = c->gtime;
    a.steplog = c->steplog;
    a.logcap = c->logcap;
    a.health = c->health;
    a.no_publish = c->tuning;
    return a;
}

constexpr size_t kCacheBytes = 256u << 20;

template <typename T>
hipError_t launch_step_t(thy_ctx *c, int slot) {
    StepArgs<T> a = make_args<T>(c);
    if (c->kernel == 0 || c->kernel == 2) {
        // Every other step takes the strips in reverse order: where the state is larger than
        // the 256 MB cache behind the L2s, a step then begins with what the last one left there
        // (4000x3000, 432 MB: 127.7 us a step in one order, 122.8 in turn; FP64 2000x2000,
        // 288 MB: 133.7 and 131.8; 2000x2000, 144 MB: no difference).  No result depends on the order.
        const int flip = c->state_bytes > kCacheBytes && c->back ? c->alone.n_deep / (8 * SW_WAVES) : 0;
        c->back = !c->back;
        hipLaunchKernelGGL((k_sweep<T>), dim3(a.n_items), dim3(64 * SW_WAVES), 0, c->stream, a, slot, flip);
        return hipGetLastError();
    }
    const int n_chunks = (a.tiles_y + c->chunk_rows - 1) / c->chunk_rows;
    const dim3 grid(((n_chunks + 7) / 8) * 8 * a.chunk), block(256);
#define THY_TILE(TX_, TY_)                                                                            \
    if (c->tx == TX_ && c->ty == TY_) {                                                              \
        hipLaunchKernelGGL((k_step<T, TX_, TY_>), grid, block, 0, c->stream, a, slot);               \
        return hipGetLastError();                                                                    \
    }
    if constexpr (sizeof(T) == 4) {
        THY_TILE(64, 16)
        THY_TILE(64, 8)
        THY_TILE(32, 16)
        THY_TILE(128, 8)
        THY_TILE(64, 12)
        THY_TILE(32, 8)
        THY_TILE(32, 24)
    } else {
        THY_TILE(32, 8)
        THY_TILE(64, 4)
    }
#undef THY_TILE
    return hipErrorInvalidValue;
}

hipError_t launch_step(thy_ctx *c) {
    c->ctrl_h_valid = false;  // the launch publishes a control block the host has not seen
    hipError_t e = c->prec ? launch_step_t<double>(c, c->slot) : launch_step_t<float>(c, c->slot);
    c->slot = (c->slot + 1) % 3;
    return e;
}

int grid_1d(int64_t n) {
    int64_t b = (n + 255) / 256;
    return (int)std::min<int64_t>(std::max<int64_t>(b, 1), 16384);
}

template <typename T>
void fill_geometry(thy_ctx *c, std::vector<RowGeo<T>> &rows, std::vector<FaceGeoY<T>> &fys) {
    const int ny = c->ny;
    // the 2s numerical-diffusion coefficient as the kernels compute it, in T
    const T cd2s = T(0.5) * (T(1) - (T)c->prm.cvis);
    rows.resize(ny);
    fys.resize(ny + 1);
    for (int j = 0; j < ny; j++) {
        const double A = c->area[j], cs = c->cosphi[j], al = c->alto[j];
        RowGeo<T> r;
        r.A = (T)A;
        r.invA = (T)(1.0 / A);
        // alto * (1/cos) rounded in T, as the device would multiply the two
        r.ilx = (T)al * (T)(1.0 / cs);
        r.valx = (T)((2.0 * (al / cs)) / (A + A));
        r.kdx = cd2s * r.valx * r.ilx;
        r.dxs = (T)c->ancho[j];
        r.dys = (T)al;
        r.kA = T(0.25) * r.A;
        rows[j] = r;
    }
    for (int g = 0; g <= ny; g++) {
        const int r0 = std::min(std::max(g - 1, 0), ny - 1), r1 = std::min(std::max(g, 0), ny - 1);
        FaceGeoY<T> f;
        const double len = c->ancho[g];
        f.len = (T)len;
        f.cos0 = (T)c->cosphi[r0];
        f.cos1 = (T)c->cosphi[r1];
        f.A0 = (T)c->area[r0];
        f.A1 = (T)c->area[r1];
        f.valy = (T)((2.0 * len) / (c->area[r0] + c->area[r1]));
        f.ic0 = (T)(1.0 / c->cosphi[r0]);
        f.ic1 = (T)(1.0 / c->cosphi[r1]);
        // in T arithmetic, each a single rounded operation as on the device
        f.gh = T(0.5) * (T)(f.cos0 + f.cos1);
        f.gd = (T)(f.cos1 - f.cos0);
        f.g1ic0 = (T)(f.cos1 * f.ic0);
        f.k0 = (T)(T(0.25) * f.cos0) * f.A0;
        f.k1 = (T)(T(0.25) * f.cos1) * f.A1;
        f.lc0 = (T)(f.len * f.cos0);
        f.kdy = cd2s * f.valy * f.len;
        f.pad = T(0);
        fys[g] = f;
    }
}

// the row tables on the device
template <typename T>
int upload_geometry(thy_ctx *ctx) {
    std::vector<RowGeo<T>> rows;
    std::vector<FaceGeoY<T>> fys;
    fill_geometry(ctx, rows, fys);
    const int ny = ctx->ny;
    std::vector<DeepRow<T>> deep(ny + 1);
    for (int r = 0; r <= ny; r++) {
        const RowGeo<T> &r0 = rows[std::min(r, ny - 1)], &r1 = rows[std::max(r - 1, 0)], &r2 = rows[std::max(r - 2, 0)];
        const FaceGeoY<T> &f0 = fys[r], &f1 = fys[std::max(r - 1, 0)];
        DeepRow<T> &d = deep[r];
        memset(&d, 0, sizeof(d));
        d.ilx = r0.ilx; d.kA = r0.kA; d.lc0 = f0.lc0; d.k0 = f0.k0; d.k1 = f0.k1; d.ic0 = f0.ic0; d.ic1 = f0.ic1;
        d.p = DeepMom<T>{r1.invA, r1.ilx, r1.kdx, f1.len, f1.cos0, f1.cos1, f1.ic0, f1.ic1, f1.gh, f1.gd, f1.g1ic0, f1.kdy};
        d.q = DeepUpdate<T>{r2.A, r2.invA};
    }
    auto put = [&](void *&dst, const auto &v) -> hipError_t {
        hipError_t e = dev_alloc(&dst, v.size() * sizeof(v[0]));
        return e == hipSuccess ? ctx_copy(ctx, dst, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice) : e;
    };
    HIPCHK(put(ctx->row, rows));
    HIPCHK(put(ctx->fy, fys));
    HIPCHK(put(ctx->deep_row, deep));
    return THY_OK;
}

int pick_tile(thy_ctx *c) {
    int tx = c->prm.tile_x, ty = c->prm.tile_y;
    if (tx == 0 || ty == 0) {
        if (c->prec) { tx = 32; ty = 8; }
        else { tx = 32; ty = 16; }
    }
    bool ok = c->prec ? tile_supported<double>(tx, ty) : tile_supported<float>(tx, ty);
    if (!ok) return fail(c, THY_ERR_INVALID, "unsupported tile shape " + std::to_string(tx) + "x" + std::to_string(ty));
    c->tx = tx;
    c->ty = ty;
    if (c->prm.kernel < 0 || c->prm.kernel > 2)
        return fail(c, THY_ERR_INVALID, "unknown step kernel " + std::to_string(c->prm.kernel));
    c->kernel = c->prm.kernel;
    if (c->prm.strip_rows < 0 || c->prm.strip_rows > 65536)
        return fail(c, THY_ERR_INVALID, "strip_rows out of range: " + std::to_string(c->prm.strip_rows));
    if (c->prm.general_rows < 0 || c->prm.general_rows > 65536)
        return fail(c, THY_ERR_INVALID, "general_rows out of range: " + std::to_string(c->prm.general_rows));
    // THYSEA_CHUNK_ROWS overrides the number of tile rows dealt to one XCD at a time
    if (const char *v = std::getenv("THYSEA_CHUNK_ROWS")) {
        const int r = std::atoi(v);
        if (r >= 1 && r <= 4096) c->chunk_rows = r;
    }
    return THY_OK;
}

// Rows per deep-water strip of a grid of `rows` segment rows (56-column segments times
// rows) that is stepped alone.  A strip's time is a chain of rows with a halo of 5: with few
// rows the step is the time of one strip, so strips are short; with many the halo's work
// counts.  Measured (us per step, coasts in the north and east): 1000x800 (14400 rows) 18.7 /
// 19.5 / 20.2 at 8 / 12 / 16 rows; 1400x1200 (30000) 29.0 / 25.8 / 29.1 at 8 / 16 / 24; 2000x2000
// (72000) 45.5 / 43.8 / 44.3 at 16 / 24 / 28, FP64 110.8 / 107.8 / 106.5 at 16 / 24 / 32;
// 2500x2500 (112500) 61.2 / 59.7 / 61.3 at 16 / 24 / 32; 4000x3000 (216000) 120.6 / 118.6 /
// 119.2 / 120.4 at 16 / 24 / 32 / 40.
int default_strip_rows(const size_t rows, const int ncu) {
    const size_t per = rows / ncu;
    return per < 80 ? 8 : (per < 200 ? 16 : (per < 560 ? 24 : 32));
}

// Rows per general tile of a grid stepped alone.  Whole tiles have the least halo.  On a
// small grid the step is the time of one tile, so tiles are lower there, the more the
// smaller it is (240x200, 3.9 segment rows a CU: 11.8 / 12.3 / 14.4 us at 3 / 4 / 8 rows;
// 1000x800, 56 rows: 18.6 / 15.9 at 4 / 8).
int default_tile_rows(const size_t rows, const int ncu) {
    return (int)std::min<size_t>(kTileRows, 3 + rows / ((size_t)ncu * 8));
}

// Listed faces (the estimate of find_coast) above which a tile of a grid stepped alone is
// made lower, down to kTileLow rows: the step would wait for the tiles along the coast.
// Above about 130 segment rows a CU no tile reaches it: many tiles share a CU there, and
// lower ones only add halo.  Us a step without this rule and with it, a coast in the north:
// 1501x607 24.3 and 17.9, 800x900 23.5 and 15.7, 731x412 16.5 and 14.5, 1000x800 24.3 and 16.4.
constexpr int kTileLow = 3;
int tile_budget(const size_t rows, const int ncu) { return (int)std::min<size_t>(100000, 5 * rows / ncu); }

// items in order, dealt in eight runs of (nearly) equal length, one per XCD: the workgroup
// at list slot b runs on XCD b mod 8, so each XCD sweeps one contiguous band and items side
// by side share their halos in that XCD's L2.  `per` items make a workgroup; runs are
// padded to whole workgroups with idle items.
std::vector<int2> xcd_runs(const std::vector<int2> &items, const int per) {
    std::vector<int2> out;
    if (items.empty()) return out;
    const int n = (int)items.size(), q = n / 8, rem = n % 8;
    const int wmax = (q + (rem > 0 ? 1 : 0) + per - 1) / per;
    out.assign((size_t)wmax * 8 * per, make_int2(-1, 0));
    for (int x = 0; x < 8; x++) {
        const int size = q + (x < rem ? 1 : 0), start = x * q + std::min(x, rem);
        for (int i = 0; i < size; i++) out[((size_t)(i / per) * 8 + x) * per + i % per] = items[start + i];
    }
    return out;
}

// The order of a step's work items, in groups of 8 that start on the same XCD.  What takes
// longest goes first, so that the short items fill in at the end: a tile takes 10 to 25 us, a
// strip of deep water about 1 us a row.  Tall strips start with the tiles, those spread
// behind, `lag` times thinner than even: tiles are bound by arithmetic, strips by memory, and
// side by side they share a CU.  With lag 0 the tiles go first.  emit(tile, i): the next item
// is the i-th of its kind, or none (i < 0).
template <typename F> void spread_items(const size_t n_tiles, const size_t n_strips, const double lag, const F &emit) {
    const size_t tg = (n_tiles + 7) / 8, dg = (n_strips + 7) / 8;
    for (size_t t = 0, d = 0; t < tg || d < dg;) {
        const bool tile = t < tg && (d >= dg || (double)t * dg * lag <= (double)d * tg);
        const size_t g = tile ? t++ : d++, n = tile ? n_tiles : n_strips;
        for (size_t k = g * 8; k < g * 8 + 8; k++) emit(tile, k < n ? (int)k : -1);
    }
}

// The items of a grid stepped alone.  Strips of up to 8 rows follow the tiles; the taller they
// are, the earlier the last of them has to start.  4000x3000, us a step at lag 1.5 / 2 / 3 / 5:
// 121.5 / 122.1 / 122.9 / 125.6 with strips of 16 rows, 126.4 / 122.3 / 118.7 / 127.5 with 32,
// 134.3 / 133.7 / 127.8 / 117.8 with 48; tiles first 139 to 154, spread evenly 128 to 145.
std::vector<int2> interleave(const std::vector<int2> &tiles, const int n_deep, const int strip_rows) {
    std::vector<int2> out;
    const double lag = strip_rows <= 8 ? 0.0 : 0.11 * strip_rows;
    spread_items(tiles.size(), n_deep, lag, [&](const bool tile, const int i) {
        if (i >= 0) out.push_back(tile ? tiles[i] : make_int2(i * SW_WAVES, 0));
    });
    return out;
}

// a list into its device buffer, which grows as needed
int put_list(thy_ctx *ctx, int2 *&dst, int &cap, const std::vector<int2> &v) {
    if (v.empty()) return THY_OK;
    if (cap < (int)v.size()) {
        dev_free(dst);
        dst = nullptr;
        cap = 0;
        HIPCHK(dev_alloc(&dst, v.size() * sizeof(int2)));
        cap = (int)v.size();
    }
    HIPCHK(ctx_copy(ctx, dst, v.data(), v.size() * sizeof(int2), hipMemcpyHostToDevice));
    return THY_OK;
}

size_t segment_rows(const thy_ctx *c) { return (size_t)((c->nx + SW_OUT - 1) / SW_OUT) * c->ny; }

// Coast along the row sweep's 56-column segments.  A segment row is coastal when any cell of
// its 64 columns is shallower than 3 hpos (or dry).  Its cost is an estimate of the faces
// that will not take the deep form: those of the wet cells shallower than hpos and of the
// cells on either side of a shoreline.  D null: no state yet, depth 0 everywhere.
template <typename T>
void find_coast(thy_ctx *c, const T *D) {
    const int nx = c->nx, ny = c->ny, P = c->pitch;
    const int nseg = (nx + SW_OUT - 1) / SW_OUT;
    const T thr = (T)(3.0 * c->prm.hpos), hpos = (T)c->prm.hpos;
    c->coastal.assign((size_t)nseg * (ny + 1), 0);
    c->cost.assign((size_t)nseg * (ny + 1), 0);
    for (int j = 0; j < ny; j++) {
        for (int sgi = 0; sgi < nseg; sgi++) {
            const int xa = std::max(0, sgi * SW_OUT - SW_HALO), xb = std::min(nx, sgi * SW_OUT + SW_OUT + SW_HALO);
            const T *d = D ? D + (size_t)j * P : nullptr;
            bool any = !D;
            for (int i = xa; i < xb && !any; i++) any = d[i] <= thr;
            int n = 0;
            for (int i = xa; d && any && i < xb; i++) {
                const bool dry = d[i] <= T(0);
                n += (!dry && d[i] <= hpos) || (i > xa && dry != (d[i - 1] <= T(0)));
            }
            const size_t k = (size_t)sgi * (ny + 1) + j;
            c->coastal[k + 1] = c->coastal[k] + (any ? 1 : 0);
            c->cost[k + 1] = c->cost[k] + std::min(SW_OUT, 3 * n);
        }
    }
}

// Work lists with deep-water strips of up to S rows and tiles of up to R rows (above
// kTileLow only as many as keep the tile's cost within `budget`).  Each
// segment's column is cut into blocks of 8 rows between the border bands; a block is deep
// when its rows y0-4 .. y1+3 and its 64 columns are clear of the grid edges (no clamping,
// no first-order band), of the sponges, and of coast.  Runs of deep blocks become strips of
// nearly equal height, the rest tiles, in order of their cost.
int build_lists(thy_ctx *ctx, WorkLists &w, int S, const int R, const int budget) {
    const int nx = ctx->nx, ny = ctx->ny;
    const int nseg = (nx + SW_OUT - 1) / SW_OUT;
    const int spi = ctx->prm.sponge_izq, spd = ctx->prm.sponge_der, sps = ctx->prm.sponge_sup, spn = ctx->prm.sponge_inf;
    S = std::min(S, 2047);
    auto between = [&](const std::vector<int> &v, const int sgi, const int y0, const int y1) {
        const int *row = &v[(size_t)sgi * (ny + 1)];
        return row[std::min(ny, y1)] - row[std::max(0, y0)];
    };
    const int ya = std::max(6, sps + 2), yb = ny - std::max(6, spn + 2);  // rows a deep block may take
    std::vector<int2> strips;
    std::vector<std::pair<int, int2>> tiles;  // (cost, tile)
    // listed faces of rows y .. y+n-1 with the halo, those of the first-order bands included
    auto cost = [&](const int sgi, const int y, const int n) {
        return between(ctx->cost, sgi, y - 2, y + n + 2) + (y < 4 ? 3 * SW_OUT : 0) + (y + n > ny - 4 ? 3 * SW_OUT : 0);
    };
    auto add_tiles = [&](const int sgi, const int y0, const int y1) {
        for (int y = y0, n; y < y1; y += n) {
            n = std::min(R, y1 - y);
            while (n > kTileLow && cost(sgi, y, n) > budget) n--;
            tiles.emplace_back(cost(sgi, y, n), make_int2(sgi * SW_OUT, y << 4 | n));
        }
    };
    for (int sgi = 0; sgi < nseg; sgi++) {
        const int x0 = sgi * SW_OUT;
        const bool xok = ctx->kernel == 0 && x0 - SW_HALO >= 2 && x0 + SW_OUT + SW_HALO - 1 <= nx - 3 &&
                         x0 - SW_HALO >= spi && x0 + SW_OUT + SW_HALO - 1 < nx - spd;
        int y = 0;  // rows before y are dealt
        for (int b = ya; xok && b < yb;) {
            int e = b;  // the run of deep blocks from row b
            while (e < yb && between(ctx->coastal, sgi, e - 4, std::min(e + 8, yb) + 4) == 0) e = std::min(e + 8, yb);
            if (e == b) {
                b += 8;
                continue;
            }
            add_tiles(sgi, y, b);
            const int n = (e - b + S - 1) / S;
            for (int k = 0; k < n; k++) {
                const int s0 = b + (int)((int64_t)(e - b) * k / n), s1 = b + (int)((int64_t)(e - b) * (k + 1) / n);
                strips.push_back(make_int2(x0, s0 << 11 | (s1 - s0)));
            }
            y = b = e;
        }
        add_tiles(sgi, y, ny);
    }
    // neighbouring strips side by side, in rows
    std::stable_sort(strips.begin(), strips.end(), [](const int2 &p, const int2 &q) { return (p.y >> 11) < (q.y >> 11); });
    std::stable_sort(tiles.begin(), tiles.end(), [](const auto &p, const auto &q) { return p.first > q.first; });
    w.tile_h.clear();
    w.tcost_h.clear();
    for (const auto &t : tiles) {
        w.tile_h.push_back(t.second);
        w.tcost_h.push_back(t.first);
    }
    const std::vector<int2> deep = xcd_runs(strips, SW_WAVES);
    const std::vector<int2> items = interleave(w.tile_h, (int)deep.size() / SW_WAVES, S);
    int r;
    if ((r = put_list(ctx, w.deep, w.deep_cap, deep)) != THY_OK || (r = put_list(ctx, w.items, w.items_cap, items)) != THY_OK)
        return r;
    w.n_deep = (int)deep.size();
    w.n_items = (int)items.size();
    return THY_OK;
}

// the lists of a run alone, with deep-water strips of S rows and tiles of R rows
int build_alone(thy_ctx *ctx, int S, const int R) {
    if (ctx->kernel == 1) return THY_OK;
    drop_graphs(ctx);  // the captured step sequences hold the old lists and grid sizes
    S = std::min(S, 2047);  // (a strip's record holds its height in 11 bits)
    ctx->srows = S;
    ctx->trows = R;
    const int budget = ctx->prm.general_rows > 0 ? INT_MAX : tile_budget(segment_rows(ctx), ctx->ncu);
    return build_lists(ctx, ctx->alone, S, R, budget);
}

// the lists of an uploaded state (D null: of the state a context has before one)
template <typename T>
int build_order(thy_ctx *ctx, const T *D) {
    if (ctx->kernel == 1) return THY_OK;
    find_coast(ctx, D);
    ctx->uploaded = D != nullptr;
    ctx->batched.n_items = 0;  // built again when a batch asks for them
    if (ctx->tuned_srows > 0) return build_alone(ctx, ctx->tuned_srows, ctx->tuned_trows);
    const size_t rows = segment_rows(ctx);
    return build_alone(ctx, ctx->prm.strip_rows > 0 ? ctx->prm.strip_rows : default_strip_rows(rows, ctx->ncu),
                       ctx->prm.general_rows > 0 ? std::min(ctx->prm.general_rows, kTileRows) : default_tile_rows(rows, ctx->ncu));
}

// a context may be stepped before a state was uploaded
int need_lists(thy_ctx *ctx) {
    if (ctx->kernel == 1 || ctx->alone.n_items > 0) return THY_OK;
    return ctx->prec ? build_order<double>(ctx, nullptr) : build_order<float>(ctx, nullptr);
}

// The lists a batch steps the scenario by.  Its scenarios fill the device whatever their
// grids: tiles are whole, and strips of 24 rows cost the least (GPU time of 24 scenarios of
// 1000x800: 88.0 / 86.3 / 85.7 ms at 16 / 24 / 32 rows; a mix of 12 grids 76.9 / 75.8 / 76.6).
int build_batched(thy_ctx *ctx) {
    const int R = ctx->prm.general_rows > 0 ? std::min(ctx->prm.general_rows, kTileRows) : kTileRows;
    return build_lists(ctx, ctx->batched, ctx->prm.strip_rows > 0 ? ctx->prm.strip_rows : 24, R, INT_MAX);
}

template <typename T>
int upload_t(thy_ctx *ctx, const double *s1, const double *s2) {
    const int nx = ctx->nx, ny = ctx->ny, P = ctx->pitch;
    const double hmin = ctx->prm.hmin;
    const size_t n = (size_t)P * ny, b = n * sizeof(T);
    ctx->batch_ready = false;  // a new state: a run prepared for it is void
    // e, D, qx, qy staged in pinned host memory (a cached block), copied asynchronously
    T *st = nullptr;
    HIPCHK(Pool::get().host_alloc((void **)&st, 4 * b));
    struct Staging {
        T *p;
        hipStream_t s;
        ~Staging() {
            (void)hipStreamSynchronize(s);  // the copies read it until they finish
            Pool::get().host_free(p);
        }
    } staging{st, ctx->stream};
    T *e = st, *D = st + n, *qx = st + 2 * n, *qy = st + 3 * n;
    for (int j = 0; j < ny; j++) {
        const size_t r = (size_t)j * nx, ro = (size_t)j * P;
        for (int i = 0; i < nx; i++) {
            const size_t c = r + i, o = ro + i;
            const double h = s1[2 * c], Hs = s1[2 * c + 1];
            if (!std::isfinite(h) || !std::isfinite(Hs) || !std::isfinite(s2[2 * c]) || !std::isfinite(s2[2 * c + 1]))
                return fail(ctx, THY_ERR_NONFINITE,
                            "non-finite input state at cell (" + std::to_string(i) + ", " + std::to_string(j) + ")");
            const double Dd = Hs + hmin;             // unshifted depth
            D[o] = (T)Dd;
            e[o] = (h > 0.0) ? (T)(h - Dd) : -(T)Dd;  // dry: e = -D exactly, so h = 0
            qx[o] = (T)s2[2 * c];
            qy[o] = (T)s2[2 * c + 1];
        }
        for (int i = nx; i < P; i++) e[ro + i] = D[ro + i] = qx[ro + i] = qy[ro + i] = T(0);
    }
    hipStream_t q = ctx->stream;
    HIPCHK(hipMemcpyAsync(ctx->e[0], e, b, hipMemcpyHostToDevice, q));
    HIPCHK(hipMemcpyAsync(ctx->D, D, b, hipMemcpyHostToDevice, q));
    HIPCHK(hipMemcpyAsync(ctx->qx[0], qx, b, hipMemcpyHostToDevice, q));
    HIPCHK(hipMemcpyAsync(ctx->qy[0], qy, b, hipMemcpyHostToDevice, q));
    HIPCHK(hipMemcpyAsync(ctx->e[1], ctx->e[0], b, hipMemcpyDeviceToDevice, q));
    HIPCHK(hipMemcpyAsync(ctx->qx[1], ctx->qx[0], b, hipMemcpyDeviceToDevice, q));
    HIPCHK(hipMemcpyAsync(ctx->qy[1], ctx->qy[0], b, hipMemcpyDeviceToDevice, q));
    ctx->cur = 0;
    HIPCHK(hipMemsetAsync(ctx->health, 0, sizeof(unsigned int), q));  // a new state is healthy until stepped
    const int r = build_order<T>(ctx, D);  // on the host while the copies run
    HIPCHK(hipStreamSynchronize(q));
    return r;
}

template <typename T>
int download_t(thy_ctx *ctx, double *s1, double *s2) {
    const int nx = ctx->nx, ny = ctx->ny, P = ctx->pitch;
    const size_t b = (size_t)P * ny * sizeof(T);
    std::vector<T> e((size_t)P * ny), D((size_t)P * ny), qx((size_t)P * ny), qy((size_t)P * ny);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    HIPCHK(ctx_copy(ctx, e.data(), ctx->e[ctx->cur], b, hipMemcpyDeviceToHost));
    HIPCHK(ctx_copy(ctx, D.data(), ctx->D, b, hipMemcpyDeviceToHost));
    HIPCHK(ctx_copy(ctx, qx.data(), ctx->qx[ctx->cur], b, hipMemcpyDeviceToHost));
    HIPCHK(ctx_copy(ctx, qy.data(), ctx->qy[ctx->cur], b, hipMemcpyDeviceToHost));
    for (int j = 0; j < ny; j++) {
        for (int i = 0; i < nx; i++) {
            const size_t c = (size_t)j * nx + i, o = (size_t)j * P + i;
            if (s1) {
                s1[2 * c] = (double)e[o] + (double)D[o];
                s1[2 * c + 1] = (double)D[o] - ctx->prm.hmin;
            }
            if (s2) {
                s2[2 * c] = (double)qx[o];
                s2[2 * c + 1] = (double)qy[o];
            }
        }
    }
    return THY_OK;
}

int read_ctrl(thy_ctx *ctx, Ctrl *c) {
    if (ctx->ctrl_h_valid) {
        *c = ctx->ctrl_h;
        return THY_OK;
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    HIPCHK(ctx_copy(ctx, c, &ctx->ctrl[ctx->slot], sizeof(Ctrl), hipMemcpyDeviceToHost));
    ctx->ctrl_h = *c;
    ctx->ctrl_h_valid = true;
    return THY_OK;
}

int write_ctrl(thy_ctx *ctx, const Ctrl &c) {
    ctx->ctrl_h_valid = false;
    HIPCHK(ctx_copy(ctx, &ctx->ctrl[ctx->slot], &c, sizeof(Ctrl), hipMemcpyHostToDevice));
    ctx->ctrl_h = c;
    ctx->ctrl_h_valid = true;
    return THY_OK;
}

// minimum over the dt partials of one launch slot, as copied to the host (kDtSlot words)
unsigned int dt_parts_min(const unsigned int *w) {
    unsigned int m = kDtNone;
    for (int p = 0; p < kDtParts; p++) m = std::min(m, w[dt_at(0, p)]);
    return m;
}

// the raw dt minimum of launch slot s
int read_dt_slot(thy_ctx *ctx, const int s, unsigned int &raw) {
    std::vector<unsigned int> w(kDtSlot);
    HIPCHK(ctx_copy(ctx, w.data(), ctx->dtmin + dt_at(s, 0), kDtSlot * sizeof(unsigned int), hipMemcpyDeviceToHost));
    raw = dt_parts_min(w.data());
    return THY_OK;
}

// every partial of launch slot s (all three slots for s < 0) back to "no cell reported"
int clear_dt_slots(thy_ctx *ctx, const int s) {
    const std::vector<unsigned int> v((s < 0 ? 3 : 1) * kDtSlot, kDtNone);
    HIPCHK(ctx_copy(ctx, ctx->dtmin + (s < 0 ? 0 : dt_at(s, 0)), v.data(), v.size() * sizeof(unsigned int),
                    hipMemcpyHostToDevice));
    return THY_OK;
}

int reset_dt_slots(thy_ctx *ctx) {
    int r;
    if ((r = clear_dt_slots(ctx, -1)) != THY_OK) return r;
    return THY_OK;
}

Ctrl idle_ctrl(thy_ctx *ctx) {
    Ctrl c;
    memset(&c, 0, sizeof(c));
    c.t = 0.0;
    c.t_end = 1e300;
    c.next_save = INFINITY;
    c.next_series = INFINITY;
    c.series_dt = 0.0;
    c.T = ctx->prm.T;
    c.cur = ctx->cur;
    c.gcap = ctx->gcap;
    return c;
}

template <typename T>
int apply_okada_t(thy_ctx *ctx, const thy_fault *f, int crop_flag, double crop_value, double *def_out) {
    const int64_t n = (int64_t)ctx->nx * ctx->ny;
    OkadaFault of;
    of.lon_c = f->lon_c; of.lat_c = f->lat_c; of.depth = f->depth_c; of.L = f->length; of.W = f->width;
    of.H = ctx->prm.H;
    of.strike = f->strike; of.dip = f->dip; of.rake = f->rake; of.slip = f->slip;
    of.lon0 = ctx->lon[0];
    of.dlon = (ctx->lon[ctx->nx - 1] - ctx->lon[0]) / (ctx->nx - 1);
    T *const e = (T *)ctx->e[ctx->cur], *const D = (T *)ctx->D, *const arr = (T *)ctx->arr;
    hipLaunchKernelGGL(k_okada_plane, dim3(1), dim3(64), 0, ctx->stream, of, ctx->okada_plane);
    HIPCHK(hipGetLastError());
    if (!def_out && crop_flag != 1) {
        hipLaunchKernelGGL((k_okada_add<T>), dim3(grid_1d(n)), dim3(256), 0, ctx->stream, of, ctx->okada_plane, ctx->okada_row, ctx->nx,
                           ctx->ny, ctx->pitch, crop_flag == 2 ? crop_value : -1.0, e, D, arr);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(ctx->stream));
        return THY_OK;
    }
    HIPCHK(hipMemsetAsync(&ctx->scratch_u[1], 0, sizeof(unsigned int), ctx->stream));
    hipLaunchKernelGGL(k_okada, dim3(grid_1d(n)), dim3(256), 0, ctx->stream, of, ctx->okada_plane, ctx->okada_row, ctx->nx, ctx->ny,
                       ctx->okada_def, &ctx->scratch_u[1]);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL((k_okada_apply<T>), dim3(grid_1d(n)), dim3(256), 0, ctx->stream, ctx->okada_def, ctx->nx,
                       ctx->ny, ctx->pitch, crop_flag, crop_value, &ctx->scratch_u[1], e, D, arr);
    HIPCHK(hipGetLastError());
    if (def_out) {
        HIPCHK(hipMemcpyAsync(def_out, ctx->okada_def, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return THY_OK;
}

template <typename T>
int init_metrics_t(thy_ctx *ctx) {
    const int64_t n = (int64_t)ctx->nx * ctx->ny;
    hipLaunchKernelGGL((k_init_metrics<T>), dim3(grid_1d(n)), dim3(256), 0, ctx->stream, (const T *)ctx->e[ctx->cur],
                       (const T *)ctx->D, ctx->nx, ctx->ny, ctx->pitch, (T)ctx->prm.eps_h, (T *)ctx->emax,
                       (T *)ctx->arr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return THY_OK;
}

template <typename T>
int initial_dt_t(thy_ctx *ctx, double *dt) {
    const int64_t n = (int64_t)ctx->nx * ctx->ny;
    StepArgs<T> a = make_args<T>(ctx);
    unsigned int big = 0x7f7fffffu;
    HIPCHK(ctx_copy(ctx, &ctx->scratch_u[0], &big, sizeof(big), hipMemcpyHostToDevice));
    hipLaunchKernelGGL((k_initial_dt<T>), dim3(grid_1d(n)), dim3(256), 0, ctx->stream, a, ctx->cur, &ctx->scratch_u[0]);
    HIPCHK(hipGetLastError());
    unsigned int r;
    HIPCHK(ctx_copy(ctx, &r, &ctx->scratch_u[0], sizeof(r), hipMemcpyDeviceToHost));
    float f;
    memcpy(&f, &r, 4);
    *dt = (double)f;
    return THY_OK;
}

// A large device buffer into the caller's pageable memory.  The runtime's own copy goes
// through one thread (or pins the caller's pages); here the data passes through pinned memory
// in chunks, and several threads copy them on, so that the page faults of a new buffer are
// taken side by side too.  The helper threads make no HIP calls and have ended on return.
// The pinned block is one of its own, of 8 chunks: 16 are no faster, and with the block that
// staged the upload, whose lines then lie in other cores' caches, the next upload took 31 ms
// instead of 21 (2000x2000) and 90 instead of 61 (4000x3000).  Four fields of 4000x3000: 19.3
// ms with the runtime's copy, 6.9 with this one; of 2000x2000 6.5 and 3.3, 1500x1450 (8.7 MB
// each) 4.2 and 2.3; of 1400x1200 (6.7 MB, below the line) the runtime's is as fast.
constexpr size_t kChunk = 2u << 20, kLargeCopy = 8u << 20;
constexpr int kCopyThreads = 8;

int read_large(thy_ctx *ctx, char *out, const char *src, const size_t bytes) {
    const int n = (int)((bytes + kChunk - 1) / kChunk);
    struct Run {
        hipStream_t q;
        char *pin = nullptr;
        std::vector<hipEvent_t> ev;        // one per slot
        std::vector<std::thread> helpers;
        std::atomic<int> ready{0}, next{0};  // chunks that have arrived; the next to be copied on
        std::unique_ptr<std::atomic<bool>[]> done;
        std::atomic<bool> stop{false};
        void join() {
            for (std::thread &t : helpers) t.join();
            helpers.clear();
        }
        ~Run() {
            stop = true;
            join();
            (void)hipStreamSynchronize(q);
            for (hipEvent_t e : ev) (void)hipEventDestroy(e);
            Pool::get().host_free(pin);
        }
    } run;
    run.q = ctx->stream;
    const size_t room = 8 * kChunk;
    HIPCHK(Pool::get().host_alloc((void **)&run.pin, room));
    const int slots = (int)std::min<size_t>({room / kChunk, (size_t)n, (size_t)64});
    run.done.reset(new std::atomic<bool>[n]);
    for (int i = 0; i < n; i++) run.done[i] = false;
    for (int i = 0; i < slots; i++) {
        hipEvent_t e;
        HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        run.ev.push_back(e);
    }
    auto size_of = [&](const int c) { return std::min(kChunk, bytes - (size_t)c * kChunk); };
    auto copy_on = [&](const int c) {
        memcpy(out + (size_t)c * kChunk, run.pin + (size_t)(c % slots) * kChunk, size_of(c));
        run.done[c] = true;
    };
    auto helper = [&] {
        for (;;) {
            const int c = run.next++;
            if (c >= n) return;
            while (run.ready <= c) {
                if (run.stop) return;
                std::this_thread::yield();
            }
            copy_on(c);
        }
    };
    try {
        const int cpus = (int)std::thread::hardware_concurrency();
        for (int t = 0; t < std::min({kCopyThreads, std::max(1, cpus / 2), n}); t++) run.helpers.emplace_back(helper);
    } catch (const std::system_error &) {
        // as many as there are; with none this thread copies
    }
    for (int c = 0, sent = 0; c < n; c++) {
        for (; sent < n && (sent < slots || run.done[sent - slots]); sent++) {
            HIPCHK(hipMemcpyAsync(run.pin + (size_t)(sent % slots) * kChunk, src + (size_t)sent * kChunk, size_of(sent),
                                  hipMemcpyDeviceToHost, ctx->stream));
            HIPCHK(hipEventRecord(run.ev[sent % slots], ctx->stream));
        }
        if (c >= sent) {  // its slot is still being copied on
            std::this_thread::yield();
            c--;
            continue;
        }
        HIPCHK(hipEventSynchronize(run.ev[c % slots]));
        run.ready = c + 1;
        if (run.helpers.empty()) copy_on(c);
    }
    run.join();
    return THY_OK;
}

template <typename T>
int get_field_t(thy_ctx *ctx, int field, float *out) {
    const int64_t n = (int64_t)ctx->nx * ctx->ny;
    if (field == THY_ARRIVAL_TIMES && !ctx->arr) {
        for (int64_t i = 0; i < n; i++) out[i] = -1.0f;
        return THY_OK;
    }
    hipLaunchKernelGGL((k_output<T>), dim3(grid_1d(n)), dim3(256), 0, ctx->stream, field, (const T *)ctx->e[ctx->cur],
                       (const T *)ctx->qx[ctx->cur], (const T *)ctx->qy[ctx->cur], (const T *)ctx->D,
                       (const T *)ctx->emax, (const T *)ctx->arr, ctx->nx, ctx->ny, ctx->pitch, (T)ctx->prm.eps_h,
                       ctx->prm.H, ctx->prm.Q, ctx->prm.T, ctx->outbuf);
    HIPCHK(hipGetLastError());
    if (n * sizeof(float) >= kLargeCopy) {
        try {
            return read_large(ctx, (char *)out, (const char *)ctx->outbuf, n * sizeof(float));
        } catch (const std::bad_alloc &) {
            return fail(ctx, THY_ERR_HOST_MEMORY, "no host memory to read a field");
        }
    }
    HIPCHK(hipMemcpyAsync(out, ctx->outbuf, n * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return THY_OK;
}

template <typename T>
int update_metrics_t(thy_ctx *ctx, double t) {
    const int64_t n = (int64_t)ctx->nx * ctx->ny;
    hipLaunchKernelGGL((k_update_metrics<T>), dim3(grid_1d(n)), dim3(256), 0, ctx->stream,
                       (const T *)ctx->e[ctx->cur], (const T *)ctx->D, ctx->nx, ctx->ny, ctx->pitch,
                       (T)ctx->prm.eps_h, (T)ctx->prm.dif_at, (T)t, (T *)ctx->emax, (T *)ctx->arr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return THY_OK;
}

// Compensated FP64 sum of h * area * cos(phi): kMassBlocks workgroup partials in the
// device buffer `partial`, copied to the host array `host` (kMassBlocks entries).
template <typename T>
int mass_t(thy_ctx *ctx, double *partial, double *host, double *mass) {
    hipLaunchKernelGGL((k_mass<T>), dim3(kMassBlocks), dim3(256), 0, ctx->stream, (const T *)ctx->e[ctx->cur],
                       (const T *)ctx->D, (const RowGeo<T> *)ctx->row, ctx->area_d, ctx->nx, ctx->ny, ctx->pitch,
                       partial);
    HIPCHK(hipGetLastError());
    HIPCHK(ctx_copy(ctx, host, partial, kMassBlocks * sizeof(double), hipMemcpyDeviceToHost));
    double s = 0.0, comp = 0.0;
    for (int k = 0; k < kMassBlocks; k++) {
        const double x = host[k];
        double t = s + x;
        if (std::fabs(s) >= std::fabs(x)) comp += (s - t) + x;
        else comp += (x - t) + s;
        s = t;
    }
    *mass = s + comp;
    return THY_OK;
}

// Capture K consecutive step launches starting at launch slot s0 (slots s0, s0+1, ...
// mod 3) into one graph, and upload it.
int capture_steps(thy_ctx *ctx, int K, int s0) {
    hipGraph_t g;
    const int slot_saved = ctx->slot;
    ctx->slot = s0;
    HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < K; k++) {
        hipError_t e = launch_step(ctx);
        if (e != hipSuccess) {
            (void)hipStreamEndCapture(ctx->stream, &g);
            ctx->slot = slot_saved;
            return fail(ctx, THY_ERR_HIP, std::string("capture: ") + hipGetErrorString(e));
        }
    }
    ctx->slot = slot_saved;
    HIPCHK(hipStreamEndCapture(ctx->stream, &g));
    hipError_t e = hipGraphInstantiate(&ctx->gexec[s0], g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    HIPCHK(e);
    HIPCHK(hipGraphUpload(ctx->gexec[s0], ctx->stream));
    return THY_OK;
}

// The step sequences replays of K steps need from the current launch slot on: with K a
// multiple of 3 every replay starts at the same slot, otherwise the replays cycle
// through all three (so any step count can be replayed without idle launches).
int build_graphs(thy_ctx *ctx, int K) {
    if (ctx->gk != K) drop_graphs(ctx);
    ctx->gk = K;
    int r;
    for (int m = 0; m < 3; m++) {
        const int s0 = (ctx->slot + m * K) % 3;
        if (!ctx->gexec[s0] && (r = capture_steps(ctx, K, s0)) != THY_OK) return r;
        if (K % 3 == 0) break;
    }
    return THY_OK;
}

// The stop predicate holds for the control block of the next launch, as seen on the
// host after a replay: finalise its dt on the host (truncation at fault times, as the
// launch would have done) and write it back, instead of replaying a sequence of launches
// that would only find the run stopped.  raw: the previous step's dt minimum.
int finalise_on_host(thy_ctx *ctx, Ctrl &c, const unsigned int raw) {
    if (c.dt_valid) return THY_OK;
    float rf;
    memcpy(&rf, &raw, 4);
    int skip;
    const double dt = step_dt(c, ctx->ftimes.data(), rf, skip);
    if (c.steps > 0 && ctx->on_step) {  // the log entry the launch would have written
        const double ent[2] = {dt, c.t};
        HIPCHK(ctx_copy(ctx, ctx->steplog + 2 * ((c.steps - 1) % ctx->logcap), ent, sizeof(ent),
                        hipMemcpyHostToDevice));
    }
    c.dt = dt;
    c.skip = skip;
    c.dt_valid = 1;
    return write_ctrl(ctx, c);
}

// Advance until the stop predicate holds; graph replays of K steps.  After each replay
// the control block, the dt partials of its last launch and the health flag are copied
// to pinned memory behind it.  While the last replay's time, steps and mean dt say that the run goes on
// for two more full replays (before t_end, max_steps, the next fault and the next
// snapshot), the next replay is queued before the one in flight is waited for, so that
// the device does not idle between replays.  When the host sees the stop predicate hold
// after a replay it finalises the control block itself; a queued replay that finds the
// run stopped idles through its launches (the stop predicate holds in every one).
int advance(thy_ctx *ctx, int K, Ctrl *out, double *ms) {
    int r;
    if ((r = build_graphs(ctx, K)) != THY_OK) return r;
    Ctrl last;
    if ((r = read_ctrl(ctx, &last)) != THY_OK) return r;
    if (must_stop(last, ctx->ftimes.data())) {  // stopped before any step
        unsigned int raw = 0;
        if (!last.dt_valid && (r = read_dt_slot(ctx, (ctx->slot + 2) % 3, raw)) != THY_OK) return r;
        if ((r = finalise_on_host(ctx, last, raw)) != THY_OK) return r;
        *out = last;
        if (ms) *ms = 0.0;
        return THY_OK;
    }
    // (a health flag raised before this call stops the first launch on the device)
    double total = 0.0, dt_mean = 0.0;
    int head = 0, queued = 0;
    auto enqueue = [&]() -> hipError_t {
        const int i = (head + queued) % 2;
        hipError_t e;
        if ((e = hipEventRecord(ctx->rev[i][0], ctx->stream)) != hipSuccess) return e;
        if ((e = hipGraphLaunch(ctx->gexec[ctx->slot], ctx->stream)) != hipSuccess) return e;
        if ((e = hipEventRecord(ctx->rev[i][1], ctx->stream)) != hipSuccess) return e;
        ctx->slot = (ctx->slot + K) % 3;
        if ((e = hipMemcpyAsync(&ctx->h_snap[i], &ctx->ctrl[ctx->slot], sizeof(Ctrl), hipMemcpyDeviceToHost,
                                ctx->stream)) != hipSuccess)
            return e;
        if ((e = hipMemcpyAsync(ctx->h_dt + (size_t)i * kDtSlot, ctx->dtmin + dt_at((ctx->slot + 2) % 3, 0),
                                kDtSlot * sizeof(unsigned int), hipMemcpyDeviceToHost, ctx->stream)) != hipSuccess)
            return e;
        if ((e = hipMemcpyAsync(&ctx->h_aux[i], ctx->health, 4, hipMemcpyDeviceToHost, ctx->stream)) !=
            hipSuccess)
            return e;
        if ((e = hipEventRecord(ctx->rev[i][2], ctx->stream)) != hipSuccess) return e;
        queued++;
        return hipSuccess;
    };
    auto goes_on = [&](const Ctrl &c) {
        if (!(dt_mean > 0.0)) return false;
        const double t2 = c.t + 2.5 * K * dt_mean;  // two replays, with a margin for dt to grow
        if (!(t2 < c.t_end) || t2 >= c.next_save) return false;
        if (c.max_steps > 0 && c.steps + 2 * (int64_t)K > c.max_steps) return false;
        if (c.k < c.nf && t2 * c.T >= ctx->ftimes[c.k]) return false;
        return true;
    };
    unsigned int raw = 0;
    auto collect = [&](Ctrl &c) -> hipError_t {
        hipError_t e = hipEventSynchronize(ctx->rev[head][2]);
        if (e != hipSuccess) return e;
        c = ctx->h_snap[head];
        raw = dt_parts_min(ctx->h_dt + (size_t)head * kDtSlot);
        if (ctx->h_aux[head]) c.nonfinite = 1;
        float f = 0.f;
        (void)hipEventElapsedTime(&f, ctx->rev[head][0], ctx->rev[head][1]);
        total += f;
        head ^= 1;
        queued--;
        return hipSuccess;
    };
    HIPCHK(enqueue());
    for (;;) {
        if (queued == 1 && goes_on(last)) HIPCHK(enqueue());
        Ctrl c;
        HIPCHK(collect(c));
        ctx->cur = c.cur;
        if (c.steps > last.steps) dt_mean = (c.t - last.t) / (double)(c.steps - last.steps);
        last = c;
        // After an executed step dt_valid is 0; it stays 1 only when a launch of this
        // replay found the stop predicate true (every later launch then idled).
        const bool host_stop = !c.dt_valid && queued == 0 && must_stop(c, ctx->ftimes.data());
        if (c.dt_valid || host_stop) {
            while (queued > 0) HIPCHK(collect(c));  // a queued replay idled: same control block
            ctx->cur = c.cur;
            if (host_stop) {
                if ((r = finalise_on_host(ctx, c, raw)) != THY_OK) return r;
            } else {
                ctx->ctrl_h = c;  // the control block the stopping launch left in this slot
                ctx->ctrl_h_valid = true;
            }
            *out = c;
            if (ms) *ms = total;
            return THY_OK;
        }
        if (queued == 0) HIPCHK(enqueue());
    }
}

// plain copy, 4 x 16 B per thread per block-chunk, chunks coalesced across the block
__global__ void __launch_bounds__(256) k_copy_probe(const float4 *__restrict__ a, float4 *__restrict__ b, int64_t n) {
    const int64_t chunk = 4 * 256;
    for (int64_t base = (int64_t)blockIdx.x * chunk; base < n; base += (int64_t)gridDim.x * chunk) {
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int64_t i = base + k * 256 + threadIdx.x;
            if (i < n) v[k] = a[i];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int64_t i = base + k * 256 + threadIdx.x;
            if (i < n) b[i] = v[k];
        }
    }
}

}  // namespace

extern "C" {

int thy_copy_probe(size_t bytes, int reps, double *ms_per_copy) {
    RelaxedCapture relaxed;
    thy_ctx *ctx = nullptr;
    const int64_t n = (int64_t)(bytes / sizeof(float4));
    if (n <= 0 || reps <= 0) return THY_ERR_INVALID;
    void *a = nullptr, *b = nullptr;
    hipEvent_t e0, e1;
    HIPCHK(hipMalloc(&a, n * sizeof(float4)));
    HIPCHK(hipMalloc(&b, n * sizeof(float4)));
    HIPCHK(hipMemset(a, 0, n * sizeof(float4)));
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    const int grid = (int)std::min<int64_t>((n + 1023) / 1024, 1 << 20);
    hipLaunchKernelGGL(k_copy_probe, dim3(grid), dim3(256), 0, 0, (const float4 *)a, (float4 *)b, n);
    HIPCHK(hipEventRecord(e0, 0));
    for (int r = 0; r < reps; r++)
        hipLaunchKernelGGL(k_copy_probe, dim3(grid), dim3(256), 0, 0, (const float4 *)a, (float4 *)b, n);
    HIPCHK(hipEventRecord(e1, 0));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    if (ms_per_copy) *ms_per_copy = ms / reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    return THY_OK;
}

int thy_probe(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return 1;
    for (int d = 0; d < n; d++) {
        hipDeviceProp_t p;
        if (hipGetDeviceProperties(&p, d) == hipSuccess && std::strncmp(p.gcnArchName, "gfx950", 6) == 0) return 0;
    }
    return 2;
}

// arrays of the state block: e, qx, qy (two buffers each), D, emax and, with arrival
// tracking, arr
static int state_arrays(const thy_params *p) { return 8 + ((p && p->track_arrival) ? 1 : 0); }

size_t thy_footprint(int nx, int ny, const thy_params *p) {
    const size_t esz = (p && p->precision) ? 8 : 4;
    const size_t pitch = ((size_t)nx + 63) / 64 * 64;
    const size_t n = pitch * ny;
    size_t bytes = (size_t)state_arrays(p) * n * esz;
    bytes += (size_t)nx * ny * (8 + 4);                 // okada scratch (double) + output staging (float)
    // row tables: geometry, deep-water records, mass weight, Okada
    const size_t row = esz == 8 ? sizeof(RowGeo<double>) + sizeof(FaceGeoY<double>) + sizeof(DeepRow<double>)
                                : sizeof(RowGeo<float>) + sizeof(FaceGeoY<float>) + sizeof(DeepRow<float>);
    bytes += (size_t)(ny + 1) * (row + sizeof(double) + sizeof(OkadaRow));
    // work lists, of a run alone and of a batch: no more items and strips than lowest tiles
    bytes += 2 * ((size_t)nx / SW_OUT + 1) * ((size_t)ny / kTileLow + 1) * sizeof(int2);
    return bytes;
}

int thy_create(const thy_grid *g, const thy_params *p, thy_ctx **out) {
    RelaxedCapture relaxed;
    if (!g || !p || !out || g->nx < 2 || g->ny < 2) return THY_ERR_INVALID;
    thy_ctx *ctx = new (std::nothrow) thy_ctx();
    if (!ctx) return THY_ERR_HOST_MEMORY;
    *out = ctx;
    ctx->nx = g->nx;
    ctx->ny = g->ny;
    ctx->prm = *p;
    ctx->prec = p->precision ? 1 : 0;
    ctx->esz = ctx->prec ? 8 : 4;
    ctx->pitch = (g->nx + 63) / 64 * 64;
    ctx->lon.assign(g->lon, g->lon + g->nx);
    ctx->lat.assign(g->lat, g->lat + g->ny);
    ctx->area.assign(g->area, g->area + g->ny);
    ctx->cosphi.assign(g->cosphi, g->cosphi + g->ny);
    ctx->ancho.assign(g->ancho, g->ancho + g->ny + 1);
    ctx->alto.assign(g->alto, g->alto + g->ny);
    int r = pick_tile(ctx);
    if (r != THY_OK) return r;
    // the row sweeps address every state array through one buffer resource over the
    // state block, with 32-bit byte offsets; a grid whose block is larger runs the tile
    // kernel
    ctx->state_bytes = (size_t)state_arrays(p) * ctx->pitch * ctx->ny * ctx->esz;
    if (ctx->kernel != 1 && ctx->state_bytes > (size_t)INT32_MAX) ctx->kernel = 1;
    HIPCHK(hipSetDevice(0));
    HIPCHK(Pool::get().get_stream(ctx->stream));
    {
        int dev = 0;
        HIPCHK(hipGetDevice(&dev));
        HIPCHK(hipDeviceGetAttribute(&ctx->ncu, hipDeviceAttributeMultiprocessorCount, dev));
        ctx->device = dev;
        // the device address of this device's copy of the allocation-free scratch, once
        // per device, with the device current
        if (dev < kScratchDevices) {
            std::lock_guard<std::mutex> lock(g_scratch_mutex);
            if (!g_scratch_ptr[dev]) {
                void *p = nullptr;
                HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
                g_scratch_ptr[dev] = (double *)p;
            }
        }
    }
    HIPCHK(hipEventCreate(&ctx->ev0));
    HIPCHK(hipEventCreate(&ctx->ev1));
    for (int i = 0; i < 2; i++) {
        HIPCHK(hipEventCreate(&ctx->rev[i][0]));
        HIPCHK(hipEventCreate(&ctx->rev[i][1]));
        HIPCHK(hipEventCreateWithFlags(&ctx->rev[i][2], hipEventDisableTiming));
    }
    HIPCHK(Pool::get().host_alloc((void **)&ctx->h_snap, 2 * sizeof(Ctrl)));
    HIPCHK(Pool::get().host_alloc((void **)&ctx->h_aux, 4 * sizeof(unsigned int)));
    HIPCHK(Pool::get().host_alloc((void **)&ctx->h_dt, 2 * kDtSlot * sizeof(unsigned int)));
    const size_t n = (size_t)ctx->pitch * ctx->ny, b = n * ctx->esz;
    HIPCHK(dev_alloc(&ctx->state, ctx->state_bytes));
    {
        char *blk = (char *)ctx->state;  // arrays of b bytes (whole 256-B rows) in a fixed order
        for (int k = 0; k < 2; k++) {
            ctx->e[k] = blk + (0 + k) * b;
            ctx->qx[k] = blk + (2 + k) * b;
            ctx->qy[k] = blk + (4 + k) * b;
        }
        ctx->D = blk + 6 * b;
        ctx->emax = blk + 7 * b;
        if (p->track_arrival) ctx->arr = blk + 8 * b;
    }
    HIPCHK(dev_alloc((void **)&ctx->okada_def, (size_t)ctx->nx * ctx->ny * sizeof(double)));
    HIPCHK(dev_alloc((void **)&ctx->outbuf, (size_t)ctx->nx * ctx->ny * sizeof(float)));
    HIPCHK(dev_alloc((void **)&ctx->ctrl, 3 * sizeof(Ctrl)));
    HIPCHK(dev_alloc((void **)&ctx->dtmin, 3 * kDtSlot * sizeof(unsigned int)));
    HIPCHK(dev_alloc((void **)&ctx->scratch_u, 4 * sizeof(unsigned int)));
    HIPCHK(dev_alloc((void **)&ctx->health, sizeof(unsigned int)));
    HIPCHK(ctx_fill(ctx, ctx->health, sizeof(unsigned int)));
    HIPCHK(dev_alloc((void **)&ctx->mass_partial, kMassBlocks * sizeof(double)));
    HIPCHK(dev_alloc((void **)&ctx->steplog, (size_t)ctx->logcap * 2 * sizeof(double)));
    HIPCHK(dev_alloc((void **)&ctx->area_d, ctx->ny * sizeof(double)));
    {
        // mass weight per row: area*cos(phi), the invariant of the discrete scheme
        std::vector<double> w(ctx->ny);
        for (int j = 0; j < ctx->ny; j++) w[j] = g->area[j] * g->cosphi[j];
        HIPCHK(ctx_copy(ctx, ctx->area_d, w.data(), ctx->ny * sizeof(double), hipMemcpyHostToDevice));
    }
    {
        // the latitudes Okada uses are uniform (src/GPU/ShallowWater.cu:215-218)
        const double lat0 = ctx->lat[0], dlat = (ctx->lat[ctx->ny - 1] - ctx->lat[0]) / (ctx->ny - 1);
        HIPCHK(dev_alloc((void **)&ctx->okada_row, ctx->ny * sizeof(OkadaRow)));
        HIPCHK(dev_alloc((void **)&ctx->okada_plane, sizeof(OkadaPlane)));
        hipLaunchKernelGGL(k_okada_rows, dim3((ctx->ny + 255) / 256), dim3(256), 0, ctx->stream, lat0, dlat, ctx->ny,
                           ctx->okada_row);
        HIPCHK(hipGetLastError());
    }
    if ((r = ctx->prec ? upload_geometry<double>(ctx) : upload_geometry<float>(ctx)) != THY_OK) return r;
    // zero state so that padding columns hold finite values
    for (int k = 0; k < 2; k++) {
        HIPCHK(ctx_fill(ctx, ctx->e[k], b));
        HIPCHK(ctx_fill(ctx, ctx->qx[k], b));
        HIPCHK(ctx_fill(ctx, ctx->qy[k], b));
    }
    HIPCHK(ctx_fill(ctx, ctx->D, b));
    HIPCHK(ctx_fill(ctx, ctx->emax, b));
    Ctrl c = idle_ctrl(ctx);
    for (int s = 0; s < 3; s++) HIPCHK(ctx_copy(ctx, &ctx->ctrl[s], &c, sizeof(c), hipMemcpyHostToDevice));
    if ((r = reset_dt_slots(ctx)) != THY_OK) return r;
    return THY_OK;
}

void thy_destroy(thy_ctx *ctx) {
    RelaxedCapture relaxed;
    if (!ctx) return;
    // no queued work may still use what goes back to the caches
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    drop_graphs(ctx);
    void *ptrs[] = {ctx->state, ctx->row, ctx->fy, ctx->deep_row, ctx->area_d, ctx->ctrl, ctx->dtmin, ctx->scratch_u,
                    ctx->ftime, ctx->gpos, ctx->gbuf, ctx->gtime, ctx->okada_def, ctx->okada_row, ctx->okada_plane, ctx->mass_partial, ctx->outbuf,
                    ctx->steplog, ctx->alone.deep, ctx->alone.items, ctx->batched.deep, ctx->batched.items, ctx->health};
    for (void *q : ptrs)
        dev_free(q);
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 3; j++)
            if (ctx->rev[i][j]) (void)hipEventDestroy(ctx->rev[i][j]);
    Pool::get().host_free(ctx->h_snap);
    Pool::get().host_free(ctx->h_aux);
    Pool::get().host_free(ctx->h_dt);
    if (ctx->stream) Pool::get().put_stream(ctx->stream);
    delete ctx;
}

const char *thy_last_error(const thy_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int thy_upload_state(thy_ctx *ctx, const double *s1, const double *s2) {
    RelaxedCapture relaxed;
    if (!ctx || !s1 || !s2) return THY_ERR_INVALID;
    return ctx->prec ? upload_t<double>(ctx, s1, s2) : upload_t<float>(ctx, s1, s2);
}

int thy_download_state(thy_ctx *ctx, double *s1, double *s2) {
    RelaxedCapture relaxed;
    if (!ctx) return THY_ERR_INVALID;
    return ctx->prec ? download_t<double>(ctx, s1, s2) : download_t<float>(ctx, s1, s2);
}

int thy_init_metrics(thy_ctx *ctx) {
    RelaxedCapture relaxed;
    if (!ctx) return THY_ERR_INVALID;
    return ctx->prec ? init_metrics_t<double>(ctx) : init_metrics_t<float>(ctx);
}

int thy_update_metrics(thy_ctx *ctx, double t) {
    RelaxedCapture relaxed;
    if (!ctx) return THY_ERR_INVALID;
    return ctx->prec ? update_metrics_t<double>(ctx, t) : update_metrics_t<float>(ctx, t);
}

int thy_apply_okada(thy_ctx *ctx, const thy_fault *f, int crop_flag, double crop_value, double *def_out) {
    RelaxedCapture relaxed;
    if (!ctx || !f || crop_flag < 0 || crop_flag > 2) return THY_ERR_INVALID;
    return ctx->prec ? apply_okada_t<double>(ctx, f, crop_flag, crop_value, def_out)
                     : apply_okada_t<float>(ctx, f, crop_flag, crop_value, def_out);
}

int thy_initial_dt(thy_ctx *ctx, double *dt) {
    RelaxedCapture relaxed;
    if (!ctx || !dt) return THY_ERR_INVALID;
    return ctx->prec ? initial_dt_t<double>(ctx, dt) : initial_dt_t<float>(ctx, dt);
}

int thy_autotune(thy_ctx *ctx, int reps, int *strip_rows, int *general_rows, double *ms_best) {
    RelaxedCapture relaxed;
    if (!ctx) return THY_ERR_INVALID;
    if (ctx->kernel == 1) return fail(ctx, THY_ERR_INVALID, "autotune covers the row-sweep kernel");
    if (!ctx->uploaded) return fail(ctx, THY_ERR_INVALID, "autotune needs an uploaded state");
    if (reps <= 0) reps = 5;
    int r;
    // the run's control blocks and dt slots are restored afterwards
    Ctrl saved[3];
    std::vector<unsigned int> saved_dt(3 * kDtSlot);
    HIPCHK(hipStreamSynchronize(ctx->stream));
    HIPCHK(ctx_copy(ctx, saved, ctx->ctrl, sizeof(saved), hipMemcpyDeviceToHost));
    HIPCHK(ctx_copy(ctx, saved_dt.data(), ctx->dtmin, saved_dt.size() * sizeof(unsigned int), hipMemcpyDeviceToHost));
    const int saved_slot = ctx->slot;
    double dt;
    if ((r = thy_initial_dt(ctx, &dt)) != THY_OK) return r;
    Ctrl c = idle_ctrl(ctx);
    c.t = saved[saved_slot].t;
    c.dt = dt;
    c.dt_valid = 1;
    c.cur = ctx->cur;
    // The heights in use, then those of a table of which none is built twice.  On a grid whose
    // default is 8 rows the table's strips are cut to 8: taller ones only leave the device
    // idle there (us a step at 8 / 16 / 24 rows: 131x97 11.8 / 13.2 / 16.3, 500x400 12.4 / 15.2 /
    // 18.4, 1000x800 15.9 / 18.1 / 22.0).  The table's name for the default is then 16.
    struct Pair { int name, strip, tile; };
    const int def = default_strip_rows(segment_rows(ctx), ctx->ncu);
    const bool own = ctx->prm.strip_rows > 0;
    const int table[][2] = {{16, 4}, {16, 8}, {24, 8}, {32, 8}, {36, 8}, {40, 8}, {48, 8}};
    std::vector<Pair> cand = {{!own && ctx->srows == 8 ? 16 : ctx->srows, ctx->srows, ctx->trows}};
    for (const auto &sg : table) {
        const Pair p{sg[0], def <= 8 ? def : sg[0], sg[1]};
        bool known = sg[0] > ctx->ny;
        for (const Pair &q : cand) known = known || (q.strip == p.strip && q.tile == p.tile);
        if (!known) cand.push_back(p);
    }
    Pair best = cand[0];
    double best_ms = 1e30;
    for (const Pair &sg : cand) {
        if ((r = build_alone(ctx, sg.strip, sg.tile)) != THY_OK) return r;
        // kSeq steps captured into one graph and replayed, as a run replays its steps.
        // The launches cycle through the three launch slots as in a run, but publish no
        // control block: every slot holds the same control block, each step reads the
        // same state and redoes the same step, and the run's state stays.
        constexpr int kSeq = 32;  // long enough that the replay launch is a small share
        hipGraph_t g = nullptr;
        hipGraphExec_t ge = nullptr;
        ctx->tuning = 1;
        ctx->slot = 0;
        HIPCHK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        for (int q = 0; q < kSeq; q++) {
            hipError_t e = launch_step(ctx);
            if (e != hipSuccess) {
                ctx->tuning = 0;
                (void)hipStreamEndCapture(ctx->stream, &g);
                if (g) (void)hipGraphDestroy(g);
                return fail(ctx, THY_ERR_HIP, std::string("autotune capture: ") + hipGetErrorString(e));
            }
        }
        ctx->tuning = 0;
        HIPCHK(hipStreamEndCapture(ctx->stream, &g));
        hipError_t ei = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        HIPCHK(ei);
        std::vector<float> t;
        const Ctrl c3[3] = {c, c, c};
        for (int k = 0; k <= reps; k++) {  // the first replay is a warm-up
            hipError_t e = hipSuccess;
            e = ctx_copy(ctx, ctx->ctrl, c3, sizeof(c3), hipMemcpyHostToDevice);
            if (e == hipSuccess) e = hipEventRecord(ctx->ev0, ctx->stream);
            if (e == hipSuccess) e = hipGraphLaunch(ge, ctx->stream);
            if (e == hipSuccess) e = hipEventRecord(ctx->ev1, ctx->stream);
            if (e == hipSuccess) e = hipEventSynchronize(ctx->ev1);
            float ms = 0.f;
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1);
            if (e != hipSuccess) {
                (void)hipGraphExecDestroy(ge);
                return fail(ctx, THY_ERR_HIP, std::string("autotune replay: ") + hipGetErrorString(e));
            }
            if (k > 0) t.push_back(ms / kSeq);
        }
        (void)hipGraphExecDestroy(ge);
        std::sort(t.begin(), t.end());
        const double med = t[t.size() / 2];
        if (med < best_ms) {
            best_ms = med;
            best = sg;
        }
    }
    if ((r = build_alone(ctx, best.strip, best.tile)) != THY_OK) return r;
    ctx->tuned_srows = best.strip;
    ctx->tuned_trows = best.tile;
    ctx->slot = saved_slot;
    HIPCHK(ctx_copy(ctx, ctx->ctrl, saved, sizeof(saved), hipMemcpyHostToDevice));
    HIPCHK(ctx_copy(ctx, ctx->dtmin, saved_dt.data(), saved_dt.size() * sizeof(unsigned int), hipMemcpyHostToDevice));
    if (strip_rows) *strip_rows = best.name;
    if (general_rows) *general_rows = best.tile;
    if (ms_best) *ms_best = best_ms;
    return THY_OK;
}

int thy_step(thy_ctx *ctx, double dt, double *dt_next) {
    RelaxedCapture relaxed;
    if (!ctx) return THY_ERR_INVALID;
    int r;
    if ((r = need_lists(ctx)) != THY_OK) return r;
    Ctrl c = idle_ctrl(ctx);
    c.dt = dt;
    c.dt_valid = 1;
    c.cur = ctx->cur;
    if ((r = write_ctrl(ctx, c)) != THY_OK) return r;
    const int s = ctx->slot;
    if ((r = clear_dt_slots(ctx, s)) != THY_OK) return r;
    hipError_t e = launch_step(ctx);
    if (e != hipSuccess) return fail(ctx, THY_ERR_HIP, std::string("step launch: ") + hipGetErrorString(e));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    Ctrl o;
    HIPCHK(ctx_copy(ctx, &o, &ctx->ctrl[ctx->slot], sizeof(Ctrl), hipMemcpyDeviceToHost));
    ctx->cur = o.cur;
    unsigned int bad = 0;
    HIPCHK(ctx_copy(ctx, &bad, ctx->health, sizeof(bad), hipMemcpyDeviceToHost));
    if (bad) return fail(ctx, THY_ERR_NONFINITE, "the step produced a non-finite eta, qx or qy");
    if (dt_next) {
        unsigned int v;
        if ((r = read_dt_slot(ctx, s, v)) != THY_OK) return r;
        float f;
        memcpy(&f, &v, 4);
        *dt_next = (double)f;
    }
    return THY_OK;
}

int thy_get_field(thy_ctx *ctx, int field, float *out) {
    RelaxedCapture relaxed;
    if (!ctx || !out || field < 0 || field > 5) return THY_ERR_INVALID;
    return ctx->prec ? get_field_t<double>(ctx, field, out) : get_field_t<float>(ctx, field, out);
}

int thy_mass(thy_ctx *ctx, double *mass) {
    RelaxedCapture relaxed;
    if (!ctx || !mass) return THY_ERR_INVALID;
    std::vector<double> host(kMassBlocks);
    return ctx->prec ? mass_t<double>(ctx, ctx->mass_partial, host.data(), mass)
                     : mass_t<float>(ctx, ctx->mass_partial, host.data(), mass);
}

int thy_mass_noalloc(thy_ctx *ctx, double *mass) {
    RelaxedCapture relaxed;
    if (!ctx || !mass) return THY_ERR_INVALID;
    if (ctx->device < 0 || ctx->device >= kScratchDevices || !g_scratch_ptr[ctx->device])
        return fail(ctx, THY_ERR_INVALID, "the allocation-free scratch of this device was not set up");
    double host[kScratchPartials];  // on the stack: no allocation on the host either
    return ctx->prec ? mass_t<double>(ctx, g_scratch_ptr[ctx->device], host, mass)
                     : mass_t<float>(ctx, g_scratch_ptr[ctx->device], host, mass);
}

int thy_last_timing(thy_ctx *ctx, double *ms) {
    if (!ctx || !ms) return THY_ERR_INVALID;
    *ms = ctx->last_ms;
    return THY_OK;
}

static int collect_gauges(thy_ctx *ctx);

int thy_get_gauges(thy_ctx *ctx, float *time, float *eta, float *u, float *v, float *eta_min, float *eta_max,
                   float *bathy) {
    RelaxedCapture relaxed;
    if (!ctx) return THY_ERR_INVALID;
    if (ctx->gauges_stale) {
        const int r = collect_gauges(ctx);
        if (r != THY_OK) return r;
        ctx->gauges_stale = false;
    }
    const int ns = ctx->nsamples, ng = ctx->ng;
    if (time) std::copy(ctx->g_time.begin(), ctx->g_time.begin() + ns, time);
    if (eta) std::copy(ctx->g_eta.begin(), ctx->g_eta.begin() + (size_t)ns * ng, eta);
    if (u) std::copy(ctx->g_u.begin(), ctx->g_u.begin() + (size_t)ns * ng, u);
    if (v) std::copy(ctx->g_v.begin(), ctx->g_v.begin() + (size_t)ns * ng, v);
    std::vector<int> pos(ng);
    if (ng) HIPCHK(ctx_copy(ctx, pos.data(), ctx->gpos, ng * sizeof(int), hipMemcpyDeviceToHost));
    if (eta_min || eta_max) {
        for (int g = 0; g < ng; g++) {
            float mn = 1e30f, mx = -1e30f;
            if (pos[g] < 0) mn = mx = -9999.0f;
            else
                for (int s = 0; s < ns; s++) {
                    float x = ctx->g_eta[(size_t)s * ng + g];
                    mn = std::min(x, mn);
                    mx = std::max(x, mx);
                }
            if (eta_min) eta_min[g] = mn;
            if (eta_max) eta_max[g] = mx;
        }
    }
    if (bathy && ng) {
        std::vector<float> field((size_t)ctx->nx * ctx->ny);
        int r = thy_get_field(ctx, THY_DEFORMED_BATHY, field.data());
        if (r != THY_OK) return r;
        for (int g = 0; g < ng; g++) bathy[g] = pos[g] < 0 ? -9999.0f : field[pos[g]];
    }
    return THY_OK;
}

// deliver finished iterations [ctx->logged, upto) to the on_step callback
static int drain_log(thy_ctx *ctx, int64_t upto) {
    if (!ctx->on_step || upto <= ctx->logged) {
        if (upto > ctx->logged) ctx->logged = upto;
        return THY_OK;
    }
    std::vector<double> buf((size_t)ctx->logcap * 2);
    HIPCHK(ctx_copy(ctx, buf.data(), ctx->steplog, buf.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int64_t it = std::max(ctx->logged, upto - ctx->logcap); it < upto; it++) {
        const int64_t li = it % ctx->logcap;
        ctx->on_step(ctx->user, it + 1, buf[2 * li], buf[2 * li + 1]);
    }
    ctx->logged = upto;
    return THY_OK;
}


static int run_loop(thy_ctx *ctx, thy_run_result *res) {
    int r;
    double total_ms = 0.0;
    for (;;) {
        Ctrl s;
        double ms = 0.0;
        if ((r = advance(ctx, ctx->K, &s, &ms)) != THY_OK) return r;
        total_ms += ms;
        // after a stop every finished iteration has its log entry; otherwise the last
        // one is completed by the next launch
        if ((r = drain_log(ctx, s.dt_valid ? s.steps : s.steps - 1)) != THY_OK) return r;
        if (s.nonfinite)
            return fail(ctx, THY_ERR_NONFINITE,
                        "non-finite eta, qx or qy after step " + std::to_string((long long)s.steps));
        if (!(s.t < s.t_end) || (s.max_steps > 0 && s.steps >= s.max_steps)) {
            res->steps = s.steps;
            res->t_final = s.t;
            ctx->nsamples = std::min(s.nsamples, ctx->gcap);
            res->n_samples = ctx->nsamples;
            break;
        }
        bool changed = false;
        // src/GPU/ShallowWater.cu:125-147: apply every fault whose time has come
        while (s.k < s.nf && s.t * s.T >= ctx->ftimes[s.k]) {
            if (ctx->on_okada) ctx->on_okada(ctx->user, s.k);
            if ((r = thy_apply_okada(ctx, &ctx->faults[s.k], ctx->crop_flag, ctx->crop_value, nullptr)) != THY_OK)
                return r;
            s.k++;
            changed = true;
        }
        // src/GPU/ShallowWater.cu:404-409: snapshot, at most one per iteration
        if (!s.snap_done && s.t >= ctx->next_save) {
            ctx->next_save += ctx->save_interval;
            s.next_save = ctx->next_save;
            s.snap_done = 1;
            if (ctx->on_snapshot) ctx->on_snapshot(ctx->user, ctx->nsnap, s.t, ctx);
            ctx->nsnap++;
            changed = true;
        }
        if (!changed) return fail(ctx, THY_ERR_INVALID, "driver stalled");
        if ((r = write_ctrl(ctx, s)) != THY_OK) return r;
    }
    res->n_snapshots = ctx->nsnap;
    res->seconds = total_ms * 1e-3;
    ctx->last_ms = total_ms;
    ctx->gauges_stale = true;  // copied to the host when thy_get_gauges asks for them
    return THY_OK;
}

// gauge samples of the finished run into host memory (read by thy_get_gauges)
static int collect_gauges(thy_ctx *ctx) {
    const int ns = ctx->nsamples, ng = ctx->ng;
    ctx->g_time.assign(ns, 0.f);
    ctx->g_eta.assign((size_t)ns * ng, 0.f);
    ctx->g_u.assign((size_t)ns * ng, 0.f);
    ctx->g_v.assign((size_t)ns * ng, 0.f);
    if (ns > 0 && ng > 0) {
        std::vector<float> buf((size_t)ns * ng * 3);
        HIPCHK(ctx_copy(ctx, buf.data(), ctx->gbuf, buf.size() * sizeof(float), hipMemcpyDeviceToHost));
        HIPCHK(ctx_copy(ctx, ctx->g_time.data(), ctx->gtime, ns * sizeof(float), hipMemcpyDeviceToHost));
        for (size_t i = 0; i < (size_t)ns * ng; i++) {
            ctx->g_eta[i] = buf[3 * i];
            ctx->g_u[i] = buf[3 * i + 1];
            ctx->g_v[i] = buf[3 * i + 2];
        }
    }
    return THY_OK;
}

// Everything thy_run does before its first step launch: schedule, gauge buffers,
// metrics, initial dt and truncation, control block in launch slot 0.
static int prepare_run(thy_ctx *ctx, const thy_run_config *cfg, thy_run_result *res) {
    if (cfg->n_faults < 0 || (cfg->n_faults > 0 && !cfg->faults) || (cfg->n_gauges > 0 && !cfg->gauge_pos))
        return fail(ctx, THY_ERR_INVALID, "bad run configuration");
    int r;
    if ((r = need_lists(ctx)) != THY_OK) return r;
    memset(res, 0, sizeof(*res));
    ctx->batch_ready = false;  // a run prepared before is replaced
    ctx->K = cfg->steps_per_sync > 0 ? cfg->steps_per_sync : 24;
    ctx->faults.assign(cfg->faults, cfg->faults + cfg->n_faults);
    ctx->ftimes.assign(std::max(1, cfg->n_faults), 0.0);
    for (int k = 0; k < cfg->n_faults; k++) ctx->ftimes[k] = cfg->faults[k].time;
    ctx->crop_flag = cfg->crop_flag;
    ctx->crop_value = cfg->crop_value;
    ctx->save_interval = cfg->save_interval;
    ctx->on_snapshot = cfg->on_snapshot;
    ctx->on_okada = cfg->on_okada;
    ctx->on_step = cfg->on_step;
    ctx->user = cfg->user;
    ctx->nsnap = 0;
    ctx->logged = 0;
    const std::vector<double> &ft = ctx->ftimes;
    if (ctx->ftime) { dev_free(ctx->ftime); ctx->ftime = nullptr; }
    HIPCHK(dev_alloc((void **)&ctx->ftime, ft.size() * sizeof(double)));
    HIPCHK(ctx_copy(ctx, ctx->ftime, ft.data(), ft.size() * sizeof(double), hipMemcpyHostToDevice));
    // gauges
    if (ctx->gpos) { dev_free(ctx->gpos); ctx->gpos = nullptr; }
    if (ctx->gbuf) { dev_free(ctx->gbuf); ctx->gbuf = nullptr; }
    if (ctx->gtime) { dev_free(ctx->gtime); ctx->gtime = nullptr; }
    ctx->ng = cfg->n_gauges;
    ctx->gcap = 0;
    if (cfg->n_gauges > 0 && cfg->series_interval >= 0.0) {
        double nsd = cfg->series_interval > 0.0 ? cfg->t_end / cfg->series_interval + 4.0 : 1e6;
        if (cfg->max_steps > 0 && cfg->series_interval <= 0.0) nsd = (double)cfg->max_steps + 2.0;
        if (nsd > 0.0) ctx->gcap = (int)std::min(nsd, 1e6);  // (a run that ends before its start has none)
    }
    HIPCHK(dev_alloc((void **)&ctx->gpos, std::max(1, ctx->ng) * sizeof(int)));
    if (ctx->ng) HIPCHK(ctx_copy(ctx, ctx->gpos, cfg->gauge_pos, ctx->ng * sizeof(int), hipMemcpyHostToDevice));
    HIPCHK(dev_alloc((void **)&ctx->gbuf, std::max<size_t>(1, (size_t)ctx->gcap * ctx->ng * 3) * sizeof(float)));
    HIPCHK(dev_alloc((void **)&ctx->gtime, std::max(1, ctx->gcap) * sizeof(float)));
    drop_graphs(ctx);

    HIPCHK(ctx_fill(ctx, ctx->health, sizeof(unsigned int)));
    // src/GPU/ShallowWater.cu:305-309: metrics from the pre-deformation state
    if ((r = thy_init_metrics(ctx)) != THY_OK) return r;
    // src/GPU/ShallowWater.cu:378-391: initial dt (pre-deformation) and truncation
    double dt0;
    if ((r = thy_initial_dt(ctx, &dt0)) != THY_OK) return r;
    res->dt_initial = dt0;
    Ctrl c = idle_ctrl(ctx);
    c.t = 0.0;
    c.t_end = cfg->t_end;
    c.max_steps = cfg->max_steps;
    c.nf = cfg->n_faults;
    c.k = 0;
    c.T = ctx->prm.T;
    c.next_save = cfg->save_interval >= 0.0 ? 0.0 : INFINITY;
    c.next_series = (cfg->series_interval >= 0.0 && ctx->ng > 0) ? 0.0 : INFINITY;
    c.series_dt = cfg->series_interval;
    c.gcap = ctx->gcap;
    ctx->next_save = c.next_save;
    double dt = dt0;
    int skip = 0;
    if (cfg->n_faults > 0) {
        // the skipping variant when the first fault is at t = 0 (src/GPU/ShallowWater.cu:382-391)
        if (ft[0] < 2.220446049250313e-16) trunc_skipping(c, ft.data(), 0.0, dt, skip);
        else trunc_plain(c, ft.data(), 0.0, dt, skip);
    }
    c.dt = dt;
    c.dt_valid = 1;
    c.skip = skip;
    c.cur = ctx->cur;
    if ((r = reset_dt_slots(ctx)) != THY_OK) return r;
    ctx->slot = 0;  // the next launch reads slot 0 (the dt slots were all reset)
    if ((r = write_ctrl(ctx, c)) != THY_OK) return r;
    ctx->run_active = true;
    return THY_OK;
}

int thy_run(thy_ctx *ctx, const thy_run_config *cfg, thy_run_result *res) {
    RelaxedCapture relaxed;
    if (!ctx || !cfg || !res) return THY_ERR_INVALID;
    int r;
    if ((r = prepare_run(ctx, cfg, res)) != THY_OK) return r;
    double dti = res->dt_initial;
    r = run_loop(ctx, res);
    res->dt_initial = dti;
    return r;
}

int thy_run_more(thy_ctx *ctx, int64_t n_steps, thy_run_result *res) {
    RelaxedCapture relaxed;
    if (!ctx || !res || n_steps < 0) return THY_ERR_INVALID;
    if (!ctx->run_active) return fail(ctx, THY_ERR_INVALID, "thy_run_more without a previous thy_run");
    int r;
    memset(res, 0, sizeof(*res));
    Ctrl c;
    if ((r = read_ctrl(ctx, &c)) != THY_OK) return r;
    c.max_steps = c.steps + n_steps;
    if ((r = write_ctrl(ctx, c)) != THY_OK) return r;
    return run_loop(ctx, res);
}

}  // extern "C"

// ===========================================================================
// Batched scenarios: many contexts advanced together, one launch per step, captured once
// for K steps.
// ===========================================================================
struct thy_batch {
    int capacity = 0;
    size_t budget = 0, used = 0;
    int K = 24;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipEvent_t ev_done = nullptr;   // end of a launch's work (admissions queue copies after it)
    std::vector<thy_ctx *> ctx;     // per slot; nullptr when free
    std::vector<size_t> bytes;      // admitted footprint per slot
    std::vector<int> srows;         // strip height of the context's own lists at admission
    std::vector<int> state;         // THY_SLOT_*
    std::vector<thy_run_result> res;
    StepArgs<float> *d_args = nullptr;
    BatchItem *d_items = nullptr;   // a workgroup's work each; the captured grid covers item_cap
    int *d_count = nullptr;         // items in the list
    int item_cap = 0;
    std::vector<BatchItem> h_items, h_back;  // of even and of odd steps: the halves of d_items
    int h_count = 0;
    Ctrl *d_ctrl = nullptr;
    Ctrl *h_ctrl = nullptr;              // pinned: control blocks gathered after a launch
    StepArgs<float> *h_args = nullptr;   // pinned: argument blocks of admitted scenarios
    hipGraphExec_t gexec = nullptr;
    bool dirty = true;
    bool in_flight = false;              // a launch is queued and not yet collected
    std::vector<char> launched;          // per slot: running when the launch was queued
    int launched_hi = 0;
    double gpu_ms = 0.0;
    std::string err;
};

namespace {

int bfail(thy_batch *b, int code, const std::string &msg) {
    b->err = msg;
    return code;
}

#define BHIPCHK(x)                                                                                        \
    do {                                                                                                 \
        hipError_t e_ = (x);                                                                             \
        if (e_ != hipSuccess)                                                                            \
            return bfail(b, e_ == hipErrorOutOfMemory ? THY_ERR_DEVICE_MEMORY : THY_ERR_HIP,             \
                         std::string(#x) + ": " + hipGetErrorString(e_));                                \
    } while (0)

// capacity of an item list: a power of two, at least 256 items
int list_cap(size_t n) {
    int c = 256;
    while ((size_t)c < n) c <<= 1;
    return c;
}

// The workgroups of the running scenarios: the general tiles of all, costliest first, spread
// among the deep-water strips, scenario by scenario, four to a workgroup in the scenario's own
// order (its runs per XCD: each scenario starts at a multiple of 8).  A scenario's writer is
// its first item.  The second half of the list, for every other step, has the strips in
// reverse where the states together exceed the cache (as in launch_step_t).  24 scenarios of
// 1000x800, GPU time: 97.2 ms with the tiles first, 89.3 spread, 88.0 with every other step
// reversed, 86.3 with strips of 24 rows too; a mix of 12 grids 85.9, 78.7, 76.9, 75.8.
int batch_items(thy_batch *b) {
    struct G { int cls; BatchItem it; };
    std::vector<G> gv;
    b->h_items.clear();
    for (int i = 0; i < b->capacity; i++) {
        if (b->state[i] != THY_SLOT_RUNNING) continue;
        const thy_ctx *c = b->ctx[i];
        // a context that was tuned after its admission is refused: its own launches replayed
        // steps on the buffers and control blocks that the batch advances
        if (c->srows != b->srows[i]) return bfail(b, THY_ERR_INVALID, "strip height changed after admission");
        const WorkLists &w = c->batched;
        for (size_t p = 0; p < w.tile_h.size(); p++)
            gv.push_back({w.tcost_h[p], BatchItem{i, p == 0 ? 1 : 0, w.tile_h[p]}});
    }
    std::stable_sort(gv.begin(), gv.end(), [](const G &x, const G &y) { return x.cls > y.cls; });
    std::vector<BatchItem> strips;
    size_t bytes = 0;
    for (int i = 0; i < b->capacity; i++) {
        if (b->state[i] != THY_SLOT_RUNNING) continue;
        const WorkLists &w = b->ctx[i]->batched;
        for (int p = 0; p < w.n_deep; p += SW_WAVES)
            strips.push_back(BatchItem{i, (p == 0 && w.tile_h.empty()) ? 1 : 0, make_int2(p, 0)});
        while (strips.size() % 8) strips.push_back(BatchItem{-1, 0, make_int2(0, 0)});
        bytes += b->ctx[i]->state_bytes;
    }
    auto fill = [&](std::vector<BatchItem> &out, const bool back) {
        const int last = (int)strips.size() / 8 - 1;
        out.clear();
        spread_items(gv.size(), strips.size(), 2.0, [&](const bool tile, const int i) {
            if (i < 0) out.push_back(BatchItem{-1, 0, make_int2(0, 0)});
            else out.push_back(tile ? gv[i].it : strips[back ? (last - i / 8) * 8 + i % 8 : i]);
        });
    };
    fill(b->h_items, false);
    fill(b->h_back, bytes > kCacheBytes);
    const int cap = list_cap(b->h_items.size());
    if (cap != b->item_cap) {
        // the captured launches hold the old list and grid size
        if (b->gexec) {
            (void)hipGraphExecDestroy(b->gexec);
            b->gexec = nullptr;
        }
        dev_free(b->d_items);
        b->d_items = nullptr;
        b->item_cap = 0;
        BHIPCHK(dev_alloc(&b->d_items, 2 * (size_t)cap * sizeof(BatchItem)));
        b->item_cap = cap;
    }
    b->h_count = (int)b->h_items.size();
    // ordered before the next launch on the batch stream; the host list lives in b
    if (!b->h_items.empty()) {
        BHIPCHK(hipMemcpyAsync(b->d_items, b->h_items.data(), b->h_items.size() * sizeof(BatchItem), hipMemcpyHostToDevice,
                               b->stream));
        BHIPCHK(hipMemcpyAsync(b->d_items + b->item_cap, b->h_back.data(), b->h_back.size() * sizeof(BatchItem),
                               hipMemcpyHostToDevice, b->stream));
    }
    BHIPCHK(hipMemcpyAsync(b->d_count, &b->h_count, sizeof(int), hipMemcpyHostToDevice, b->stream));
    BHIPCHK(hipStreamSynchronize(b->stream));
    b->dirty = false;
    return THY_OK;
}

// K steps (launch slots 0, 1, 2, ...), captured once, one launch each
int batch_graph(thy_batch *b) {
    if (b->gexec) return THY_OK;
    BatchArgs q;
    q.args = b->d_args;
    q.n_items = b->d_count;
    hipGraph_t g;
    BHIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < b->K; k++) {
        q.items = b->d_items + (k % 2) * b->item_cap;
        hipLaunchKernelGGL(k_batch, dim3(b->item_cap), dim3(64 * SW_WAVES), 0, b->stream, q, k % 3);
    }
    BHIPCHK(hipStreamEndCapture(b->stream, &g));
    BHIPCHK(hipGraphInstantiate(&b->gexec, g, nullptr, nullptr, 0));
    (void)hipGraphDestroy(g);
    return THY_OK;
}

// apply every fault of a scenario whose time has come; Ctrl c is its control block
// faults that came due at the control block's time: Okada, then the control block
// rewritten into launch slot 0; errors are the context's
int ctx_faults(thy_ctx *ctx, Ctrl &cb, bool &changed) {
    changed = false;
    while (cb.k < cb.nf && cb.t * cb.T >= ctx->ftimes[cb.k]) {
        const int r = thy_apply_okada(ctx, &ctx->faults[cb.k], ctx->crop_flag, ctx->crop_value, nullptr);
        if (r != THY_OK) return fail(ctx, r, std::string("okada: ") + thy_last_error(ctx));
        cb.k++;
        changed = true;
    }
    if (changed) {
        HIPCHK(hipStreamSynchronize(ctx->stream));
        ctx->slot = 0;
        return write_ctrl(ctx, cb);
    }
    return THY_OK;
}

int batch_faults(thy_batch *b, thy_ctx *c, Ctrl &cb, bool &changed) {
    const int r = ctx_faults(c, cb, changed);
    return r == THY_OK ? r : bfail(b, r, thy_last_error(c));
}

// the context-local part of admission: run configuration, metrics, initial dt, faults
// due at t = 0 (src/GPU/ShallowWater.cu:305-391)
int prepare_for_batch(thy_ctx *ctx, const thy_run_config *cfg, thy_run_result &res) {
    if (ctx->prec != 0 || ctx->kernel == 1)
        return fail(ctx, THY_ERR_INVALID, "batched scenarios run the FP32 row-sweep kernel only");
    if (cfg->save_interval >= 0.0) return fail(ctx, THY_ERR_INVALID, "batched scenarios take no snapshots");
    if (!ctx->uploaded) return fail(ctx, THY_ERR_INVALID, "scenario state not uploaded");
    int r;
    if (ctx->batched.n_items == 0 && (r = build_batched(ctx)) != THY_OK) return r;
    if ((r = prepare_run(ctx, cfg, &res)) != THY_OK) return r;
    Ctrl cb;
    if ((r = read_ctrl(ctx, &cb)) != THY_OK) return r;
    bool changed;
    return ctx_faults(ctx, cb, changed);
}

}  // namespace

extern "C" {

int thy_batch_create(int capacity, size_t hbm_budget, int steps_per_sync, thy_batch **out) {
    RelaxedCapture relaxed;
    if (!out || capacity < 1 || capacity > 65536) return THY_ERR_INVALID;
    thy_batch *b = new (std::nothrow) thy_batch();
    if (!b) return THY_ERR_HOST_MEMORY;
    *out = b;
    b->capacity = capacity;
    b->budget = hbm_budget;
    b->K = steps_per_sync > 0 ? ((steps_per_sync + 2) / 3) * 3 : 24;
    b->ctx.assign(capacity, nullptr);
    b->bytes.assign(capacity, 0);
    b->srows.assign(capacity, 0);
    b->state.assign(capacity, THY_SLOT_FREE);
    b->res.assign(capacity, thy_run_result{});
    b->launched.assign(capacity, 0);
    // (a cached stream: creating and destroying streams with every batch would shift how
    // the runtime spreads streams over the hardware queues)
    BHIPCHK(Pool::get().get_stream(b->stream));
    BHIPCHK(hipEventCreate(&b->ev0));
    BHIPCHK(hipEventCreate(&b->ev1));
    BHIPCHK(hipEventCreateWithFlags(&b->ev_done, hipEventDisableTiming));
    BHIPCHK(dev_alloc(&b->d_args, (size_t)capacity * sizeof(StepArgs<float>)));
    BHIPCHK(hipMemsetAsync(b->d_args, 0, (size_t)capacity * sizeof(StepArgs<float>), b->stream));
    BHIPCHK(dev_alloc(&b->d_count, sizeof(int)));
    BHIPCHK(hipMemsetAsync(b->d_count, 0, sizeof(int), b->stream));
    BHIPCHK(dev_alloc(&b->d_ctrl, (size_t)capacity * sizeof(Ctrl)));
    BHIPCHK(Pool::get().host_alloc((void **)&b->h_ctrl, (size_t)capacity * sizeof(Ctrl)));
    BHIPCHK(Pool::get().host_alloc((void **)&b->h_args, (size_t)capacity * sizeof(StepArgs<float>)));
    return THY_OK;
}

void thy_batch_destroy(thy_batch *b) {
    RelaxedCapture relaxed;
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    Pool::get().host_free(b->h_ctrl);
    Pool::get().host_free(b->h_args);
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    void *ptrs[] = {b->d_args, b->d_items, b->d_count, b->d_ctrl};
    for (void *p : ptrs)
        dev_free(p);
    hipEvent_t evs[] = {b->ev0, b->ev1, b->ev_done};
    for (hipEvent_t e : evs)
        if (e) (void)hipEventDestroy(e);
    if (b->stream) Pool::get().put_stream(b->stream);
    delete b;
}

const char *thy_batch_last_error(thy_batch *b) { return b ? b->err.c_str() : "null batch"; }

int thy_batch_prepare(thy_ctx *ctx, const thy_run_config *cfg) {
    RelaxedCapture relaxed;
    if (!ctx || !cfg) return THY_ERR_INVALID;
    ctx->batch_ready = false;
    const int r = prepare_for_batch(ctx, cfg, ctx->prep_res);
    if (r == THY_OK) ctx->batch_ready = true;
    return r;
}

int thy_batch_add(thy_batch *b, thy_ctx *ctx, const thy_run_config *cfg, int *slot_out) {
    RelaxedCapture relaxed;
    if (!b || !ctx || !slot_out) return THY_ERR_INVALID;
    if (!cfg && !ctx->batch_ready) return bfail(b, THY_ERR_INVALID, "context not prepared (thy_batch_prepare)");
    for (int i = 0; i < b->capacity; i++)
        if (b->ctx[i] == ctx && b->state[i] != THY_SLOT_FREE) return bfail(b, THY_ERR_INVALID, "context already admitted");
    int slot = -1;
    for (int i = 0; i < b->capacity && slot < 0; i++)
        if (b->state[i] == THY_SLOT_FREE) slot = i;
    if (slot < 0) return bfail(b, THY_ERR_BUDGET, "no free scenario slot");
    const size_t need = thy_footprint(ctx->nx, ctx->ny, &ctx->prm);
    if (b->budget > 0 && b->used + need > b->budget) return bfail(b, THY_ERR_BUDGET, "HBM budget exceeded");
    thy_run_result res;
    if (cfg) {
        const int r = prepare_for_batch(ctx, cfg, res);
        if (r != THY_OK) return bfail(b, r, thy_last_error(ctx));
    } else {
        res = ctx->prep_res;
    }
    ctx->batch_ready = false;
    ctx->ctrl_h_valid = false;  // the batch's launches advance its control blocks
    const StepArgs<float> a = make_args<float>(ctx, true);
    // ordered after a launch in flight, which does not read this free slot
    b->h_args[slot] = a;
    BHIPCHK(hipMemcpyAsync(b->d_args + slot, b->h_args + slot, sizeof(a), hipMemcpyHostToDevice, b->stream));
    b->ctx[slot] = ctx;
    b->srows[slot] = ctx->srows;
    b->bytes[slot] = need;
    b->used += need;
    b->state[slot] = THY_SLOT_RUNNING;
    b->launched[slot] = 0;  // not in a launch in flight: it joins the next one
    b->res[slot] = res;
    b->dirty = true;
    *slot_out = slot;
    return THY_OK;
}

int thy_batch_launch(thy_batch *b) {
    RelaxedCapture relaxed;
    if (!b) return THY_ERR_INVALID;
    if (b->in_flight) return bfail(b, THY_ERR_INVALID, "a launch is in flight");
    int r;
    if (b->dirty && (r = batch_items(b)) != THY_OK) return r;
    int hi = 0;
    for (int i = 0; i < b->capacity; i++) {
        b->launched[i] = b->state[i] == THY_SLOT_RUNNING;
        if (b->launched[i]) hi = i + 1;
    }
    if (hi == 0) return THY_OK;
    if ((r = batch_graph(b)) != THY_OK) return r;
    BHIPCHK(hipEventRecord(b->ev0, b->stream));
    BHIPCHK(hipGraphLaunch(b->gexec, b->stream));
    BHIPCHK(hipEventRecord(b->ev1, b->stream));
    // K is a multiple of 3: the next launch reads slot 0 again
    hipLaunchKernelGGL(k_gather_ctrl, dim3((hi + 63) / 64), dim3(64), 0, b->stream, b->d_args, hi, 0, b->d_ctrl);
    BHIPCHK(hipGetLastError());
    BHIPCHK(hipMemcpyAsync(b->h_ctrl, b->d_ctrl, (size_t)hi * sizeof(Ctrl), hipMemcpyDeviceToHost, b->stream));
    BHIPCHK(hipEventRecord(b->ev_done, b->stream));
    b->launched_hi = hi;
    b->in_flight = true;
    return THY_OK;
}

int thy_batch_ready(thy_batch *b, int *done) {
    RelaxedCapture relaxed;
    if (!b || !done) return THY_ERR_INVALID;
    if (!b->in_flight) {
        *done = 1;
        return THY_OK;
    }
    // the launch's own work: copies that admissions queued after it do not count
    const hipError_t e = hipEventQuery(b->ev_done);
    if (e != hipSuccess && e != hipErrorNotReady) BHIPCHK(e);
    *done = e == hipSuccess ? 1 : 0;
    return THY_OK;
}

int thy_batch_wait(thy_batch *b, int *n_running) {
    RelaxedCapture relaxed;
    if (!b) return THY_ERR_INVALID;
    int r;
    if (b->in_flight) {
        b->in_flight = false;
        BHIPCHK(hipStreamSynchronize(b->stream));
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, b->ev0, b->ev1);
        b->gpu_ms += ms;
        for (int i = 0; i < b->launched_hi; i++) {
            if (!b->launched[i] || b->state[i] != THY_SLOT_RUNNING) continue;
            thy_ctx *c = b->ctx[i];
            Ctrl cb = b->h_ctrl[i];
            c->cur = cb.cur;
            b->res[i].steps = cb.steps;  // progress, final once it has finished
            b->res[i].t_final = cb.t;
            if (!cb.dt_valid) continue;  // stepped through the whole sequence
            if (cb.nonfinite) {
                // the health check stopped it: retired as failed, the batch goes on
                c->err = "non-finite eta, qx or qy after step " + std::to_string((long long)cb.steps);
                b->state[i] = THY_SLOT_FAILED;
                b->dirty = true;
                BHIPCHK(hipMemsetAsync(b->d_args + i, 0, sizeof(StepArgs<float>), b->stream));
                continue;
            }
            // stopped: finished, or a fault is due (the only other stop a batched run has)
            if (!(cb.t < cb.t_end) || (cb.max_steps > 0 && cb.steps >= cb.max_steps)) {
                c->nsamples = std::min(cb.nsamples, c->gcap);
                c->gauges_stale = true;  // read by thy_get_gauges, on the caller's thread
                thy_run_result &res = b->res[i];
                res.steps = cb.steps;
                res.t_final = cb.t;
                res.n_samples = c->nsamples;
                b->state[i] = THY_SLOT_FINISHED;
                b->dirty = true;
                // no later launch or gather reads a finished scenario
                BHIPCHK(hipMemsetAsync(b->d_args + i, 0, sizeof(StepArgs<float>), b->stream));
                continue;
            }
            bool changed;
            if ((r = batch_faults(b, c, cb, changed)) != THY_OK) return r;
            if (!changed) return bfail(b, THY_ERR_INVALID, "batched scenario stalled");
        }
        BHIPCHK(hipStreamSynchronize(b->stream));
    }
    if (n_running) {
        int running = 0;
        for (int i = 0; i < b->capacity; i++) running += b->state[i] == THY_SLOT_RUNNING;
        *n_running = running;
    }
    return THY_OK;
}

int thy_batch_advance(thy_batch *b, int *n_running) {
    RelaxedCapture relaxed;
    int r = thy_batch_launch(b);
    if (r != THY_OK) return r;
    return thy_batch_wait(b, n_running);
}

int thy_batch_status(thy_batch *b, int slot, int *state, thy_run_result *res) {
    if (!b || slot < 0 || slot >= b->capacity) return THY_ERR_INVALID;
    if (state) *state = b->state[slot];
    if (res) *res = b->res[slot];
    return THY_OK;
}

int thy_batch_remove(thy_batch *b, int slot) {
    RelaxedCapture relaxed;
    if (!b || slot < 0 || slot >= b->capacity || b->state[slot] == THY_SLOT_FREE) return THY_ERR_INVALID;
    if (b->state[slot] == THY_SLOT_RUNNING) {
        // a launch in flight may be stepping it: wait, and take it out of every later one
        BHIPCHK(hipStreamSynchronize(b->stream));
        BHIPCHK(hipMemsetAsync(b->d_args + slot, 0, sizeof(StepArgs<float>), b->stream));
    }
    // a finished slot's argument block was cleared when it finished; a launch in flight
    // (already waited for) must not be collected for this slot, nor for a scenario
    // admitted to it later
    b->launched[slot] = 0;
    b->ctx[slot]->run_active = false;
    b->used -= b->bytes[slot];
    b->bytes[slot] = 0;
    b->ctx[slot] = nullptr;
    b->state[slot] = THY_SLOT_FREE;
    b->dirty = true;
    return THY_OK;
}

void thy_release_cached(void) {
    RelaxedCapture relaxed;
    Pool::get().trim();
}

int thy_batch_info(thy_batch *b, int *running, size_t *bytes_used, double *gpu_seconds) {
    if (!b) return THY_ERR_INVALID;
    int n = 0;
    for (int i = 0; i < b->capacity; i++) n += b->state[i] == THY_SLOT_RUNNING;
    if (running) *running = n;
    if (bytes_used) *bytes_used = b->used;
    if (gpu_seconds) *gpu_seconds = b->gpu_ms * 1e-3;
    return THY_OK;
}

}  // extern "C"
