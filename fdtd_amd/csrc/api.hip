// api.hip -- the C ABI declared in include/fdtd.h.
//
// Replaces the reference's host orchestration, marchingLoop
// (fdtdrav.h:3425-4387), and its per-step driver, solver (fdtdrav.h:3188-3422),
// for one device: the z-slab split and ghost-plane copies of the reference
// collapse into a single domain whose neighbour planes are plain HBM reads.
// All work goes to one non-blocking stream, with no host synchronisation
// between steps: a step is the E sweep then the H sweep, a launch each; one pass
// over large FP32 grids; and small grids run many steps in one launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/fdtd.h"
#include "internal.h"

namespace fdtd {
hipError_t launch_half_step(bool efield, int storage, int mode, const KArgs &a, int m, hipStream_t s);
hipError_t launch_adj(bool efield, int mode, int euni, int huni, const KArgs &a, const AArgs &b, int m, int fstep,
                      int sten, hipStream_t s);
hipError_t launch_snap(int storage, const KArgs &a, float *hist, int slot, hipStream_t s);
bool adj_stores_quantities(int nx);
void adj_fuse_tiles(const KArgs &a, const std::vector<int> &e_first, const std::vector<int> &h_first,
                    const int sb[6], std::vector<int> &quiet, std::vector<int> &noisy);
hipError_t launch_pair_half_step(bool efield, int storage, int mode, const KArgs &a, int m, hipStream_t s,
                                 bool gen_cells);
hipError_t launch_step(int em, int hm, const KArgs &a, int m, hipStream_t s);
int fused_rows();
size_t persist_lds(int units, int sx);
int persist_max_units();
bool persist_fits(int storage, int units, int tiles, size_t lds, int device);
hipError_t launch_persist(int storage, const KArgs &a, const PArgs &p, int tiles, size_t lds, hipStream_t s);
hipError_t launch_unpack(int storage, const void *f, const std::uint8_t *q, float *out, std::uint32_t g0, std::uint32_t n,
                         int nx, int px, float scale, hipStream_t s);
size_t adj_persist_lds(int units, int sx, int events);
int adj_persist_max_units();
bool adj_persist_fits(int units, int tiles, size_t lds, int device);
hipError_t launch_adj_persist(const KArgs &a, const AArgs &b, const RArgs &p, int tiles, size_t lds, hipStream_t s);
hipError_t launch_dft(const KArgs &a, int nprobe, int m0, int n, hipStream_t s);
int tile_rows();
int tile_cols();
int pair_tile_cols();
}  // namespace fdtd

using namespace fdtd;

struct fdtd_ctx {
    SceneIn in;
    bool cpml_set = false;
    bool finalized = false;
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    Built built;
    KArgs ka{};
    int e_mode = 0, h_mode = 0;
    int steps_done = 0;
    bool broken = false;            // a launch gave up a wait: no valid state until a reset or a restore
    bool has_port = false;          // fdtd_set_port: its samples are probes port_base ..
    int port_base = 0;
    PortPlan port;
    double last_run_ms = 0.0, e_ms = 0.0, h_ms = 0.0;
    size_t esz = 4;                 // bytes per stored value
    i64 field_elems = 0;            // per field allocation, guard planes included
    std::vector<void *> allocs;     // every device allocation
    long n_allocs = 0;              // device allocations attempted (failure injection)
    long n_coops = 0;               // cooperative launches attempted (likewise)
    // Field and psi allocation bases (the sweeps update them in place).
    void *fields[6] = {};
    void *psi[12] = {};
    // block-scaled storage: the E and H exponent arrays (BQ_STRIDE bytes per
    // 8 x-cells: the x, y, z components' exponents), guard planes included,
    // and the component pointers into them (qexp[f] = qarr[f / 3] + f % 3)
    std::uint8_t *qarr[2] = {};
    std::uint8_t *qexp[6] = {};
    size_t qarr_bytes = 0;          // per array
    bool pair = false;              // 16-bit storage: two cells per thread in the half-step kernels
    bool pair_gen_cells = false;    // ... except the general variant, which runs one cell per thread
    int pair_tiles_x = 0, pair_kchunk = 0;
    int kchunk_h = 0;               // planes per block of the one-cell H sweep (E: ka.kchunk)
    int box[3][6] = {};             // interior tile box per sweep (0 = E, 1 = H, 2 = the fused step)
    // fused step: the other buffer of each field and of each psi of the E
    // sweep, swapped with the current one after a step
    bool fused = false;
    int kchunk_f = 0;               // planes per block
    void *fields2[6] = {};
    void *psi2[12] = {};            // (psi_h: null, updated in place)
    // many steps in one launch (persist.hip): its arguments, tiles, LDS bytes
    // and the exchange rows' bytes
    bool persist = false;
    bool unchecked = false;         // a launch that waits was made since its flag was read
    PArgs pa{};
    int ptiles = 0;
    size_t plds = 0, pll = 0;
    // reverse steps likewise (adj_persist.hip; on persist's tiles and rows)
    bool radj = false;
    RArgs ra{};
    size_t rlds = 0;
    double step_ms = 0.0;
    size_t psi_elems[12] = {};
    uint64_t dev_bytes = 0;
    // SI coefficient tables for the adjoint
    const float4 *etab_si = nullptr, *htab_si = nullptr;
    const SrcEdge *srcs_si = nullptr;
    const float4 *dcoef = nullptr;
    double adj_fwd_ms = 0.0, adj_total_ms = 0.0;
    int adj_segments = 0;
    uint64_t adj_bytes = 0;         // peak device memory of the last adjoint run
    hipEvent_t adj_ev[3] = {};      // timing events of the adjoint (made at create)
    float *stage = nullptr;         // pinned memory of fdtd_get_field, up to two pieces
    hipEvent_t stage_ev[2] = {};
    unsigned char *scratch = nullptr;   // this device's copy of the static scratch
};

// Device scratch of fdtd_adjoint_gradient_noalloc: a file-scope device array,
// one copy per GPU, held from the library's first use on that GPU until the
// process ends.  Its name is a host-side stand-in, never a device address:
// host code uses only the per-device address hipGetSymbolAddress returns
// (scratch_address), for kernel arguments, memsets and copies.  Every call
// on one GPU shares that GPU's copy, and it keeps the last call's contents.
static __device__ __align__(256) unsigned char scratch[FDTD_NOALLOC_SCRATCH_BYTES];

namespace {

// Text of the last refused fdtd_create on this thread (no context to hold it).
thread_local char g_create_err[256] = "no error";

int create_fail(int rc, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(g_create_err, sizeof g_create_err, fmt, ap);
    va_end(ap);
    return rc;
}

// The address of this device's copy of scratch, looked up once per device
// with that device current (fdtd_create's device); nullptr on failure.
unsigned char *scratch_address(int device)
{
    static std::mutex mu;
    static std::vector<unsigned char *> addr;
    static std::vector<char> looked;
    std::lock_guard<std::mutex> lock(mu);
    if (device < 0) return nullptr;
    if ((size_t)device >= addr.size()) {
        addr.resize((size_t)device + 1, nullptr);
        looked.resize((size_t)device + 1, 0);
    }
    if (!looked[(size_t)device]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) == hipSuccess) {
            addr[(size_t)device] = (unsigned char *)p;
            looked[(size_t)device] = 1;
        } else {
            (void)hipGetLastError();   // not cached: a later context may retry
        }
    }
    return addr[(size_t)device];
}

int fail(fdtd_ctx *c, int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}

#define HIPCHK(c, expr)                                                                      \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return fail(c, e_ == hipErrorOutOfMemory ? FDTD_E_NOMEM : FDTD_E_DEVICE, "%s: %s", \
                        #expr, hipGetErrorString(e_));                                       \
    } while (0)

int dev_alloc(fdtd_ctx *c, void **p, size_t bytes)
{
    *p = nullptr;
    if (bytes == 0) bytes = 256;
    // failure injection: FDTD_FAIL_ALLOC=n makes the context's n-th device
    // allocation fail as out of memory (tests of the error paths)
    ++c->n_allocs;
    if (const char *fa = std::getenv("FDTD_FAIL_ALLOC"))
        if (std::atol(fa) == c->n_allocs)
            return fail(c, FDTD_E_NOMEM, "hipMalloc(%zu) failed: injected (FDTD_FAIL_ALLOC=%s)", bytes, fa);
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(c, FDTD_E_NOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    }
    c->allocs.push_back(*p);
    c->dev_bytes += bytes;
    return FDTD_OK;
}

int upload(fdtd_ctx *c, void **p, const void *src, size_t bytes)
{
    int rc = dev_alloc(c, p, bytes);
    if (rc) return rc;
    if (bytes && src) HIPCHK(c, hipMemcpyAsync(*p, src, bytes, hipMemcpyHostToDevice, c->stream));
    return FDTD_OK;
}

void free_device(fdtd_ctx *c)
{
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (void *p : c->allocs) (void)hipFree(p);
    c->allocs.clear();
    c->dev_bytes = 0;
    for (auto &f : c->fields) f = nullptr;
    for (auto &p : c->psi) p = nullptr;
    for (auto &q : c->qexp) q = nullptr;
    for (auto &q : c->qarr) q = nullptr;
    for (auto &f : c->fields2) f = nullptr;
    for (auto &p : c->psi2) p = nullptr;
    c->fused = c->persist = c->radj = c->unchecked = false;
}

// The buffers holding the current state.
void *fld(const fdtd_ctx *c, int f) { return c->fields[f]; }
void *psv(const fdtd_ctx *c, int q) { return c->psi[q]; }

bool box_in_grid(const fdtd_ctx *c, int i, int j, int k)
{
    return i >= 0 && j >= 0 && k >= 0 && i < c->in.nx && j < c->in.ny && k < c->in.nz;
}

// Zero every piece of time-dependent state.  (Not the fused step's second
// buffers, cleared when they are made: a step writes every value of theirs that
// is ever read, and nothing writes the rest.)
int zero_state(fdtd_ctx *c)
{
    for (int f = 0; f < 6; ++f) {
        if (c->fields[f]) HIPCHK(c, hipMemsetAsync(c->fields[f], 0, (size_t)c->field_elems * c->esz, c->stream));
    }
    for (int q = 0; q < 2; ++q)
        if (c->qarr[q]) HIPCHK(c, hipMemsetAsync(c->qarr[q], 0, c->qarr_bytes, c->stream));
    for (int p = 0; p < 12; ++p)
        if (c->psi_elems[p] && c->psi[p])
            HIPCHK(c, hipMemsetAsync(c->psi[p], 0, c->psi_elems[p] * c->esz, c->stream));
    const size_t np = c->in.probes.size(), nf = c->in.freqs.size();
    if (np) HIPCHK(c, hipMemsetAsync(c->ka.probe_hist, 0, np * (size_t)c->in.steps_cap * sizeof(float), c->stream));
    if (np && nf) HIPCHK(c, hipMemsetAsync(c->ka.dft, 0, np * nf * sizeof(double2), c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->steps_done = 0;
    c->broken = false;
    return FDTD_OK;
}

// Upload the material-dependent tables (class map, E/H tables, sources).
void bind_sets(const fdtd_ctx *c, KArgs &a);
int upload_tables(fdtd_ctx *c);

// Planes per z-march block.  Many short marches keep every CU's wave slots
// full through the tail of a launch; each block re-reads one plane of the
// carried z-neighbour, so a block of `planes` costs 1/planes extra on that
// stream.  Measured: the FP32 sweeps are fastest at 4 planes (us per step, H
// at 2 / at 4: 203x149x97 magnetic 66.9 / 64.4, 200^3 154 / 145, 320x320x130
// magnetic 221 / 207), the 16-bit pair sweeps at 8 (FDTD_CHUNKS overrides all
// three with a number of blocks along z; FDTD_E_PLANES, FDTD_H_PLANES and
// FDTD_PAIR_PLANES set one sweep's planes per block before the small-grid
// halving).
int choose_chunks(const fdtd_ctx *c, int tiles, int planes, const char *planes_env, long min_wg = 1024)
{
    const char *ov = std::getenv("FDTD_CHUNKS");
    if (const char *pe = std::getenv(planes_env)) planes = std::max(1, std::atoi(pe));
    // Small grids: halve the planes per block until a launch has 1024
    // workgroups (4 per CU), down to one plane (FDTD_MIN_WG overrides 1024).
    // Measured: 64^3 FP32 18.4 -> 22.7 G, FP16 10.3 -> 22.3 G; 128x128x64
    // FP32 keeps its 4-plane E blocks (2-plane ones measured 3.5 % slower).
    if (const char *mw = std::getenv("FDTD_MIN_WG")) min_wg = std::atol(mw);
    while (planes > 1 && (long)tiles * (c->in.nz / planes) < min_wg) planes /= 2;
    int nchunks = ov ? std::atoi(ov)
                     : std::min((32 * 1024 * 8 / planes + tiles - 1) / tiles, c->in.nz / planes);
    nchunks = std::max(1, std::min(nchunks, c->in.nz));
    return (c->in.nz + nchunks - 1) / nchunks;
}

// Interior tile box of one sweep (tiles tile_cols wide and tile_rows() high,
// z-blocks of kchunk planes): along each axis, the run of tiles whose cell
// range reaches neither a CPML slab nor an outer face (nor the grid's end).
// The x-edge variant takes the tiles beside the box in x, the general
// variant the rows and z-blocks outside it.  Where no column of tiles is
// interior (nx up to two tiles and a slab), the x-edge variant takes every
// column of the box's rows and z-blocks -- with 128-cell tiles where they
// leave no 64 columns idle that the general variant's 64-cell tiles would not
// (or one in six).  us per step, general variant alone / so: FP16 220x220x200
// 117 / 93, 250x150x60 38.6 / 36.2, 128x200x200 62 / 55; block-scaled int16
// 220x220x200 170 / 134, 128x128x100 42.7 / 38.6; with 64 idle columns of 256
// FP16 180x180x160 66.3 / 67.4, 160x160x150 55 / 59; FP32 112x150x200 74 / 70,
// 100x80x70 19.9 / 18.2.  128-cell tiles do so only where half of them lie in
// those rows and z-blocks, or the z-blocks are long: a pair tile beside two of the
// general variant's is the longer wait.  By the share of the tiles: block-scaled
// 212x45x91 (0.31) 29.4 / 31.5, 97x48x83 (0.37) 19.8 / 23.0, 115x54x60 (0.47) 18.8 /
// 19.4, 73x198x76 (0.53) 45.9 / 43.9, 203x70x160 (0.65) 56.4 / 51.3; of 18 grids
// below a half 13 were slower so, of 52 others 3 (by 4 % at most); blocks of nine
// planes: FP16 232x243x74 (0.39) 66.3 / 59.9.  FDTD_INTERIOR=0, or a y or z
// axis without interior tiles, leaves the box empty (z range [0, 0)) and every
// tile to the general variant.
// beyond: cells past the tile's high sides that must lie off the slabs too
// (the fused step evaluates one).
void sweep_split(fdtd_ctx *c, int sweep, int tile_cols, int by, int kchunk, int beyond = 0)
{
    const SceneIn &in = c->in;
    const int *L = in.cpml.thick;
    int *ib = c->box[sweep];
    for (int q = 0; q < 6; ++q) ib[q] = 0;
    const char *ev = std::getenv("FDTD_INTERIOR");
    if (ev && std::strcmp(ev, "0") == 0) return;
    const int nts[3] = {(in.nx + tile_cols - 1) / tile_cols, (in.ny + by - 1) / by, (in.nz + kchunk - 1) / kchunk};
    const int w[3] = {tile_cols, by, kchunk}, nn[3] = {in.nx, in.ny, in.nz};
    int box[6];
    bool edge_only = false;
    for (int ax = 0; ax < 3; ++ax) {
        const int lo_cells = std::max(L[2 * ax], 1), hi_cells = nn[ax] - std::max(L[2 * ax + 1], 1);
        int lo = nts[ax], hi = 0;
        for (int t = 0; t < nts[ax]; ++t)
            if (t * w[ax] >= lo_cells && (t + 1) * w[ax] + beyond <= hi_cells) {
                lo = std::min(lo, t);
                hi = t + 1;
            }
        if (hi <= lo) {
            const int t64 = (in.nx + 63) / 64;
            if (ax > 0 || sweep == 2 || (tile_cols > 64 && t64 % 2 != 0 && t64 < 5)) return;
            lo = hi = 0;
            edge_only = true;
        }
        box[ax] = lo;
        box[ax + 3] = hi;
    }
    if (edge_only && tile_cols > 64 && kchunk < 8 &&
        2L * (box[4] - box[1]) * (box[5] - box[2]) < (long)nts[1] * nts[2])
        return;
    for (int q = 0; q < 6; ++q) ib[q] = box[q];
}

// Whether one of the switches is set.
bool any_set(std::initializer_list<const char *> names)
{
    for (const char *n : names)
        if (std::getenv(n)) return true;
    return false;
}

// The fused step's second buffers: the fields and the psi of the E sweep.
size_t second_bytes(const fdtd_ctx *c)
{
    size_t b = 6 * (size_t)c->field_elems * c->esz;
    for (int p : {0, 1, 4, 5, 8, 9}) b += std::max<size_t>(c->psi_elems[p], 1) * c->esz;
    return b;
}

// The fused step's tiling and its second buffers; without the memory for
// them the context steps with the two sweeps.
//
// The rule: FP32 grids of 24 M cells or more (60 M where the H coefficients
// differ by cell, which costs the fused kernel 16 registers) whose interior
// tiles hold 3/8 of the cells (3/5).  The fused pass gains on interior tiles
// and where the fields are read from HBM; its general variant, with both
// half-steps' slab state, does not, and its workgroups are fewer and longer.
// Measured, us per step, sweeps / fused: 512x512x256 1061 / 937, 384x384x200
// 488 / 446, 448x256x256 468 / 430, 300^3 463 / 448; below the line 288^3 400
// / 409, 512x300x150 380 / 363, 260x260x300 376 / 398, 320x320x160 254 / 271,
// 256^3 262 / 277.  Magnetic, by the share of the interior: 512x512x240 (0.61) 1092
// / 988, 900x300x250 (0.65) 1116 / 1102, 400^3 (0.68) 1110 / 1061, but 1000x260x250
// (0.66) 1060 / 1088; below the line 512x512x256 (0.56) 1093 / 1102, 900x300x250
// with a thicker CPML (0.55) 1244 / 1268, 640x400x256 (0.54) 1144 / 1143, 400^3 (0.46)
// 1185 / 1227; below 60 M 512x512x200 900 / 922, 512x512x128 573 / 634.
// FDTD_FUSED=0 / 1 overrides it; a switch that only the sweeps have asks for
// those.  The second buffers take at most an eighth of the memory that is free:
// what a program allocates next, another context or a tensor, fits as before but
// for that eighth.  Blocks of 16 planes, halved until a launch
// has 4096 workgroups (256^3: 8 planes 281 us, 16 planes 296).
void setup_fused(fdtd_ctx *c)
{
    const SceneIn &in = c->in;
    c->fused = false;
    const char *fv = std::getenv("FDTD_FUSED");
    const bool force = fv && std::strcmp(fv, "1") == 0;
    if (in.storage != FDTD_STORE_F32 || (fv && std::strcmp(fv, "0") == 0)) return;
    if (!force && any_set({"FDTD_STREAM", "FDTD_E_PLANES", "FDTD_H_PLANES"})) return;
    const int by = fused_rows(), tx = (in.nx + tile_cols() - 1) / tile_cols(), ty = (in.ny + by - 1) / by;
    c->kchunk_f = choose_chunks(c, tx * ty, 16, "FDTD_F_PLANES", 4096);
    sweep_split(c, 2, tile_cols(), by, c->kchunk_f, 1);
    const int *ib = c->box[2];
    const double cells = (double)in.nx * in.ny * in.nz;
    const double inner = (double)(ib[3] - ib[0]) * tile_cols() * (ib[4] - ib[1]) * by * (ib[5] - ib[2]) * c->kchunk_f;
    const bool uni = c->h_mode == CLS_UNIFORM;
    if (!force && (cells < (uni ? 24e6 : 60e6) || inner < (uni ? 0.375 : 0.6) * cells)) return;

    size_t freeb = 0, totb = 0;
    if (!force && (hipMemGetInfo(&freeb, &totb) != hipSuccess || second_bytes(c) > freeb / 8)) {
        (void)hipGetLastError();
        return;
    }

    const size_t n_allocs = c->allocs.size();
    const uint64_t bytes = c->dev_bytes;
    const std::string err = c->err;
    int rc = FDTD_OK;
    for (int f = 0; f < 6 && !rc; ++f) rc = dev_alloc(c, &c->fields2[f], (size_t)c->field_elems * c->esz);
    for (int p : {0, 1, 4, 5, 8, 9})
        if (!rc) rc = dev_alloc(c, &c->psi2[p], std::max<size_t>(c->psi_elems[p], 1) * c->esz);
    for (int f = 0; f < 6 && !rc; ++f)
        if (hipMemsetAsync(c->fields2[f], 0, (size_t)c->field_elems * c->esz, c->stream) != hipSuccess) rc = FDTD_E_DEVICE;
    for (int p : {0, 1, 4, 5, 8, 9})
        if (!rc && c->psi_elems[p] &&
            hipMemsetAsync(c->psi2[p], 0, c->psi_elems[p] * c->esz, c->stream) != hipSuccess)
            rc = FDTD_E_DEVICE;
    if (rc) {
        (void)hipGetLastError();
        (void)hipStreamSynchronize(c->stream);
        while (c->allocs.size() > n_allocs) {
            (void)hipFree(c->allocs.back());
            c->allocs.pop_back();
        }
        for (auto &f : c->fields2) f = nullptr;
        for (auto &p : c->psi2) p = nullptr;
        c->dev_bytes = bytes;
        c->err = err;
        return;
    }
    c->fused = true;
}

// Give the fused step's second buffers back; the context steps with the two
// sweeps from here on (same bits).
void release_fused(fdtd_ctx *c)
{
    (void)hipStreamSynchronize(c->stream);
    auto drop = [c](void *&p, size_t bytes) {
        if (!p) return;
        (void)hipFree(p);
        c->allocs.erase(std::find(c->allocs.begin(), c->allocs.end(), p));
        c->dev_bytes -= bytes;
        p = nullptr;
    };
    for (auto &f : c->fields2) drop(f, (size_t)c->field_elems * c->esz);
    for (int p = 0; p < 12; ++p) drop(c->psi2[p], std::max<size_t>(c->psi_elems[p], 1) * c->esz);
    c->fused = false;
}

// Reverse steps in one launch: on the tiles of the forward ones (ty x tz rows
// of sx segments, gy of them along y), whose exchange rows are taken from the
// forward units.  Rule: wherever the forward steps run in one launch and a
// tile's units and events fit 160 KB of LDS (76 units; any storage form: the
// reverse state is FP32).  All of it is faster that way; a reverse step, us,
// launched / in one launch: 28x24x22 13.4 / 5.4, 64^3 18.4 / 6.0, 127x100x50 30.8 /
// 13.3, 300x60x40 34.8 / 17.0, 128x128x64 44.0 / 21.1, 112x96x90 43.1 / 26.7, 96^3
// 43.2 / 26.5.  FDTD_ADJ_PERSIST=0 turns it off.
void setup_radj(fdtd_ctx *c, const std::vector<PTile> &ptiles, const std::vector<PUnit> (&units)[2], int gy, int tz)
{
    const SceneIn &in = c->in;
    const Built &bt = c->built;
    const int nx = in.nx, ny = in.ny, nz = in.nz, ty = c->pa.ty, sx = c->pa.sx, U = c->pa.units;
    const char *ev = std::getenv("FDTD_ADJ_PERSIST");
    if ((ev && std::strcmp(ev, "0") == 0) || U > adj_persist_max_units() || sx >= 1 << (31 - RU_SEG) || ny > 0xFFFF ||
        nz > 0xFFFF)
        return;
    // a tile's units: those on its high sides first, on its low sides last
    // (high and low: last); at[u]: where unit u comes
    const int tiles = c->ptiles;
    std::vector<RUnit> ru((size_t)tiles * U, RUnit{});
    std::vector<PTile> pt(ptiles);
    std::vector<const PUnit *> pe(U), ph(U);
    std::vector<std::vector<REvent>> le(U), lh(U);   // a tile's events, by unit
    std::vector<REvent> events;
    int max_ev = 0;
    // E events and source edges by tile
    struct At { int i, j, k, u; Event e; std::uint32_t cls; };
    std::vector<std::vector<At>> per(tiles);
    auto tile_of = [&](int j, int k) { return (k / tz) * gy + j / ty; };
    auto unit_of = [&](int i, int j, int k) { return ((k % tz) * ty + j % ty) * sx + i / 64; };
    for (const Event &e : bt.events) {
        if (e.kind < 0) break;   // (the H events follow)
        if (e.kind != EV_SOURCE && e.kind > EV_PROBE + 2) continue;
        const int i = e.col % nx, j = e.col / nx;
        per[tile_of(j, e.k)].push_back(At{i, j, e.k, unit_of(i, j, e.k), e, bt.src_cls[&e - bt.events.data()]});
    }
    // source gathers: of the cell itself, of (i-1, j) and of (i, j-1), the
    // latter in the tile below when j is its first row
    std::vector<std::vector<std::pair<int, REvent>>> gather(tiles);
    std::vector<char> third((size_t)ny * nz * sx, 0);   // rows (by segment) posted with dJ/dEz
    for (int q = 0; q < 3; ++q)
        for (int t = 0; t < tiles; ++t)
            for (const At &s : per[t]) {
                if (s.e.kind != EV_SOURCE) continue;
                const int i = q == 1 ? s.i - 1 : s.i, j = q == 2 ? s.j - 1 : s.j;
                if (i < 0 || j < 0) continue;
                const SrcEdge &se = bt.srcs_si[s.e.id];
                const size_t cl = bt.e_uniform ? 0 : s.cls;
                const float *ez = bt.etab_si.data() + (cl * 3 + 2) * 4;
                const int *L = in.cpml.thick;
                auto slab = [](int v, int n, int lo, int hi) { return (v > 0 && v < lo) || (v >= n - hi && v < n - 1); };
                const float kx = slab(s.i, nx, L[0], L[1]) ? bt.prof[0][4 * (size_t)s.i + 2] : 1.0f;
                const float ky = slab(s.j, ny, L[2], L[3]) ? bt.prof[1][4 * (size_t)s.j + 2] : 1.0f;
                const int to = tile_of(j, s.k);
                REvent r{i, q, to == t ? (int)(&s - per[t].data()) : -1, 0, se.cezhy, se.cezhx, ez[1] / kx, ez[2] / ky};
                if (to != t) third[((size_t)s.k * ny + s.j) * sx + s.i / 64] = 1;
                gather[to].push_back({unit_of(i, j, s.k), r});
            }
    for (int t = 0; t < tiles; ++t) {
        std::fill(pe.begin(), pe.end(), nullptr);
        std::fill(ph.begin(), ph.end(), nullptr);
        const int nu = ptiles[t].nu;
        for (int n = 0; n < nu; ++n) {
            const PUnit &e = units[0][(size_t)t * U + n], &h = units[1][(size_t)t * U + n];
            pe[e.lds / (6 * 64)] = &e;
            ph[h.lds / (6 * 64)] = &h;
        }
        pt[t].ev = (int)events.size();
        std::vector<int> where(per[t].size());   // of each E event
        std::vector<int> evw(U, 0), hvw(U, 0);
        for (int u = 0; u < U; ++u) {
            const int first = (int)events.size() - pt[t].ev;
            for (size_t x = 0; x < per[t].size(); ++x) {
                const At &s = per[t][x];
                if (s.u != u) continue;
                where[x] = (int)events.size() - pt[t].ev;
                const float c0 = s.e.kind == EV_SOURCE ? bt.srcs_si[s.e.id].ceze : 0.f;
                events.push_back(REvent{s.i, s.e.kind, s.e.id, 0, c0, 0.f, 0.f, 0.f});
            }
            evw[u] = first | ((int)events.size() - pt[t].ev - first) << 16;
        }
        for (int u = 0; u < U; ++u) {
            const int first = (int)events.size() - pt[t].ev;
            for (const auto &g : gather[t]) {
                if (g.first != u) continue;
                events.push_back(g.second);
                if (g.second.id >= 0) events.back().id = where[g.second.id];
            }
            hvw[u] = first | ((int)events.size() - pt[t].ev - first) << 16;
        }
        pt[t].nev = (int)events.size() - pt[t].ev;
        if (pt[t].nev > 0x7FFF) return;   // (16-bit fields of RUnit)
        max_ev = std::max(max_ev, pt[t].nev);
        int n = 0;
        for (int pass = 0; pass < 3; ++pass)
            for (int u = 0; u < U; ++u) {
                if (!pe[u]) continue;
                const PUnit &e = *pe[u], &h = *ph[u];
                const bool lo = !(e.flags & PU_IJ) || !(e.flags & PU_IK), hi = !(h.flags & PU_IJ) || !(h.flags & PU_IK);
                if ((lo ? 2 : hi ? 0 : 1) != pass) continue;
                auto f = [](int from, int bit, int to) { return from & bit ? to : 0; };
                // (third words: of rows that another tile waits for)
                const bool se = (e.flags & PU_GJ) && third[((size_t)e.k * ny + e.j) * sx + e.i0 / 64];
                const bool sh = (h.flags & PU_GJ) && third[((size_t)h.k * ny + h.j + 1) * sx + h.i0 / 64];
                RUnit &r = ru[(size_t)t * U + n++];
                r.w[RW_UNIT] = u;
                r.w[RW_FLAGS] = f(e.flags, PU_JLO, RU_JLO) | f(e.flags, PU_JHI, RU_JHI) | f(e.flags, PU_KLO, RU_KLO) |
                                f(e.flags, PU_KHI, RU_KHI) | f(e.flags, PU_XS, RU_XS) | f(e.flags, PU_YS, RU_YSE) |
                                f(h.flags, PU_YS, RU_YSH) | f(e.flags, PU_ZS, RU_ZSE) | f(h.flags, PU_ZS, RU_ZSH) |
                                f(e.flags, PU_GJ, RU_GJE) | f(e.flags, PU_GK, RU_GKE) | f(h.flags, PU_GJ, RU_GJH) |
                                f(h.flags, PU_GK, RU_GKH) | f(e.flags, PU_IJ, RU_IJE) | f(e.flags, PU_IK, RU_IKE) |
                                f(h.flags, PU_IJ, RU_IJH) | f(h.flags, PU_IK, RU_IKH) | f(e.flags, PU_XL, RU_XLE) |
                                f(h.flags, PU_XL, RU_XLH) | (se ? RU_SRE : 0) | (sh ? RU_SRH : 0) |
                                (int)((unsigned)(e.i0 / 64) << RU_SEG);
                r.w[RW_JK] = (int)((unsigned)e.j | (unsigned)e.k << 16);
                r.w[RW_PSX] = e.psx;
                r.w[RW_PSY] = e.psy;
                r.w[RW_PSZ] = e.psz;
                r.w[RW_WJE] = e.wj; r.w[RW_WKE] = e.wk; r.w[RW_OJE] = e.oj; r.w[RW_OKE] = e.ok;
                r.w[RW_WJH] = h.wj; r.w[RW_WKH] = h.wk; r.w[RW_OJH] = h.oj; r.w[RW_OKH] = h.ok;
                r.w[RW_EVE] = evw[u];
                r.w[RW_EVH] = hvw[u];
            }
    }
    const size_t lds = adj_persist_lds(U, sx, max_ev);
    if (lds > 160 * 1024 || !adj_persist_fits(U, c->ptiles, lds, c->device)) return;
    const size_t n_allocs = c->allocs.size();
    const uint64_t bytes = c->dev_bytes;
    const std::string err = c->err;
    void *dt = nullptr, *du = nullptr, *de = nullptr;
    int rc = upload(c, &dt, pt.data(), pt.size() * sizeof(PTile));
    if (!rc) rc = upload(c, &du, ru.data(), ru.size() * sizeof(RUnit));
    if (!rc) rc = upload(c, &de, events.data(), events.size() * sizeof(REvent));
    if (hipStreamSynchronize(c->stream) != hipSuccess) rc = FDTD_E_DEVICE;   // (the host vectors go out of scope)
    if (rc) {
        (void)hipGetLastError();
        while (c->allocs.size() > n_allocs) {
            (void)hipFree(c->allocs.back());
            c->allocs.pop_back();
        }
        c->dev_bytes = bytes;
        c->err = err;
        return;
    }
    RArgs &r = c->ra;
    r = RArgs{};
    r.ty = ty;
    r.sx = sx;
    r.units = U;
    r.cls16 = c->pa.cls16;
    r.euni = bt.e_uniform ? 1 : 0;
    r.failed = c->pa.failed;
    r.ll = c->pa.ll;
    r.tiles = (const PTile *)dt;
    r.u = (const RUnit *)du;
    r.events = (const REvent *)de;
    c->rlds = lds;
    c->radj = true;
}

// Reads of a neighbour's row before a wait is given up (some seconds);
// FDTD_PERSIST_POLLS, looked up at each launch, overrides it.
int poll_limit()
{
    const char *mp = std::getenv("FDTD_PERSIST_POLLS");
    return mp ? std::atoi(mp) : 1 << 22;
}

// Failure injection: FDTD_FAIL_COOP=n makes the context's n-th cooperative launch
// (the first is the trial of setup_persist) fail as refused.
bool coop_refused(fdtd_ctx *c)
{
    ++c->n_coops;
    const char *fc = std::getenv("FDTD_FAIL_COOP");
    return fc && std::atol(fc) == c->n_coops;
}

// Many steps in one launch; one that is refused (nothing has run then) leaves
// the context to the sweeps from here on, as at set-up.
hipError_t launch_steps(fdtd_ctx *c, const KArgs &a)
{
    const hipError_t e = coop_refused(c) ? hipErrorCooperativeLaunchTooLarge
                                         : launch_persist(c->in.storage, a, c->pa, c->ptiles, c->plds, c->stream);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        c->persist = c->radj = false;
    }
    return e;
}

// Tiles, exchange rows and event lists of the steps in one launch; a context
// they do not fit, or without the memory, steps with the sweeps.
//
// The rule: FP32, FP16 or BF16 storage, one H class, and a tiling of at most
// 256 tiles of 80 row segments (about 1.3 M cells), each with at most
// P_MAX_EVENTS source edges and probes.  Every such grid measured is faster in
// one launch, us per step, sweeps / one launch of 300 steps: 64^3 12.2 / 3.9,
// 300x60x40 18.0 / 11.4, 110x150x53 22.0 / 14.6, 128x128x64 19.4 / 14.5 (FP16 22.4 /
// 16.5), 128x128x80 22.9 / 17.2, 96^3 19.6 / 14.1, 12x9x8 8.0 / 3.0; and from 6 to 10 steps
// on (persist_min_steps).  FDTD_PERSIST=0 turns it off, and so does a switch of
// the launched sweeps, which asks for those.
void setup_persist(fdtd_ctx *c)
{
    const SceneIn &in = c->in;
    c->persist = c->radj = false;
    const char *ev = std::getenv("FDTD_PERSIST");
    if (in.storage == FDTD_STORE_BQ16 || c->h_mode != CLS_UNIFORM || c->fused || (ev && std::strcmp(ev, "0") == 0) ||
        any_set({"FDTD_PAIR", "FDTD_GEN16", "FDTD_CHUNKS", "FDTD_INTERIOR", "FDTD_STREAM", "FDTD_MIN_WG",
                 "FDTD_E_PLANES", "FDTD_H_PLANES", "FDTD_PAIR_PLANES"}))
        return;
    // the tiling: at most one tile per CU and 160 KB of LDS each, the fewest
    // units (64-cell row segments) per tile, then the fewest rows exchanged
    const size_t lds_max = 160 * 1024;
    const int cus = 256, sx = (in.nx + 63) / 64;
    if ((double)in.ny * in.nz * sx > (double)cus * persist_max_units()) return;
    int ty = 0, tz = 0;
    double best = 0.0;
    for (int z = 1; z <= in.nz && z <= 64; ++z)
        for (int y = 1; y <= in.ny && y <= 64; ++y) {
            if (((in.ny + y - 1) / y) * ((in.nz + z - 1) / z) > cus || y * z * sx > persist_max_units() ||
                persist_lds(y * z * sx, sx) > lds_max)
                continue;
            const double cost = y * z * sx + 0.25 * (y + z) * sx;
            if (ty == 0 || cost < best) {
                best = cost;
                ty = y;
                tz = z;
            }
        }
    if (ty == 0) return;
    const int gy = (in.ny + ty - 1) / ty, gz = (in.nz + tz - 1) / tz, tiles = gy * gz, U = ty * tz * sx;
    const size_t lds = persist_lds(U, sx);
    if (!persist_fits(in.storage, U, tiles, lds, c->device)) return;
    // events of each tile's units: E events, then (after their terminator) H events
    const int nx = in.nx, ny = in.ny, nz = in.nz, XS = sx * 64;
    const int *L = in.cpml.thick;
    std::vector<std::vector<PEvent>> per((size_t)tiles * 2 * U);
    int half = 0;
    for (const Event &e : c->built.events) {
        if (e.kind < 0) {
            ++half;
            continue;
        }
        const int i = e.col % nx, j = e.col / nx;
        const int tile = (e.k / tz) * gy + j / ty, u = ((e.k % tz) * ty + j % ty) * sx + i / 64;
        PEvent q{i, e.kind, e.id, 0, 0.f, 0.f, 0.f, 0.f};
        if (e.kind == EV_SOURCE) {
            const SrcEdge &se = c->built.srcs[e.id];
            q.wave = se.wave;
            q.ceze = se.ceze; q.cezhy = se.cezhy; q.cezhx = se.cezhx; q.cezj = se.cezj;
        }
        per[((size_t)tile * 2 + half) * U + u].push_back(q);
    }
    // exchange rows, [2][XS] words each: H of a tile's last row (hx, hz) and
    // last plane (hx, hy), E of its first row (ex, ez; [3][XS], the third for
    // the reverse steps) and plane (ex, ey)
    const size_t wj = (size_t)gy * nz * XS, wk = (size_t)gz * ny * XS;
    const size_t o_hj = 0, o_hk = 2 * wj, o_ej = o_hk + 2 * wk, o_ek = o_ej + 3 * wj, words = o_ek + 2 * wk;
    std::vector<PTile> pt(tiles);
    std::vector<PUnit> units[2];
    std::vector<PEvent> events;
    for (auto &v : units) v.assign((size_t)tiles * U, PUnit{});
    for (int t = 0; t < tiles; ++t) {
        const int tj = t % gy, tk = t / gy, j0 = tj * ty, k0 = tk * tz;
        const int nyt = std::min(ty, ny - j0), nzt = std::min(tz, nz - k0);
        pt[t] = PTile{nyt * nzt * sx, (int)events.size(), 0, 0};
        for (int h = 0; h < 2; ++h) {
            int n = 0;
            for (int pass = 0; pass < 2; ++pass)
                for (int u = 0; u < U; ++u) {
                    const int jt = (u / sx) % ty, kt = u / sx / ty, j = j0 + jt, k = k0 + kt, i0 = (u % sx) * 64;
                    if (jt >= nyt || kt >= nzt) continue;
                    const bool sj = h == 0 ? jt == 0 : jt == nyt - 1, sk = h == 0 ? kt == 0 : kt == nzt - 1;
                    if ((sj || sk) != (pass == 1)) continue;   // units that wait come last
                    PUnit q{};
                    q.lds = u * 6 * 64;
                    q.i0 = i0;
                    q.j = j;
                    q.k = k;
                    const bool gj = sj && (h == 0 ? j > 0 : j < ny - 1), gk = sk && (h == 0 ? k > 0 : k < nz - 1);
                    const bool lo = h == 0;   // the E slabs leave out cell 0 (fdtdrav.h:752, 402)
                    const bool ys = ((!lo || j > 0) && j < L[2]) || (j >= ny - L[3] && j < ny - 1);
                    const bool zs = ((!lo || k > 0) && k < L[4]) || (k >= nz - L[5] && k < nz - 1);
                    const bool xs = i0 < L[0] || i0 + 64 > nx - L[1];
                    const bool xl = h == 0 ? i0 > 0 : i0 + 64 < XS;
                    q.flags = (j > 0 ? PU_JLO : 0) | (j < ny - 1 ? PU_JHI : 0) | (k > 0 ? PU_KLO : 0) |
                              (k < nz - 1 ? PU_KHI : 0) | (ys ? PU_YS : 0) | (zs ? PU_ZS : 0) | (xs ? PU_XS : 0) |
                              (gj ? PU_GJ : 0) | (gk ? PU_GK : 0) | (!sj ? PU_IJ : 0) | (!sk ? PU_IK : 0) |
                              (xl ? PU_XL : 0);
                    q.psx = (k * ny + j) * (L[0] + L[1]);
                    q.psy = (k * (L[2] + L[3]) + (j < L[2] ? j : j - (ny - L[3]) + L[2])) * in.px + i0;
                    q.psz = ((k < L[4] ? k : k - (nz - L[5]) + L[4]) * ny + j) * in.px + i0;
                    const int dj = h == 0 ? tj - 1 : tj + 1, dk = h == 0 ? tk - 1 : tk + 1;
                    // of a tile in y (in z), the row in plane k (the row j) from cell i0
                    auto hj = [&](int tile_) { return (int)(o_hj + ((size_t)tile_ * nz + k) * 2 * XS + i0); };
                    auto ej = [&](int tile_) { return (int)(o_ej + ((size_t)tile_ * nz + k) * 3 * XS + i0); };
                    auto hk = [&](int tile_) { return (int)(o_hk + ((size_t)tile_ * ny + j) * 2 * XS + i0); };
                    auto ek = [&](int tile_) { return (int)(o_ek + ((size_t)tile_ * ny + j) * 2 * XS + i0); };
                    if (gj) {
                        q.wj = h == 0 ? hj(dj) : ej(dj);
                        q.oj = h == 0 ? ej(tj) : hj(tj);
                    }
                    if (gk) {
                        q.wk = h == 0 ? hk(dk) : ek(dk);
                        q.ok = h == 0 ? ek(tk) : hk(tk);
                    }
                    q.ev = (int)events.size() - pt[t].ev;
                    for (const PEvent &e : per[((size_t)t * 2 + h) * U + u]) events.push_back(e);
                    q.nev = (int)events.size() - pt[t].ev - q.ev;
                    units[h][(size_t)t * U + n++] = q;
                }
        }
        pt[t].nev = (int)events.size() - pt[t].ev;
        if (pt[t].nev > P_MAX_EVENTS) return;
    }

    const size_t n_allocs = c->allocs.size();
    const uint64_t bytes = c->dev_bytes;
    const std::string err = c->err;
    void *ll = nullptr, *fd = nullptr, *dt = nullptr, *du[2] = {}, *de = nullptr;
    c->pll = words * sizeof(std::uint64_t);
    int rc = c->pll < ((size_t)1 << 31) ? dev_alloc(c, &ll, c->pll) : FDTD_E_UNSUPPORTED;
    if (!rc) rc = dev_alloc(c, &fd, sizeof(int));
    if (!rc) rc = upload(c, &dt, pt.data(), pt.size() * sizeof(PTile));
    for (int h = 0; h < 2 && !rc; ++h) rc = upload(c, &du[h], units[h].data(), units[h].size() * sizeof(PUnit));
    if (!rc) rc = upload(c, &de, events.data(), events.size() * sizeof(PEvent));
    if (!rc && (hipMemsetAsync(ll, 0, c->pll, c->stream) != hipSuccess ||
                hipMemsetAsync(fd, 0, sizeof(int), c->stream) != hipSuccess))
        rc = FDTD_E_DEVICE;
    if (hipStreamSynchronize(c->stream) != hipSuccess) rc = FDTD_E_DEVICE;   // (the host vectors go out of scope)
    auto drop = [&]() {
        (void)hipGetLastError();
        while (c->allocs.size() > n_allocs) {
            (void)hipFree(c->allocs.back());
            c->allocs.pop_back();
        }
        c->dev_bytes = bytes;
        c->err = err;
    };
    if (rc) return drop();
    PArgs &p = c->pa;
    p = PArgs{};
    p.ty = ty;
    p.sx = sx;
    p.units = U;
    p.cls16 = c->built.mode == CLS_U16 ? 1 : 0;
    p.epoch = 1;
    p.max_polls = poll_limit();
    p.failed = (int *)fd;
    p.ll = (std::uint64_t *)ll;
    p.tiles = (const PTile *)dt;
    p.units_e = (const PUnit *)du[0];
    p.units_h = (const PUnit *)du[1];
    p.events = (const PEvent *)de;
    c->ptiles = tiles;
    c->plds = lds;
    // A launch of no steps (it stores the state that it read): cooperative
    // launches are refused while another process on the card has made some,
    // and the sweeps are used then.
    KArgs ka = c->ka;
    bind_sets(c, ka);
    ka.snap = nullptr;
    if (launch_steps(c, ka) != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess) return drop();
    p.epoch += 1;
    c->persist = true;
    if (!in.design_eps.empty()) setup_radj(c, pt, units, gy, tz);
}

int do_finalize(fdtd_ctx *c)
{
    const SceneIn &in = c->in;
    Built &b = c->built;
    std::string err;
    {
        // The sweep kernels address every array with 32-bit byte offsets:
        // refuse a field array (with its two guard planes) of 4 GiB or more
        // before building anything.
        const size_t fb = (size_t)in.px * in.ny * (in.nz + 2) * (in.storage == FDTD_STORE_F32 ? 4 : 2);
        if (fb >= ((size_t)1 << 32))
            return fail(c, FDTD_E_UNSUPPORTED,
                        "grid too large: each field array (with its two guard planes) must be under 4 GiB "
                        "(%zu bytes per field)", fb);
    }
    if (build_scene(in, b, err) != 0) return fail(c, FDTD_E_INVALID, "%s", err.c_str());
    c->e_mode = b.e_uniform ? CLS_UNIFORM : b.mode;
    c->h_mode = b.h_uniform ? CLS_UNIFORM : b.mode;
    c->esz = in.storage == FDTD_STORE_F32 ? 4 : 2;

    KArgs &a = c->ka;
    a = KArgs{};
    a.nx = in.nx; a.ny = in.ny; a.nz = in.nz; a.px = in.px;
    a.plane = (i64)in.px * in.ny;
    for (int q = 0; q < 6; ++q) a.L[q] = in.cpml.thick[q];
    a.Lx = a.L[0] + a.L[1];
    a.Ly = a.L[2] + a.L[3];
    a.Lz = a.L[4] + a.L[5];
    a.d[0] = (float)in.dx; a.d[1] = (float)in.dy; a.d[2] = (float)in.dz;
    a.steps_cap = in.steps_cap;
    a.nfreq = (int)in.freqs.size();
    for (int q = 0; q < 6; ++q) a.probe_unscale[q] = b.probe_unscale[q];
    a.tiles_x = (in.nx + tile_cols() - 1) / tile_cols();
    a.tiles_y = (in.ny + tile_rows() - 1) / tile_rows();
    a.kchunk = choose_chunks(c, a.tiles_x * a.tiles_y, 4, "FDTD_E_PLANES");
    c->kchunk_h = choose_chunks(c, a.tiles_x * a.tiles_y, 4, "FDTD_H_PLANES");
    // 16-bit storage (FP16, BF16, block-scaled int16) sweeps a cell pair per
    // thread (128-cell tile rows); FDTD_PAIR=0 selects the one-cell kernels
    // instead (same stored bits)
    const char *pv = std::getenv("FDTD_PAIR");
    c->pair = in.storage != FDTD_STORE_F32 && !(pv && std::strcmp(pv, "0") == 0);
    // The pair sweeps' general variant (slab rows and z-blocks) runs as the
    // one-cell kernel (same stored bits): on 512x512x256 FP16 the step took
    // 0.772 ms against 0.788 with the pair kernel's own general variant,
    // which holds two cells of slab state per thread.  FDTD_GEN16=pair
    // selects the latter.
    const char *gv = std::getenv("FDTD_GEN16");
    c->pair_gen_cells = !(gv && std::strcmp(gv, "pair") == 0);
    c->pair_tiles_x = (in.nx + pair_tile_cols() - 1) / pair_tile_cols();
    // planes in whole blocks of p off the z slabs and faces
    auto inner = [&](int p) {
        const int lo = std::max(in.cpml.thick[4], 1), hi = in.nz - std::max(in.cpml.thick[5], 1);
        return std::max(0, hi / p * p - (lo + p - 1) / p * p);
    };
    // Block-scaled storage: 16 planes a block where as many planes stay off the
    // general variant; us per step, 8 / 16: 512x512x256 791 / 780, 384^3 675 /
    // 643, 256^3 212 / 205; where fewer do: 512x512x120 402 / 421, 300x200x200
    // 147 / 149.  (FP16, where as many do: 512x512x256 657 / 668, 256^3 178 / 173.)
    const int pp = in.storage == FDTD_STORE_BQ16 && inner(16) >= inner(8) ? 16 : 8;
    c->pair_kchunk = choose_chunks(c, c->pair_tiles_x * a.tiles_y, pp, "FDTD_PAIR_PLANES");
    a.rec = 1;
    a.snap = nullptr;

    // fields: one zero guard plane below and above
    c->field_elems = a.plane * (in.nz + 2);
    // The sweep kernels address every array with 32-bit byte offsets.
    const size_t cls_bytes = (size_t)a.plane * in.nz * (b.mode == CLS_U32 ? 4 : 2);
    if ((size_t)c->field_elems * c->esz >= ((size_t)1 << 32) || cls_bytes >= ((size_t)1 << 32))
        return fail(c, FDTD_E_UNSUPPORTED,
                    "grid too large: each field array (with its two guard planes) and the class map "
                    "must be under 4 GiB (%zu bytes per field)", (size_t)c->field_elems * c->esz);
    for (int f = 0; f < 6; ++f) {
        int rc = dev_alloc(c, &c->fields[f], (size_t)c->field_elems * c->esz);
        if (rc) return rc;
    }
    if (in.storage == FDTD_STORE_BQ16) {
        // BQ_STRIDE exponent bytes per 8 x-cells of E and of H (px is a
        // multiple of 64)
        c->qarr_bytes = (size_t)c->field_elems / BQ_BLOCK * BQ_STRIDE;
        for (int q = 0; q < 2; ++q) {
            void *d = nullptr;
            int rc = dev_alloc(c, &d, c->qarr_bytes);
            if (rc) return rc;
            c->qarr[q] = (std::uint8_t *)d;
        }
        for (int f = 0; f < 6; ++f) c->qexp[f] = c->qarr[f / 3] + f % 3;
    }
    // interior / general split of the two sweeps
    {
        const int tcols = c->pair ? pair_tile_cols() : tile_cols();
        sweep_split(c, 0, tcols, tile_rows(), c->pair ? c->pair_kchunk : a.kchunk);
        sweep_split(c, 1, tcols, tile_rows(), c->pair ? c->pair_kchunk : c->kchunk_h);
    }
    // psi slabs
    const size_t px_elems = (size_t)in.nz * in.ny * a.Lx;
    const size_t py_elems = (size_t)in.nz * a.Ly * in.px;
    const size_t pz_elems = (size_t)a.Lz * in.ny * in.px;
    for (int p = 0; p < 12; ++p) {
        c->psi_elems[p] = p < 4 ? px_elems : p < 8 ? py_elems : pz_elems;
        int rc = dev_alloc(c, &c->psi[p], std::max<size_t>(c->psi_elems[p], 1) * c->esz);
        if (rc) return rc;
    }
    // The half-steps go past the caches with the swept field's own values
    // (V_STREAM) once the state -- fields, psi, class map -- is larger than
    // 300 MB: below that most of it stays in the 256 MB Infinity Cache for the
    // next half-step.  us per step, past the caches / through them: FP32 150^3
    // (128 MB) 71 / 54, 190^3 (217) 107 / 88, 200^3 (320: rows of 256) 144 /
    // 153, 224^3 191 / 205; FP16 230^3 147 / 119, 256^3 (268) 177 / 161,
    // 512x512x64 (325) 198 / 201, 270^3 (370) 242 / 256; block-scaled int16
    // 256^3 (284) 220 / 209, 270^3 307 / 320.  FDTD_STREAM=0 / 1 overrides it.
    {
        size_t bytes = 6 * (size_t)c->field_elems * c->esz + 2 * c->qarr_bytes + (b.mode == CLS_UNIFORM ? 0 : cls_bytes);
        for (int p = 0; p < 12; ++p) bytes += c->psi_elems[p] * c->esz;
        const char *sv = std::getenv("FDTD_STREAM");
        a.stream = sv ? std::atoi(sv) != 0 : bytes > 300000000;
    }
    a.e_uni = b.e_uniform ? 1 : 0;
    a.h_uni = b.h_uniform ? 1 : 0;
    int rc;
    void *tmp;
    for (int ax = 0; ax < 3; ++ax) {
        if ((rc = upload(c, &tmp, b.prof[ax].data(), b.prof[ax].size() * sizeof(float)))) return rc;
        (ax == 0 ? a.px_prof : ax == 1 ? a.py_prof : a.pz_prof) = (const float4 *)tmp;
    }
    if ((rc = upload(c, &tmp, b.e_first.data(), b.e_first.size() * sizeof(int)))) return rc;
    a.e_first = (const int *)tmp;
    if ((rc = upload(c, &tmp, b.h_first.data(), b.h_first.size() * sizeof(int)))) return rc;
    a.h_first = (const int *)tmp;
    if ((rc = upload(c, &tmp, b.events.data(), b.events.size() * sizeof(Event)))) return rc;
    a.events = (const Event *)tmp;
    if ((rc = upload(c, &tmp, b.vpn.data(), b.vpn.size() * sizeof(float)))) return rc;
    a.vpn = (const float *)tmp;
    if ((rc = upload(c, &tmp, b.phasor.data(), b.phasor.size() * sizeof(double)))) return rc;
    a.phasor = (const double2 *)tmp;
    const size_t np = in.probes.size(), nf = in.freqs.size();
    if ((rc = dev_alloc(c, &tmp, np * (size_t)in.steps_cap * sizeof(float)))) return rc;
    a.probe_hist = (float *)tmp;
    if ((rc = dev_alloc(c, &tmp, np * nf * sizeof(double2)))) return rc;
    a.dft = (double2 *)tmp;
    if ((rc = upload_tables(c))) return rc;
    setup_fused(c);
    setup_persist(c);
    if ((rc = zero_state(c))) return rc;
    c->finalized = true;
    return FDTD_OK;
}

int upload_tables(fdtd_ctx *c)
{
    Built &b = c->built;
    KArgs &a = c->ka;
    int rc;
    void *tmp;
    if ((rc = upload(c, &tmp, b.etab.data(), b.etab.size() * sizeof(float)))) return rc;
    a.etab = (const float4 *)tmp;
    if ((rc = upload(c, &tmp, b.htab.data(), b.htab.size() * sizeof(float)))) return rc;
    a.htab = (const float4 *)tmp;
    if ((rc = upload(c, &tmp, b.srcs.data(), b.srcs.size() * sizeof(SrcEdge)))) return rc;
    a.srcs = (const SrcEdge *)tmp;
    if ((rc = upload(c, &tmp, b.etab_si.data(), b.etab_si.size() * sizeof(float)))) return rc;
    c->etab_si = (const float4 *)tmp;
    if ((rc = upload(c, &tmp, b.htab_si.data(), b.htab_si.size() * sizeof(float)))) return rc;
    c->htab_si = (const float4 *)tmp;
    if ((rc = upload(c, &tmp, b.srcs_si.data(), b.srcs_si.size() * sizeof(SrcEdge)))) return rc;
    c->srcs_si = (const SrcEdge *)tmp;
    c->dcoef = nullptr;
    if (!b.dcoef.empty()) {
        if ((rc = upload(c, &tmp, b.dcoef.data(), b.dcoef.size() * sizeof(float)))) return rc;
        c->dcoef = (const float4 *)tmp;
    }
    a.cls = nullptr;
    if (b.mode == CLS_U16) {
        std::vector<uint16_t> m16(b.cls.size());
        for (size_t q = 0; q < b.cls.size(); ++q) m16[q] = (uint16_t)b.cls[q];
        if ((rc = upload(c, &tmp, m16.data(), m16.size() * sizeof(uint16_t)))) return rc;
        HIPCHK(c, hipStreamSynchronize(c->stream));
        a.cls = tmp;
    } else if (b.mode == CLS_U32) {
        if ((rc = upload(c, &tmp, b.cls.data(), b.cls.size() * sizeof(uint32_t)))) return rc;
        a.cls = tmp;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    b.src_cls.assign(b.events.size(), 0);
    for (size_t q = 0; q < b.events.size() && !b.cls.empty(); ++q) {
        const Event &e = b.events[q];
        if (e.kind == EV_SOURCE)
            b.src_cls[q] = b.cls[((size_t)e.k * a.ny + e.col / a.nx) * a.px + e.col % a.nx];
    }
    std::vector<uint32_t>().swap(b.cls);   // host copy no longer needed
    return FDTD_OK;
}

// Point a kernel argument block at the field and psi buffers; the sweeps
// read and write them in place.
void bind_sets(const fdtd_ctx *c, KArgs &a)
{
    const size_t g = (size_t)c->ka.plane * c->esz;   // guard plane
    void **rd[6] = {&a.ex, &a.ey, &a.ez, &a.hx, &a.hy, &a.hz};
    for (int f = 0; f < 6; ++f) *rd[f] = (char *)c->fields[f] + g;
    std::uint8_t **qd[6] = {&a.qex, &a.qey, &a.qez, &a.qhx, &a.qhy, &a.qhz};
    for (int f = 0; f < 6; ++f)
        *qd[f] = c->qexp[f] ? c->qexp[f] + (size_t)c->ka.plane / BQ_BLOCK * BQ_STRIDE : nullptr;
    void **pr[12] = {&a.psi_eyx, &a.psi_ezx, &a.psi_hyx, &a.psi_hzx, &a.psi_exy, &a.psi_ezy,
                     &a.psi_hxy, &a.psi_hzy, &a.psi_exz, &a.psi_eyz, &a.psi_hxz, &a.psi_hyz};
    for (int p = 0; p < 12; ++p) *pr[p] = c->psi[p];
    if (c->fused) {
        void **nd[6] = {&a.nex, &a.ney, &a.nez, &a.nhx, &a.nhy, &a.nhz};
        for (int f = 0; f < 6; ++f) *nd[f] = (char *)c->fields2[f] + g;
        a.npsi_eyx = c->psi2[0]; a.npsi_ezx = c->psi2[1];
        a.npsi_exy = c->psi2[4]; a.npsi_ezy = c->psi2[5];
        a.npsi_exz = c->psi2[8]; a.npsi_eyz = c->psi2[9];
    }
}

// One time step m.  base carries the per-call flags (rec, snapshot); the
// tile geometry and buffer pointers are filled in here.
hipError_t do_step(fdtd_ctx *c, const KArgs &base, int m, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr,
                   hipEvent_t ev2 = nullptr, hipEvent_t ev3 = nullptr)
{
    hipError_t e;
    KArgs a = base;
    a.tiles_x = c->pair ? c->pair_tiles_x : c->ka.tiles_x;
    a.tiles_y = c->ka.tiles_y;
    a.kchunk = c->pair ? c->pair_kchunk : c->ka.kchunk;
    bind_sets(c, a);
    if (c->fused && a.lc[3] == 0) {   // (light-cone steps sweep their box in place)
        a.tiles_x = c->ka.tiles_x;
        a.tiles_y = (a.ny + fused_rows() - 1) / fused_rows();
        a.kchunk = c->kchunk_f;
        for (int q = 0; q < 6; ++q) a.ib[q] = c->box[2][q];
        a.sub[3] = 0;
        if (ev0) (void)hipEventRecord(ev0, c->stream);
        e = launch_step(c->e_mode, c->h_mode, a, m, c->stream);
        if (ev1) (void)hipEventRecord(ev1, c->stream);
        if (ev2) (void)hipEventRecord(ev2, c->stream);
        if (ev3) (void)hipEventRecord(ev3, c->stream);
        for (int f = 0; f < 6; ++f) std::swap(c->fields[f], c->fields2[f]);
        for (int p : {0, 1, 4, 5, 8, 9}) std::swap(c->psi[p], c->psi2[p]);
        return e;
    }
    auto half = [c](bool efield, int storage, int mode, const KArgs &ka, int mm, hipStream_t st) {
        return c->pair ? launch_pair_half_step(efield, storage, mode, ka, mm, st, c->pair_gen_cells)
                       : launch_half_step(efield, storage, mode, ka, mm, st);
    };
    auto split = [&](int sweep) {
        for (int q = 0; q < 6; ++q) a.ib[q] = c->box[sweep][q];
        a.sub[3] = 0;
        if (a.lc[3] > 0) {   // light-cone box: its tiles of this sweep's tiling, general variant
            for (int q = 0; q < 6; ++q) a.ib[q] = 0;
            const int tc = c->pair ? pair_tile_cols() : tile_cols(), by = tile_rows();
            a.sub[0] = a.lc[0] / tc;
            a.sub[3] = (a.lc[3] + tc - 1) / tc - a.sub[0];
            a.sub[1] = a.lc[1] / by;
            a.sub[4] = (a.lc[4] + by - 1) / by - a.sub[1];
            a.sub[2] = a.lc[2] / a.kchunk;
            a.sub[5] = (a.lc[5] + a.kchunk - 1) / a.kchunk - a.sub[2];
        }
    };
    split(0);
    if (ev0) (void)hipEventRecord(ev0, c->stream);
    if ((e = half(true, c->in.storage, c->e_mode, a, m, c->stream)) != hipSuccess) return e;
    if (ev1) (void)hipEventRecord(ev1, c->stream);
    if (ev2) (void)hipEventRecord(ev2, c->stream);
    if (!c->pair) a.kchunk = c->kchunk_h;
    split(1);
    e = half(false, c->in.storage, c->h_mode, a, m, c->stream);
    if (ev3) (void)hipEventRecord(ev3, c->stream);
    return e;
}

// The fewest steps that pay for one launch -- the launch itself, loading and
// storing the tiles, reading its flag -- by the units a wave holds.  us per
// fdtd_run, launched / in one launch, around the line: 64^3 (one unit) 5 steps 103
// / 108, 6 steps 115 / 112; 64x120x60 (two) 122 / 123, 138 / 129; 300x60x40 (three)
// 6 steps 153 / 160, 7 steps 171 / 170, FP16 169 / 174, 190 / 187; 128x128x64 (four)
// 8 steps 205 / 211, 9 steps 225 / 225; 100x96x90 (five) 9 steps 215 / 215, 10
// steps 234 / 228.
int units_per_wave(const fdtd_ctx *c) { return (5 * c->pa.units - 1) / persist_max_units() + 1; }
int persist_min_steps(const fdtd_ctx *c)
{
    static const int least[5] = {6, 6, 7, 9, 10};
    return least[units_per_wave(c) - 1];
}

// Before a launch of n steps: start over when the step numbers run out.
hipError_t new_epochs(fdtd_ctx *c, int n)
{
    if (c->pa.epoch <= 0xFFFFFFFFu - (std::uint32_t)n - 2u) return hipSuccess;
    c->pa.epoch = 1;
    return hipMemsetAsync(c->pa.ll, 0, c->pll, c->stream);
}

// Steps m0 .. m0 + n - 1, in one launch where the context has the tiles for it
// and the call `least` steps.
hipError_t advance(fdtd_ctx *c, const KArgs &base, int m0, int n, int least)
{
    hipError_t e = hipSuccess;
    if (c->persist && base.lc[3] == 0 && n >= least) {
        PArgs &p = c->pa;
        if ((e = new_epochs(c, n)) != hipSuccess) return e;
        KArgs a = base;
        bind_sets(c, a);
        p.m0 = m0;
        p.n = n;
        p.max_polls = poll_limit();
        if (launch_steps(c, a) == hipSuccess) {
            c->unchecked = true;
            p.epoch += (std::uint32_t)n + 1u;
            return a.rec ? launch_dft(a, (int)c->in.probes.size(), m0, n, c->stream) : hipSuccess;
        }
    }
    for (int m = m0; m < m0 + n && e == hipSuccess; ++m) e = do_step(c, base, m);
    return e;
}

// A context whose last launch gave up a wait holds no state to run on, read
// or save.
int check_state(fdtd_ctx *c)
{
    return c->broken ? fail(c, FDTD_E_STATE, "the state is not valid: a launch gave up a wait (fdtd_reset or "
                            "fdtd_checkpoint_restore starts over)") : FDTD_OK;
}

// After a synchronisation: whether a launch of advance gave up a wait.  The
// flag and the exchange rows are cleared in the order of the context's stream
// (it does not wait for the null stream's work).
int check_advance(fdtd_ctx *c)
{
    if (!c->unchecked) return FDTD_OK;
    int failed = 0;
    HIPCHK(c, hipMemcpy(&failed, c->pa.failed, sizeof failed, hipMemcpyDeviceToHost));
    c->unchecked = false;
    if (!failed) return FDTD_OK;
    c->broken = true;
    HIPCHK(c, hipMemsetAsync(c->pa.failed, 0, sizeof failed, c->stream));
    HIPCHK(c, hipMemsetAsync(c->pa.ll, 0, c->pll, c->stream));
    c->pa.epoch = 1;
    return fail(c, FDTD_E_DEVICE, "a workgroup waited too long for a neighbour's rows; the state is not valid "
                "(fdtd_reset starts over)");
}

// The context's device current on this thread, for a scope.
struct DeviceGuard {
    int was = -1;
    explicit DeviceGuard(int device)
    {
        if (hipGetDevice(&was) != hipSuccess || was == device || hipSetDevice(device) != hipSuccess) was = -1;
    }
    ~DeviceGuard()
    {
        if (was >= 0) (void)hipSetDevice(was);
    }
};

// A stream of one call, drained and destroyed on every return path.
struct StreamGuard {
    hipStream_t s = nullptr;
    ~StreamGuard()
    {
        if (s) {
            (void)hipStreamSynchronize(s);
            (void)hipStreamDestroy(s);
        }
    }
};

// The events of one call, destroyed on every return path.
struct EventSet {
    std::vector<hipEvent_t> v;
    ~EventSet()
    {
        for (hipEvent_t e : v)
            if (e) (void)hipEventDestroy(e);
    }
};

int run_steps(fdtd_ctx *c, int nsteps, bool profile)
{
    if (!c->finalized) return fail(c, FDTD_E_STATE, "fdtd_finalize has not been called");
    if (int rc = check_state(c)) return rc;
    if (nsteps < 0) return fail(c, FDTD_E_INVALID, "nsteps < 0");
    if (c->steps_done + nsteps > c->in.steps_cap)
        return fail(c, FDTD_E_RANGE, "run past the finalized horizon (%d + %d > %d)", c->steps_done, nsteps,
                    c->in.steps_cap);
    EventSet all;
    all.v.assign(2 + (profile ? (size_t)4 * nsteps : 0), nullptr);
    for (auto &e : all.v) HIPCHK(c, hipEventCreate(&e));
    hipEvent_t t0 = all.v[0], t1 = all.v[1];
    hipEvent_t *evs = all.v.data() + 2;
    const int m0 = c->steps_done;
    HIPCHK(c, hipEventRecord(t0, c->stream));
    if (!profile) HIPCHK(c, advance(c, c->ka, m0, nsteps, persist_min_steps(c)));
    for (int s = 0; profile && s < nsteps; ++s)
        HIPCHK(c, do_step(c, c->ka, m0 + s, evs[4 * s + 0], evs[4 * s + 1], evs[4 * s + 2], evs[4 * s + 3]));
    HIPCHK(c, hipEventRecord(t1, c->stream));
    HIPCHK(c, hipEventSynchronize(t1));
    float ms = 0.f;
    HIPCHK(c, hipEventElapsedTime(&ms, t0, t1));
    c->last_run_ms = ms;
    if (int rc = check_advance(c)) return rc;
    if (profile && nsteps > 0) {
        double se = 0, sh = 0;
        for (int s = 0; s < nsteps; ++s) {
            float a = 0, b = 0;
            HIPCHK(c, hipEventElapsedTime(&a, evs[4 * s + 0], evs[4 * s + 1]));
            HIPCHK(c, hipEventElapsedTime(&b, evs[4 * s + 2], evs[4 * s + 3]));
            se += a;
            sh += b;
        }
        c->e_ms = se / nsteps;
        c->h_ms = sh / nsteps;
        c->step_ms = c->e_ms + c->h_ms;
    }
    c->steps_done = m0 + nsteps;
    // blow-up detection on the probe samples of this call
    const size_t np = c->in.probes.size();
    if (np && nsteps > 0) {
        std::vector<float> h(np * (size_t)nsteps);
        HIPCHK(c, hipMemcpy2D(h.data(), (size_t)nsteps * sizeof(float), c->ka.probe_hist + m0,
                              (size_t)c->in.steps_cap * sizeof(float), (size_t)nsteps * sizeof(float), np,
                              hipMemcpyDeviceToHost));
        for (size_t q = 0; q < h.size(); ++q)
            if (!std::isfinite(h[q]))
                return fail(c, FDTD_E_NONFINITE, "probe %zu is non-finite at step %zu", q / nsteps,
                            m0 + q % nsteps);
    }
    return FDTD_OK;
}

uint64_t fnv1a(const unsigned char *p, size_t n, uint64_t h = 1469598103934665603ull)
{
    for (size_t q = 0; q < n; ++q) { h ^= p[q]; h *= 1099511628211ull; }
    return h;
}

struct CkHeader {
    char magic[8];
    int32_t version, nx, ny, nz, storage, step, nprobe, nfreq, steps_cap, pad;
    uint64_t payload, checksum;
};

}  // namespace


// ---- adjoint orchestration --------------------------------------------------
namespace {

// Device memory the forward state occupies (fields + psi), per checkpoint.
size_t state_bytes(const fdtd_ctx *c)
{
    size_t b = 6 * (size_t)c->field_elems * c->esz;
    for (int q = 0; q < 12; ++q) b += c->psi_elems[q] * c->esz;
    return b;
}

int copy_state(fdtd_ctx *c, char *dst, bool save)
{
    size_t off = 0;
    for (int f = 0; f < 6; ++f) {
        const size_t n = (size_t)c->field_elems * c->esz;
        if (save) HIPCHK(c, hipMemcpyAsync(dst + off, fld(c, f), n, hipMemcpyDeviceToDevice, c->stream));
        else HIPCHK(c, hipMemcpyAsync(fld(c, f), dst + off, n, hipMemcpyDeviceToDevice, c->stream));
        off += n;
    }
    for (int q = 0; q < 12; ++q) {
        const size_t n = c->psi_elems[q] * c->esz;
        if (!n) continue;
        if (save) HIPCHK(c, hipMemcpyAsync(dst + off, psv(c, q), n, hipMemcpyDeviceToDevice, c->stream));
        else HIPCHK(c, hipMemcpyAsync(psv(c, q), dst + off, n, hipMemcpyDeviceToDevice, c->stream));
        off += n;
    }
    return FDTD_OK;
}

// The device buffers of one adjoint call: hipMalloc'd and freed on return,
// or (arena set) carved in 256-byte-aligned pieces from the static scratch,
// with no allocation at all.
struct DevBuf {
    std::vector<void *> ptrs;
    uint64_t bytes = 0;
    unsigned char *arena = nullptr;
    size_t arena_cap = 0;
    hipStream_t stream = nullptr;   // the arena's work is queued here
    static size_t rounded(size_t b) { return (std::max<size_t>(b, 256) + 255) / 256 * 256; }
    ~DevBuf()
    {
        // an early return may leave work queued on these buffers
        if (!ptrs.empty()) (void)hipDeviceSynchronize();
        for (void *p : ptrs) (void)hipFree(p);
        if (arena && bytes && stream) (void)hipStreamSynchronize(stream);
    }
    void *get(size_t bytes_)
    {
        const size_t b = rounded(bytes_);
        if (arena) {
            if (bytes + b > arena_cap) return nullptr;
            void *p = arena + bytes;
            bytes += b;
            return p;
        }
        void *p = nullptr;
        if (hipMalloc(&p, b) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        ptrs.push_back(p);
        bytes += b;
        return p;
    }
};

}  // namespace

// Reverse steps in one launch were refused: the call starts over without them.
constexpr int ADJ_AGAIN = 1;

// arena: nullptr allocates the call's buffers with hipMalloc; otherwise they
// are carved from arena (the static scratch, arena_cap bytes), which allows
// one segment only (no checkpoint pool, no second stream).
static int adjoint_call(fdtd_ctx *c, const fdtd_objective *obj, int n_steps, int K, double *J_out, double *grad_out,
                        size_t n_grad, unsigned char *arena, size_t arena_cap)
{
    if (!c->finalized) return fail(c, FDTD_E_STATE, "fdtd_finalize has not been called");
    const SceneIn &in = c->in;
    if (in.design_eps.empty() || !c->dcoef) return fail(c, FDTD_E_STATE, "no design region");
    if (in.storage == FDTD_STORE_BQ16)
        return fail(c, FDTD_E_UNSUPPORTED, "the adjoint runs with FP32, FP16 or BF16 storage, not block-scaled int16");
    if (n_steps < 1 || n_steps > in.steps_cap) return fail(c, FDTD_E_RANGE, "n_steps outside [1, %d]", in.steps_cap);
    // the adjoint sweeps address their FP32 arrays (two guard planes
    // included) and the class map with 32-bit byte offsets
    if ((size_t)c->field_elems * 4 >= ((size_t)1 << 32))
        return fail(c, FDTD_E_UNSUPPORTED, "grid too large for the adjoint: each FP32 adjoint array (with its two "
                    "guard planes) must be under 4 GiB (%zu bytes)", (size_t)c->field_elems * 4);
    const int *d = in.design;
    const int dnx = d[3] - d[0], dny = d[4] - d[1], dnz = d[5] - d[2];
    if (n_grad < (size_t)dnx * dny * dnz) return fail(c, FDTD_E_INVALID, "gradient buffer too small");
    const int *L = in.cpml.thick;
    const int nx = in.nx, ny = in.ny, nz = in.nz;
    // the dilated design box must be updated, CPML-free E edges
    if (d[0] < std::max(1, L[0]) || d[3] >= nx - std::max(1, L[1]) || d[1] < std::max(1, L[2]) ||
        d[4] >= ny - std::max(1, L[3]) || d[2] < std::max(1, L[4]) || d[5] >= nz - std::max(1, L[5]))
        return fail(c, FDTD_E_RANGE, "design region (dilated by one edge) must lie outside the CPML");
    for (const Source &s : in.sources)
        for (int k = s.b[2]; k < s.b[5]; ++k)
            for (int j = s.b[1]; j <= s.b[4]; ++j)
                for (int i = s.b[0]; i <= s.b[3]; ++i)
                    if (i >= d[0] && i <= d[3] && j >= d[1] && j <= d[4] && k >= d[2] && k < d[5])
                        return fail(c, FDTD_E_INVALID, "a source edge touches the design region");
    const int np = (int)in.probes.size(), nf = (int)in.freqs.size();
    if (obj->n_terms < 1) return fail(c, FDTD_E_INVALID, "empty objective");
    for (int t = 0; t < obj->n_terms; ++t) {
        const int p = obj->probe[t], f = obj->freq[t];
        if (p < 0 || p >= np || f < 0 || f >= nf) return fail(c, FDTD_E_RANGE, "objective term %d out of range", t);
        const Probe &pr = in.probes[p];
        if (pr.comp > 2) return fail(c, FDTD_E_INVALID, "objective probes must sample E");
        if (pr.i < std::max(1, L[0]) || pr.i >= nx - std::max(1, L[1]) || pr.j < std::max(1, L[2]) ||
            pr.j >= ny - std::max(1, L[3]) || pr.k < std::max(1, L[4]) || pr.k >= nz - std::max(1, L[5]))
            return fail(c, FDTD_E_INVALID, "objective probe %d lies in the CPML or on a face", p);
    }
    const int n = n_steps;
    const int bx = dnx + 1, by = dny + 1, bz = dnz + 1;
    const i64 nb = (i64)bx * by * bz;
    // adjoint fields (6) and, on narrow grids, every cell's transposed
    // quantities (12 arrays), guard planes included
    const int nq = adj_stores_quantities(nx) ? 12 : 0;
    const size_t adj_bytes = (6 + nq) * (size_t)c->field_elems * 4 + [&] {
        size_t t = 0;
        for (int q = 0; q < 12; ++q) t += c->psi_elems[q] * 4;
        return t;
    }();
    size_t freeb = 0, totb = 0;
    if (K < 0) {
        // automatic: the design history of the whole run when it fits in half
        // the free device memory (no recompute), else checkpoints every
        // ceil(sqrt(n)) steps.  (The fused step's second buffers count as free:
        // they are given back below where the gradient needs them.)
        HIPCHK(c, hipMemGetInfo(&freeb, &totb));
        if (c->fused) freeb += second_bytes(c);
        const size_t all = (size_t)(n + 1) * 3 * nb * sizeof(float) + adj_bytes + (size_t)std::max(np, 1) * n * 4;
        K = all < freeb / 2 ? 0 : (int)std::ceil(std::sqrt((double)n));
    }
    int Kseg = K > 0 ? std::min(K, n) : n;
    const int nseg = (n + Kseg - 1) / Kseg;
    // Small grids: the recompute of a segment in one launch where its steps pay
    // for one (no flag is read after it, so from 4 steps on up to two units a
    // wave), before the reverse steps on the one stream: it holds every CU's LDS,
    // and beside it they slow down by more than it hides.  Shorter segments sweep
    // the light cone.  ms of a gradient of 128 steps, design 6x6x6 (64^3: 8x8x8),
    // in one launch / light cone, by segment length: 64^3 (one unit) 4: 8.7 / 9.1,
    // 6: 6.9 / 7.3, 16: 4.1 / 5.4; 300x60x40 (three) 6: 10.9 / 10.3, 8: 9.3 / 9.3, 16:
    // 7.7 / 8.1; 128x128x64 (four) 8: 11.2 / 10.9, 16: 9.1 / 9.5, 64: 7.9 / 9.1; 100x96x90
    // (five) 8: 11.7 / 11.7, 16: 9.5 / 10.2.
    const int upw = c->persist ? units_per_wave(c) : 0;
    const int least = !c->persist ? 0 : upw <= 2 ? 4 : persist_min_steps(c);
    const bool whole = c->persist && Kseg >= least;
    // All reverse steps of a segment in one launch (a switch of the launched sweeps
    // asks for those), but not of segments of one step, or two up to two units a
    // wave: launched beside the recompute / in one launch after it, ms as above,
    // of one step: 64^3 20.8 / 22.4, 100x96x90 27.3 / 30.9, 128x128x64 27.9 / 28.9; of
    // two: 64^3 12.6 / 13.0, 28x24x22 12.0 / 12.4, 128x128x64 19.4 / 18.8.
    const bool radj = c->radj && Kseg > (upw <= 2 ? 2 : 1) &&
                      !any_set({"FDTD_ADJ_GATHER", "FDTD_ADJ_CHUNKS", "FDTD_ADJ_FUSE", "FDTD_INTERIOR"});
    const size_t hist_bytes = (size_t)(Kseg + 1) * 3 * nb * sizeof(float);
    const size_t ck_bytes = state_bytes(c);
    // segmented runs double-buffer the history: with launched reverse sweeps,
    // segment s-1 is recomputed beside the reverse sweep of segment s
    const int nhist = nseg > 1 ? 2 : 1;
    if (arena) {
        if (nseg > 1)
            return fail(c, FDTD_E_INVALID, "the no-allocation adjoint stores the design history of the whole run: "
                        "checkpoint_every must be 0 or >= n_steps");
        // exactly the pieces carved below, each rounded to 256 bytes
        size_t carve = (6 + nq) * DevBuf::rounded((size_t)c->field_elems * 4) + DevBuf::rounded(hist_bytes) +
                       DevBuf::rounded(3 * nb * sizeof(double)) +
                       DevBuf::rounded((size_t)std::max(np, 1) * n * sizeof(float));
        for (int q = 0; q < 12; ++q) carve += DevBuf::rounded(std::max<size_t>(c->psi_elems[q], 1) * 4);
        if (carve > arena_cap)
            return fail(c, FDTD_E_NOMEM, "the no-allocation adjoint needs %zu bytes of device scratch for this "
                        "run; the static scratch holds %zu (FDTD_NOALLOC_SCRATCH_BYTES)", carve, arena_cap);
    } else {
        HIPCHK(c, hipMemGetInfo(&freeb, &totb));
        const size_t need = nhist * hist_bytes + (size_t)(nseg - 1) * ck_bytes + adj_bytes +
                            (size_t)np * n * 4 + 3 * nb * 8;
        if ((double)need > 0.9 * (double)freeb && c->fused) {   // (memory before the one-pass step)
            release_fused(c);
            HIPCHK(c, hipMemGetInfo(&freeb, &totb));
        }
        if ((double)need > 0.9 * (double)freeb)
            return fail(c, FDTD_E_NOMEM, "adjoint needs %.2f GB of device memory, %.2f GB free; use a larger "
                        "checkpoint interval", need / 1e9, freeb / 1e9);
    }

    DevBuf mem;
    mem.arena = arena;
    mem.arena_cap = arena_cap;
    mem.stream = c->stream;
    AArgs b{};
    for (int q = 0; q < 3; ++q) {
        char *e = (char *)mem.get((size_t)c->field_elems * 4);
        char *h = (char *)mem.get((size_t)c->field_elems * 4);
        if (!e || !h) return fail(c, FDTD_E_NOMEM, "adjoint field allocation failed");
        HIPCHK(c, hipMemsetAsync(e, 0, (size_t)c->field_elems * 4, c->stream));
        HIPCHK(c, hipMemsetAsync(h, 0, (size_t)c->field_elems * 4, c->stream));
        b.eb[q] = (float *)(e + (size_t)c->ka.plane * 4);
        b.hb[q] = (float *)(h + (size_t)c->ka.plane * 4);
        b.ebn[q] = b.eb[q];   // in place unless the fused interior sweep is set up below
        b.hbn[q] = b.hb[q];
    }
    for (int q = 0; q < (radj ? 0 : nq); ++q) {   // (one launch keeps them in LDS)
        char *t = (char *)mem.get((size_t)c->field_elems * 4);
        if (!t) return fail(c, FDTD_E_NOMEM, "adjoint transposed-quantity allocation failed");
        HIPCHK(c, hipMemsetAsync(t, 0, (size_t)c->field_elems * 4, c->stream));
        (q < 6 ? b.hq[q] : b.eq[q - 6]) = (float *)(t + (size_t)c->ka.plane * 4);
    }
    for (int q = 0; q < 12; ++q) {
        b.pb[q] = (float *)mem.get(std::max<size_t>(c->psi_elems[q], 1) * 4);
        if (!b.pb[q]) return fail(c, FDTD_E_NOMEM, "adjoint psi allocation failed");
        HIPCHK(c, hipMemsetAsync(b.pb[q], 0, std::max<size_t>(c->psi_elems[q], 1) * 4, c->stream));
    }
    float *hbuf[2] = {(float *)mem.get(hist_bytes), nhist > 1 ? (float *)mem.get(hist_bytes) : nullptr};
    float *hist = hbuf[0];
    double *gedge = (double *)mem.get(3 * nb * sizeof(double));
    float *gdev = (float *)mem.get((size_t)std::max(np, 1) * n * sizeof(float));
    char *pool = nseg > 1 ? (char *)mem.get((size_t)(nseg - 1) * ck_bytes) : nullptr;
    if (!hist || (nhist > 1 && !hbuf[1]) || !gedge || !gdev || (nseg > 1 && !pool))
        return fail(c, FDTD_E_NOMEM, "adjoint buffers");
    for (int q = 0; q < nhist; ++q) HIPCHK(c, hipMemsetAsync(hbuf[q], 0, hist_bytes, c->stream));
    HIPCHK(c, hipMemsetAsync(gedge, 0, 3 * nb * sizeof(double), c->stream));
    b.gsteps = n;
    b.g = gdev;
    b.hist = hist;
    b.dcoef = c->dcoef;
    b.gedge = gedge;
    b.sb[0] = d[0]; b.sb[1] = d[1]; b.sb[2] = d[2]; b.sb[3] = bx; b.sb[4] = by; b.sb[5] = bz;
    b.src_j0 = c->built.src_j0;
    b.src_j1 = c->built.src_j1;

    int rc = zero_state(c);
    if (rc) return rc;
    KArgs fa = c->ka;               // forward arguments
    fa.sb[0] = d[0]; fa.sb[1] = d[1]; fa.sb[2] = d[2]; fa.sb[3] = bx; fa.sb[4] = by; fa.sb[5] = bz;
    KArgs aa = c->ka;               // adjoint arguments: SI tables
    if (const char *ov = std::getenv("FDTD_ADJ_CHUNKS")) {
        const int nch = std::max(1, std::min(std::atoi(ov), nz));
        aa.kchunk = (nz + nch - 1) / nch;
    } else {
        // z-blocks of the adjoint sweeps: those of the forward E sweep, halved
        // until a launch has 2048 workgroups (8 per CU: the reverse sweeps of a
        // small grid are latency-bound).  Measured on 128x128x64, 1000 steps,
        // stored history: 4-plane blocks 83.0 ms, 2-plane 78.3, 1-plane 78.2.
        const int tiles = ((nx + tile_cols() - 1) / tile_cols()) * ((ny + tile_rows() - 1) / tile_rows());
        while (aa.kchunk > 1 && (long)tiles * ((nz + aa.kchunk - 1) / aa.kchunk) < 2048) aa.kchunk /= 2;
    }
    aa.etab = c->etab_si;
    aa.htab = c->htab_si;
    aa.srcs = c->srcs_si;
    // interior / general split of the adjoint sweeps (FDTD_INTERIOR=0: general only)
    {
        const char *ev = std::getenv("FDTD_INTERIOR");
        aa.ib[0] = (ev && std::strcmp(ev, "0") == 0) ? -1 : 0;
    }
    const int mode = c->built.mode;
    const int euni = c->built.e_uniform ? 1 : 0, huni = c->built.h_uniform ? 1 : 0;
    // fused interior sweep (LDS gather path, one H class, FDTD_ADJ_FUSE=0
    // disables): its tile columns and the others, and the second dJ/dE,
    // dJ/dH buffers it writes (the pair is swapped after every step).  Not
    // with the no-allocation scratch, nor when the pair would take more than
    // half the free memory, nor where all steps of a segment run in one launch
    // (in place: a swap would leave the next segment the zeros of the second
    // buffers).
    bool pp = false;
    {
        const char *fv = std::getenv("FDTD_ADJ_FUSE");
        const bool want = !(fv && std::strcmp(fv, "0") == 0);
        std::vector<int> quiet, noisy;
        if (want && !arena && !radj && huni && !adj_stores_quantities(nx) && aa.ib[0] >= 0)
            adj_fuse_tiles(aa, c->built.e_first, c->built.h_first, b.sb, quiet, noisy);
        const size_t pair_bytes = 6 * (size_t)c->field_elems * 4 + (quiet.size() + noisy.size() + 2) * 4;
        if (!quiet.empty()) HIPCHK(c, hipMemGetInfo(&freeb, &totb));
        if (!quiet.empty() && c->fused && pair_bytes >= freeb / 2 && pair_bytes < (freeb + second_bytes(c)) / 2) {
            release_fused(c);   // (the same choice as without them)
            HIPCHK(c, hipMemGetInfo(&freeb, &totb));
        }
        if (!quiet.empty() && pair_bytes < freeb / 2) {
            for (int q = 0; q < 6; ++q) {
                char *f = (char *)mem.get((size_t)c->field_elems * 4);
                if (!f) return fail(c, FDTD_E_NOMEM, "adjoint field allocation failed");
                HIPCHK(c, hipMemsetAsync(f, 0, (size_t)c->field_elems * 4, c->stream));
                (q < 3 ? b.ebn[q] : b.hbn[q - 3]) = (float *)(f + (size_t)c->ka.plane * 4);
            }
            int *fl = (int *)mem.get(quiet.size() * 4);
            int *tl = (int *)mem.get(std::max<size_t>(noisy.size(), 1) * 4);
            if (!fl || !tl) return fail(c, FDTD_E_NOMEM, "adjoint tile lists");
            HIPCHK(c, hipMemcpyAsync(fl, quiet.data(), quiet.size() * 4, hipMemcpyHostToDevice, c->stream));
            if (!noisy.empty())
                HIPCHK(c, hipMemcpyAsync(tl, noisy.data(), noisy.size() * 4, hipMemcpyHostToDevice, c->stream));
            HIPCHK(c, hipStreamSynchronize(c->stream));   // the host vectors go out of scope
            b.fl = fl;
            b.nfl = (int)quiet.size();
            b.tl = tl;
            b.ntl = (int)noisy.size();
            pp = true;
        }
    }
    // after a step the buffers just written hold the current state
    auto swap_e = [&]() { for (int q = 0; q < 3; ++q) std::swap(b.eb[q], b.ebn[q]); };
    auto swap_h = [&]() { for (int q = 0; q < 3; ++q) std::swap(b.hb[q], b.hbn[q]); };

    hipEvent_t t0 = c->adj_ev[0], t1 = c->adj_ev[1], t2 = c->adj_ev[2];
    // second stream (default priority) for the reverse sweeps of a segmented
    // run, and the events that order it against the recompute stream:
    // ready[q] = history buffer q filled, freed[q] = its reverse sweep done
    StreamGuard rsg;
    EventSet sync;
    hipStream_t rs = c->stream;
    if (nseg > 1) {
        if (!whole && !radj) {
            HIPCHK(c, hipStreamCreateWithFlags(&rsg.s, hipStreamNonBlocking));
            rs = rsg.s;
        }
        sync.v.assign(4, nullptr);
        for (auto &e : sync.v) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    HIPCHK(c, hipEventRecord(t0, c->stream));
    // ---- forward pass: DFT at the probes; checkpoints at segment starts, or
    // the whole design history when there is a single segment
    fa.rec = 1;
    fa.snap = nseg == 1 ? hist : nullptr;
    fa.snap_base = 0;
    for (int m = 0; m < n; m += Kseg) {
        if (nseg > 1 && m > 0)
            if ((rc = copy_state(c, pool + (size_t)(m / Kseg - 1) * ck_bytes, true))) return rc;
        HIPCHK(c, advance(c, fa, m, std::min(Kseg, n - m), least));
    }
    HIPCHK(c, hipEventRecord(t1, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if ((rc = check_advance(c))) return rc;
    c->steps_done = n;
    // ---- objective J = sum w |X|^2 and dJ/ds[m] = sum w 2 Re(conj(X) phasor[m])
    std::vector<double> X((size_t)np * nf * 2);
    if (np && nf) HIPCHK(c, hipMemcpy(X.data(), c->ka.dft, X.size() * sizeof(double), hipMemcpyDeviceToHost));
    std::vector<float> g((size_t)np * n, 0.0f);
    std::vector<double> gd((size_t)np * n, 0.0);
    double J = 0.0;
    for (int t = 0; t < obj->n_terms; ++t) {
        const int p = obj->probe[t], f = obj->freq[t];
        const double w = obj->weight ? obj->weight[t] : 1.0;
        const double xr = X[((size_t)p * nf + f) * 2], xi = X[((size_t)p * nf + f) * 2 + 1];
        J += w * (xr * xr + xi * xi);
        for (int m = 0; m < n; ++m) {
            const double pr = c->built.phasor[((size_t)m * nf + f) * 2], pi = c->built.phasor[((size_t)m * nf + f) * 2 + 1];
            gd[(size_t)p * n + m] += w * 2.0 * (xr * pr + xi * pi);
        }
    }
    for (size_t q = 0; q < g.size(); ++q) g[q] = (float)gd[q];
    HIPCHK(c, hipMemcpyAsync(gdev, g.data(), g.size() * sizeof(float), hipMemcpyHostToDevice, c->stream));
    // ---- reverse sweep, segment by segment.  Segmented: the forward state of
    // segment sgi is recomputed from its checkpoint on c->stream into history
    // buffer sgi % 2 while the reverse sweep of segment sgi + 1 runs on rs.
    // A step moves information one cell per axis (E reads H at i-1, H reads E
    // at i+1), so over a segment of at most Kseg steps the design history
    // depends only on the checkpoint within Kseg + 1 cells of the snapshot
    // box: the recompute sweeps that box alone, dilated by Kseg + 2 at a
    // segment's first step and a cell less at each later one, whenever the
    // step's box holds under 60 % of the grid's cells (the light-cone tiles
    // run the general variant; a larger box runs the whole grid).
    // FDTD_LIGHTCONE=0: the whole grid always; FDTD_LIGHTCONE=fixed: the
    // first box for every step.  Cells outside it keep stale values, and every
    // segment restarts from a full checkpoint.
    const char *lce = std::getenv("FDTD_LIGHTCONE");
    const bool lc_on = nseg > 1 && !whole && !(lce && std::strcmp(lce, "0") == 0);
    const bool lc_fixed = lce && std::strcmp(lce, "fixed") == 0;
    // the box dilated by R, or all zero (the whole grid)
    auto cone = [&](int R, int lc[6]) {
        const int lo[3] = {std::max(0, d[0] - R), std::max(0, d[1] - R), std::max(0, d[2] - R)};
        const int hi[3] = {std::min(nx, d[0] + bx + R), std::min(ny, d[1] + by + R), std::min(nz, d[2] + bz + R)};
        const double frac = (double)(hi[0] - lo[0]) * (hi[1] - lo[1]) * (hi[2] - lo[2]) / ((double)nx * ny * nz);
        const bool use = lc_on && frac < 0.6;
        for (int v = 0; v < 3; ++v) {
            lc[v] = use ? lo[v] : 0;
            lc[v + 3] = use ? hi[v] : 0;
        }
    };
    auto recompute = [&](int sgi) -> int {
        const int s0 = sgi * Kseg, s1 = std::min(n, s0 + Kseg), q = sgi % 2;
        if (sgi + 2 < nseg) HIPCHK(c, hipStreamWaitEvent(c->stream, sync.v[2 + q], 0));   // buffer q free
        if (sgi == 0) {
            for (int f = 0; f < 6; ++f)
                HIPCHK(c, hipMemsetAsync(fld(c, f), 0, (size_t)c->field_elems * c->esz, c->stream));
            for (int p = 0; p < 12; ++p)
                if (c->psi_elems[p]) HIPCHK(c, hipMemsetAsync(psv(c, p), 0, c->psi_elems[p] * c->esz, c->stream));
        } else {
            const int r = copy_state(c, pool + (size_t)(sgi - 1) * ck_bytes, false);
            if (r) return r;
        }
        KArgs ra = fa;
        ra.rec = 0;
        ra.snap = hbuf[q];
        ra.snap_base = s0;
        cone(Kseg + 2, ra.lc);
        bind_sets(c, ra);
        HIPCHK(c, launch_snap(in.storage, ra, hbuf[q], 0, c->stream));
        for (int m = s0, runs = 0; m < s1; m += runs) {
            runs = 1;
            // the cone narrows a cell per step: step m feeds only the
            // snapshots of steps m .. s1-1, so the design box dilated by
            // s1 - m + 2 (Kseg + 2 at most) suffices
            if (!lc_fixed) cone(s1 - m + 2, ra.lc);
            if (whole) runs = s1 - m;
            HIPCHK(c, advance(c, ra, m, runs, least));
        }
        HIPCHK(c, hipEventRecord(sync.v[q], c->stream));   // buffer q ready
        return FDTD_OK;
    };
    if (nseg > 1 && (rc = recompute(nseg - 1))) return rc;
    for (int sgi = nseg - 1; sgi >= 0; --sgi) {
        const int s0 = sgi * Kseg, s1 = std::min(n, s0 + Kseg), q = sgi % 2;
        if (nseg > 1) HIPCHK(c, hipStreamWaitEvent(rs, sync.v[q], 0));
        b.hist = hbuf[q];
        b.hist_base = s0;
        if (radj) {
            RArgs &r = c->ra;
            HIPCHK(c, new_epochs(c, s1 - s0));
            r.m1 = s1 - 1;
            r.n = s1 - s0;
            r.max_polls = poll_limit();
            r.epoch = c->pa.epoch;
            if (coop_refused(c) || launch_adj_persist(aa, b, r, c->ptiles, c->rlds, rs) != hipSuccess) {
                (void)hipGetLastError();
                c->persist = c->radj = false;
                return ADJ_AGAIN;
            }
            c->unchecked = true;
            c->pa.epoch += (std::uint32_t)r.n + 1u;
        }
        for (int m = s1 - 1; !radj && m >= s0; --m) {
            const int fst = m < s1 - 1 ? m + 1 : -1;
            HIPCHK(c, launch_adj(true, mode, euni, huni, aa, b, m, fst, 1, rs));
            HIPCHK(c, launch_adj(false, mode, euni, huni, aa, b, m, -1, 1, rs));
            if (pp) {
                swap_e();
                swap_h();
            }
        }
        if (!radj) HIPCHK(c, launch_adj(true, mode, euni, huni, aa, b, s0, s0, 0, rs));
        if (pp) swap_e();
        if (nseg > 1) {
            HIPCHK(c, hipEventRecord(sync.v[2 + q], rs));   // buffer q free
            if (sgi > 0 && (rc = recompute(sgi - 1))) return rc;
        }
    }
    if (nseg > 1) {
        HIPCHK(c, hipEventRecord(sync.v[2], rs));
        HIPCHK(c, hipStreamWaitEvent(c->stream, sync.v[2], 0));
    }
    HIPCHK(c, hipEventRecord(t2, c->stream));
    HIPCHK(c, hipEventSynchronize(t2));
    if ((rc = check_advance(c))) return rc;
    float ms1 = 0.f, ms2 = 0.f;
    HIPCHK(c, hipEventElapsedTime(&ms1, t0, t1));
    HIPCHK(c, hipEventElapsedTime(&ms2, t0, t2));
    c->adj_fwd_ms = ms1;
    c->adj_total_ms = ms2;
    c->adj_segments = nseg;
    c->adj_bytes = c->dev_bytes + mem.bytes;
    // ---- chain rule through the 4-cell averages (fdtdrav.h:1135-1177)
    std::vector<double> ge((size_t)3 * nb);
    HIPCHK(c, hipMemcpy(ge.data(), gedge, ge.size() * sizeof(double), hipMemcpyDeviceToHost));
    auto q = [&](int a_, int b_, int c_) { return (size_t)(a_ + (i64)bx * (b_ + (i64)by * c_)); };
    for (int k = 0; k < dnz; ++k)
        for (int j = 0; j < dny; ++j)
            for (int i = 0; i < dnx; ++i) {
                double acc = 0.0;
                for (int u = 0; u < 2; ++u)
                    for (int v = 0; v < 2; ++v) {
                        acc += ge[q(i, j + u, k + v)];
                        acc += ge[(size_t)nb + q(i + u, j, k + v)];
                        acc += ge[(size_t)2 * nb + q(i + u, j + v, k)];
                    }
                grad_out[i + (size_t)dnx * (j + (size_t)dny * k)] = 0.25 * acc;
            }
    *J_out = J;
    // leave the context as after an uninterrupted forward run of n steps
    // when there was a single segment; otherwise rewind it
    if (nseg > 1) return zero_state(c);
    return FDTD_OK;
}

int run_adjoint(fdtd_ctx *c, const fdtd_objective *obj, int n_steps, int K, double *J_out, double *grad_out,
                size_t n_grad, unsigned char *arena = nullptr, size_t arena_cap = 0)
{
    const int rc = adjoint_call(c, obj, n_steps, K, J_out, grad_out, n_grad, arena, arena_cap);
    return rc == ADJ_AGAIN ? adjoint_call(c, obj, n_steps, K, J_out, grad_out, n_grad, arena, arena_cap) : rc;
}

// ============================================================================
extern "C" {

const char *fdtd_last_error(const fdtd_ctx *ctx) { return ctx ? ctx->err.c_str() : g_create_err; }

int fdtd_create(const fdtd_grid *g, int storage, fdtd_ctx **out)
{
    if (!out) return create_fail(FDTD_E_INVALID, "null output pointer");
    *out = nullptr;
    if (!g) return create_fail(FDTD_E_INVALID, "null grid");
    if (g->nx < 4 || g->ny < 4 || g->nz < 4)
        return create_fail(FDTD_E_INVALID, "the grid needs at least 4 cells along each axis (got %d x %d x %d)", g->nx,
                           g->ny, g->nz);
    if (!(g->dx > 0) || !(g->dy > 0) || !(g->dz > 0))
        return create_fail(FDTD_E_INVALID, "cell sizes must be positive");
    if (storage < FDTD_STORE_F32 || storage > FDTD_STORE_BQ16)
        return create_fail(FDTD_E_INVALID, "unknown storage form %d", storage);
    double eps0 = g->eps0 > 0 ? g->eps0 : 8.854187817e-12;
    double mu0 = g->mu0 > 0 ? g->mu0 : 4.0 * M_PI * 1e-7;
    double dt = g->dt;
    const double cfl = 1.0 / ((1.0 / std::sqrt(mu0 * eps0)) *
                              std::sqrt(1.0 / (g->dx * g->dx) + 1.0 / (g->dy * g->dy) + 1.0 / (g->dz * g->dz)));
    if (!(dt > 0)) {
        if (!(g->courant > 0) || g->courant > 1.0)
            return create_fail(FDTD_E_INVALID, "courant must lie in (0, 1] when dt is not given");
        dt = g->courant * cfl;
    } else if (dt > cfl * (1.0 + 4.0 * FLT_EPSILON)) {
        // above the 3-D Courant limit: unstable.  A dt computed in float at
        // Courant factor 1 (source.cu:45-46 built as C++, where sqrt of a
        // float is a float) lands a few float ulps either side of the double
        // limit, so the test allows float resolution.
        return create_fail(FDTD_E_INVALID, "dt %.9g s is above the 3-D Courant limit %.9g s", dt, cfl);
    }
    fdtd_ctx *c = new (std::nothrow) fdtd_ctx();
    if (!c) return create_fail(FDTD_E_NOMEM, "out of host memory");
    SceneIn &in = c->in;
    in.nx = g->nx; in.ny = g->ny; in.nz = g->nz;
    in.px = (g->nx + 63) / 64 * 64;
    in.dx = g->dx; in.dy = g->dy; in.dz = g->dz;
    in.dt = dt; in.eps0 = eps0; in.mu0 = mu0;
    in.storage = storage;
    in.cpml = CpmlParams{{0, 0, 0, 0, 0, 0}, 3.0, {0, 0, 0}, 1.5, 5.0, 0.05, 0.0};
    for (int q = 0; q < 6; ++q) in.design[q] = 0;
    in.steps_cap = 0;
    if (hipGetDevice(&c->device) != hipSuccess ||
        hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        (void)hipGetLastError();
        delete c;
        return create_fail(FDTD_E_DEVICE, "no HIP device");
    }
    for (hipEvent_t &e : c->adj_ev)
        if (hipEventCreate(&e) != hipSuccess) {
            (void)hipGetLastError();
            fdtd_destroy(c);
            return create_fail(FDTD_E_DEVICE, "hipEventCreate failed");
        }
    // the no-allocation adjoint's scratch on this (current) device
    c->scratch = scratch_address(c->device);
    *out = c;
    return FDTD_OK;
}

int fdtd_destroy(fdtd_ctx *c)
{
    if (!c) return FDTD_E_INVALID;
    free_device(c);
    for (hipEvent_t e : c->adj_ev)
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : c->stage_ev)
        if (e) (void)hipEventDestroy(e);
    if (c->stage) (void)hipHostFree(c->stage);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return FDTD_OK;
}

int fdtd_set_cpml(fdtd_ctx *c, const fdtd_cpml *p)
{
    if (!c || !p) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    const int n[3] = {c->in.nx, c->in.ny, c->in.nz};
    for (int a = 0; a < 3; ++a) {
        const int lo = p->thick[2 * a], hi = p->thick[2 * a + 1];
        if (lo < 0 || hi < 0 || lo + hi > n[a] - 2)
            return fail(c, FDTD_E_INVALID, "CPML widths %d+%d do not fit axis %d of %d cells", lo, hi, a, n[a]);
    }
    if (!(p->order >= 0) || !(p->kappa_max >= 1) || !(p->alpha_max >= 0) || !(p->alpha_min >= 0))
        return fail(c, FDTD_E_INVALID, "invalid CPML grading parameters");
    CpmlParams &q = c->in.cpml;
    for (int a = 0; a < 6; ++a) q.thick[a] = p->thick[a];
    q.order = p->order;
    for (int a = 0; a < 3; ++a) q.sigma_max[a] = p->sigma_max[a];
    q.sigma_factor = p->sigma_factor > 0 ? p->sigma_factor : 1.5;
    q.kappa_max = p->kappa_max;
    q.alpha_max = p->alpha_max;
    q.alpha_min = p->alpha_min;
    c->cpml_set = true;
    return FDTD_OK;
}

int fdtd_add_box(fdtd_ctx *c, int is, int js, int ks, int ie, int je, int ke, const float eps_r[3],
                 const float sigma_e[3], const float mu_r[3], const float sigma_m[3])
{
    if (!c || !eps_r || !sigma_e || !mu_r || !sigma_m) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    for (int q = 0; q < 3; ++q) {
        if (!(eps_r[q] > 0) || !(mu_r[q] > 0) || !(sigma_e[q] >= 0) || !(sigma_m[q] >= 0) ||
            !std::isfinite(eps_r[q]) || !std::isfinite(mu_r[q]) || !std::isfinite(sigma_e[q]) ||
            !std::isfinite(sigma_m[q]))
            return fail(c, FDTD_E_INVALID, "invalid material values");
    }
    Box b;
    b.b[0] = is; b.b[1] = js; b.b[2] = ks; b.b[3] = ie; b.b[4] = je; b.b[5] = ke;
    for (int q = 0; q < 3; ++q) {
        b.mat[q] = eps_r[q];
        b.mat[3 + q] = sigma_e[q];
        b.mat[6 + q] = mu_r[q];
        b.mat[9 + q] = sigma_m[q];
    }
    c->in.boxes.push_back(b);
    return FDTD_OK;
}

int fdtd_add_sector(fdtd_ctx *c, int i0, int j0, int i1, int j1, int i2, int j2, int kz, float radius, int max_x,
                    int max_y, float sigma_x, float sigma_y)
{
    if (!c) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (!(radius > 0) || !std::isfinite(radius)) return fail(c, FDTD_E_INVALID, "sector radius must be > 0");
    if (!(sigma_x >= 0) || !(sigma_y >= 0) || !std::isfinite(sigma_x) || !std::isfinite(sigma_y))
        return fail(c, FDTD_E_INVALID, "invalid sector sigma");
    if (kz < 1 || kz > c->in.nz - 2 || max_x < 0 || max_x >= c->in.nx || max_y < 0 || max_y >= c->in.ny)
        return fail(c, FDTD_E_RANGE, "sector plane %d or extent (%d, %d) outside the grid", kz, max_x, max_y);
    const int lim = 1 << 24;   // node coordinates stay exact in float
    for (int v : {i0, j0, i1, j1, i2, j2})
        if (v <= -lim || v >= lim) return fail(c, FDTD_E_RANGE, "sector point index out of range");
    c->in.sectors.push_back(Sector{{i0, j0, i1, j1, i2, j2}, kz, max_x, max_y, radius, {sigma_x, sigma_y}});
    return FDTD_OK;
}

int fdtd_add_plate(fdtd_ctx *c, int axis, int is, int js, int ks, int ie, int je, int ke, const float sigma[3])
{
    if (!c || !sigma) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (axis < 1 || axis > 3) return fail(c, FDTD_E_INVALID, "plate axis must be 1, 2 or 3");
    for (int q = 0; q < 3; ++q)
        if (!(sigma[q] >= 0) || !std::isfinite(sigma[q])) return fail(c, FDTD_E_INVALID, "invalid plate sigma");
    if (is < 0 || js < 0 || ks < 0 || ie >= c->in.nx || je >= c->in.ny || ke >= c->in.nz || is > ie || js > je ||
        ks > ke)
        return fail(c, FDTD_E_RANGE, "plate (%d,%d,%d)-(%d,%d,%d) outside the grid", is, js, ks, ie, je, ke);
    Plate p{axis, {is, js, ks, ie, je, ke}, {sigma[0], sigma[1], sigma[2]}};
    c->in.plates.push_back(p);
    return FDTD_OK;
}

int fdtd_add_resistor(fdtd_ctx *c, int dir, int is, int js, int ks, int ie, int je, int ke, double R)
{
    if (!c) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (dir != 3) return fail(c, FDTD_E_UNSUPPORTED, "only z-directed resistors (dir = 3) are built");
    if (!(R > 0) || !std::isfinite(R)) return fail(c, FDTD_E_INVALID, "resistance must be > 0");
    const SceneIn &in = c->in;
    if (is < 1 || js < 1 || ks < 0 || ie > in.nx - 2 || je > in.ny - 2 || ke > in.nz - 1 || is > ie || js > je ||
        ks >= ke)
        return fail(c, FDTD_E_RANGE, "resistor edges (%d,%d,%d)-(%d,%d,%d) outside the updated Ez edges", is, js, ks,
                    ie, je, ke);
    Resistor r{{is, js, ks, ie, je, ke}, R};
    c->in.resistors.push_back(r);
    return FDTD_OK;
}

int fdtd_add_lumped_source(fdtd_ctx *c, int dir, int is, int js, int ks, int ie, int je, int ke, double R,
                           const fdtd_waveform *w)
{
    if (!c || !w) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (dir != 3 && dir != 1) return fail(c, FDTD_E_UNSUPPORTED, "lumped sources are x- (dir = 1) or z-directed (dir = 3)");
    if (!(R > 0) || !std::isfinite(R)) return fail(c, FDTD_E_INVALID, "source resistance must be > 0");
    if (w->type < FDTD_WAVE_GAUSSIAN || w->type > FDTD_WAVE_SINE)
        return fail(c, FDTD_E_INVALID, "unknown waveform type %d", w->type);
    if ((w->type != FDTD_WAVE_SINE && !(w->tau > 0)) || !std::isfinite(w->amp))
        return fail(c, FDTD_E_INVALID, "invalid waveform parameters");
    if (dir == 1) {
        // defineSourceX's loaded edges: is<=i<ie, js<=j<=ie, ks<=k<=ke, all updated Ex
        // edges (i<nx-1, 0<j<ny-1, 0<k<nz-1); calc_e's Ez injection still runs on the
        // box's Ez edges is<=i<=ie, js<=j<=je, ks<=k<ke (none when ks == ke)
        if (is >= ie || js > ie || js > je || ks > ke) return fail(c, FDTD_E_INVALID, "empty x-source box (needs ie > is)");
        if (is < 1 || ie > c->in.nx - 2 || js < 1 || std::max(ie, je) > c->in.ny - 2 || ks < 1 || ke > c->in.nz - 2)
            return fail(c, FDTD_E_RANGE, "x-source box outside the updated Ex / Ez region");
    } else {
        if (is > ie || js > je || ks >= ke) return fail(c, FDTD_E_INVALID, "empty source box");
        // every edge must be an updated Ez edge: 0<i<nx-1, 0<j<ny-1, k<nz-1
        if (is < 1 || ie > c->in.nx - 2 || js < 1 || je > c->in.ny - 2 || ks < 0 || ke > c->in.nz - 1)
            return fail(c, FDTD_E_RANGE, "source box outside the updated Ez region");
    }
    Source s;
    s.dir = dir;
    s.b[0] = is; s.b[1] = js; s.b[2] = ks; s.b[3] = ie; s.b[4] = je; s.b[5] = ke;
    s.R = R;
    s.wtype = w->type;
    s.amp = w->amp; s.t0 = w->t0; s.tau = w->tau; s.freq = w->freq;
    c->in.sources.push_back(s);
    return FDTD_OK;
}

int fdtd_add_probe(fdtd_ctx *c, int comp, int i, int j, int k, int *index)
{
    if (!c) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (comp < FDTD_EX || comp > FDTD_HZ) return fail(c, FDTD_E_INVALID, "invalid component %d", comp);
    if (!box_in_grid(c, i, j, k)) return fail(c, FDTD_E_RANGE, "probe (%d,%d,%d) outside the grid", i, j, k);
    if (index) *index = (int)c->in.probes.size();
    c->in.probes.push_back(Probe{comp, i, j, k});
    return FDTD_OK;
}

int fdtd_set_dft(fdtd_ctx *c, int nfreq, const double *freqs)
{
    if (!c || nfreq < 0 || (nfreq > 0 && !freqs)) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    for (int f = 0; f < nfreq; ++f)
        if (!std::isfinite(freqs[f])) return fail(c, FDTD_E_INVALID, "non-finite DFT frequency");
    c->in.freqs.assign(freqs, freqs + nfreq);
    return FDTD_OK;
}

int fdtd_set_design_region(fdtd_ctx *c, int is, int js, int ks, int ie, int je, int ke)
{
    if (!c) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (is < 0 || js < 0 || ks < 0 || ie > c->in.nx || je > c->in.ny || ke > c->in.nz || is >= ie || js >= je ||
        ks >= ke)
        return fail(c, FDTD_E_RANGE, "design region outside the grid or empty");
    int *d = c->in.design;
    d[0] = is; d[1] = js; d[2] = ks; d[3] = ie; d[4] = je; d[5] = ke;
    c->in.design_eps.assign((size_t)(ie - is) * (je - js) * (ke - ks), 1.0f);
    return FDTD_OK;
}

int fdtd_set_design_eps(fdtd_ctx *c, const float *eps, size_t n)
{
    if (!c || !eps) return FDTD_E_INVALID;
    if (c->in.design_eps.empty()) return fail(c, FDTD_E_STATE, "no design region");
    if (n != c->in.design_eps.size()) return fail(c, FDTD_E_INVALID, "design eps has %zu cells, expected %zu", n,
                                                  c->in.design_eps.size());
    for (size_t q = 0; q < n; ++q)
        if (!(eps[q] > 0) || !std::isfinite(eps[q])) return fail(c, FDTD_E_INVALID, "invalid design eps_r");
    std::memcpy(c->in.design_eps.data(), eps, n * sizeof(float));
    if (!c->finalized) return FDTD_OK;
    // rebuild every table on the new materials and restart from step 0
    free_device(c);
    c->finalized = false;
    const int rc = do_finalize(c);
    if (rc) free_device(c);
    return rc;
}

int fdtd_finalize(fdtd_ctx *c, int n_steps)
{
    if (!c) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "already finalized");
    if (n_steps < 1) return fail(c, FDTD_E_INVALID, "n_steps must be >= 1");
    c->in.steps_cap = n_steps;
    int rc = do_finalize(c);
    if (rc) free_device(c);
    return rc;
}

int fdtd_run(fdtd_ctx *c, int nsteps)
{
    if (!c) return FDTD_E_INVALID;
    return run_steps(c, nsteps, false);
}

int fdtd_step(fdtd_ctx *c)
{
    if (!c) return FDTD_E_INVALID;
    return run_steps(c, 1, false);
}

int fdtd_profile(fdtd_ctx *c, int nsteps)
{
    if (!c) return FDTD_E_INVALID;
    return run_steps(c, nsteps, true);
}

int fdtd_reset(fdtd_ctx *c)
{
    if (!c) return FDTD_E_INVALID;
    if (!c->finalized) return fail(c, FDTD_E_STATE, "fdtd_finalize has not been called");
    return zero_state(c);
}

int fdtd_get_info(const fdtd_ctx *c, fdtd_info *o)
{
    if (!c || !o) return FDTD_E_INVALID;
    std::memset(o, 0, sizeof *o);
    o->nx = c->in.nx; o->ny = c->in.ny; o->nz = c->in.nz;
    o->steps_done = c->steps_done;
    o->steps_capacity = c->in.steps_cap;
    o->n_probes = (int)c->in.probes.size();
    o->n_freqs = (int)c->in.freqs.size();
    o->n_sources = (int)c->in.sources.size();
    o->n_classes = c->built.ncls;
    o->storage = c->in.storage;
    o->dt = c->in.dt;
    o->last_run_ms = c->last_run_ms;
    o->e_kernel_ms = c->e_ms;
    o->h_kernel_ms = c->h_ms;
    o->step_kernel_ms = c->step_ms;
    o->interior_split = c->box[0][5] > c->box[0][2] ? 1 : 0;
    o->device_bytes = c->dev_bytes;
    // algorithmic bytes per cell: E sweep reads E, H and writes E (9 values);
    // H sweep likewise; plus one class index per cell in a classed sweep and
    // psi read+write over the slabs (averaged over the grid).
    // block-scaled storage: 2 bytes per value plus BQ_STRIDE exponent bytes
    // per 8 cells of the three components; its psi is FP16
    const double s = c->in.storage == FDTD_STORE_BQ16 ? 2.0 + (double)BQ_STRIDE / (3 * BQ_BLOCK) : (double)c->esz;
    const double sp = (double)c->esz;
    const double fx = (double)(c->in.cpml.thick[0] + c->in.cpml.thick[1]) / c->in.nx;
    const double fy = (double)(c->in.cpml.thick[2] + c->in.cpml.thick[3]) / c->in.ny;
    const double fz = (double)(c->in.cpml.thick[4] + c->in.cpml.thick[5]) / c->in.nz;
    const double psi = 4.0 * sp * (fx + fy + fz);
    const double cls = c->built.mode == CLS_U16 ? 2.0 : c->built.mode == CLS_U32 ? 4.0 : 0.0;
    o->adjoint_forward_ms = c->adj_fwd_ms;
    o->adjoint_total_ms = c->adj_total_ms;
    o->adjoint_segments = c->adj_segments;
    o->adjoint_device_bytes = c->adj_bytes;
    o->bytes_per_cell_e = (uint64_t)std::llround(9 * s + (c->e_mode ? cls : 0.0) + psi);
    o->bytes_per_cell_h = (uint64_t)std::llround(9 * s + (c->h_mode ? cls : 0.0) + psi);
    return FDTD_OK;
}

int fdtd_get_probes(fdtd_ctx *c, float *out, size_t n)
{
    if (!c || (!out && n)) return FDTD_E_INVALID;
    if (!c->finalized) return fail(c, FDTD_E_STATE, "not finalized");
    if (int rc = check_state(c)) return rc;
    const size_t np = c->in.probes.size(), ns = (size_t)c->steps_done;
    if (n < np * ns) return fail(c, FDTD_E_INVALID, "output holds %zu values, need %zu", n, np * ns);
    if (np && ns)
        HIPCHK(c, hipMemcpy2D(out, ns * sizeof(float), c->ka.probe_hist, (size_t)c->in.steps_cap * sizeof(float),
                              ns * sizeof(float), np, hipMemcpyDeviceToHost));
    return FDTD_OK;
}

int fdtd_set_port(fdtd_ctx *c, int vdir, int vis, int vjs, int vks, int vie, int vje, int vke, int idir, int iis,
                  int ijs, int iks, int iie, int ije, int ike)
{
    if (!c) return FDTD_E_INVALID;
    if (c->finalized) return fail(c, FDTD_E_STATE, "scene is finalized");
    if (c->has_port) return fail(c, FDTD_E_STATE, "the port is already set (one port per context)");
    PortDef d{vdir, {vis, vjs, vks, vie, vje, vke}, idir, {iis, ijs, iks, iie, ije, ike}};
    std::string err;
    const SceneIn &in = c->in;
    int rc = port_plan(d, in.nx, in.ny, in.nz, (float)in.dx, (float)in.dy, (float)in.dz, c->port, err);
    if (rc != FDTD_OK) return fail(c, rc, "%s", err.c_str());
    c->port_base = (int)c->in.probes.size();
    c->in.probes.insert(c->in.probes.end(), c->port.samples.begin(), c->port.samples.end());
    c->has_port = true;
    return FDTD_OK;
}

// V and averaged I of the steps run so far (host copies of the port's probe
// histories, reduced by port_series).
static int port_read(fdtd_ctx *c, std::vector<float> &v, std::vector<float> &cur)
{
    if (!c->finalized) return fail(c, FDTD_E_STATE, "not finalized");
    if (!c->has_port) return fail(c, FDTD_E_STATE, "no port was set");
    if (int rc = check_state(c)) return rc;
    const size_t np = c->port.samples.size(), ns = (size_t)c->steps_done;
    v.assign(ns, 0.f);
    cur.assign(ns, 0.f);
    if (!ns) return FDTD_OK;
    std::vector<float> hist(np * ns);
    HIPCHK(c, hipMemcpy2D(hist.data(), ns * sizeof(float), c->ka.probe_hist + (size_t)c->port_base * c->in.steps_cap,
                          (size_t)c->in.steps_cap * sizeof(float), ns * sizeof(float), np, hipMemcpyDeviceToHost));
    port_series(c->port, hist.data(), ns, v.data(), cur.data());
    return FDTD_OK;
}

int fdtd_get_port(fdtd_ctx *c, float *v, float *i, size_t n)
{
    if (!c || ((!v || !i) && n)) return FDTD_E_INVALID;
    std::vector<float> vv, ii;
    if (int rc = port_read(c, vv, ii)) return rc;
    if (n < vv.size()) return fail(c, FDTD_E_INVALID, "output holds %zu values, need %zu", n, vv.size());
    std::copy(vv.begin(), vv.end(), v);
    std::copy(ii.begin(), ii.end(), i);
    return FDTD_OK;
}

int fdtd_port_spectrum(fdtd_ctx *c, double z0, int nfreq, const double *freqs, double *out, size_t n)
{
    if (!c || nfreq < 0 || (nfreq && (!freqs || !out))) return FDTD_E_INVALID;
    if (!(z0 > 0.0) || !std::isfinite(z0)) return fail(c, FDTD_E_INVALID, "z0 must be positive");
    if (n < 8 * (size_t)nfreq) return fail(c, FDTD_E_INVALID, "output holds %zu values, need %zu", n, 8 * (size_t)nfreq);
    std::vector<float> vv, ii;
    if (int rc = port_read(c, vv, ii)) return rc;
    port_spectrum(vv.data(), ii.data(), vv.size(), c->in.dt, z0, nfreq, freqs, out);
    return FDTD_OK;
}

int fdtd_save_port(fdtd_ctx *c, const char *vpath, const char *ipath)
{
    if (!c || !vpath || !ipath) return FDTD_E_INVALID;
    std::vector<float> vv, ii;
    if (int rc = port_read(c, vv, ii)) return rc;
    if (port_save(vv.data(), vv.size(), vpath) != FDTD_OK) return fail(c, FDTD_E_INVALID, "cannot write %s", vpath);
    if (port_save(ii.data(), ii.size(), ipath) != FDTD_OK) return fail(c, FDTD_E_INVALID, "cannot write %s", ipath);
    return FDTD_OK;
}

int fdtd_get_dft(fdtd_ctx *c, double *out, size_t n)
{
    if (!c || (!out && n)) return FDTD_E_INVALID;
    if (!c->finalized) return fail(c, FDTD_E_STATE, "not finalized");
    if (int rc = check_state(c)) return rc;
    const size_t cnt = c->in.probes.size() * c->in.freqs.size() * 2;
    if (n < cnt) return fail(c, FDTD_E_INVALID, "output holds %zu values, need %zu", n, cnt);
    if (cnt) HIPCHK(c, hipMemcpy(out, c->ka.dft, cnt * sizeof(double), hipMemcpyDeviceToHost));
    return FDTD_OK;
}

int fdtd_get_field(fdtd_ctx *c, int comp, float *out, size_t n)
{
    if (!c || !out) return FDTD_E_INVALID;
    if (!c->finalized) return fail(c, FDTD_E_STATE, "not finalized");
    if (int rc = check_state(c)) return rc;
    if (comp < 0 || comp > 5) return fail(c, FDTD_E_INVALID, "invalid component");
    const int nx = c->in.nx, ny = c->in.ny, nz = c->in.nz, px = c->in.px;
    const size_t cells = (size_t)nx * ny * nz;
    if (n < cells) return fail(c, FDTD_E_INVALID, "output too small");
    DeviceGuard dg(c->device);
    // two pieces of pinned memory, made at the first call and kept: the GPU packs
    // and converts one while the other is copied out.  Through a copy of the
    // padded array in pageable memory and a loop here, the six fields of
    // 150x131x118 took 14.5 ms; so 6.3, most of it the copy out (9 GB/s).  The
    // host's first use of the pieces costs 1.7 us for each 4 KB of them, so they
    // are no larger than the reads after it need: us, a context's first read / six
    // later ones, pieces of 2^16, 2^17 and 2^20 values: 64^3 350 / 355, 560 / 325,
    // 535 / 390; 100x96x90 490 / 1050, 670 / 850, 1530 / 1150; 150x131x118 960 / 2860,
    // 1100 / 2440, 3470 / 2550; 2^17, 2^19, 2^20: 160^3 1390 / 4460, 2500 / 4170, 3810 /
    // 4150; 256x256x200 3170 / 14900, 3590 / 12000, 5170 / 11500.
    const size_t piece = cells <= (size_t)1 << 20 ? 1 << 16 : cells <= (size_t)3 << 20 ? 1 << 17 : 1 << 19;
    const size_t stage = std::min(cells, 2 * piece);
    if (!c->stage) {
        for (auto &e : c->stage_ev)
            if (!e) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
        if (hipHostMalloc((void **)&c->stage, stage * sizeof(float), hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            c->stage = nullptr;
            return fail(c, FDTD_E_NOMEM, "pinned host memory (%zu bytes)", stage * sizeof(float));
        }
    }
    const char *base = (const char *)c->fields[comp] + (size_t)c->ka.plane * c->esz;
    const std::uint8_t *qe = c->qexp[comp] ? c->qexp[comp] + (size_t)c->ka.plane / BQ_BLOCK * BQ_STRIDE : nullptr;
    const float un = c->built.probe_unscale[comp];
    const size_t pieces = (cells + piece - 1) / piece;
    for (size_t p = 0; p <= pieces; ++p) {
        if (p < pieces) {
            const size_t g = p * piece, len = std::min(piece, cells - g);
            HIPCHK(c, launch_unpack(c->in.storage, base, qe, c->stage + p % 2 * piece, (std::uint32_t)g,
                                    (std::uint32_t)len, nx, px, un, c->stream));
            HIPCHK(c, hipEventRecord(c->stage_ev[p % 2], c->stream));
        }
        if (p > 0) {
            const size_t g = (p - 1) * piece, len = std::min(piece, cells - g);
            HIPCHK(c, hipEventSynchronize(c->stage_ev[(p - 1) % 2]));
            std::memcpy(out + g, c->stage + (p - 1) % 2 * piece, len * sizeof(float));
        }
    }
    return FDTD_OK;
}

// ---- checkpoint -------------------------------------------------------------
int fdtd_checkpoint_size(const fdtd_ctx *c, size_t *bytes)
{
    if (!c || !bytes) return FDTD_E_INVALID;
    if (!c->finalized) return FDTD_E_STATE;
    size_t p = 6 * (size_t)c->field_elems * c->esz + 2 * c->qarr_bytes;
    for (int q = 0; q < 12; ++q) p += c->psi_elems[q] * c->esz;
    p += c->in.probes.size() * (size_t)c->in.steps_cap * sizeof(float);
    p += c->in.probes.size() * c->in.freqs.size() * sizeof(double2);
    *bytes = sizeof(CkHeader) + p;
    return FDTD_OK;
}

int fdtd_checkpoint_save(fdtd_ctx *c, void *buf, size_t bytes)
{
    if (!c || !buf) return FDTD_E_INVALID;
    size_t need = 0;
    int rc = fdtd_checkpoint_size(c, &need);
    if (rc) return fail(c, rc, "not finalized");
    if ((rc = check_state(c))) return rc;
    if (bytes < need) return fail(c, FDTD_E_INVALID, "checkpoint buffer holds %zu bytes, need %zu", bytes, need);
    HIPCHK(c, hipStreamSynchronize(c->stream));
    unsigned char *p = (unsigned char *)buf + sizeof(CkHeader);
    auto get = [&](const void *dev, size_t n) -> int {
        if (n) HIPCHK(c, hipMemcpy(p, dev, n, hipMemcpyDeviceToHost));
        p += n;
        return FDTD_OK;
    };
    for (int f = 0; f < 6; ++f)
        if ((rc = get(fld(c, f), (size_t)c->field_elems * c->esz))) return rc;
    for (int q = 0; q < 2; ++q)
        if ((rc = get(c->qarr[q], c->qarr_bytes))) return rc;
    for (int q = 0; q < 12; ++q)
        if ((rc = get(psv(c, q), c->psi_elems[q] * c->esz))) return rc;
    if ((rc = get(c->ka.probe_hist, c->in.probes.size() * (size_t)c->in.steps_cap * sizeof(float)))) return rc;
    if ((rc = get(c->ka.dft, c->in.probes.size() * c->in.freqs.size() * sizeof(double2)))) return rc;
    CkHeader h{};
    std::memcpy(h.magic, "FDTDCKP1", 8);
    h.version = 1;
    h.nx = c->in.nx; h.ny = c->in.ny; h.nz = c->in.nz;
    h.storage = c->in.storage;
    h.step = c->steps_done;
    h.nprobe = (int)c->in.probes.size();
    h.nfreq = (int)c->in.freqs.size();
    h.steps_cap = c->in.steps_cap;
    h.payload = need - sizeof(CkHeader);
    h.checksum = fnv1a((const unsigned char *)buf + sizeof(CkHeader), h.payload);
    std::memcpy(buf, &h, sizeof h);
    return FDTD_OK;
}

int fdtd_checkpoint_restore(fdtd_ctx *c, const void *buf, size_t bytes)
{
    if (!c || !buf) return FDTD_E_INVALID;
    size_t need = 0;
    int rc = fdtd_checkpoint_size(c, &need);
    if (rc) return fail(c, rc, "not finalized");
    if (bytes < need) return fail(c, FDTD_E_CHECKSUM, "checkpoint truncated");
    CkHeader h;
    std::memcpy(&h, buf, sizeof h);
    if (std::memcmp(h.magic, "FDTDCKP1", 8) != 0 || h.version != 1 || h.nx != c->in.nx || h.ny != c->in.ny ||
        h.nz != c->in.nz || h.storage != c->in.storage || h.nprobe != (int)c->in.probes.size() ||
        h.nfreq != (int)c->in.freqs.size() || h.steps_cap != c->in.steps_cap || h.payload != need - sizeof h ||
        h.step < 0 || h.step > c->in.steps_cap)
        return fail(c, FDTD_E_CHECKSUM, "checkpoint does not match this context");
    if (fnv1a((const unsigned char *)buf + sizeof h, h.payload) != h.checksum)
        return fail(c, FDTD_E_CHECKSUM, "checkpoint checksum mismatch");
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const unsigned char *p = (const unsigned char *)buf + sizeof h;
    auto put = [&](void *dev, size_t n) -> int {
        if (n) HIPCHK(c, hipMemcpy(dev, p, n, hipMemcpyHostToDevice));
        p += n;
        return FDTD_OK;
    };
    for (int f = 0; f < 6; ++f)
        if ((rc = put(fld(c, f), (size_t)c->field_elems * c->esz))) return rc;
    for (int q = 0; q < 2; ++q)
        if ((rc = put(c->qarr[q], c->qarr_bytes))) return rc;
    for (int q = 0; q < 12; ++q)
        if ((rc = put(psv(c, q), c->psi_elems[q] * c->esz))) return rc;
    if ((rc = put(c->ka.probe_hist, c->in.probes.size() * (size_t)c->in.steps_cap * sizeof(float)))) return rc;
    if ((rc = put(c->ka.dft, c->in.probes.size() * c->in.freqs.size() * sizeof(double2)))) return rc;
    c->steps_done = h.step;
    c->broken = false;
    return FDTD_OK;
}

int fdtd_adjoint_gradient(fdtd_ctx *c, const fdtd_objective *obj, int n_steps, int checkpoint_every,
                          double *J_out, double *grad_out, size_t n_grad)
{
    if (!c || !obj || !J_out || !grad_out) return FDTD_E_INVALID;
    return run_adjoint(c, obj, n_steps, checkpoint_every, J_out, grad_out, n_grad);
}

int fdtd_adjoint_gradient_noalloc(fdtd_ctx *c, const fdtd_objective *obj, int n_steps, double *J_out,
                                  double *grad_out, size_t n_grad)
{
    if (!c || !obj || !J_out || !grad_out) return FDTD_E_INVALID;
    if (!c->scratch)
        return fail(c, FDTD_E_DEVICE, "the static scratch has no device address on device %d", c->device);
    return run_adjoint(c, obj, n_steps, 0, J_out, grad_out, n_grad, c->scratch, FDTD_NOALLOC_SCRATCH_BYTES);
}

}  // extern "C"
