// Host-side internals shared by the single-scene library (openem_hip.hip) and the serving pool
// (oem_pool.hip): error reporting, the resident-scene context, and the arena hooks a pool
// context allocates through.

#pragma once

#include "../../include/openem_hip.h"
#include "oem_kernels.h"

#include <mutex>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

namespace oemi {

// One message per host thread; the C ABI returns a code and oem_last_error reads this.
inline thread_local std::string g_err;

inline int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

struct Monitor {
    MonDev d;
    size_t count;         // ncomp*nf*npts
    bool fused = false;   // the fused step writes its snapshots; `patch` lists the points an
    int *patch = nullptr; // E-side point list corrects afterwards, snapped again
    int n_patch = 0;
    bool blk = false;     // the E sweep's work-groups write its snapshots
};

struct TimeMonitor {
    TimeMonDev d;
    size_t count;     // nc*slots*cells elements of the field type
};

struct FluxTimeMonitor {
    FluxTimeDev d;
};

// One grouped point list (dipoles or TF/SF face corrections) and which field it updates.
enum { PT_DIPOLE = 0, PT_TFSF = 1, PT_MODE = 2 };

// From this size (cells) on every scene takes the fused H+E step by default (march_pays).
#define OEM_FUSE_MIN_CELLS (10u << 20)

struct Points {
    PointsDev d;
    int magnetic;       // 1: applied to H after update_h; 0: to E after update_e
    int kind;           // PT_*: launch order H: dipole, TF/SF, mode; E: TF/SF, mode, dipole
    std::vector<int> cells, comps;   // the group cells and components (host copies)
};

// Kernel family of a point list (profiling ids of include/openem_hip.h).
inline int points_kid(const Points &p) {
    if (p.kind == PT_MODE) return p.magnetic ? OEM_K_MODE_H : OEM_K_MODE_E;
    if (p.kind == PT_TFSF) return p.magnetic ? OEM_K_TFSF_H : OEM_K_TFSF_E;
    return p.magnetic ? OEM_K_DIPOLE_H : OEM_K_DIPOLE_E;
}

// Position of a point list in the step (0..5): H side dipole, TF/SF, mode; E side TF/SF,
// mode, dipole -- the reference's order (`openem/solver.py:876-968`).
inline int points_slot(const Points &p) {
    static const int h[3] = {0, 1, 2}, e[3] = {5, 3, 4};
    return p.magnetic ? h[p.kind] : e[p.kind];
}

// Arena of a serving pool (oem_pool.hip).
int pool_arena_alloc(oem_pool *pool, size_t bytes, void **out);
void pool_arena_free(oem_pool *pool, void *p);

}  // namespace oemi

namespace oemi {
// Held while a stream is captured into a graph (begin to instantiate) and around every call
// that may synchronise the device (hipFree, hipHostFree, hipStreamDestroy, hipMalloc):
// contexts step on several host threads at once (serving lanes, designs in flight), and a
// device-wide synchronisation issued by one thread while another thread's stream is capturing
// invalidates that capture.  For the same reason no copy here goes through the legacy stream:
// every host copy is hipMemcpyAsync on the context's (or pool's) own stream, then a
// synchronisation of that stream.
std::mutex &device_sync_mutex();
}

struct oem_reduce_state;            // energy / flux reduction tables (oem_reduce.hip)
struct oem_adjoint_state;           // checkpoints, adjoint fields, design gradient (oem_adjoint.hip)
namespace oemi {
void reduce_state_free(oem_reduce_state *r);
void adjoint_state_free(oem_adjoint_state *a);
}

using oemi::fail;
using oemi::Monitor;
using oemi::TimeMonitor;
using oemi::FluxTimeMonitor;
using oemi::Points;
using oemi::PT_DIPOLE;
using oemi::PT_MODE;
using oemi::PT_TFSF;

#define HIP_OK(expr)                                                                     \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess)                                                            \
            return fail(e_ == hipErrorOutOfMemory ? OEM_ENOMEM : OEM_EHIP, "%s: %s (%s:%d)", \
                        #expr, hipGetErrorString(e_), __FILE__, __LINE__);               \
    } while (0)

#define TRY(expr)                  \
    do {                           \
        int rc_ = (expr);          \
        if (rc_) return rc_;       \
    } while (0)

struct oem_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    oem_dims dims{};
    size_t ncell = 0;           // cells of the grid (the ABI's flat index space)
    int pz = 0;                 // row pitch of the device arrays (row_pitch)
    size_t nst = 0;             // cells of one device component, nx*ny*pz
    size_t n_laid = 0;          // allocations up to the fields' (lay_out)
    bool written = false;       // oem_write_field was called
    float *stage = nullptr;     // dense rows of a padded field on their way to or from the host
    bool cplx = false;          // Bloch: complex fields, (re, im) interleaved
    size_t esz = 1;             // floats per field element
    float *E = nullptr, *H = nullptr;
    PsiDev psi{};
    // fused H+E step: a second set of fields and psi; after s steps the state is in set s % 2
    bool fused = false;
    float *E2 = nullptr, *H2 = nullptr;
    PsiDev psi2{};
    float *cur_E() const { return (fused && (step & 1)) ? E2 : E; }
    float *cur_H() const { return (fused && (step & 1)) ? H2 : H; }
    GridDev g{};
    GridDev fg{};               // launch geometry of the fused H+E step
    bool fuse_plain = false;    // its stores keep their lines in the caches (march_bytes)
    FuseSnap fsnap{};           // the DFT monitors the fused step snaps
    FusePts fpts{};             // the E-side points the E update applies (n = 0: none)
    bool fsnap_multi = false;   // some work-group meets more than one of them
    BlkPts blk_h{}, blk_e{};    // the point lists the H and the E sweep apply (t.n = 0: none)
    BlkSnap blk_snap{};         // the monitors the E sweep snaps
    bool e_swept = false;       // the E sweep's work-groups leave the step's final E
    bool axis_set[3] = {false, false, false};
    bool unit_masks = true;     // every real mask of the axes is 0 or +-1
    MatDev mat{};
    bool mat_set = false;
    std::vector<char> class_flagged;   // LUT classes that read the ADE history term
    DispDev disp{};
    bool has_disp = false;
    int64_t disp_n_pole = 0;           // poles over all entries (the pole state's length)
    PlaneSrcDev pw{};
    std::vector<Points> points;
    std::vector<Monitor> mons;
    std::vector<TimeMonitor> tmons;
    std::vector<FluxTimeMonitor> ftmons;
    int *d_step = nullptr;      // steps taken, up to the captured or pooled block under way
    int64_t step = 0;
    int pending = 0;
    bool pre_ready = false;     // ADE: hist/P already advanced by the previous fused step
    bool prepared = false;
    int chunk_req = 0;          // x-planes per work-group requested (0: heuristic)
    int form_req = 0;           // step form requested: 0 the library's choice, 1 two sweeps, 2 fused
    bool mons_off = false;      // adjoint recomputation: no DFT snapshots or flushes
    // adjoint forward recording (oem_adjoint_forward): after each step, E at the design cells
    // goes to row (step + 1 - base) of rec
    struct RecHook {
        bool on = false;
        const int *comp = nullptr, *cell = nullptr;
        int n = 0;
        float *rec = nullptr;       // of the field type (two floats per value on complex fields)
        int64_t base = 0;
        BlkTab tab{};               // its entries by work-group of the E sweep (n = 0: a launch)
    } rec_hook;
    struct oem_adjoint_state *adj = nullptr;
    hipGraphExec_t graph[2] = {nullptr, nullptr};   // a block's steps, by the parity of its first
    void drop_graphs() {
        for (hipGraphExec_t &g : graph) {
            if (g) (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
    }
    std::vector<void *> allocs;
    oem_reduce_state *red = nullptr;

    // serving pool membership (oem_pool.hip); pool == nullptr for a standalone context
    oem_pool *pool = nullptr;
    bool attached = false;
    int64_t done_block = -1;    // pool block in which the last step runs (-1: not scheduled)
    int64_t retire_after = -1;  // memory is reclaimed once this pool block has completed

    ~oem_ctx() {
        drop_graphs();
        if (red) oemi::reduce_state_free(red);
        if (adj) oemi::adjoint_state_free(adj);
        // arena ranges before the capture lock: the pool's lock is never taken under it
        if (pool)
            for (void *p : allocs) oemi::pool_arena_free(pool, p);
        std::lock_guard<std::mutex> hold(oemi::device_sync_mutex());
        if (!pool)
            for (void *p : allocs) (void)hipFree(p);
        if (stream) (void)hipStreamDestroy(stream);
    }

    template <typename T>
    int alloc(T **out, size_t n, bool zero) {
        void *p = nullptr;
        if (n == 0) n = 1;
        if (pool) {
            TRY(oemi::pool_arena_alloc(pool, n * sizeof(T), &p));
        } else {
            std::lock_guard<std::mutex> hold(oemi::device_sync_mutex());
            const hipError_t e = hipMalloc(&p, n * sizeof(T));
            if (e != hipSuccess) {
                (void)hipGetLastError();    // reported here, not by the thread's next launch check
                return fail(e == hipErrorOutOfMemory ? OEM_ENOMEM : OEM_EHIP, "hipMalloc of %zu bytes: %s",
                            n * sizeof(T), hipGetErrorString(e));
            }
        }
        allocs.push_back(p);
        if (zero) HIP_OK(hipMemsetAsync(p, 0, n * sizeof(T), stream));
        *out = static_cast<T *>(p);
        return OEM_OK;
    }

    // give back an allocation of a standalone context
    int release(void *p) {
        auto it = std::find(allocs.begin(), allocs.end(), p);
        if (it == allocs.end()) return OEM_OK;
        HIP_OK(hipStreamSynchronize(stream));
        allocs.erase(it);
        std::lock_guard<std::mutex> hold(oemi::device_sync_mutex());
        HIP_OK(hipFree(p));
        return OEM_OK;
    }

    // flat cell of the ABI -> flat cell of the pitched device arrays
    size_t dev_cell(size_t id) const {
        const size_t nz = (size_t)dims.nz;
        return pz == dims.nz ? id : id / nz * (size_t)pz + id % nz;
    }

    // `rows` rows of nz elements of a caller's array -> the pitched rows of an uploaded one
    template <typename T>
    int upload_rows(T **out, const T *host, size_t rows) {
        const size_t nz = (size_t)dims.nz;
        if (pz == dims.nz) return upload(out, host, rows * nz);
        std::vector<T> v(rows * (size_t)pz, T(0));
        for (size_t r = 0; r < rows; ++r) std::memcpy(&v[r * pz], host + r * nz, nz * sizeof(T));
        return upload(out, (const T *)v.data(), v.size());
    }

    template <typename T>
    int upload(T **out, const T *host, size_t n) {
        int rc = alloc(out, n, false);
        if (rc) return rc;
        HIP_OK(hipMemcpyAsync(*out, host, n * sizeof(T), hipMemcpyHostToDevice, stream));
        HIP_OK(hipStreamSynchronize(stream));
        return OEM_OK;
    }
};

#define CHECK_CTX(c)                                                           \
    do {                                                                       \
        if (!(c)) return fail(OEM_EINVAL, "null context");                     \
        HIP_OK(hipSetDevice((c)->device));                                     \
    } while (0)

// The work-groups the chip holds at once, the share of a larger launch's that may have a tail, and the
// most items of a table (build_blk).
#define OEM_BLK_RESIDENT 1024
#define OEM_BLK_SHARE 8
#define OEM_BLK_ITEMS 320000
// Tables of the items of several lists by the work-group that owns them: blk(l, t) of the n[l]
// items of list l.  False, and the lists keep their own launches, when out of memory or when too
// many work-groups would end with a tail of dependent loads: a grid whose work-groups all run at
// once hides them behind each other (120 x 120 x 44, mode source, planes and design: E sweep 11.2
// us with 11.8 us of launches after it, 12.5 with the lists), a larger one pays them per round
// (160^3 with a z plane, in every work-group: 42.7 us against 35.6 and a launch of 5; 400 x 400 x
// 48 with a 160 x 160 design, in a sixth of them: 99.9 against 79.3 and 5.2).  Nor with more than
// OEM_BLK_ITEMS items: a step saves a launch, 3 us whatever its size, and the tables cost the context
// 4 to 8 ns an item (TF/SF box of 100^3 with a box monitor of 593,000 points: 49.2 against 46.4 us a
// step, oem_prepare 4.5 against 10.2 ms; 120^3 with three of 1.1 M 109.7 / 112.5 us, 6.3 / 34.5 ms).
template <typename Fn>
bool build_blk(oem_ctx *ctx, int nblocks, const std::vector<int> &n, Fn blk, BlkTab *out,
               int resident = OEM_BLK_RESIDENT) {
    const size_t nl = n.size();
    size_t total = 0;
    for (size_t l = 0; l < nl; ++l) total += (size_t)n[l];
    if (total > OEM_BLK_ITEMS) return false;
    // a few thousand of the items first: they mostly tell when there are too many work-groups
    for (const size_t step : {std::max<size_t>(1, total >> 13), (size_t)1}) {
        if (nblocks <= resident) break;
        std::vector<char> hit((size_t)nblocks, 0);
        int touched = 0;
        for (size_t l = 0; l < nl; ++l)
            for (size_t t = 0; t < (size_t)n[l]; t += step) {
                char &h = hit[(size_t)blk((int)l, (int)t)];
                touched += !h;
                h = 1;
            }
        if (touched > nblocks / OEM_BLK_SHARE) return false;
    }
    std::vector<int> ofs((size_t)nblocks * nl + 1, 0), row, idx(total);
    row.reserve(total);
    for (size_t l = 0; l < nl; ++l)
        for (int t = 0; t < n[l]; ++t) {
            row.push_back((int)((size_t)blk((int)l, t) * nl + l));
            ++ofs[(size_t)row.back() + 1];
        }
    for (size_t q = 1; q < ofs.size(); ++q) ofs[q] += ofs[q - 1];
    std::vector<int> at(ofs.begin(), ofs.end() - 1);
    size_t q = 0;
    for (size_t l = 0; l < nl; ++l)
        for (int t = 0; t < n[l]; ++t) idx[at[row[q++]]++] = t;
    int *d_ofs = nullptr, *d_idx = nullptr;
    if (ctx->upload(&d_ofs, ofs.data(), ofs.size()) || ctx->upload(&d_idx, idx.data(), idx.size()))
        return false;
    *out = BlkTab{(int)nl, d_ofs, d_idx};
    return true;
}

// Row pitch (cells) of a context's device arrays, from the dimensions and the step form requested.
int row_pitch(const oem_dims *d, bool pooled, int form);

// Shared by oem_ctx_create and oem_pool_ctx_create: validate dims and allocate the fields,
// psi slabs and counters of a context (through the pool's arena when ctx->pool is set).
int ctx_init(oem_ctx *c, const oem_dims *d, int32_t device);

// Pool hooks used by the single-scene entry points (oem_pool.hip), and the point-list builder
// and step launcher shared with the adjoint (openem_hip.hip).
namespace oemi {
int build_points(oem_ctx *ctx, int magnetic, int kind, int tfsf, int cplx_amp, int32_t n_pts,
                 const int32_t *comp, const int32_t *cell, const float *coef, const int32_t *col,
                 const float *phase, int32_t ncol, const double *tab, size_t tab_doubles,
                 Points *out);
// One eager step, no flush, no profiling: the step at the device counter plus off, which then
// moves by adv.
int launch_one_step(oem_ctx *ctx, bool last, int off, int adv);
// The entries of a cell list by work-group of the E sweep; false: they keep a launch of their own.
bool plan_sweep_record(oem_ctx *ctx, const int32_t *cell, int n, BlkTab *out);
int pool_retire(oem_ctx *ctx);                  // oem_ctx_destroy of a pool context
int pool_wait_done(oem_ctx *ctx);               // before reading a pool context's results
}
