// clm_api.hip -- C ABI (include/clm_hip.h) of the MI355X cell-list engine.
//
// One context owns a HIP stream, the particle data and grow-only device buffers.
// The pipeline per cell-list update is
//   k_bin_bucket -> k_scan_pair (cell counts) -> k_cell_sort
// (or, on the first build of a layout and in captured graphs, the two passes k_bin_count ->
// scans -> k_bin_scatter -> k_cell_sort), and per operator call
//   ([k_scan_pair (homes)], cached per sweep mode) -> sweep -> k_read_back.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "clm_box.hpp"
#include "clm_sweep.hpp"
#include "clm_hip.h"

using namespace clm;

namespace {

struct DBuf {
    void *p = nullptr;
    size_t bytes = 0;
};

struct Pending {
    std::string name;
    hipEvent_t a, b;
};

}  // namespace

struct clm_ctx {
    int device = 0, dtype = CLM_F32, dim = 3;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    std::string err;
    int num_cus = 256;

    // geometry: one entry per system (a single system unless clm_set_systems was used)
    bool has_box = false;
    int celltype = CLM_ORTHORHOMBIC, lcell = 1;
    double cutoff_in = 0;
    int nsys = 1;
    std::vector<HostBox<float>> hbf;
    std::vector<HostBox<double>> hbd;
    std::vector<int64_t> sys_n;
    std::vector<int> h_rowoff, h_celloff;
    bool layout_dirty = true;
    DBuf sys_desc, sys_of, rowoff, systasks, systasks_all;
    int systasks_homes = 0;  // homes per task of systasks (0: not built)
    int waves_per_cu = 0;  // persistent sweep grid; 0 = as many as fit
    int sweep_variant = 1;  // 0 = union rows (k_sweep), 1 = windows (k_sweep_win)
    int sweep_group = 0;    // entries per lane per step of k_sweep_win in mode B (0: the default, SWEEP_GROUP; 2, 4, 8)
    int sweep_lanes = 8;    // lanes per home of the last sweep prepared (choose_lanes)
    int parts_variant = -1;  // the sweep variant the grid was laid out for
    bool parts = false;      // some cells of the grid are cut into parts
    bool whole_cells = false;  // the grid is laid out for a neighbour list (choose_parts)

    // captured pipeline (update + energy/forces) for replay, and what it was captured
    // against: the device address of every buffer it may touch, the particle count and
    // the box epoch (a replay after any of them changed is refused)
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    std::vector<void *> graph_ptrs;
    int64_t graph_n = -1;
    int graph_box_epoch = -1;
    bool graph_bucketed = false;
    bool graph_ordered = false;  // it bins in the order of order[]

    // particles
    int64_t n = 0;
    bool has_pos = false, dirty = true;
    DBuf pos, types, vel;
    bool has_types = false;
    int64_t n_vel = -1;  // velocities set (-1: none)

    // cell list
    bool cl_valid = false;
    int ncells = 0, nrows = 0;
    int64_t n_entries = 0;
    DBuf xw, home_cell, cnt, creal, cstart, cur_real, cur_ghost, E, E_raw, rstart, real_pos, order, flags, cnt64, maxcnt;
    DBuf limits;    // open box: limits of the coordinates (k_limits)
    DBuf vq0, vq1;  // histogram: neighbour velocities in entry order (k_entry_velocities)
    bool order_valid = false;  // order[] holds the particles in the cell order of the last build
    // triclinic boxes: the cell-sorted entries split into the real ones and the ghost ones
    // (written by k_cell_sort with E; split_valid when the last sort wrote them)
    DBuf E_real, E_ghost;
    bool split_valid = false;
    int bucket = 0;  // entries per cell bucket of the single-pass binning; 0 = not sized yet, -1 = off
    int64_t e_cap = 0;
    DBuf hstart[3], tstart[3];
    bool mode_valid[3] = {false, false, false};  // hstart
    bool rows_valid[3] = {false, false, false};  // tstart
    DBuf counters, scan_tmp;
    bool counters_zeroed = false;  // the caller zeroed the sweep's task counters with its own fill
    DBuf scan_st[3];  // state of the single-pass scans: cells, rows, neighbour-list chunks

    // operator buffers
    DBuf nl_i, nl_j, nl_d, nl_count, outbuf, acc, hist, md_best;
    DBuf sp_i, sp_j, sp_d, ch_used, ch_hstart, ch_mstart;
    // host memory of the read-backs, READ_WORDS long: [0, 4) status of a build read at once, [4, 8) of a
    // deferred build, the rest an operator's results.  Pinned where h_mapped (kernels write to it).
    uint32_t *h_flags = nullptr;
    bool h_mapped = false;
    // A single-pass build enqueued without reading its status block back (bin_pending):
    // the next synchronisation reads it with whatever the operator reads back.
    bool bin_pending = false;
    bool no_defer = false;  // the next build reads its status back first (after an overflow)

    // second particle set (two-set / cross mode): a sub-context on the same stream and
    // box holding the y positions and their cell list
    clm_ctx *ysub = nullptr;
    bool two_set = false;
    clm_ctx *root = nullptr;  // set in a sub-context: the owner (profiling, box)
    int box_epoch = 0, sub_epoch = -1;

    // measurement
    bool prof = false;
    std::vector<Pending> pending;
    std::vector<hipEvent_t> ev_pool;
    std::map<std::string, std::pair<double, int64_t>> prof_acc;

    // events of clm_join_stream (created on first use, timing off)
    hipEvent_t join_ev[2] = {nullptr, nullptr};
};

namespace {

// Internal: the cell list was found invalid after the fact (a deferred build overflowed);
// the entry point runs again on a rebuilt list.  Never returned through the ABI.
constexpr clm_status CLM_REDO = (clm_status)15;

clm_status fail(clm_ctx *c, clm_status s, const std::string &msg) {
    if (c) c->err = msg;
    return s;
}

clm_status hip_fail(clm_ctx *c, hipError_t e, const char *where) {
    return fail(c, CLM_ERR_HIP, std::string(where) + ": " + hipGetErrorString(e));
}

#define HIPCHK(c, expr)                                      \
    do {                                                     \
        hipError_t e_ = (expr);                              \
        if (e_ != hipSuccess) return hip_fail(c, e_, #expr); \
    } while (0)

// Device memory of an allocation-free call (clm_energy_forces_noalloc): while `on`,
// ensure() carves buffers out of the per-device scratch array instead of allocating
// (a buffer that must grow takes a new block; nothing is freed), and reports an
// exhausted arena as an allocation failure.
struct ScratchArena {
    char *base = nullptr;
    size_t cap = 0, used = 0;
    bool on = false, exhausted = false;
};
thread_local ScratchArena g_arena;

// What destroyed contexts leave for the next ones of the same device: device memory, streams and
// their pinned read-back blocks.  A program that makes a context for every call (neighborlist) paid
// for them on each: creating a context 390 us, destroying it 1000, an allocation 25 to 130 (list of
// 5e4 points from host arrays 1.21 ms without the pool, 0.89 with it, a call after the other; 1.0 to
// 1.3 among calls of other sizes, first touch of the result arrays included).  At
// most POOL_BYTES in POOL_BLOCKS blocks and POOL_STREAMS streams are kept; what goes beyond is given
// back at once, and all of the memory when an allocation fails.  A context leaves its memory after
// the device has finished all work, so that the next one may use it on any stream.  ensure() takes
// from the pool of the current device, so every entry point that allocates makes its context's
// device the current one first.
constexpr size_t POOL_BYTES = (size_t)256 << 20;
constexpr size_t POOL_BLOCKS = 256, POOL_STREAMS = 8;
struct Pool {
    struct Block { void *p; size_t bytes; };
    struct Stream { hipStream_t stream; uint32_t *host; };
    std::mutex lock;
    std::vector<Block> blocks;
    std::vector<Stream> streams;
    size_t bytes = 0;

    // A block of at least `want` bytes and at most twice that; null when there is none.
    void *take(size_t want, size_t &got) {
        std::lock_guard<std::mutex> g(lock);
        size_t at = blocks.size();
        for (size_t k = 0; k < blocks.size(); ++k)
            if (blocks[k].bytes >= want && blocks[k].bytes <= 2 * want && (at == blocks.size() || blocks[k].bytes < blocks[at].bytes))
                at = k;
        if (at == blocks.size()) return nullptr;
        const Block b = blocks[at];
        blocks[at] = blocks.back();
        blocks.pop_back();
        bytes -= b.bytes;
        got = b.bytes;
        return b.p;
    }
    // Whether the block is kept.
    bool leave(void *p, size_t n) {
        std::lock_guard<std::mutex> g(lock);
        if (blocks.size() >= POOL_BLOCKS || n > POOL_BYTES - bytes) return false;
        blocks.push_back({p, n});
        bytes += n;
        return true;
    }
    bool give_back() {
        std::vector<Block> all;
        {
            std::lock_guard<std::mutex> g(lock);
            all.swap(blocks);
            bytes = 0;
        }
        for (const Block &b : all) hipFree(b.p);
        return !all.empty();
    }
    bool take_stream(Stream &s) {
        std::lock_guard<std::mutex> g(lock);
        if (streams.empty()) return false;
        s = streams.back();
        streams.pop_back();
        return true;
    }
    bool leave_stream(const Stream &s) {
        std::lock_guard<std::mutex> g(lock);
        if (streams.size() >= POOL_STREAMS) return false;
        streams.push_back(s);
        return true;
    }
};
// The pool of a device (null beyond POOL_DEVICES).  Never destroyed: at the end of the process
// the runtime may be gone before it.
constexpr int POOL_DEVICES = 64;
Pool *device_pool(int device) {
    static Pool *pools = new Pool[POOL_DEVICES];
    return device >= 0 && device < POOL_DEVICES ? pools + device : nullptr;
}

hipError_t ensure(DBuf &b, size_t bytes) {
    if (bytes <= b.bytes && b.p) return hipSuccess;
    if (g_arena.on) {
        const size_t off = (g_arena.used + 255) & ~(size_t)255;
        const size_t want = std::max<size_t>(bytes, 256);
        if (off > g_arena.cap || want > g_arena.cap - off) {
            g_arena.exhausted = true;
            return hipErrorOutOfMemory;
        }
        b.p = g_arena.base + off;
        b.bytes = want;
        g_arena.used = off + want;
        return hipSuccess;
    }
    if (b.p) hipFree(b.p);
    b.p = nullptr;
    b.bytes = 0;
    size_t want = std::max<size_t>(bytes + bytes / 4, 256);
    int device = -1;
    Pool *pool = hipGetDevice(&device) == hipSuccess ? device_pool(device) : nullptr;
    if (pool && (b.p = pool->take(want, b.bytes))) return hipSuccess;
    hipError_t e = hipMalloc(&b.p, want);
    if (e == hipErrorOutOfMemory && pool && pool->give_back()) {
        (void)hipGetLastError();
        e = hipMalloc(&b.p, want);
    }
    if (e == hipSuccess) b.bytes = want;
    else b.p = nullptr;
    return e;
}

hipEvent_t take_event(clm_ctx *c) {
    if (!c->ev_pool.empty()) {
        hipEvent_t e = c->ev_pool.back();
        c->ev_pool.pop_back();
        return e;
    }
    hipEvent_t e;
    hipEventCreate(&e);
    return e;
}

void collect_profile(clm_ctx *c) {
    for (auto &p : c->pending) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
            auto &acc = c->prof_acc[p.name];
            acc.first += ms;
            acc.second += 1;
        }
        c->ev_pool.push_back(p.a);
        c->ev_pool.push_back(p.b);
    }
    c->pending.clear();
}

template <typename F>
hipError_t timed(clm_ctx *c, const char *name, F &&launch) {
    hipEvent_t a = nullptr, b = nullptr;
    if (c->root) c = c->root;  // a sub-context's kernels are timed by its owner
    if (c->prof) {
        a = take_event(c);
        b = take_event(c);
        hipEventRecord(a, c->stream);
    }
    launch();
    hipError_t e = hipGetLastError();
    if (c->prof) {
        hipEventRecord(b, c->stream);
        c->pending.push_back({name, a, b});
    }
    return e;
}

#define LAUNCH(c, name, ...)                                            \
    do {                                                                \
        hipError_t e_ = timed(c, name, [&] { __VA_ARGS__; });           \
        if (e_ != hipSuccess) return hip_fail(c, e_, name);             \
    } while (0)

clm_status check_flags(clm_ctx *c, uint32_t fl);
clm_status check_deferred_build(clm_ctx *c, const uint32_t *status);

constexpr int READ_WORDS = 2048;
constexpr int READ_RESULTS = 12;  // first word of an operator's results (y's build status before it)
static_assert(LIMITS_BLOCKS * sizeof(Limits<double>) / sizeof(uint32_t) <= READ_WORDS - READ_RESULTS, "limits are read back at once");

// Synchronises the stream after copying `words` words from src (device) to where result_words
// points, and the status of builds not yet checked; those are then checked.
clm_status sync(clm_ctx *c, const void *src = nullptr, int words = 0) {
    clm_ctx *y = c->two_set ? c->ysub : nullptr;
    const bool px = c->bin_pending, py = y && y->bin_pending;
    ReadList r;
    std::memset(&r, 0, sizeof(r));
    auto add = [&](const void *p, int n) {
        r.p[r.count] = (const uint32_t *)p;
        r.n[r.count++] = n;
    };
    // contiguous from word 4 on: x's status, y's status, the results
    add(px ? c->flags.p : nullptr, px ? 4 : 0);
    add(py ? y->flags.p : nullptr, py ? 4 : 0);
    add(src, words);
    int at[3];
    for (int k = 0, o = 4; k < 3; o += r.n[k++]) at[k] = o;
    if (words > READ_WORDS - READ_RESULTS) return fail(c, CLM_ERR_ARG, "read-back too long");
    if (px || py || words) {
        if (c->h_mapped) {
            LAUNCH(c, "k_read_back", hipLaunchKernelGGL(k_read_back, dim3(1), dim3(256), 0, c->stream, r, c->h_flags + 4));
        } else {
            for (int k = 0; k < 3; ++k)
                if (r.n[k])
                    HIPCHK(c, hipMemcpyAsync(c->h_flags + at[k], r.p[k], sizeof(uint32_t) * r.n[k], hipMemcpyDeviceToHost,
                                             c->stream));
        }
    }
    hipError_t e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return hip_fail(c, e, "hipStreamSynchronize");
    clm_ctx *o = c->root ? c->root : c;
    if (o->prof) collect_profile(o);
    // the results move to their fixed place, out of the way of the statuses
    uint32_t st[8];
    std::memcpy(st, c->h_flags + 4, sizeof(st));
    if (words) std::memmove(c->h_flags + READ_RESULTS, c->h_flags + at[2], sizeof(uint32_t) * words);
    clm_status s = CLM_OK;
    if (px) {
        c->bin_pending = false;
        s = check_deferred_build(c, st);
    }
    if (py) {
        y->bin_pending = false;
        const clm_status sy = check_deferred_build(y, st + (px ? 4 : 0));
        if (sy && (s == CLM_OK || s == CLM_REDO)) s = sy == CLM_REDO ? sy : fail(c, sy, y->err);
    }
    return s;
}

// The operator's results read by the last sync().
const uint32_t *result_words(const clm_ctx *c) { return c->h_flags + READ_RESULTS; }

inline unsigned blocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

clm_status fill_int(clm_ctx *c, void *p, int64_t n, int v) {
    if (n <= 0) return CLM_OK;
    LAUNCH(c, "k_fill_int", hipLaunchKernelGGL(k_fill_int, dim3(blocks(n, 256)), dim3(256), 0, c->stream, (int *)p, (int)n, v));
    return CLM_OK;
}

clm_status fill_zero(clm_ctx *c, std::initializer_list<std::pair<void *, int64_t>> bufs) {
    FillList f;
    std::memset(&f, 0, sizeof(f));
    int64_t mx = 0;
    for (auto &b : bufs) {
        if (b.second <= 0) continue;
        if (f.count == 8) return fail(c, CLM_ERR_ARG, "fill list too long");
        f.p[f.count] = (int *)b.first;
        f.n[f.count] = (int)b.second;
        mx = std::max(mx, b.second);
        ++f.count;
    }
    if (!f.count) return CLM_OK;
    LAUNCH(c, "k_fill_int", hipLaunchKernelGGL(k_fill_multi, dim3(std::min<unsigned>(blocks(mx, 256), 1024)), dim3(256), 0,
                                               c->stream, f));
    return CLM_OK;
}

clm_status scan_int(clm_ctx *c, const int *in, int *out, int n) {
    size_t need = 0;
    hipcub::DeviceScan::ExclusiveSum(nullptr, need, in, out, n, c->stream);
    HIPCHK(c, ensure(c->scan_tmp, need));
    size_t have = c->scan_tmp.bytes;
    LAUNCH(c, "scan", hipcub::DeviceScan::ExclusiveSum(c->scan_tmp.p, have, in, out, n, c->stream));
    return CLM_OK;
}

template <typename T>
std::vector<HostBox<T>> &hboxes(clm_ctx *c);
template <>
std::vector<HostBox<float>> &hboxes<float>(clm_ctx *c) { return c->hbf; }
template <>
std::vector<HostBox<double>> &hboxes<double>(clm_ctx *c) { return c->hbd; }
template <typename T>
HostBox<T> &hbox(clm_ctx *c) { return hboxes<T>(c)[0]; }

template <typename T>
DevBox<T> dev_box(const HostBox<T> &hb) {
    DevBox<T> b;
    std::memset(&b, 0, sizeof(b));
    for (int k = 0; k < 9; ++k) { b.input[k] = hb.input.a[k]; b.rot[k] = hb.rot.a[k]; }
    const int D = hb.dim;
    const int nimg = D == 3 ? 27 : 9;
    for (int m = 0; m < nimg; ++m) {
        T kv[3] = {T(m % 3 - 1), T((m / 3) % 3 - 1), D == 3 ? T(m / 9 - 1) : T(0)};
        for (int i = 0; i < D; ++i) {
            // aligned * k in the order of translation_image (CellOperations.jl:138-139)
            T s = hb.aligned(i, 0) * kv[0];
            for (int j = 1; j < D; ++j) s = s + hb.aligned(i, j) * kv[j];
            b.shift[m][i] = s;
        }
    }
    for (int k = 0; k < 3; ++k) {
        b.cbmin[k] = hb.cbmin[k];
        b.cbmax[k] = hb.cbmax[k];
        b.cs[k] = hb.cs[k];
        b.nc[k] = hb.nc[k];
    }
    b.rc2 = hb.cutoff_sqr;
    b.lcell = hb.lcell;
    b.celltype = hb.celltype;
    b.dim = hb.dim;
    b.sub = hb.sub;
    return b;
}

template <typename T>
int build_host_box(int dim, const double *cell, int celltype, double cutoff, int lcell, const double *origin,
                   HostBox<T> &hb) {
    if (dim != 2 && dim != 3) return BOX_BAD_DIM;
    T c[9], o[3] = {0, 0, 0};
    for (int k = 0; k < dim * dim; ++k) c[k] = T(cell[k]);
    if (celltype == CLM_ORTHORHOMBIC || celltype == CLM_NONPERIODIC)
        for (int i = 0; i < dim; ++i)
            for (int j = 0; j < dim; ++j)
                if (i != j) c[i + dim * j] = T(0);
    if (origin)
        for (int k = 0; k < dim; ++k) o[k] = T(origin[k]);
    return build_box<T>(dim, c, celltype, T(cutoff), lcell, o, hb);
}

template <typename T>
void box_info(const HostBox<T> &hb, clm_box_info *out) {
    std::memset(out, 0, sizeof(*out));
    out->dim = hb.dim;
    out->celltype = hb.celltype;
    out->lcell = hb.lcell;
    for (int k = 0; k < 3; ++k) {
        out->nc[k] = hb.nc[k];
        out->cell_size[k] = hb.cs[k];
        out->cbmin[k] = hb.cbmin[k];
        out->cbmax[k] = hb.cbmax[k];
        out->origin[k] = hb.origin[k];
    }
    for (int k = 0; k < 9; ++k) {
        out->input[k] = hb.input.a[k];
        out->aligned[k] = hb.aligned.a[k];
        out->rotation[k] = hb.rot.a[k];
        out->inv_rotation[k] = hb.invrot.a[k];
    }
    out->cutoff = hb.cutoff;
    out->cutoff_sqr = hb.cutoff_sqr;
}

clm_status box_status(clm_ctx *c, int rc) {
    if (rc == BOX_OK) return CLM_OK;
    if (rc == BOX_BAD_LCELL) return fail(c, CLM_ERR_ARG, "lcell must be greater or equal to 1");
    if (rc == BOX_BAD_DIM) return fail(c, CLM_ERR_DIM, "dimension must be 2 or 3");
    return fail(c, CLM_ERR_CELL, "Unit cell matrix does not satisfy required conditions "
                                 "(distance between cell planes must exceed 2*cutoff)");
}

// limits(x) + _sides_from_limits (CellOperations.jl:262-297, Box.jl:38) for the
// non-periodic box, found on the device (k_limits).
// With two sets the limits cover both (limits(x, y), CellOperations.jl:312-324).
template <typename T>
clm_status nonperiodic_box(clm_ctx *c) {
    const int D = c->dim;
    clm_ctx *y = c->two_set ? c->ysub : nullptr;
    const int64_t ny = y ? y->n : 0;
    const int64_t ntot = c->n + ny;
    T mn[3] = {0, 0, 0}, mx[3] = {0, 0, 0};
    if (ntot > 0) {
        const int nb = (int)std::min<int64_t>(LIMITS_BLOCKS, (ntot + 255) / 256);
        HIPCHK(c, ensure(c->limits, sizeof(Limits<T>) * nb));
        LAUNCH(c, "k_limits", hipLaunchKernelGGL(k_limits<T>, dim3(nb), dim3(256), 0, c->stream, (const T *)c->pos.p, (long long)c->n,
                                                 y ? (const T *)y->pos.p : nullptr, (long long)ny, D, (Limits<T> *)c->limits.p));
        clm_status s = sync(c, c->limits.p, (int)(sizeof(Limits<T>) / sizeof(uint32_t)) * nb);
        if (s) return s;
        for (int k = 0; k < D; ++k) { mn[k] = INFINITY; mx[k] = -INFINITY; }
        for (int b = 0; b < nb; ++b) {
            Limits<T> l;
            std::memcpy(&l, result_words(c) + b * (sizeof(l) / sizeof(uint32_t)), sizeof(l));
            if (l.nan != T(0)) return fail(c, CLM_ERR_NAN, "Invalid coordinates found (NaN)");
            for (int k = 0; k < D; ++k) {
                mn[k] = std::min(mn[k], l.lo[k]);
                mx[k] = std::max(mx[k], l.hi[k]);
            }
        }
    }
    const T rc = T(c->cutoff_in);
    const T pad = (T(210) * rc) / T(100);
    double cell[9] = {0}, origin[3] = {0, 0, 0};
    for (int k = 0; k < D; ++k) {
        cell[k + D * k] = double((mx[k] - mn[k]) + pad);
        origin[k] = double(mn[k]);
    }
    hboxes<T>(c).resize(1);
    int rcode = build_host_box<T>(D, cell, CLM_NONPERIODIC, c->cutoff_in, c->lcell, origin, hbox<T>(c));
    return box_status(c, rcode);
}

// Entries of the widest window of a stencil row of b for n particles spread over its cells.
template <typename T>
double window_entries(const HostBox<T> &b, int64_t n) {
    double section = 1, volume = 1;
    for (int k = 0; k < b.dim; ++k) {
        volume *= (double)b.cs[k] * std::max(b.nc[k] - 2 * b.lcell, 1);
        if (k > 0) section *= (double)b.cs[k] / b.sub;
    }
    return 2.0 * (double)b.cutoff * section * (double)n / std::max(volume, 1e-300);
}

// Parts of the cells along y and z (DevBox::sub).  Thinner rows follow the cutoff sphere more
// closely (entries tested per pair at lcell 1: 2.98 with whole cells, 1.87 with 2 parts, 1.55 with
// 3), but there are more of them, each to be started.  So the cells are cut while their rows'
// windows hold more than PARTS_WINDOW entries, up to four parts to a cutoff (gradient of 2e5 at
// lcell 1, 345 entries: the sweep takes 573 us whole, 414 in 2 parts, 460 in 3; clustered 4M at
// lcell 2, 1000 entries: 52.6 ms, 50.7 in 2, 54.8 in 3, and the cell sort 4.4 ms, 2.4; 1M at lcell
// 2, 86 entries: 1413 us, 1682 in 2; with lists of windows 1210 and 1400); not in small systems (a sweep of which lasts as long as its
// longest task), nor for the union-row sweep, nor where the call has no more than its scratch.
constexpr double PARTS_WINDOW = 160;
constexpr int64_t PARTS_MIN = 20000;
template <typename T>
void choose_parts(clm_ctx *c) {
    std::vector<HostBox<T>> &hb = hboxes<T>(c);
    const int64_t ny = c->two_set && c->ysub ? c->ysub->n : 0;
    bool changed = false;
    int64_t cells = 0;
    for (size_t k = 0; k < hb.size(); ++k) {
        HostBox<T> &b = hb[k];
        const int was = b.sub;
        b.sub = 1;
        const int64_t n = hb.size() == 1 ? std::max(c->n, ny) : c->sys_n[k];
        if (c->sweep_variant == 1 && !g_arena.on && !c->whole_cells && c->n >= PARTS_MIN)
            while (window_entries(b, n) > PARTS_WINDOW && (b.sub + 1) * b.lcell <= 4) ++b.sub;
        cells += (int64_t)b.nc[0] * b.nc[1] * b.nc[2] * b.sub * b.sub;
        changed = changed || b.sub != was;
    }
    if (cells > ((int64_t)1 << 28))
        for (HostBox<T> &b : hb) b.sub = 1;
    if (changed) ++c->box_epoch;  // captured graphs and the second set's list are of another grid
    c->parts = false;
    for (const HostBox<T> &b : hb) c->parts = c->parts || b.sub > 1;
    c->parts_variant = c->sweep_variant;
}

// Cell/row offsets of every system and the device system table.
template <typename T>
clm_status layout_systems(clm_ctx *c) {
    std::vector<HostBox<T>> &hb = hboxes<T>(c);
    const int ns = (int)hb.size();
    c->h_celloff.assign(ns + 1, 0);
    c->h_rowoff.assign(ns + 1, 0);
    int64_t cells = 0, rows = 0, pos = 0;
    if (!c->root) choose_parts<T>(c);  // (a second set's boxes come from the owner with their parts)
    std::vector<SysDesc<T>> desc(ns);
    for (int k = 0; k < ns; ++k) {
        c->h_celloff[k] = (int)cells;
        c->h_rowoff[k] = (int)rows;
        desc[k].box = dev_box(hb[k]);
        for (int q = 0; q < 9; ++q) desc[k].invrot[q] = hb[k].invrot.a[q];
        desc[k].cell_off = (int)cells;
        desc[k].row_off = (int)rows;
        desc[k].pos_off = (int)pos;
        desc[k].n = (int)(ns == 1 ? c->n : c->sys_n[k]);
        cells += (int64_t)hb[k].nc[0] * grid_rows(desc[k].box);
        rows += grid_rows(desc[k].box);
        pos += desc[k].n;
        if (cells > ((int64_t)1 << 30)) return fail(c, CLM_ERR_ARG, "too many computing cells");
    }
    c->h_celloff[ns] = (int)cells;
    c->h_rowoff[ns] = (int)rows;
    c->ncells = (int)cells;
    c->nrows = (int)rows;
    HIPCHK(c, ensure(c->sys_desc, sizeof(SysDesc<T>) * ns));
    HIPCHK(c, ensure(c->rowoff, sizeof(int) * (ns + 1)));
    HIPCHK(c, hipMemcpyAsync(c->sys_desc.p, desc.data(), sizeof(SysDesc<T>) * ns, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(c->rowoff.p, c->h_rowoff.data(), sizeof(int) * (ns + 1), hipMemcpyHostToDevice, c->stream));
    clm_status s = sync(c);
    if (s) return s;
    c->layout_dirty = false;
    c->systasks_homes = 0;
    return CLM_OK;
}

template <typename T>
clm_status ensure_bin_buffers(clm_ctx *c) {
    const int64_t n = c->n;
    const int nc1 = c->ncells + 1;
    for (DBuf *b : {&c->cnt, &c->creal, &c->cstart, &c->cur_real, &c->cur_ghost, &c->rstart})
        HIPCHK(c, ensure(*b, sizeof(int) * nc1));
    HIPCHK(c, ensure(c->real_pos, sizeof(int) * std::max<int64_t>(n, 1)));
    HIPCHK(c, ensure(c->order, sizeof(int) * std::max<int64_t>(n, 1)));
    HIPCHK(c, ensure(c->xw, sizeof(Ent<T>) * std::max<int64_t>(n, 1)));
    HIPCHK(c, ensure(c->home_cell, sizeof(int) * std::max<int64_t>(n, 1)));
    HIPCHK(c, ensure(c->flags, sizeof(uint32_t) * 4));
    return CLM_OK;
}

const int *sys_of_ptr(clm_ctx *c) { return c->nsys > 1 ? (const int *)c->sys_of.p : nullptr; }

constexpr int TASK_INTS = TASK_COUNTERS * TASK_COUNTER_STRIDE;

enum { SCAN_CELLS = 0, SCAN_ROWS = 1, SCAN_CHUNKS = 2 };

// State of one single-pass scan site for n elements: the ticket and done counters, then
// one status word per tile.  Zeroed when allocated (never inside a graph capture: the
// capture sizes it first); every launch leaves it zeroed again.
clm_status scan_state(clm_ctx *c, int site, long long n, ScanState &st) {
    const size_t bytes = sizeof(unsigned long long) * (size_t)(scan_tiles(n) + 1);
    DBuf &b = c->scan_st[site];
    if (!b.p || b.bytes < bytes) {
        HIPCHK(c, ensure(b, bytes));
        HIPCHK(c, hipMemsetAsync(b.p, 0, b.bytes, c->stream));
    }
    st.ticket = (unsigned int *)b.p;
    st.done = st.ticket + 1;
    st.status = (unsigned long long *)b.p + 1;
    return CLM_OK;
}

// k_bin_count + scan of the cell counts (no host synchronisation).
template <typename T>
clm_status enqueue_count(clm_ctx *c) {
    const int64_t n = c->n;
    const int nc1 = c->ncells + 1;
    clm_status s;
    if ((s = fill_zero(c, {{c->cnt.p, nc1}, {c->creal.p, nc1}, {c->flags.p, 4}}))) return s;
    const SysDesc<T> *sd = (const SysDesc<T> *)c->sys_desc.p;
    if (n > 0) {
        if (c->dim == 3)
            LAUNCH(c, "k_bin_count", hipLaunchKernelGGL((k_bin_count<T, 3>), dim3(blocks(n, 256)), dim3(256), 0, c->stream,
                                                        (const T *)c->pos.p, (int)n, sd, sys_of_ptr(c), (Ent<T> *)c->xw.p,
                                                        (int *)c->home_cell.p, (int *)c->cnt.p, (int *)c->creal.p,
                                                        (uint32_t *)c->flags.p));
        else
            LAUNCH(c, "k_bin_count", hipLaunchKernelGGL((k_bin_count<T, 2>), dim3(blocks(n, 256)), dim3(256), 0, c->stream,
                                                        (const T *)c->pos.p, (int)n, sd, sys_of_ptr(c), (Ent<T> *)c->xw.p,
                                                        (int *)c->home_cell.p, (int *)c->cnt.p, (int *)c->creal.p,
                                                        (uint32_t *)c->flags.p));
    }
    if ((s = scan_int(c, (const int *)c->creal.p, (int *)c->rstart.p, nc1))) return s;
    return scan_int(c, (const int *)c->cnt.p, (int *)c->cstart.p, nc1);
}

// The triclinic sweep of one set walks the real and the ghost entries in separate arrays.
bool wants_split(const clm_ctx *c) { return c->celltype == CLM_TRICLINIC && !c->root; }

// Makes room in an entry array of the cell list.  A larger block holds nothing of the list, which
// is then built again before the next operator walks it.
hipError_t ensure_entries(clm_ctx *c, DBuf &b, size_t bytes) {
    if (bytes > b.bytes) c->cl_valid = c->split_valid = false;
    return ensure(b, bytes);
}

// Sizes the split arrays for the current entry capacity (before a sort is enqueued or
// captured).
template <typename T>
clm_status ensure_split(clm_ctx *c) {
    if (!wants_split(c)) return CLM_OK;
    HIPCHK(c, ensure_entries(c, c->E_real, sizeof(Ent<T>) * (std::max<int64_t>(c->n, 1) + SWEEP_PAD)));
    HIPCHK(c, ensure_entries(c, c->E_ghost, sizeof(Ent<T>) * (std::max<int64_t>(c->e_cap, 1) + SWEEP_PAD)));
    return CLM_OK;
}

// Particles below which the binning takes a thread per particle and image (k_bin_images): each
// makes its one claim as soon as it knows the cell (1000 particles, 5300 entries: 9.8 us
// against 32.5 with k_bin_bucket, which goes through the 27 directions one by one; 10000: 15.6
// against 35.5; 20000: 31 against 29, the claims then being the bound, and k_bin_bucket makes one
// per cell and wave).
constexpr int64_t BIN_IMAGES_MAX = 20000;

// There the cells' counters lie on cache lines of their own (2^4 words apart): claims on one
// line queue, whichever of its counters they take (1000 particles: 22 us with 16 to a line).
int counter_shift(const clm_ctx *c) { return c->n < BIN_IMAGES_MAX && c->ncells <= 8192 ? 4 : 0; }

// Threads per entry of the cell sort: a cell's entries are compared with each other, one after
// another; while there are too few entries to fill the chip, several threads share the
// comparisons of one (20000 particles of 170 to a cell: 33 us with one, 20 with 4; 1e5: 21.9 with
// one, 19.6 with 2; 2e5: 32 with one, 36 with 2).
int sort_threads(int64_t entries) { return entries <= 100000 ? 4 : entries <= 250000 ? 2 : 1; }

// Order every cell by x into E and list the real particles' positions (k_cell_sort); the
// unsorted entries are in E_raw, compact (bucket 0) or in cell buckets.
// threads: an upper bound of the entry count (the count itself when known on the host, the
// entry capacity inside a captured graph).
template <typename T>
clm_status enqueue_sort(clm_ctx *c, int bucket, int64_t threads) {
    c->split_valid = false;
    if (c->ncells <= 0 || threads <= 0) {
        c->order_valid = false;
        return CLM_OK;
    }
    // the split arrays, when wanted and sized for this capacity (ensure_split)
    const bool split = wants_split(c) && c->E_real.bytes >= sizeof(Ent<T>) * (size_t)std::max<int64_t>(c->n, 1) &&
                       c->E_ghost.bytes >= sizeof(Ent<T>) * (size_t)std::max<int64_t>(c->e_cap, 1);
    const int q = sort_threads(threads);
    auto kernel = q == 4 ? k_cell_sort<T, 4> : q == 2 ? k_cell_sort<T, 2> : k_cell_sort<T, 1>;
    LAUNCH(c, "k_cell_sort", hipLaunchKernelGGL(kernel, dim3(blocks(threads * q, 256)), dim3(256), 0, c->stream,
                                                c->ncells, (const int *)c->cstart.p, (const int *)c->rstart.p,
                                                (const Ent<T> *)c->E_raw.p, bucket, c->e_cap, (Ent<T> *)c->E.p,
                                                (int *)c->real_pos.p, (int *)c->order.p, (int *)c->home_cell.p,
                                                split ? (Ent<T> *)c->E_real.p : nullptr,
                                                split ? (Ent<T> *)c->E_ghost.p : nullptr));
    c->order_valid = true;
    c->split_valid = split;
    return CLM_OK;
}

// k_bin_scatter into E (capacity c->e_cap; overflow raises FLAG_OVERFLOW).
template <typename T>
clm_status enqueue_scatter(clm_ctx *c) {
    const int64_t n = c->n;
    const int nc1 = c->ncells + 1;
    clm_status s;
    if ((s = fill_zero(c, {{c->cur_real.p, nc1}, {c->cur_ghost.p, nc1}}))) return s;
    const SysDesc<T> *sd = (const SysDesc<T> *)c->sys_desc.p;
    if (n > 0) {
        const int *tp = c->has_types ? (const int *)c->types.p : nullptr;
        if (c->dim == 3)
            LAUNCH(c, "k_bin_scatter", hipLaunchKernelGGL((k_bin_scatter<T, 3>), dim3(blocks(n, 256)), dim3(256), 0, c->stream,
                                                          (int)n, sd, sys_of_ptr(c), (const Ent<T> *)c->xw.p,
                                                          (const int *)c->home_cell.p, (const int *)c->cstart.p,
                                                          (const int *)c->creal.p, tp, (int *)c->cur_real.p,
                                                          (int *)c->cur_ghost.p, (Ent<T> *)c->E_raw.p, c->e_cap,
                                                          (uint32_t *)c->flags.p));
        else
            LAUNCH(c, "k_bin_scatter", hipLaunchKernelGGL((k_bin_scatter<T, 2>), dim3(blocks(n, 256)), dim3(256), 0, c->stream,
                                                          (int)n, sd, sys_of_ptr(c), (const Ent<T> *)c->xw.p,
                                                          (const int *)c->home_cell.p, (const int *)c->cstart.p,
                                                          (const int *)c->creal.p, tp, (int *)c->cur_real.p,
                                                          (int *)c->cur_ghost.p, (Ent<T> *)c->E_raw.p, c->e_cap,
                                                          (uint32_t *)c->flags.p));
    }
    return enqueue_sort<T>(c, 0, c->e_cap);
}

// A build may skip its status read-back: a periodic context whose bucket size and entry
// capacity are known, unless the last deferred build overflowed.
bool can_defer(const clm_ctx *c) {
    return !c->no_defer && c->celltype != CLM_NONPERIODIC && c->bucket > 0 && c->e_cap > 0 &&
           c->sweep_variant == 1;
}

clm_status check_flags(clm_ctx *c, uint32_t fl) {
    if (fl & FLAG_SCAN) return fail(c, CLM_ERR_HIP, "a single-pass scan did not complete (internal error)");
    if (fl & FLAG_NAN) return fail(c, CLM_ERR_NAN, "Invalid coordinates found (NaN or Inf)");
    if (fl & FLAG_RANGE)
        return fail(c, CLM_ERR_RANGE, "a particle maps outside the computing grid (the reference raises a BoundsError)");
    return CLM_OK;
}

// Entries per bucket for a fullest cell of mx entries: a power of two with 25 % headroom;
// -1 (single-pass binning off) when the buckets would take more than sixteen times the
// compact cell list and 1 GiB.
int bucket_size(const clm_ctx *c, int mx, size_t esize) {
    int64_t b = 8;
    while (b < (int64_t)mx + mx / 4 + 4) b *= 2;
    const double need = (double)c->ncells * (double)b * (double)esize;
    const double limit = std::max(16.0 * (double)(c->n_entries + 1) * (double)esize, 1024.0 * 1024 * 1024);
    if (need > limit || b > (1 << 20)) return -1;
    return (int)b;
}

// Status of a build enqueued without its read-back (the status block copied by sync()):
// errors are reported as from a synchronous build; an overflow (a cell past its bucket,
// or more entries than the list holds) invalidates the list, and CLM_REDO tells the entry
// point to run again on a list rebuilt with its status read first.  The sweeps skip such
// a list on the device (SweepArgs::bin_flags), so nothing read it out of range.
clm_status check_deferred_build(clm_ctx *c, const uint32_t *status) {
    const uint32_t fl = status[0];
    const int mx = (int)status[1], total = (int)status[2];
    clm_status s = check_flags(c, fl);
    if (s) {
        c->cl_valid = false;
        c->order_valid = false;
        return s;
    }
    if ((fl & FLAG_OVERFLOW) || (int64_t)total > c->e_cap) {
        c->cl_valid = false;
        c->dirty = true;
        c->order_valid = false;  // cells past the capacity were not sorted
        c->no_defer = true;
        if (fl & FLAG_OVERFLOW) c->bucket = bucket_size(c, mx, c->dtype == CLM_F32 ? sizeof(Ent<float>) : sizeof(Ent<double>));
        return CLM_REDO;
    }
    c->n_entries = total;
    return CLM_OK;
}

// The first two launches of a single-pass build: zeroed counters and status block,
// k_bin_bucket into the cell buckets, then k_scan_cells (per-cell counts, both scans, the
// fullest cell and the entry total).  Status block c->flags: [0] flags, [1] fullest cell,
// [2] entry total.
template <typename T>
clm_status enqueue_bucket_pass(clm_ctx *c) {
    const int64_t n = c->n;
    const SysDesc<T> *sd = (const SysDesc<T> *)c->sys_desc.p;
    const int *tp = c->has_types ? (const int *)c->types.p : nullptr;
    const int *ord = c->order_valid ? (const int *)c->order.p : nullptr;
    clm_status s;
    if ((s = fill_zero(c, {{c->cnt64.p, (2 * (int64_t)c->ncells) << counter_shift(c)}, {c->flags.p, 4}}))) return s;
    if (n > 0) {
        const bool split = n < BIN_IMAGES_MAX;
        auto kernel = c->dim == 3 ? (split ? k_bin_images<T, 3> : k_bin_bucket<T, 3>)
                                  : (split ? k_bin_images<T, 2> : k_bin_bucket<T, 2>);
        const dim3 block(split ? 64 : 256);
        const dim3 grid(blocks(n, block.x), !split ? 1 : c->dim == 3 ? 27 : 9);
        LAUNCH(c, "k_bin_bucket", hipLaunchKernelGGL(kernel, grid, block, 0, c->stream, (const T *)c->pos.p, (int)n, ord, sd,
                                                     sys_of_ptr(c), tp, (unsigned long long *)c->cnt64.p,
                                                     counter_shift(c), (Ent<T> *)c->E_raw.p, c->bucket, (uint32_t *)c->flags.p));
    }
    ScanState st;
    if ((s = scan_state(c, SCAN_CELLS, c->ncells, st))) return s;
    ProdCells pc{(const unsigned long long *)c->cnt64.p, counter_shift(c), (int *)c->cnt.p, (int *)c->creal.p};
    LAUNCH(c, "k_scan_cells", hipLaunchKernelGGL((k_scan_pair<ProdCells>), dim3((unsigned)scan_tiles_for<ProdCells>(c->ncells)),
                                                 dim3(SCAN_THREADS), 0, c->stream, (long long)c->ncells, pc,
                                                 ScanValue{}, (int *)c->cstart.p, (int *)c->rstart.p,
                                                 (int *)c->flags.p + 1, (int *)c->flags.p + 2, st, (unsigned int *)c->flags.p,
                                                 FLAG_SCAN));
    return CLM_OK;
}

// Single-pass binning (k_bin_bucket + k_scan_pair + k_cell_sort).  With a bucket size and
// an entry capacity known from an earlier build, nothing is read back: the sort covers the
// capacity (it reads the count on the device) and the status is checked at the next
// synchronisation.  Otherwise one host synchronisation reads the status first.
// done = false when the buckets cannot be sized within the memory limit (the caller then
// bins in two passes).
template <typename T>
clm_status bin_bucketed(clm_ctx *c, bool &done) {
    done = false;
    HIPCHK(c, ensure(c->cnt64, (sizeof(unsigned long long) * std::max(c->ncells, 1)) << counter_shift(c)));
    HIPCHK(c, ensure(c->maxcnt, sizeof(int) * 2));
    for (int attempt = 0; attempt < 4; ++attempt) {
        if (c->bucket <= 0) return CLM_OK;
        HIPCHK(c, ensure(c->E_raw, sizeof(Ent<T>) * (size_t)c->ncells * (size_t)c->bucket));
        clm_status s;
        if ((s = enqueue_bucket_pass<T>(c))) return s;
        if (can_defer(c)) {
            if ((s = ensure_split<T>(c))) return s;
            if ((s = enqueue_sort<T>(c, c->bucket, c->e_cap))) return s;
            c->bin_pending = true;
            done = true;
            return CLM_OK;
        }
        HIPCHK(c, hipMemcpyAsync(c->h_flags, c->flags.p, 4 * sizeof(uint32_t), hipMemcpyDeviceToHost, c->stream));
        if ((s = sync(c))) return s;
        if ((s = check_flags(c, c->h_flags[0]))) return s;
        const int mx = (int)c->h_flags[1], total = (int)c->h_flags[2];
        c->n_entries = total;
        if (c->h_flags[0] & FLAG_OVERFLOW) {  // a cell outgrew its bucket: larger buckets, again
            c->bucket = bucket_size(c, mx, sizeof(Ent<T>));
            continue;
        }
        HIPCHK(c, ensure(c->E, sizeof(Ent<T>) * ((int64_t)total + SWEEP_PAD)));
        c->e_cap = (int64_t)(c->E.bytes / sizeof(Ent<T>)) - SWEEP_PAD;
        if ((s = ensure_split<T>(c))) return s;
        if ((s = enqueue_sort<T>(c, c->bucket, total))) return s;
        done = true;
        return CLM_OK;
    }
    c->bucket = -1;
    return CLM_OK;
}

// A new cell list: its home and task tables are to be built again.
void forget_modes(clm_ctx *c) {
    for (bool &m : c->mode_valid) m = false;
    for (bool &m : c->rows_valid) m = false;
}

template <typename T>
clm_status update_cell_list_t(clm_ctx *c) {
    if (!c->has_box) return fail(c, CLM_ERR_STATE, "no box set");
    if (!c->has_pos) return fail(c, CLM_ERR_STATE, "no positions set");
    if (c->n >= (int64_t)IDX_LIMIT) return fail(c, CLM_ERR_ARG, "too many particles (limit 2^28-1)");
    clm_status s;
    if (c->celltype == CLM_NONPERIODIC && !c->root) {  // a sub-context gets its box from the owner
        if ((s = nonperiodic_box<T>(c))) return s;
        c->layout_dirty = true;
        ++c->box_epoch;
    }
    if (!c->root && c->parts_variant != c->sweep_variant) c->layout_dirty = true;
    if (c->layout_dirty) {
        if ((s = layout_systems<T>(c))) return s;
        c->bucket = 0;  // re-sized on the first two-pass build of the new layout
        c->order_valid = false;
    }
    if ((s = ensure_bin_buffers<T>(c))) return s;
    bool done = false;
    if (c->bucket > 0 && (s = bin_bucketed<T>(c, done))) return s;
    if (!done) {
        // two passes: count (+ the fullest cell, which sizes the buckets of later builds),
        // scan, scatter
        if ((s = enqueue_count<T>(c))) return s;
        HIPCHK(c, ensure(c->maxcnt, sizeof(int) * 2));
        if ((s = fill_int(c, c->maxcnt.p, 1, 0))) return s;
        LAUNCH(c, "k_count_max", hipLaunchKernelGGL(k_count_max, dim3(std::min<unsigned>(blocks(c->ncells + 1, 256), 512)),
                                                    dim3(256), 0, c->stream,
                                                    c->ncells, (const int *)c->cnt.p, (int *)c->maxcnt.p));
        int total = 0, mx = 0;
        uint32_t fl = 0;
        const void *src[3] = {(int *)c->cstart.p + c->ncells, c->maxcnt.p, c->flags.p};
        void *dst[3] = {&total, &mx, &fl};
        if (c->h_mapped) {  // one launch, not three copies to pageable memory of ~20 us each
            ReadList r;
            std::memset(&r, 0, sizeof(r));
            for (int k = 0; k < 3; ++k) {
                r.p[k] = (const uint32_t *)src[k];
                r.n[k] = 1;
            }
            r.count = 3;
            LAUNCH(c, "k_read_back", hipLaunchKernelGGL(k_read_back, dim3(1), dim3(256), 0, c->stream, r, c->h_flags + READ_RESULTS));
        } else {
            for (int k = 0; k < 3; ++k)
                HIPCHK(c, hipMemcpyAsync(dst[k], src[k], sizeof(uint32_t), hipMemcpyDeviceToHost, c->stream));
        }
        if ((s = sync(c))) return s;
        if (c->h_mapped)
            for (int k = 0; k < 3; ++k) std::memcpy(dst[k], result_words(c) + k, sizeof(uint32_t));
        if ((s = check_flags(c, fl))) return s;
        c->n_entries = total;
        HIPCHK(c, ensure(c->E, sizeof(Ent<T>) * ((int64_t)total + SWEEP_PAD)));
        HIPCHK(c, ensure(c->E_raw, c->E.bytes));
        c->e_cap = (int64_t)(std::min(c->E.bytes, c->E_raw.bytes) / sizeof(Ent<T>)) - SWEEP_PAD;
        if ((s = ensure_split<T>(c))) return s;
        if ((s = enqueue_scatter<T>(c))) return s;
        if (c->bucket == 0) c->bucket = bucket_size(c, mx, sizeof(Ent<T>));
    }
    if (!c->bin_pending) c->no_defer = false;
    c->cl_valid = true;
    c->dirty = false;
    forget_modes(c);
    return CLM_OK;
}

clm_status ensure_cell_list(clm_ctx *c) {
    if (c->cl_valid && !c->dirty) return CLM_OK;
    return c->dtype == CLM_F32 ? update_cell_list_t<float>(c) : update_cell_list_t<double>(c);
}

// Both cell lists of a two-set context on one box (CellListPair, CellLists.jl:590-605):
// the x list first (for a non-periodic box it sizes the box from both sets), then the
// owner's box is handed to the y sub-context.
clm_status ensure_cross(clm_ctx *c) {
    clm_ctx *y = c->ysub;
    if (!c->two_set || !y) return fail(c, CLM_ERR_STATE, "no second set of positions");
    if (c->nsys != 1) return fail(c, CLM_ERR_ARG, "two sets need a single system");
    if (!y->has_pos) return fail(c, CLM_ERR_STATE, "no y positions set");
    if (c->celltype == CLM_NONPERIODIC && y->dirty) c->dirty = true;
    clm_status s = ensure_cell_list(c);
    if (s) return s;
    if (c->sub_epoch != c->box_epoch) {
        y->hbf = c->hbf;
        y->hbd = c->hbd;
        y->nsys = 1;
        y->celltype = c->celltype;
        y->cutoff_in = c->cutoff_in;
        y->lcell = c->lcell;
        y->parts = c->parts;
        y->has_box = true;
        y->layout_dirty = true;
        y->dirty = true;
        c->sub_epoch = c->box_epoch;
    }
    y->waves_per_cu = c->waves_per_cu;
    y->sweep_variant = c->sweep_variant;
    y->stream = c->stream;
    if ((s = ensure_cell_list(y))) return fail(c, s, y->err);
    return CLM_OK;
}

int mode_a(const clm_ctx *c) { return c->celltype == CLM_TRICLINIC ? MODE_A_TRIC : MODE_A_ORTHO; }

// Per-cell home counts and per-row wave tasks of a sweep mode (no host synchronisation).
// Home tables: the two-set modes share those of the one-set modes with the same homes.
inline int mode_table(int mode) {
    return mode == MODE_X_ORTHO ? MODE_A_ORTHO : (mode == MODE_X_REAL ? MODE_B : mode);
}

// Homes per cell, scanned: the real-particle scan of the binning (rstart) when the homes
// are the real particles, else a scan of all entries of cells holding a real particle.
const int *home_start(const clm_ctx *c, int mode) {
    mode = mode_table(mode);
    return mode_all_entries(mode) ? (const int *)c->hstart[mode].p : (const int *)c->rstart.p;
}

// Cells up to which their homes are counted and scanned in one launch: the tiles of that scan take
// numbers from one counter and wait for each other in turn, 58 ns each, which costs more than a launch
// where there are many (closest pair of 5000 particles in a grid of 1e5 cells: 97 us against 98 in
// three launches, 3e5: 108 and 105, 1e6: 159 and 140, 1e7: 527 and 348, 6.3e7: 2764 and 1304).
constexpr int HOMES_ONE_LAUNCH = 300000;

// Home starts of the modes whose homes are all entries of the real cells.
template <typename T>
clm_status enqueue_homes(clm_ctx *c, int mode) {
    HIPCHK(c, ensure(c->hstart[mode], sizeof(int) * (c->ncells + 1)));
    ScanState st;
    clm_status s;
    ProdHomes<T> ph{(const int *)c->cnt.p, (const int *)c->creal.p, (const SysDesc<T> *)c->sys_desc.p, c->nsys, c->parts};
    if (c->ncells > HOMES_ONE_LAUNCH) {
        int *counts = (int *)c->cur_real.p;  // (scratch of the two-pass build)
        LAUNCH(c, "k_home_counts", hipLaunchKernelGGL(k_home_counts<T>, dim3(blocks(c->ncells + 1, 256)), dim3(256), 0, c->stream,
                                                      c->ncells, ph, counts));
        return scan_int(c, counts, (int *)c->hstart[mode].p, c->ncells + 1);
    }
    if ((s = scan_state(c, SCAN_CELLS, c->ncells, st))) return s;
    LAUNCH(c, "k_scan_homes", hipLaunchKernelGGL((k_scan_pair<ProdHomes<T>>), dim3((unsigned)scan_tiles_for<ProdHomes<T>>(c->ncells)),
                                                 dim3(SCAN_THREADS), 0, c->stream, (long long)c->ncells, ph,
                                                 ScanValue{}, (int *)c->hstart[mode].p, (int *)nullptr,
                                                 (int *)nullptr, (int *)nullptr, st, (unsigned int *)c->flags.p, FLAG_SCAN));
    return CLM_OK;
}

// Wave tasks per row and their scan (the union-row sweep).
template <typename T>
clm_status enqueue_rows(clm_ctx *c, int mode) {
    HIPCHK(c, ensure(c->tstart[mode], sizeof(int) * (c->nrows + 1)));
    ScanState st;
    clm_status s;
    if ((s = scan_state(c, SCAN_ROWS, c->nrows, st))) return s;
    ProdRows<T> pr{(const SysDesc<T> *)c->sys_desc.p, (const int *)c->rowoff.p, home_start(c, mode), c->nsys};
    LAUNCH(c, "k_scan_rows", hipLaunchKernelGGL((k_scan_pair<ProdRows<T>>), dim3((unsigned)scan_tiles_for<ProdRows<T>>(c->nrows)),
                                                dim3(SCAN_THREADS), 0, c->stream, (long long)c->nrows, pr,
                                                ScanValue{}, (int *)c->tstart[mode].p, (int *)nullptr, (int *)nullptr, (int *)nullptr, st,
                                                (unsigned int *)c->flags.p, FLAG_SCAN));
    return CLM_OK;
}

// Lanes per home of the windowed sweep (homes of c, neighbours of nb).  With few homes the
// chip is filled by more lanes on each: 32 below 20000 homes (1000 particles, energy and
// forces: 165 us a call against 194 with 8; 10000 at float64: 203 against 216).  Above, the
// fewer lanes the less is done per home besides testing entries, but the longer the wait for
// home with the most entries: 8 for windows of 160 entries and more (list of 1e5, 340
// entries: the sweep takes 119 us, 134 with 4; clustered, 1000 entries: 49.6 ms against 56.3),
// else 4 (1M at lcell 2, 86 entries: list 1188 us against 1235, forces 1210 against 1248;
// batch 6.48 ms against 6.80).
int choose_lanes(const clm_ctx *c, const clm_ctx *nb) {
    if (c->n < 20000 && !c->parts) return 32;
    double w = 0;
    for (int k = 0; k < c->nsys; ++k) {
        const int64_t n = c->nsys == 1 ? nb->n : c->sys_n[k];
        w = std::max(w, c->dtype == CLM_F32 ? window_entries(c->hbf[k], n) : window_entries(c->hbd[k], n));
    }
    return w < 160 ? 4 : 8;
}

// First wave task of each system of a batch, for the current task shape: from the host where
// the homes are the particles (nothing to launch), else scanned on the device.
template <typename T>
clm_status prepare_systasks(clm_ctx *c, int mode) {
    const int homes = task_homes(c->sweep_variant, c->sweep_lanes);
    if (c->nsys <= 1) return CLM_OK;
    if (mode_all_entries(mode)) {
        int shift = 0;
        while ((1 << shift) < homes) ++shift;
        HIPCHK(c, ensure(c->systasks_all, sizeof(int) * (c->nsys + 1)));
        ScanState st;
        clm_status s;
        if ((s = scan_state(c, SCAN_ROWS, c->nsys, st))) return s;
        ProdSystems<T> ps{(const SysDesc<T> *)c->sys_desc.p, home_start(c, mode), c->nsys, c->ncells, shift};
        LAUNCH(c, "k_scan_systems", hipLaunchKernelGGL((k_scan_pair<ProdSystems<T>>), dim3((unsigned)scan_tiles_for<ProdSystems<T>>(c->nsys)),
                                                       dim3(SCAN_THREADS), 0, c->stream, (long long)c->nsys, ps,
                                                       ScanValue{}, (int *)c->systasks_all.p, (int *)nullptr,
                                                       (int *)nullptr, (int *)nullptr, st, (unsigned int *)c->flags.p, FLAG_SCAN));
        return CLM_OK;
    }
    if (c->systasks_homes == homes) return CLM_OK;
    std::vector<int> first(c->nsys + 1, 0);
    for (int k = 0; k < c->nsys; ++k) first[k + 1] = first[k] + (int)((c->sys_n[k] + homes - 1) / homes);
    HIPCHK(c, ensure(c->systasks, sizeof(int) * first.size()));
    HIPCHK(c, hipMemcpyAsync(c->systasks.p, first.data(), sizeof(int) * first.size(), hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    c->systasks_homes = homes;
    return CLM_OK;
}

// The tables a sweep of homes of c against nb needs besides the cell lists.
clm_status prepare_mode(clm_ctx *c, int mode, const clm_ctx *nb) {
    mode = mode_table(mode);
    c->sweep_lanes = choose_lanes(c, nb);
    clm_status s;
    if (mode_all_entries(mode) && !c->mode_valid[mode]) {
        if ((s = c->dtype == CLM_F32 ? enqueue_homes<float>(c, mode) : enqueue_homes<double>(c, mode))) return s;
        c->mode_valid[mode] = true;
    }
    if (c->sweep_variant == 0) {
        if (c->rows_valid[mode]) return CLM_OK;
        s = c->dtype == CLM_F32 ? enqueue_rows<float>(c, mode) : enqueue_rows<double>(c, mode);
        if (!s) c->rows_valid[mode] = true;
        return s;
    }
    return c->dtype == CLM_F32 ? prepare_systasks<float>(c, mode) : prepare_systasks<double>(c, mode);
}

template <typename T>
SweepArgs<T> sweep_args(clm_ctx *c, int mode) {
    mode = mode_table(mode);
    SweepArgs<T> sa;
    sa.hstart = home_start(c, mode);
    sa.tstart = (const int *)c->tstart[mode].p;
    sa.real_pos = (const int *)c->real_pos.p;
    sa.real_cell = (const int *)c->home_cell.p;
    sa.systasks = (const int *)(mode_all_entries(mode) ? c->systasks_all.p : c->systasks.p);
    sa.ncells = c->ncells;
    sa.nhomes = (int)c->n;
    sa.rowoff = (const int *)c->rowoff.p;
    sa.sys = (const SysDesc<T> *)c->sys_desc.p;
    sa.task_counter = (int *)c->counters.p;
    sa.nrows = c->nrows;
    sa.nsys = c->nsys;
    return sa;
}

SweepShape sweep_shape(const clm_ctx *c) {
    return {c->dim, c->sweep_variant, c->sweep_lanes, c->parts, c->sweep_group, c->waves_per_cu, c->num_cus};
}

// Upper bound of the wave tasks of a sweep (the entry count may be that of an earlier build).
int64_t max_tasks(const clm_ctx *c, int mode) {
    const int64_t homes = mode_all_entries(mode) ? std::max<int64_t>(c->n_entries, c->n) : c->n;
    return homes / task_homes(c->sweep_variant, c->sweep_lanes) + (c->sweep_variant == 0 ? c->nrows : c->nsys) + 1;
}

// Waves of a sweep: no more than it has tasks, in whole rounds over the 8 XCDs.
template <typename T, int MODE, typename Op>
int sweep_waves(const clm_ctx *c) {
    const int64_t tasks = (max_tasks(c, MODE) + 7) / 8 * 8;
    return (int)std::min<int64_t>(sweep_grid<T, MODE, Op>(sweep_shape(c)), tasks);
}

// Sweep with homes from context c and neighbours from context nb (nb == c for one set).
template <typename T, int MODE, typename Op>
clm_status run_sweep_on(clm_ctx *c, clm_ctx *nb, const char *name, const Op &op, int grid) {
    HIPCHK(c, ensure(c->counters, sizeof(int) * TASK_INTS));
    clm_status s;
    if (!c->counters_zeroed && (s = fill_int(c, c->counters.p, TASK_INTS, 0))) return s;
    c->counters_zeroed = false;
    SweepArgs<T> sa = sweep_args<T>(c, MODE);
    if (grid <= 0) grid = sweep_waves<T, MODE, Op>(c);
    const Ent<T> *E = (const Ent<T> *)c->E.p;
    const int *cs = (const int *)c->cstart.p;
    const Ent<T> *En = (const Ent<T> *)nb->E.p;
    const int *csn = (const int *)nb->cstart.p;
    sa.en_bytes = (uint32_t)std::min<size_t>(nb->E.bytes, 0xFFFFFFF0u);
    if (c->sweep_variant == 1 && nb->E.bytes > 0xFFFFFFF0u)
        return fail(c, CLM_ERR_ARG, "cell list above 4 GiB: use sweep variant 0");
    // a build whose status is still to be read: the sweep checks it on the device first
    sa.bin_flags = c->bin_pending ? (const uint32_t *)c->flags.p : nullptr;
    sa.e_cap = c->e_cap;
    sa.bin_flags_n = nb != c && nb->bin_pending ? (const uint32_t *)nb->flags.p : nullptr;
    sa.e_cap_n = nb->e_cap;
    sa.reals = (const Ent<T> *)c->E_real.p;
    sa.ghosts = (const Ent<T> *)c->E_ghost.p;
    sa.reals_bytes = (uint32_t)std::min<size_t>(c->E_real.bytes, 0xFFFFFFF0u);
    sa.ghosts_bytes = (uint32_t)std::min<size_t>(c->E_ghost.bytes, 0xFFFFFFF0u);
    if (MODE == MODE_A_TRIC && c->sweep_variant == 1) {
        if (!c->split_valid) return fail(c, CLM_ERR_STATE, "the split entry arrays of the triclinic sweep are not built");
        if (c->E_ghost.bytes > 0xFFFFFFF0u) return fail(c, CLM_ERR_ARG, "cell list above 4 GiB: use sweep variant 0");
    }
    LAUNCH(c, name, (sweep_launch<T, MODE, Op>(sweep_shape(c), grid, c->stream, E, cs, En, csn, sa, op)));
    return CLM_OK;
}

template <typename T, int MODE, typename Op>
clm_status run_sweep(clm_ctx *c, const char *name, const Op &op, int grid) {
    return run_sweep_on<T, MODE>(c, c, name, op, grid);
}

// The sweep that visits every pair once in the reference's orientation: one set
// (self.jl) or two (cross.jl, x homes against the y list).
int mode_once(const clm_ctx *c) {
    if (c->two_set) return c->celltype == CLM_TRICLINIC ? MODE_X_REAL : MODE_X_ORTHO;
    return mode_a(c);
}

clm_status prepare_once(clm_ctx *c) {
    clm_status s = c->two_set ? ensure_cross(c) : ensure_cell_list(c);
    if (s) return s;
    return prepare_mode(c, mode_once(c), c->two_set ? c->ysub : c);
}

template <typename T, typename Op>
clm_status run_mode_a(clm_ctx *c, const char *name, const Op &op, int grid) {
    switch (mode_once(c)) {
        case MODE_A_TRIC: return run_sweep<T, MODE_A_TRIC>(c, name, op, grid);
        case MODE_X_ORTHO: return run_sweep_on<T, MODE_X_ORTHO>(c, c->ysub, name, op, grid);
        case MODE_X_REAL: return run_sweep_on<T, MODE_X_REAL>(c, c->ysub, name, op, grid);
        default: return run_sweep<T, MODE_A_ORTHO>(c, name, op, grid);
    }
}

template <typename T, typename Op>
int once_waves(clm_ctx *c) {
    switch (mode_once(c)) {
        case MODE_A_TRIC: return sweep_waves<T, MODE_A_TRIC, Op>(c);
        case MODE_X_ORTHO: return sweep_waves<T, MODE_X_ORTHO, Op>(c);
        case MODE_X_REAL: return sweep_waves<T, MODE_X_REAL, Op>(c);
        default: return sweep_waves<T, MODE_A_ORTHO, Op>(c);
    }
}

template <typename T>
clm_status neighborlist_t(clm_ctx *c, int32_t *oi, int32_t *oj, void *od, int64_t cap, int64_t *npairs, int on_device) {
    clm_status s;
    // (a list whose grid is laid out now takes whole cells: writing the pairs bounds it, and it
    // gains nothing from thinner rows: 1e5 particles 119 us, 144 in parts, 2e4 at float64 103 and 155.
    // The grid stays what the first operator after a change of box or count made it; an open box is
    // laid out whenever its positions change, by whatever asks first, which may be clm_get_box)
    c->whole_cells = true;
    s = prepare_once(c);
    c->whole_cells = false;
    if (s) return s;
    int32_t *di = oi, *dj = oj;
    T *dd = (T *)od;
    if (!on_device) {
        HIPCHK(c, ensure(c->nl_i, sizeof(int32_t) * std::max<int64_t>(cap, 1)));
        HIPCHK(c, ensure(c->nl_j, sizeof(int32_t) * std::max<int64_t>(cap, 1)));
        HIPCHK(c, ensure(c->nl_d, sizeof(T) * std::max<int64_t>(cap, 1)));
        di = (int32_t *)c->nl_i.p;
        dj = (int32_t *)c->nl_j.p;
        dd = (T *)c->nl_d.p;
    }
    // persistent grid and a bound on the slots left unused in partially filled chunks
    const int grid = once_waves<T, OpNeighborList<T>>(c);
    const int64_t active = grid;
    // the slots of a chunk: an eighth of what a wave writes, so that it leaves few empty, up to
    // NL_CHUNK (list of 1e5: sweep and moves 163 + 25 us; a third: 160 + 40; a sixteenth: 173 + 27)
    int chunk = 64;
    while (chunk < NL_CHUNK && cap > 8 * chunk * active) chunk *= 2;
    // Spill slots beyond the capacity: every wave holds at most one partial and one unused
    // prefetched chunk, and the interleaved counters can run ahead of each other by a few
    // standard deviations of sqrt(active) chunks each.  Counted in chunks of up to SPILL_CHUNK slots
    // (17M slots with 5120 waves, 0.2 GB at float32): longer ones are handed out as much more
    // seldom, and waves that end do not all hold a full one (lists of 26M to 353M pairs without a
    // slot to spare, even, in clusters and in clumps within a gas: one sweep each).  A pair beyond the
    // spill raises the overflow word; the sweep is then repeated with twice the spill.
    constexpr int SPILL_CHUNK = 512;
    int64_t scap = ((int64_t)3 * active + 4 * NL_COUNTERS * ((int64_t)std::sqrt((double)active) + 1) + NL_COUNTERS) *
                   std::min(chunk, SPILL_CHUNK);
    const int nctr = NL_COUNTERS * NL_COUNTER_STRIDE;  // chunk counters, then pair counts, the pair count and the overflow word
    HIPCHK(c, ensure(c->nl_count, sizeof(unsigned long long) * (2 * nctr + 2)));
    unsigned long long *ctr = (unsigned long long *)c->nl_count.p;
    unsigned long long *tot = ctr + 2 * nctr;
    unsigned int *ovf = (unsigned int *)(ctr + 2 * nctr + 1);
    unsigned long long cnt = 0;
    int64_t nchunks = 0;
    NLOut<T> out;
    for (int attempt = 0;; ++attempt) {
        nchunks = (cap + scap + chunk - 1) / chunk + 1;
        HIPCHK(c, ensure(c->sp_i, sizeof(int32_t) * scap));
        HIPCHK(c, ensure(c->sp_j, sizeof(int32_t) * scap));
        HIPCHK(c, ensure(c->sp_d, sizeof(T) * scap));
        for (DBuf *b : {&c->ch_used, &c->ch_hstart, &c->ch_mstart})
            HIPCHK(c, ensure(*b, sizeof(int) * (nchunks + 1)));
        HIPCHK(c, ensure(c->counters, sizeof(int) * TASK_INTS));
        if ((s = fill_zero(c, {{c->nl_count.p, 2 * (int64_t)(2 * nctr + 2)}, {c->ch_used.p, nchunks + 1}, {c->counters.p, TASK_INTS}})))
            return s;
        c->counters_zeroed = true;  // the sweep below skips its own fill
        out.oi = di; out.oj = dj; out.od = dd;
        out.si = (int32_t *)c->sp_i.p; out.sj = (int32_t *)c->sp_j.p; out.sd = (T *)c->sp_d.p;
        out.cap = cap;
        out.scap = scap;
        out.overflow = ovf;
        OpNeighborList<T> op;
        std::memset((void *)&op, 0, sizeof(op));
        op.out = out;
        op.chunk_counter = ctr;
        op.total = ctr + nctr;
        op.chunk_used = (int *)c->ch_used.p;
        op.max_chunks = nchunks;
        op.chunk = chunk;
        op.ordered = mode_once(c) == MODE_A_TRIC;
        s = run_mode_a<T>(c, "k_sweep_neighborlist", op, grid);
        c->counters_zeroed = false;
        if (s) return s;
        // compaction (a no-op on the device when the pairs exceed the capacity), then one
        // host synchronisation for the count and the overflow word
        ScanState st;
        if ((s = scan_state(c, SCAN_CHUNKS, nchunks, st))) return s;
        ProdHoles ph{(const int *)c->ch_used.p, (long long)cap, chunk};
        LAUNCH(c, "k_scan_holes", hipLaunchKernelGGL((k_scan_pair<ProdHoles>), dim3((unsigned)scan_tiles_for<ProdHoles>(nchunks)),
                                                     dim3(SCAN_THREADS), 0, c->stream, (long long)nchunks, ph,
                                                     ScanValue{ctr + nctr, NL_COUNTERS, NL_COUNTER_STRIDE, tot},
                                                     (int *)c->ch_hstart.p, (int *)c->ch_mstart.p, (int *)nullptr,
                                                     (int *)nullptr, st, ovf, 2u));
        LAUNCH(c, "k_nl_fill", hipLaunchKernelGGL((k_nl_fill<T>), dim3(std::max(1, std::min(2048, c->num_cus * 8))), dim3(256),
                                                  0, c->stream, (long long)nchunks, chunk, (const int *)c->ch_used.p,
                                                  (const int *)c->ch_hstart.p, (const int *)c->ch_mstart.p, tot, out));
        if ((s = sync(c, tot, 3))) return s;  // pair count, then the overflow word
        std::memcpy(&cnt, result_words(c), sizeof(cnt));
        const unsigned int h_ovf = result_words(c)[2];
        if (h_ovf & 2u) return fail(c, CLM_ERR_HIP, "a single-pass scan did not complete (internal error)");
        if (!h_ovf || (int64_t)cnt > cap) break;
        if (attempt >= 3) return fail(c, CLM_ERR_HIP, "neighbor list spill area overflow");
        scap *= 2;
    }
    *npairs = (int64_t)cnt;
    if (!on_device && cnt > 0 && (int64_t)cnt <= cap) {
        const int64_t m = (int64_t)cnt;
        HIPCHK(c, hipMemcpyAsync(oi, di, sizeof(int32_t) * m, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipMemcpyAsync(oj, dj, sizeof(int32_t) * m, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipMemcpyAsync(od, dd, sizeof(T) * m, hipMemcpyDeviceToHost, c->stream));
        if ((s = sync(c))) return s;
    }
    if ((int64_t)cnt > cap) return fail(c, CLM_ERR_CAPACITY, "neighbor list capacity too small");
    return CLM_OK;
}

template <typename T>
SoftParams<T> soft_params(const clm_softcore *p) {
    SoftParams<T> sp;
    std::memset(&sp, 0, sizeof(sp));
    const int nt = p->ntypes > 0 ? p->ntypes : 1;
    sp.ntypes = p->ntypes > 0 ? p->ntypes : 0;
    const bool lj = p->form == CLM_POT_LJ;
    sp.a = lj ? T(0) : T(1);
    sp.c = lj ? T(2) : T(1);
    sp.c3 = lj ? T(6) : T(3);
    for (int a = 0; a < nt; ++a) {
        sp.eps_t[a] = T(p->eps[a]);
        for (int b = 0; b < nt; ++b) {
            const int t = sp.ntypes ? a * 8 + b : 0;
            const double e = std::sqrt(p->eps[a] * p->eps[b]);
            const double sg = (p->sigma[a] + p->sigma[b]) / 2.0;
            sp.eps[t] = T(e);
            sp.isig[t] = T(1.0 / sg);
            sp.sig2[t] = T(sg * sg);
        }
    }
    return sp;
}

clm_status check_softcore(clm_ctx *c, const clm_softcore *p) {
    if (!p) return fail(c, CLM_ERR_ARG, "NULL soft-core parameters");
    if (p->ntypes < 0 || p->ntypes > 8) return fail(c, CLM_ERR_ARG, "ntypes must be in 0..8");
    if (p->form != CLM_POT_SOFTCORE && p->form != CLM_POT_LJ) return fail(c, CLM_ERR_ARG, "unknown potential form");
    if (p->ntypes > 0 && !c->has_types) return fail(c, CLM_ERR_STATE, "typed parameters need clm_set_types");
    if (p->ntypes > 0 && c->two_set && !(c->ysub && c->ysub->has_types))
        return fail(c, CLM_ERR_STATE, "typed parameters need clm_set_types_y for the second set");
    return CLM_OK;
}

// The energy alone of one set takes every pair once (the sweep of the neighbour list,
// modes A, at weight 1); forces and gradients take every pair from both sides (mode B),
// so that each lane writes its own particle's result without atomics.
// c->acc: the energies (per system; of one system ACC_SLOTS copies), then the copies of the
// per-type gradients.
int64_t acc_energies(const clm_ctx *c) { return c->nsys > 1 ? c->nsys : ACC_SLOTS * ACC_STRIDE; }
int64_t acc_size(const clm_ctx *c) { return acc_energies(c) + ACC_SLOTS * ACC_STRIDE; }
double acc_energy(const clm_ctx *c, const double *acc, int k) {
    if (c->nsys > 1) return acc[k];
    double e = 0;
    for (int s = 0; s < ACC_SLOTS; ++s) e += acc[s * ACC_STRIDE];
    return e;
}
double acc_gradient(const clm_ctx *c, const double *acc, int k) {
    double g = 0;
    for (int s = 0; s < ACC_SLOTS; ++s) g += acc[acc_energies(c) + s * ACC_STRIDE + k];
    return g;
}

// Reads the first n doubles of c->acc, synchronising.
clm_status sync_acc(clm_ctx *c, int64_t n, std::vector<double> &acc) {
    acc.resize(n);
    if (2 * n <= READ_WORDS - READ_RESULTS && c->h_mapped) {
        clm_status s = sync(c, c->acc.p, (int)(2 * n));
        if (!s) std::memcpy(acc.data(), result_words(c), sizeof(double) * n);
        return s;
    }
    HIPCHK(c, hipMemcpyAsync(acc.data(), c->acc.p, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
    return sync(c);
}

template <bool FORCES, bool ADJ>
int softcore_mode(const clm_ctx *c) {
    return (!FORCES && !ADJ && !c->two_set) ? mode_once(c) : MODE_B;
}

template <typename T, bool FORCES, bool ADJ, bool TYPED>
clm_status enqueue_potential(clm_ctx *c, const clm_softcore *p, T *df) {
    clm_status s;
    const int64_t nacc = acc_size(c);
    HIPCHK(c, ensure(c->acc, sizeof(double) * nacc));
    HIPCHK(c, ensure(c->counters, sizeof(int) * TASK_INTS));
    if ((s = fill_zero(c, {{c->acc.p, 2 * nacc}, {c->counters.p, TASK_INTS}}))) return s;
    c->counters_zeroed = true;  // the first sweep below skips its own fill
    OpSoftCore<T, FORCES, ADJ, TYPED> op;
    std::memset((void *)&op, 0, sizeof(op));
    op.prm = soft_params<T>(p);
    op.forces = df;
    op.energy = (double *)c->acc.p;
    op.grad = (double *)c->acc.p + acc_energies(c);
    op.nsys = c->nsys;
    op.dim = c->dim;
    const char *name = ADJ ? "k_sweep_energy_adjoint" : (FORCES ? "k_sweep_energy_forces" : "k_sweep_energy");
    if constexpr (!ADJ) {
        if (c->two_set) {
            // x homes against the y list: every x-y pair once (energy, forces on x); then,
            // for forces, y homes against the x list (forces on y, written after the x rows)
            op.escale = 1.0;
            if ((s = run_sweep_on<T, MODE_X_REAL>(c, c->ysub, name, op, 0))) return s;
            if (!FORCES) return CLM_OK;
            op.escale = 0.0;
            op.forces = df + (size_t)c->n * c->dim;
            if ((s = run_sweep_on<T, MODE_X_REAL>(c->ysub, c, name, op, 0))) return fail(c, s, c->ysub->err);
            return CLM_OK;
        }
    }
    if constexpr (!FORCES && !ADJ) {
        op.escale = 1.0;  // every pair once
        if (c->celltype == CLM_TRICLINIC) return run_sweep<T, MODE_A_TRIC>(c, name, op, 0);
        return run_sweep<T, MODE_A_ORTHO>(c, name, op, 0);
    } else {
        op.escale = 0.5;  // MODE_B sees every pair from both sides
        return run_sweep<T, MODE_B>(c, name, op, 0);
    }
}

// Launch the soft-core sweep writing forces/gradients to df and the per-system energies
// + per-type gradients to c->acc (no host synchronisation).
template <typename T, bool FORCES, bool ADJ>
clm_status enqueue_softcore(clm_ctx *c, const clm_softcore *p, T *df) {
    return p->ntypes ? enqueue_potential<T, FORCES, ADJ, true>(c, p, df) : enqueue_potential<T, FORCES, ADJ, false>(c, p, df);
}

template <typename T, bool FORCES, bool ADJ>
clm_status softcore_t(clm_ctx *c, const clm_softcore *p, double *energies, int per_system, void *fout, double *deps,
                      double *dsig, int on_device) {
    clm_status s;
    if ((s = check_softcore(c, p))) return s;
    if (c->two_set) {
        if (ADJ) return fail(c, CLM_ERR_ARG, "the energy adjoint is for one set of particles");
        if ((s = ensure_cross(c))) return s;
        if ((s = prepare_mode(c, MODE_X_REAL, c->ysub))) return s;
        if (FORCES && (s = prepare_mode(c->ysub, MODE_X_REAL, c))) return fail(c, s, c->ysub->err);
    } else {
        if ((s = ensure_cell_list(c))) return s;
        if ((s = prepare_mode(c, softcore_mode<FORCES, ADJ>(c), c))) return s;
    }
    const int D = c->dim;
    const int64_t nrows_out = c->n + (c->two_set ? c->ysub->n : 0);  // y rows follow the x rows
    T *df = (T *)fout;
    if ((FORCES || ADJ) && (!on_device || !fout)) {
        HIPCHK(c, ensure(c->outbuf, sizeof(T) * std::max<int64_t>(nrows_out * D, 1)));
        df = (T *)c->outbuf.p;
    }
    if ((s = enqueue_softcore<T, FORCES, ADJ>(c, p, df))) return s;
    if ((FORCES || ADJ) && fout && !on_device && nrows_out > 0)
        HIPCHK(c, hipMemcpyAsync(fout, df, sizeof(T) * nrows_out * D, hipMemcpyDeviceToHost, c->stream));
    std::vector<double> acc;
    if ((s = sync_acc(c, ADJ ? acc_size(c) : acc_energies(c), acc))) return s;
    if (energies) {
        if (per_system) {
            for (int k = 0; k < c->nsys; ++k) energies[k] = acc_energy(c, acc.data(), k);
        } else {
            double e = 0;
            for (int k = 0; k < c->nsys; ++k) e += acc_energy(c, acc.data(), k);
            *energies = e;
        }
    }
    const int nt = p->ntypes > 0 ? p->ntypes : 1;
    if (ADJ) {
        for (int k = 0; k < nt; ++k) {
            if (deps) deps[k] = acc_gradient(c, acc.data(), k);
            if (dsig) dsig[k] = acc_gradient(c, acc.data(), 8 + k);
        }
    }
    return CLM_OK;
}

// Device addresses of every context buffer a captured graph references (one- and
// two-pass binning, the soft-core sweep, and the mode-B row tasks, which only the union-row sweep
// reads but which every capture sizes, so that trying that sweep leaves a graph valid), in a fixed order.
std::vector<void *> graph_buffers(clm_ctx *c) {
    std::vector<void *> v;
    for (DBuf *b : {&c->sys_desc, &c->sys_of, &c->rowoff, &c->pos, &c->types, &c->xw, &c->home_cell, &c->cnt, &c->creal,
                    &c->cstart, &c->cur_real, &c->cur_ghost, &c->E, &c->E_raw, &c->rstart, &c->real_pos, &c->order,
                    &c->flags, &c->cnt64, &c->E_real, &c->E_ghost, &c->counters, &c->scan_tmp, &c->outbuf, &c->acc,
                    &c->tstart[MODE_B], &c->systasks, &c->scan_st[SCAN_ROWS], &c->scan_st[SCAN_CELLS]})
        v.push_back(b->p);
    return v;
}

void drop_graph(clm_ctx *c) {
    if (c->graph_exec) { hipGraphExecDestroy(c->graph_exec); c->graph_exec = nullptr; }
    if (c->graph) { hipGraphDestroy(c->graph); c->graph = nullptr; }
    c->graph_ptrs.clear();
    c->graph_n = -1;
    c->graph_box_epoch = -1;
}

// Records update + energy/forces (device forces array) into a HIP graph.  The cell list
// must have been built once eagerly (it sizes the buckets and the entry buffer, with
// headroom).  The graph bins in one pass (k_bin_bucket + k_scan_cells + k_cell_sort) when
// the context has a bucket size, else in two (count, scans, scatter).  A replay whose cells
// outgrow their buckets or whose entries exceed the captured capacity reports
// CLM_ERR_CAPACITY (its sweep skips the list on the device) and must be re-captured; so must
// a replay after any buffer the graph references was reallocated or the box or the
// particle count changed (CLM_ERR_STATE).  The caller's forces array must outlive the graph.
template <typename T>
clm_status graph_capture_t(clm_ctx *c, const clm_softcore *p, void *forces) {
    clm_status s;
    if ((s = check_softcore(c, p))) return s;
    if (c->celltype == CLM_NONPERIODIC) return fail(c, CLM_ERR_ARG, "graph capture needs a periodic box");
    if (c->two_set) return fail(c, CLM_ERR_ARG, "graph capture is for one set of particles");
    drop_graph(c);
    if ((s = ensure_cell_list(c))) return s;
    if (c->bin_pending && (s = sync(c))) return s;  // CLM_REDO: captured again on a rebuilt list
    const bool bucketed = c->bucket > 0 && c->sweep_variant == 1;
    // headroom for fluctuating ghost counts between replays; the bucket storage and the
    // compact list sized so that eager builds between replays reuse them
    const int64_t want = c->n_entries + c->n_entries / 8 + 1024;
    if (c->e_cap < want) {
        HIPCHK(c, ensure_entries(c, c->E, sizeof(Ent<T>) * (want + SWEEP_PAD)));
        c->e_cap = (int64_t)(c->E.bytes / sizeof(Ent<T>)) - SWEEP_PAD;
    }
    const size_t raw = std::max(c->E.bytes, bucketed ? sizeof(Ent<T>) * (size_t)c->ncells * (size_t)c->bucket : 0);
    HIPCHK(c, ensure(c->E_raw, raw));
    c->e_cap = std::min<int64_t>(c->e_cap, (int64_t)(c->E_raw.bytes / sizeof(Ent<T>)) - SWEEP_PAD);
    if ((s = ensure_split<T>(c))) return s;
    const int64_t nD = std::max<int64_t>(c->n * c->dim, 1);
    HIPCHK(c, ensure(c->outbuf, sizeof(T) * nD));
    HIPCHK(c, ensure(c->cnt64, (sizeof(unsigned long long) * std::max(c->ncells, 1)) << counter_shift(c)));
    HIPCHK(c, ensure(c->tstart[MODE_B], sizeof(int) * (c->nrows + 1)));
    HIPCHK(c, ensure(c->counters, sizeof(int) * TASK_INTS));
    HIPCHK(c, ensure(c->acc, sizeof(double) * acc_size(c)));
    {  // scan states (zeroed here, outside the capture)
        ScanState st;
        if ((s = scan_state(c, SCAN_ROWS, c->nrows, st))) return s;
        if ((s = scan_state(c, SCAN_CELLS, c->ncells, st))) return s;
    }
    {  // size the scan scratch for the largest scan before capturing
        size_t need = 0;
        hipcub::DeviceScan::ExclusiveSum(nullptr, need, (const int *)nullptr, (int *)nullptr, c->ncells + 1, c->stream);
        HIPCHK(c, ensure(c->scan_tmp, need));
    }
    c->sweep_lanes = choose_lanes(c, c);
    if ((s = prepare_systasks<T>(c, MODE_B))) return s;
    HIPCHK(c, hipStreamSynchronize(c->stream));  // the zeroed scan states before the first replay
    // what is recorded has not run: the list stays what it is
    const bool prof = c->prof, order_valid = c->order_valid, split_valid = c->split_valid;
    c->prof = false;  // no events inside the capture
    HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    clm_status cs = CLM_OK;
    // the build with its status left on the device: the sweep checks it before walking the list
    // (the homes of a build with a NaN are fewer than the particles that the sweep counts on), the
    // replay's read-back reports it
    if (bucketed) {
        cs = enqueue_bucket_pass<T>(c);
        if (!cs) cs = enqueue_sort<T>(c, c->bucket, c->e_cap);
    } else {
        cs = enqueue_count<T>(c);
        if (!cs) cs = enqueue_scatter<T>(c);
    }
    c->bin_pending = true;  // the sweep takes the status block (SweepArgs::bin_flags)
    if (!cs && c->sweep_variant == 0) cs = enqueue_rows<T>(c, MODE_B);
    T *df = forces ? (T *)forces : (T *)c->outbuf.p;
    if (!cs) cs = enqueue_softcore<T, true, false>(c, p, df);
    c->bin_pending = false;
    hipError_t e = hipStreamEndCapture(c->stream, &c->graph);
    c->prof = prof;
    c->order_valid = order_valid;
    c->split_valid = split_valid;
    if (cs) { drop_graph(c); return cs; }
    if (e != hipSuccess) { drop_graph(c); return hip_fail(c, e, "hipStreamEndCapture"); }
    HIPCHK(c, hipGraphInstantiate(&c->graph_exec, c->graph, nullptr, nullptr, 0));
    c->graph_ptrs = graph_buffers(c);
    c->graph_n = c->n;
    c->graph_box_epoch = c->box_epoch;
    c->graph_bucketed = bucketed;
    c->graph_ordered = bucketed && order_valid;
    return CLM_OK;
}

clm_status graph_launch(clm_ctx *c, double *energies) {
    if (!c->graph_exec) return fail(c, CLM_ERR_STATE, "no captured graph");
    if (c->layout_dirty || c->n != c->graph_n || c->box_epoch != c->graph_box_epoch || graph_buffers(c) != c->graph_ptrs) {
        drop_graph(c);
        return fail(c, CLM_ERR_STATE,
                    "the captured graph is stale (the box, the particle count or a buffer it uses changed); capture again");
    }
    // a build that failed since (a NaN, an overflow) left some particles out of the order and others twice
    if (c->graph_ordered && !c->order_valid && c->n > 0)
        LAUNCH(c, "k_iota", hipLaunchKernelGGL(k_iota, dim3(blocks(c->n, 256)), dim3(256), 0, c->stream, (int *)c->order.p, (int)c->n));
    HIPCHK(c, hipGraphLaunch(c->graph_exec, c->stream));
    std::vector<double> acc;
    if (c->graph_bucketed) {
        // the replay's build status, as for a deferred eager build: an overflow marks the
        // list for a rebuild (and re-sizes the buckets) and asks for a new capture
        c->bin_pending = true;
        clm_status s = energies ? sync_acc(c, acc_energies(c), acc) : sync(c);
        if (s == CLM_REDO) return fail(c, CLM_ERR_CAPACITY, "cells or entries exceed the captured capacity; capture again");
        if (s) return s;
    } else {
        int total = 0;
        HIPCHK(c, hipMemcpyAsync(c->h_flags, c->flags.p, sizeof(uint32_t), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipMemcpyAsync(&total, (int *)c->cstart.p + c->ncells, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        clm_status s = energies ? sync_acc(c, acc_energies(c), acc) : sync(c);
        if (s) return s;
        s = check_flags(c, *c->h_flags);
        if (s || total > c->e_cap || (*c->h_flags & FLAG_OVERFLOW)) {
            c->cl_valid = false;
            c->order_valid = false;
            if (s) return s;
            c->dirty = true;
            return fail(c, CLM_ERR_CAPACITY, "entries exceed the captured capacity; capture again");
        }
        c->n_entries = total;
    }
    c->cl_valid = true;
    c->dirty = c->parts_variant != c->sweep_variant;
    c->order_valid = true;
    c->split_valid = wants_split(c);
    forget_modes(c);
    if (energies)
        for (int k = 0; k < c->nsys; ++k) energies[k] = acc_energy(c, acc.data(), k);
    return CLM_OK;
}

template <typename T>
clm_status histogram_t(clm_ctx *c, int nbins, double width, int64_t *counts, double *vsum) {
    clm_status s;
    if (nbins < 1 || nbins > OpHistogram<T>::MAXB) return fail(c, CLM_ERR_ARG, "nbins must be in 1..512");
    if (!(width > 0)) return fail(c, CLM_ERR_ARG, "bin width must be positive");
    auto has_vel = [](const clm_ctx *k) { return k && k->n_vel >= k->n; };
    if (vsum && !has_vel(c)) return fail(c, CLM_ERR_STATE, "velocities not set");
    if (c->two_set && vsum && !has_vel(c->ysub)) return fail(c, CLM_ERR_STATE, "y velocities not set");
    if (c->nsys != 1) return fail(c, CLM_ERR_ARG, "histograms are per system (nsys must be 1)");
    if ((s = prepare_once(c))) return s;
    const int64_t nhist = (int64_t)HIST_COPIES * nbins;
    HIPCHK(c, ensure(c->hist, sizeof(unsigned long long) * 2 * nhist));  // counts, then velocity sums
    HIPCHK(c, ensure(c->counters, sizeof(int) * TASK_INTS));
    if ((s = fill_zero(c, {{c->hist.p, (vsum ? 4 : 2) * nhist}, {c->counters.p, TASK_INTS}}))) return s;
    OpHistogram<T> op;
    op.nbins = nbins;
    op.width = T(width);
    op.inv_width = T(1) / T(width);
    op.vel = vsum ? (const T *)c->vel.p : nullptr;
    const HostBox<T> &hb = hbox<T>(c);
    for (int k = 0; k < 9; ++k) op.rot[k] = hb.rot.a[k];
    op.tric = c->celltype == CLM_TRICLINIC;
    op.vq0 = op.vq1 = nullptr;
    if (vsum) {
        // the neighbour velocities in the order of the entry arrays the sweep walks: the
        // real and the ghost entries of the triclinic split, else the neighbour set's entries
        const int mode = mode_once(c);
        clm_ctx *nb = (mode == MODE_X_ORTHO || mode == MODE_X_REAL) ? c->ysub : c;
        const T *vn = (const T *)nb->vel.p;
        const long long nvel = nb->n;
        OpRot<T> rot;
        for (int k = 0; k < 9; ++k) rot.m[k] = op.rot[k];
        rot.tric = op.tric;
        const uint32_t *bf = nb->bin_pending ? (const uint32_t *)nb->flags.p : nullptr;
        auto gather = [&](DBuf &dst, const DBuf &src, const int *ta, const int *tb, const char *name) -> clm_status {
            const long long cap = (long long)(src.bytes / sizeof(Ent<T>));
            HIPCHK(c, ensure(dst, sizeof(vec4<T>) * (size_t)std::max<long long>(cap, 1)));
            const unsigned grid = (unsigned)std::min<long long>(std::max<long long>((cap + 255) / 256, 1), 8192);
            LAUNCH(c, name, hipLaunchKernelGGL((k_entry_velocities<T>), dim3(grid), dim3(256), 0, c->stream, (const Ent<T> *)src.p, ta, tb,
                                               cap, vn, nvel, c->dim, rot, (vec4<T> *)dst.p, bf, nb->e_cap));
            return CLM_OK;
        };
        const int nc = c->ncells;
        if (mode == MODE_A_TRIC && c->sweep_variant >= 1) {
            if ((s = gather(c->vq0, c->E_real, (const int *)c->rstart.p + nc, nullptr, "k_entry_velocities"))) return s;
            if ((s = gather(c->vq1, c->E_ghost, (const int *)c->cstart.p + nc, (const int *)c->rstart.p + nc,
                            "k_entry_velocities")))
                return s;
            op.vq0 = (const vec4<T> *)c->vq0.p;
            op.vq1 = (const vec4<T> *)c->vq1.p;
        } else {
            if ((s = gather(c->vq0, nb->E, (const int *)nb->cstart.p + nb->ncells, nullptr, "k_entry_velocities"))) return s;
            op.vq0 = op.vq1 = (const vec4<T> *)c->vq0.p;
        }
    }
    op.dim = c->dim;
    op.counts = (unsigned long long *)c->hist.p;
    op.vsum = (double *)c->hist.p + nhist;
    c->counters_zeroed = true;
    s = run_mode_a<T>(c, "k_sweep_histogram", op, 0);
    c->counters_zeroed = false;
    if (s) return s;
    LAUNCH(c, "k_hist_sum", hipLaunchKernelGGL(k_hist_sum, dim3(blocks(nbins, 256)), dim3(256), 0, c->stream, nbins, op.counts,
                                               vsum ? op.vsum : nullptr));
    if (vsum) HIPCHK(c, hipMemcpyAsync(vsum, op.vsum, sizeof(double) * nbins, hipMemcpyDeviceToHost, c->stream));
    static_assert(2 * OpHistogram<T>::MAXB <= READ_WORDS - READ_RESULTS, "the read-back holds the longest histogram");
    if ((s = sync(c, op.counts, 2 * nbins))) return s;
    std::memcpy(counts, result_words(c), sizeof(int64_t) * nbins);
    return CLM_OK;
}

template <typename T>
clm_status mindist_t(clm_ctx *c, int64_t *oi, int64_t *oj, double *od) {
    clm_status s;
    if (c->nsys != 1) return fail(c, CLM_ERR_ARG, "minimum distance is per system (nsys must be 1)");
    if ((s = prepare_once(c))) return s;
    const int grid = once_waves<T, OpMinDist<T>>(c);
    HIPCHK(c, ensure(c->md_best, sizeof(MinDistBest<T>) * grid));
    OpMinDist<T> op;
    op.best = (MinDistBest<T> *)c->md_best.p;
    op.cross = c->two_set ? 1 : 0;
    if ((s = run_mode_a<T>(c, "k_sweep_mindist", op, grid))) return s;
    LAUNCH(c, "k_mindist_best", hipLaunchKernelGGL((k_mindist_best<T>), dim3(1), dim3(256), 0, c->stream, op.best, grid));
    if ((s = sync(c, op.best, (int)(sizeof(MinDistBest<T>) / sizeof(uint32_t))))) return s;
    MinDistBest<T> w;
    std::memcpy(&w, result_words(c), sizeof(w));
    const T best = w.d2;
    const int ba = w.a, bb = w.b;
    if (std::isinf(best)) {
        *oi = -1; *oj = -1; *od = INFINITY;
    } else {
        *oi = ba; *oj = bb; *od = (double)std::sqrt(best);
    }
    return CLM_OK;
}

}  // namespace

// ------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------

// Runs an entry point, and once more if it found its cell list invalid (CLM_REDO): the
// second run rebuilds the list with its status read first, so it cannot ask again.  A call that
// fails before it has read the status of a build it enqueued (x's, where y's build fails) leaves no
// build to be judged by the next synchronisation: nothing is known of that list, which is built again.
template <typename F>
clm_status with_redo(clm_ctx *c, F f) {
    clm_status s = f();
    if (s == CLM_REDO) s = f();
    if (s == CLM_REDO) s = fail(c, CLM_ERR_HIP, "cell list rebuild did not settle");
    for (clm_ctx *k : {c, c->ysub})
        if (s && k && k->bin_pending) k->bin_pending = k->cl_valid = k->order_valid = false;
    return s;
}

// ---------------------------------------------------------------------------
// Allocation-free soft-core energy / forces (clm_energy_forces_noalloc)
// ---------------------------------------------------------------------------

// Scratch of the allocation-free entry point: cell list, counters, scans and task
// tables of one call.  Every GPU the library runs on holds its own copy until the
// process ends.  Host code never uses this name as an address (it is a host-side
// stand-in): the device address comes from hipGetSymbolAddress, per device.
constexpr size_t CLM_SCRATCH_BYTES = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[CLM_SCRATCH_BYTES];

namespace {

constexpr int CLM_MAX_DEVICES = 64;
struct ScratchSlot {
    std::once_flag once;
    void *ptr = nullptr;
    hipError_t err = hipSuccess;
};
ScratchSlot g_scratch[CLM_MAX_DEVICES];
thread_local std::string g_noalloc_err;

// The scratch array's address on device dev (current): looked up once per device.
hipError_t scratch_ptr(int dev, void **out) {
    ScratchSlot &sl = g_scratch[dev];
    std::call_once(sl.once, [&] { sl.err = hipGetSymbolAddress(&sl.ptr, HIP_SYMBOL(scratch)); });
    *out = sl.ptr;
    return sl.err;
}

clm_status noalloc_fail(clm_status s, const std::string &msg) {
    g_noalloc_err = msg;
    return s;
}

template <typename T>
clm_status energy_forces_noalloc_t(int dim, const void *x, int64_t n, const double *cell, int celltype, double cutoff,
                                   int lcell, const clm_softcore *p, double *energy, void *forces, hipStream_t stream,
                                   int dev, void *base) {
    // a context on the stack: the caller's stream and positions, pageable status words,
    // every other buffer from the scratch arena
    clm_ctx c;
    uint32_t flags_host[64] = {0};  // (no results are read into it: see sync_acc)
    c.device = dev;
    c.dtype = std::is_same<T, float>::value ? CLM_F32 : CLM_F64;
    c.dim = dim;
    c.stream = stream;
    c.own_stream = false;
    c.h_flags = flags_host;
    int ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && ncu > 0) c.num_cus = ncu;
    clm_status s = clm_set_box(&c, cell, celltype, cutoff, lcell);
    if (s) return noalloc_fail(s, c.err);
    c.pos.p = const_cast<void *>(x);
    c.pos.bytes = sizeof(T) * (size_t)dim * (size_t)n;
    c.n = n;
    c.has_pos = true;
    c.dirty = true;
    g_arena = ScratchArena{(char *)base, CLM_SCRATCH_BYTES, 0, true, false};
    s = with_redo(&c, [&] {
        return forces ? softcore_t<T, true, false>(&c, p, energy, 0, forces, nullptr, nullptr, 1)
                      : softcore_t<T, false, false>(&c, p, energy, 0, nullptr, nullptr, nullptr, 1);
    });
    const bool exhausted = g_arena.exhausted;
    g_arena = ScratchArena{};
    c.pos = DBuf{};  // the caller's positions and the arena blocks are not the context's to free
    if (exhausted) {
        hipStreamSynchronize(stream);  // nothing of the call left running on the scratch
        return noalloc_fail(CLM_ERR_CAPACITY, "the system needs more than the " +
                                                  std::to_string(CLM_SCRATCH_BYTES >> 20) +
                                                  " MiB scratch of the allocation-free entry point");
    }
    if (s) return noalloc_fail(s, c.err);
    g_noalloc_err.clear();
    return CLM_OK;
}

}  // namespace

extern "C" {

const char *clm_version(void) { return "celllistmap-hip 0.1.0 (gfx950)"; }

clm_status clm_create(clm_ctx **out, int device, int dtype, int dim) {
    if (!out) return CLM_ERR_ARG;
    *out = nullptr;
    if (dtype != CLM_F32 && dtype != CLM_F64) return CLM_ERR_ARG;
    if (dim != 2 && dim != 3) return CLM_ERR_DIM;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= device || device < 0) return CLM_ERR_HIP;
    if (hipSetDevice(device) != hipSuccess) return CLM_ERR_HIP;
    clm_ctx *c = new clm_ctx();
    c->device = device;
    c->dtype = dtype;
    c->dim = dim;
    Pool *pool = device_pool(device);
    Pool::Stream kept{nullptr, nullptr};
    if (pool && pool->take_stream(kept)) {
        c->stream = kept.stream;
        c->h_flags = kept.host;
    } else if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return CLM_ERR_HIP;
    }
    c->own_stream = true;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess && prop.multiProcessorCount > 0) c->num_cus = prop.multiProcessorCount;
    if (!c->h_flags && hipHostMalloc((void **)&c->h_flags, sizeof(uint32_t) * READ_WORDS, hipHostMallocDefault) != hipSuccess) {
        hipStreamDestroy(c->stream);
        delete c;
        return CLM_ERR_HIP;
    }
    c->h_mapped = true;
    *out = c;
    return CLM_OK;
}

clm_status clm_destroy(clm_ctx *c) {
    if (!c) return CLM_OK;
    hipSetDevice(c->device);
    if (c->stream) hipStreamSynchronize(c->stream);
    // (as hipFree does: work on a stream that the context had earlier may still use its memory)
    Pool *pool = hipDeviceSynchronize() == hipSuccess ? device_pool(c->device) : nullptr;
    if (c->ysub) {
        c->ysub->stream = nullptr;  // the owner's stream
        c->ysub->own_stream = false;
        c->ysub->root = nullptr;
        clm_destroy(c->ysub);
        c->ysub = nullptr;
    }
    DBuf *bufs[] = {&c->pos, &c->types, &c->vel, &c->xw, &c->home_cell, &c->cnt, &c->creal, &c->cstart,
                    &c->cur_real, &c->cur_ghost, &c->E, &c->flags, &c->systasks, &c->systasks_all, &c->hstart[0],
                    &c->hstart[1], &c->hstart[2], &c->tstart[0], &c->tstart[1], &c->tstart[2], &c->counters,
                    &c->scan_tmp, &c->nl_i, &c->nl_j, &c->nl_d, &c->nl_count, &c->outbuf, &c->acc,
                    &c->hist, &c->md_best, &c->sp_i, &c->sp_j, &c->sp_d,
                    &c->ch_used, &c->ch_hstart, &c->ch_mstart, &c->sys_desc,
                    &c->sys_of, &c->rowoff, &c->E_raw, &c->rstart, &c->real_pos, &c->cnt64, &c->maxcnt, &c->order,
                    &c->E_real, &c->E_ghost, &c->scan_st[0], &c->scan_st[1], &c->scan_st[2], &c->vq0, &c->vq1,
                    &c->limits};
    for (DBuf *b : bufs)
        if (b->p && !(pool && pool->leave(b->p, b->bytes))) hipFree(b->p);
    for (auto &p : c->pending) { hipEventDestroy(p.a); hipEventDestroy(p.b); }
    for (hipEvent_t e : c->ev_pool) hipEventDestroy(e);
    if (c->graph_exec) hipGraphExecDestroy(c->graph_exec);
    if (c->graph) hipGraphDestroy(c->graph);
    for (hipEvent_t e : c->join_ev)
        if (e) hipEventDestroy(e);
    const bool own = c->own_stream && c->stream;
    if (!(own && c->h_flags && pool && pool->leave_stream({c->stream, c->h_flags}))) {
        if (c->h_flags) hipHostFree(c->h_flags);
        if (own) hipStreamDestroy(c->stream);
    }
    delete c;
    return CLM_OK;
}

const char *clm_last_error(const clm_ctx *c) { return c ? c->err.c_str() : g_noalloc_err.c_str(); }

clm_status clm_join_stream(clm_ctx *c, void *other, int both) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    hipStream_t o = (hipStream_t)other;
    if (o == c->stream) return CLM_OK;
    for (hipEvent_t &e : c->join_ev)
        if (!e) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (both < 0 || both > 2) return fail(c, CLM_ERR_ARG, "join_stream: both must be 0, 1 or 2");
    if (both >= 1) {
        HIPCHK(c, hipEventRecord(c->join_ev[0], o));
        HIPCHK(c, hipStreamWaitEvent(c->stream, c->join_ev[0], 0));
    }
    if (both <= 1) {
        HIPCHK(c, hipEventRecord(c->join_ev[1], c->stream));
        HIPCHK(c, hipStreamWaitEvent(o, c->join_ev[1], 0));
    }
    return CLM_OK;
}

clm_status clm_get_stream(clm_ctx *c, void **stream) {
    if (!c || !stream) return CLM_ERR_ARG;
    *stream = (void *)c->stream;
    return CLM_OK;
}

clm_status clm_set_stream(clm_ctx *c, void *stream) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    if (stream) {
        if (c->own_stream && c->stream) {
            hipStreamSynchronize(c->stream);
            hipStreamDestroy(c->stream);
        }
        c->stream = (hipStream_t)stream;
        c->own_stream = false;
    } else if (!c->own_stream) {
        if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) return CLM_ERR_HIP;
        c->own_stream = true;
    }
    if (c->ysub) c->ysub->stream = c->stream;
    return CLM_OK;
}

clm_status clm_box_compute(int dtype, int dim, const double *cell, int celltype, double cutoff, int lcell,
                           const double *origin, clm_box_info *out) {
    if (!cell || !out) return CLM_ERR_ARG;
    if (celltype < 0 || celltype > 2) return CLM_ERR_ARG;
    int rc;
    if (dtype == CLM_F32) {
        HostBox<float> hb;
        rc = build_host_box<float>(dim, cell, celltype, cutoff, lcell, origin, hb);
        if (rc == BOX_OK) box_info(hb, out);
    } else if (dtype == CLM_F64) {
        HostBox<double> hb;
        rc = build_host_box<double>(dim, cell, celltype, cutoff, lcell, origin, hb);
        if (rc == BOX_OK) box_info(hb, out);
    } else {
        return CLM_ERR_ARG;
    }
    if (rc == BOX_BAD_LCELL) return CLM_ERR_ARG;
    if (rc == BOX_BAD_DIM) return CLM_ERR_DIM;
    if (rc == BOX_BAD_CELL) return CLM_ERR_CELL;
    return CLM_OK;
}

clm_status clm_set_box(clm_ctx *c, const double *cell, int celltype, double cutoff, int lcell) {
    if (!c) return CLM_ERR_ARG;
    if (celltype < 0 || celltype > 2) return fail(c, CLM_ERR_ARG, "unknown cell type");
    if (lcell < 1) return fail(c, CLM_ERR_ARG, "lcell must be greater or equal to 1");
    if (!(cutoff > 0) || !std::isfinite(cutoff)) return fail(c, CLM_ERR_ARG, "cutoff must be positive and finite");
    const int D = c->dim;
    if (celltype != CLM_NONPERIODIC) {
        if (!cell) return fail(c, CLM_ERR_ARG, "NULL unit cell");
        HostBox<float> bf;
        HostBox<double> bd;
        int rc = c->dtype == CLM_F32 ? build_host_box<float>(D, cell, celltype, cutoff, lcell, nullptr, bf)
                                     : build_host_box<double>(D, cell, celltype, cutoff, lcell, nullptr, bd);
        clm_status s = box_status(c, rc);
        if (s) return s;
        c->hbf.assign(1, bf);
        c->hbd.assign(1, bd);
    }
    c->nsys = 1;
    c->sys_n.clear();
    c->celltype = celltype;
    c->cutoff_in = cutoff;
    c->lcell = lcell;
    c->has_box = true;
    c->dirty = true;
    c->layout_dirty = true;
    ++c->box_epoch;
    return CLM_OK;
}

clm_status clm_set_systems(clm_ctx *c, int nsys, const int64_t *n, const double *cells, int celltype,
                           const double *cutoffs, const int *lcells) {
    if (!c) return CLM_ERR_ARG;
    if (nsys < 1 || !n || !cells || !cutoffs || !lcells) return fail(c, CLM_ERR_ARG, "bad system description");
    if (celltype != CLM_ORTHORHOMBIC && celltype != CLM_TRICLINIC)
        return fail(c, CLM_ERR_ARG, "systems of a batch must be periodic (orthorhombic or triclinic)");
    if (c->two_set) return fail(c, CLM_ERR_ARG, "a batch of systems holds one set of particles per system");
    const int D = c->dim;
    std::vector<HostBox<float>> vf(nsys);
    std::vector<HostBox<double>> vd(nsys);
    int64_t total = 0;
    for (int k = 0; k < nsys; ++k) {
        if (n[k] < 0) return fail(c, CLM_ERR_ARG, "negative particle count");
        if (lcells[k] < 1) return fail(c, CLM_ERR_ARG, "lcell must be greater or equal to 1");
        const double *cell = cells + (size_t)k * D * D;
        int rc = c->dtype == CLM_F32 ? build_host_box<float>(D, cell, celltype, cutoffs[k], lcells[k], nullptr, vf[k])
                                     : build_host_box<double>(D, cell, celltype, cutoffs[k], lcells[k], nullptr, vd[k]);
        clm_status s = box_status(c, rc);
        if (s) {
            c->err = "system " + std::to_string(k) + ": " + c->err;
            return s;
        }
        total += n[k];
    }
    if (total >= (int64_t)IDX_LIMIT) return fail(c, CLM_ERR_ARG, "too many particles (limit 2^28-1)");
    hipSetDevice(c->device);
    std::vector<int> sof(std::max<int64_t>(total, 1));
    for (int k = 0, o = 0; k < nsys; ++k)
        for (int64_t q = 0; q < n[k]; ++q) sof[o++] = k;
    HIPCHK(c, ensure(c->sys_of, sizeof(int) * sof.size()));
    HIPCHK(c, hipMemcpyAsync(c->sys_of.p, sof.data(), sizeof(int) * sof.size(), hipMemcpyHostToDevice, c->stream));
    clm_status s = sync(c);
    if (s) return s;
    c->hbf = vf;
    c->hbd = vd;
    c->nsys = nsys;
    c->sys_n.assign(n, n + nsys);
    c->celltype = celltype;
    c->cutoff_in = cutoffs[0];
    c->lcell = lcells[0];
    c->has_box = true;
    c->dirty = true;
    c->layout_dirty = true;
    ++c->box_epoch;
    return CLM_OK;
}

clm_status clm_get_box(clm_ctx *c, clm_box_info *out) {
    return clm_get_system_box(c, 0, out);
}

clm_status clm_get_system_box(clm_ctx *c, int k, clm_box_info *out) {
    if (!c || !out) return CLM_ERR_ARG;
    if (!c->has_box) return fail(c, CLM_ERR_STATE, "no box set");
    if (k < 0 || k >= c->nsys) return fail(c, CLM_ERR_ARG, "system index out of range");
    if (c->celltype == CLM_NONPERIODIC) {
        hipSetDevice(c->device);
        clm_status s = c->two_set ? ensure_cross(c) : ensure_cell_list(c);
        if (s) return s;
    }
    if (c->dtype == CLM_F32) box_info(c->hbf[k], out);
    else box_info(c->hbd[k], out);
    return CLM_OK;
}

clm_status clm_set_tuning(clm_ctx *c, int waves_per_cu) {
    if (!c || waves_per_cu < 0) return CLM_ERR_ARG;
    c->waves_per_cu = waves_per_cu;
    return CLM_OK;
}

clm_status clm_set_sweep_group(clm_ctx *c, int group) {
    if (!c) return CLM_ERR_ARG;
    if (group != 0 && group != 2 && group != 4 && group != 8)
        return fail(c, CLM_ERR_ARG, "sweep group must be 0 (the default), 2, 4 or 8");
    c->sweep_group = group;
    return CLM_OK;
}

clm_status clm_set_sweep_variant(clm_ctx *c, int variant) {
    if (!c) return CLM_ERR_ARG;
    if (variant != 0 && variant != 1) return fail(c, CLM_ERR_ARG, "sweep variant must be 0 or 1");
    if (variant != c->sweep_variant) c->dirty = true;  // the grid may be another one (choose_parts)
    c->sweep_variant = variant;
    if (c->ysub) c->ysub->sweep_variant = variant;
    return CLM_OK;
}

clm_status clm_set_positions(clm_ctx *c, const void *x, int64_t n, int on_device) {
    if (!c) return CLM_ERR_ARG;
    if (n < 0 || (n > 0 && !x)) return fail(c, CLM_ERR_ARG, "bad positions");
    if (c->nsys > 1) {
        int64_t tot = 0;
        for (int64_t v : c->sys_n) tot += v;
        if (n != tot) return fail(c, CLM_ERR_DIM, "positions must hold every particle of every system");
    }
    hipSetDevice(c->device);
    const size_t es = c->dtype == CLM_F32 ? 4 : 8;
    const size_t bytes = es * (size_t)c->dim * (size_t)n;
    HIPCHK(c, ensure(c->pos, std::max<size_t>(bytes, 16)));
    if (bytes)
        HIPCHK(c, hipMemcpyAsync(c->pos.p, x, bytes, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c->stream));
    if (!on_device) {
        clm_status s = sync(c);
        if (s) return s;
    }
    if (n != c->n) {
        c->has_types = false;
        c->layout_dirty = true;
    }
    c->n = n;
    c->has_pos = true;
    c->dirty = true;
    return CLM_OK;
}

clm_status clm_set_types(clm_ctx *c, const int32_t *t, int64_t n, int on_device) {
    if (!c) return CLM_ERR_ARG;
    if (!c->has_pos || n != c->n) return fail(c, CLM_ERR_DIM, "types must have one entry per particle");
    hipSetDevice(c->device);
    HIPCHK(c, ensure(c->types, sizeof(int32_t) * std::max<int64_t>(n, 1)));
    if (n) HIPCHK(c, hipMemcpyAsync(c->types.p, t, sizeof(int32_t) * n, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c->stream));
    if (!on_device) {
        clm_status s = sync(c);
        if (s) return s;
    }
    c->has_types = true;
    c->dirty = true;
    return CLM_OK;
}

clm_status clm_set_velocities(clm_ctx *c, const void *v, int64_t n, int on_device) {
    if (!c) return CLM_ERR_ARG;
    if (!c->has_pos || n != c->n) return fail(c, CLM_ERR_DIM, "velocities must have one entry per particle");
    hipSetDevice(c->device);
    const size_t es = c->dtype == CLM_F32 ? 4 : 8;
    const size_t bytes = es * c->dim * (size_t)n;
    HIPCHK(c, ensure(c->vel, std::max<size_t>(bytes, 16)));
    if (bytes) HIPCHK(c, hipMemcpyAsync(c->vel.p, v, bytes, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c->stream));
    if (!on_device) {
        clm_status s = sync(c);
        if (s) return s;
    }
    c->n_vel = n;
    return CLM_OK;
}

clm_status clm_update_cell_list(clm_ctx *c) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    c->dirty = true;
    if (c->two_set && c->ysub) c->ysub->dirty = true;
    return with_redo(c, [&] {
        clm_status s = c->two_set ? ensure_cross(c) : ensure_cell_list(c);
        if (s) return s;
        return sync(c);
    });
}

// Second set of particles (xpositions/ypositions of ParticleSystem, ParticleSystem.jl:149-214).
clm_status clm_set_positions_y(clm_ctx *c, const void *y, int64_t n, int on_device) {
    if (!c) return CLM_ERR_ARG;
    if (c->root) return fail(c, CLM_ERR_ARG, "not an owner context");
    if (c->nsys != 1) return fail(c, CLM_ERR_ARG, "a batch of systems holds one set of particles per system");
    hipSetDevice(c->device);
    if (!c->ysub) {
        clm_ctx *y2 = new clm_ctx();
        y2->device = c->device;
        y2->dtype = c->dtype;
        y2->dim = c->dim;
        y2->num_cus = c->num_cus;
        y2->stream = c->stream;
        y2->own_stream = false;
        y2->root = c;
        if (hipHostMalloc((void **)&y2->h_flags, sizeof(uint32_t) * READ_WORDS, hipHostMallocDefault) != hipSuccess) {
            delete y2;
            return fail(c, CLM_ERR_HIP, "hipHostMalloc");
        }
        y2->h_mapped = true;
        c->ysub = y2;
        c->sub_epoch = -1;
    }
    c->ysub->stream = c->stream;
    clm_status s = clm_set_positions(c->ysub, y, n, on_device);
    if (s) return fail(c, s, c->ysub->err);
    c->two_set = true;
    if (c->celltype == CLM_NONPERIODIC) c->dirty = true;
    return CLM_OK;
}

clm_status clm_clear_positions_y(clm_ctx *c) {
    if (!c) return CLM_ERR_ARG;
    c->two_set = false;
    return CLM_OK;
}

clm_status clm_set_types_y(clm_ctx *c, const int32_t *t, int64_t n, int on_device) {
    if (!c) return CLM_ERR_ARG;
    if (!c->two_set || !c->ysub) return fail(c, CLM_ERR_STATE, "no second set of positions");
    clm_status s = clm_set_types(c->ysub, t, n, on_device);
    return s ? fail(c, s, c->ysub->err) : CLM_OK;
}

clm_status clm_set_velocities_y(clm_ctx *c, const void *v, int64_t n, int on_device) {
    if (!c) return CLM_ERR_ARG;
    if (!c->two_set || !c->ysub) return fail(c, CLM_ERR_STATE, "no second set of positions");
    clm_status s = clm_set_velocities(c->ysub, v, n, on_device);
    return s ? fail(c, s, c->ysub->err) : CLM_OK;
}

}  // extern "C"

template <typename T>
clm_status cell_list_info(clm_ctx *c, int64_t *out4) {
    clm_status s = ensure_cell_list(c);
    if (s) return s;
    std::vector<int> cr(c->ncells), cst(c->ncells + 1);
    HIPCHK(c, hipMemcpyAsync(cr.data(), c->creal.p, sizeof(int) * c->ncells, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipMemcpyAsync(cst.data(), c->cstart.p, sizeof(int) * (c->ncells + 1), hipMemcpyDeviceToHost, c->stream));
    if ((s = sync(c))) return s;
    int64_t withreal = 0, withp = 0, cells = 0;
    for (int k = 0; k < c->nsys; ++k) {
        const HostBox<T> &b = hboxes<T>(c)[k];
        const int S = b.sub, sz = b.dim == 3 ? S : 1;
        const int64_t ny = (int64_t)b.nc[1] * S;
        for (int z = 0; z < b.nc[2]; ++z)
            for (int y = 0; y < b.nc[1]; ++y)
                for (int x = 0; x < b.nc[0]; ++x) {
                    bool real = false, any = false;  // over the parts of the cell
                    for (int t = 0; t < S * sz; ++t) {
                        const int64_t q = c->h_celloff[k] + ((z * sz + t / S) * ny + y * S + t % S) * b.nc[0] + x;
                        real = real || cr[q] > 0;
                        any = any || cst[q + 1] > cst[q];
                    }
                    withreal += real;
                    withp += any;
                    ++cells;
                }
    }
    out4[0] = cst[c->ncells];
    out4[1] = withreal;
    out4[2] = withp;
    out4[3] = cells;
    return CLM_OK;
}

extern "C" {

clm_status clm_cell_list_info(clm_ctx *c, int64_t *out4) {
    if (!c || !out4) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return with_redo(c, [&] { return c->dtype == CLM_F32 ? cell_list_info<float>(c, out4) : cell_list_info<double>(c, out4); });
}

clm_status clm_neighborlist(clm_ctx *c, int32_t *i, int32_t *j, void *d, int64_t capacity, int64_t *npairs, int on_device) {
    if (!c || !npairs || capacity < 0) return CLM_ERR_ARG;
    if (capacity > 0 && (!i || !j || !d)) return fail(c, CLM_ERR_ARG, "NULL output arrays");
    hipSetDevice(c->device);
    return with_redo(c, [&] {
        return c->dtype == CLM_F32 ? neighborlist_t<float>(c, i, j, d, capacity, npairs, on_device)
                                   : neighborlist_t<double>(c, i, j, d, capacity, npairs, on_device);
    });
}

clm_status clm_energy_forces(clm_ctx *c, const clm_softcore *p, double *energy, void *forces, int on_device, int64_t *npairs) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    if (npairs) *npairs = -1;
    return with_redo(c, [&] {
        if (forces)
            return c->dtype == CLM_F32 ? softcore_t<float, true, false>(c, p, energy, 0, forces, nullptr, nullptr, on_device)
                                       : softcore_t<double, true, false>(c, p, energy, 0, forces, nullptr, nullptr, on_device);
        return c->dtype == CLM_F32 ? softcore_t<float, false, false>(c, p, energy, 0, nullptr, nullptr, nullptr, on_device)
                                   : softcore_t<double, false, false>(c, p, energy, 0, nullptr, nullptr, nullptr, on_device);
    });
}

clm_status clm_energy_forces_batch(clm_ctx *c, const clm_softcore *p, double *energies, void *forces, int on_device) {
    if (!c || !energies) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return with_redo(c, [&] {
        if (forces)
            return c->dtype == CLM_F32 ? softcore_t<float, true, false>(c, p, energies, 1, forces, nullptr, nullptr, on_device)
                                       : softcore_t<double, true, false>(c, p, energies, 1, forces, nullptr, nullptr, on_device);
        return c->dtype == CLM_F32 ? softcore_t<float, false, false>(c, p, energies, 1, nullptr, nullptr, nullptr, on_device)
                                   : softcore_t<double, false, false>(c, p, energies, 1, nullptr, nullptr, nullptr, on_device);
    });
}

clm_status clm_energy_adjoint(clm_ctx *c, const clm_softcore *p, double *energy, void *dedx, double *deps, double *dsig,
                              int on_device) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return with_redo(c, [&] {
        return c->dtype == CLM_F32 ? softcore_t<float, true, true>(c, p, energy, 0, dedx, deps, dsig, on_device)
                                   : softcore_t<double, true, true>(c, p, energy, 0, dedx, deps, dsig, on_device);
    });
}

clm_status clm_graph_capture_energy_forces(clm_ctx *c, const clm_softcore *p, void *forces) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return with_redo(c, [&] { return c->dtype == CLM_F32 ? graph_capture_t<float>(c, p, forces) : graph_capture_t<double>(c, p, forces); });
}

clm_status clm_graph_launch(clm_ctx *c, double *energies) {
    if (!c) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return graph_launch(c, energies);
}

clm_status clm_histogram(clm_ctx *c, int nbins, double width, int64_t *counts, double *vsum) {
    if (!c || !counts) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return with_redo(c, [&] {
        return c->dtype == CLM_F32 ? histogram_t<float>(c, nbins, width, counts, vsum)
                                   : histogram_t<double>(c, nbins, width, counts, vsum);
    });
}

clm_status clm_min_distance(clm_ctx *c, int64_t *i, int64_t *j, double *d) {
    if (!c || !i || !j || !d) return CLM_ERR_ARG;
    hipSetDevice(c->device);
    return with_redo(c, [&] { return c->dtype == CLM_F32 ? mindist_t<float>(c, i, j, d) : mindist_t<double>(c, i, j, d); });
}

clm_status clm_profile_enable(clm_ctx *c, int enable) {
    if (!c) return CLM_ERR_ARG;
    c->prof = enable != 0;
    return CLM_OK;
}

clm_status clm_profile_get(clm_ctx *c, const char *name, double *total_ms, int64_t *count) {
    if (!c || !name || !total_ms || !count) return CLM_ERR_ARG;
    if (c->prof && !c->pending.empty()) {
        hipStreamSynchronize(c->stream);
        collect_profile(c);
    }
    auto it = c->prof_acc.find(name);
    *total_ms = it == c->prof_acc.end() ? 0.0 : it->second.first;
    *count = it == c->prof_acc.end() ? 0 : it->second.second;
    return CLM_OK;
}

clm_status clm_profile_reset(clm_ctx *c) {
    if (!c) return CLM_ERR_ARG;
    if (!c->pending.empty()) {
        hipStreamSynchronize(c->stream);
        collect_profile(c);
    }
    c->prof_acc.clear();
    return CLM_OK;
}

clm_status clm_energy_forces_noalloc(int dtype, int dim, const void *x, int64_t n, const double *cell, int celltype,
                                     double cutoff, int lcell, const clm_softcore *p, double *energy, void *forces,
                                     void *stream) {
    if (dtype != CLM_F32 && dtype != CLM_F64) return noalloc_fail(CLM_ERR_ARG, "dtype must be CLM_F32 or CLM_F64");
    if (dim != 2 && dim != 3) return noalloc_fail(CLM_ERR_DIM, "dimension must be 2 or 3");
    if (n < 0 || (n > 0 && !x) || !cell || !p) return noalloc_fail(CLM_ERR_ARG, "bad positions, cell or parameters");
    if (celltype != CLM_ORTHORHOMBIC && celltype != CLM_TRICLINIC)
        return noalloc_fail(CLM_ERR_ARG, "the allocation-free entry point needs a periodic cell");
    if (p->ntypes != 0) return noalloc_fail(CLM_ERR_ARG, "the allocation-free entry point takes untyped parameters");
    // the positions, the cell list (entries, the unsorted copy) and the per-particle tables
    // must fit at the least: reject what cannot before launching anything
    const size_t es = dtype == CLM_F32 ? sizeof(Ent<float>) : sizeof(Ent<double>);
    const size_t least = (size_t)n * (2 * es + 4 * sizeof(int));
    if (n >= (int64_t)IDX_LIMIT || least > CLM_SCRATCH_BYTES)
        return noalloc_fail(CLM_ERR_CAPACITY, "too many particles for the " + std::to_string(CLM_SCRATCH_BYTES >> 20) +
                                                  " MiB scratch of the allocation-free entry point");
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= CLM_MAX_DEVICES)
        return noalloc_fail(CLM_ERR_HIP, "no current device");
    void *base = nullptr;
    hipError_t e = scratch_ptr(dev, &base);
    if (e != hipSuccess || !base)
        return noalloc_fail(CLM_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    return dtype == CLM_F32 ? energy_forces_noalloc_t<float>(dim, x, n, cell, celltype, cutoff, lcell, p, energy, forces,
                                                             (hipStream_t)stream, dev, base)
                            : energy_forces_noalloc_t<double>(dim, x, n, cell, celltype, cutoff, lcell, p, energy, forces,
                                                              (hipStream_t)stream, dev, base);
}

}  // extern "C"
