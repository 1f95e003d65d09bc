// clm_kernels.hpp -- HIP kernels of the cell-list engine for gfx950.
//
//   k_bin_bucket  wrap + rotate each particle, place it and its ghost images in the
//                 buckets of their cells (add_particles! / replicate_particle!,
//                 CellLists.jl:940-1057, Box.jl:556-566); k_bin_count / k_bin_scatter
//                 are the two-pass form
//   k_bin_images  the same for small systems, a thread per particle and image
//   k_limits      extremes of the coordinates (open boxes)
//   k_scan_pair   single-pass scans: cell counts, homes per cell, wave tasks, output chunks
//   k_cell_sort   order every cell by x (and split real / ghost entries)
//   k_sweep_win<Op> / k_sweep<Op>   the cell-pair sweep (self.jl:106-184,
//                 vicinal_cells.jl:4-75) with a fixed device operator Op in place of the
//                 user closure
//   k_nl_fill     compaction of the chunked neighbour-list output
//
// Sweep mapping of k_sweep_win: see there.  Of k_sweep: one wave (64 lanes) takes up to 64 consecutive home entries of one
// x-row of cells.  For each of the (2L+1)^2 (3D) stencil rows the union of the lanes'
// x-ranges is one contiguous slice of E; every lane walks the same entry j (a
// wave-uniform load) and keeps it if j lies in its own stencil range, the pair filter
// of the mode holds and d2 <= rc^2.  Modes:
//   MODE_A_ORTHO  each pair once, reference orientation for orthorhombic/non-periodic
//                 boxes: homes = all entries of cells holding a real particle, forward
//                 stencil, later entries of the own cell, skip ghost-ghost pairs.
//   MODE_A_TRIC   each pair once for triclinic boxes: homes = real particles, full
//                 stencil, keep index_i < index_j.  The windowed sweep takes the same
//                 pairs in two parts: pairs of two real particles from the home earlier
//                 in the cell order (a half stencil over the real entries alone), pairs
//                 with a ghost image by the index rule (full stencil over the ghost
//                 entries alone, rows without ghost images skipped).
//   MODE_B        each pair from both sides (homes = real particles, full stencil,
//                 index_i != index_j); operators accumulate only into the home
//                 particle, so no atomics are needed for forces.
// Two sets (cross.jl): the homes come from the cell list of one set and the
// neighbours from the cell list of the other (same box and grid).
//   MODE_X_ORTHO  reference orientation for orthorhombic/non-periodic boxes: homes =
//                 all entries of cells holding a real particle, full stencil; in the
//                 cell of the same index the home must be real, elsewhere at least one
//                 of the two (cross.jl:81-130).
//   MODE_X_REAL   homes = real particles, full stencil, every neighbour entry: each
//                 pair once per real home (the triclinic cross sweep, and the force
//                 sweeps of either set for any box).
#pragma once

#include <type_traits>

#include "clm_device.hpp"

namespace clm {

enum { MODE_A_ORTHO = 0, MODE_A_TRIC = 1, MODE_B = 2, MODE_X_ORTHO = 3, MODE_X_REAL = 4 };
constexpr bool mode_all_entries(int m) { return m == MODE_A_ORTHO || m == MODE_X_ORTHO; }
enum { NONPER_FLAG = 2 };

// ------------------------------------------------------------------------------
// binning
// ------------------------------------------------------------------------------

// Per-system description for the device: the box, the inverse rotation used for
// outputs, and where the system's cells, rows and particles start in the global arrays.
// A single system is a table with one entry; a batch of independent systems (each with
// its own box, cutoff and lcell) is one table, processed by the same kernels.
template <typename T>
struct SysDesc {
    DevBox<T> box;
    T invrot[9];
    int cell_off;
    int row_off;
    int pos_off;
    int n;
};

// Largest k in [lo, hi) with a[k] <= v (a non-decreasing, a[lo] <= v).
__device__ inline int last_le(const int *__restrict__ a, int lo, int hi, int v) {
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (a[mid] <= v) lo = mid;
        else hi = mid;
    }
    return lo;
}

template <typename T, int D>
__global__ void __launch_bounds__(256) k_bin_count(const T *__restrict__ x, int n, const SysDesc<T> *__restrict__ sys,
                                                   const int *__restrict__ sys_of, Ent<T> *__restrict__ xw,
                                                   int *__restrict__ home_cell, int *__restrict__ cnt,
                                                   int *__restrict__ creal, uint32_t *__restrict__ gflags) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int si = sys_of ? sys_of[i] : 0;
    const DevBox<T> &b = sys[si].box;
    const int coff = sys[si].cell_off;
    const bool periodic = b.celltype != NONPER_FLAG;
    T xi[3] = {T(0), T(0), T(0)};
    bool finite = true;
    for (int k = 0; k < D; ++k) {
        xi[k] = x[(size_t)i * D + k];
        finite = finite && dev_finite(xi[k]);
    }
    uint32_t flags = 0;
    if (!finite) {
        atomicOr(gflags, FLAG_NAN);
        home_cell[i] = -1;
        return;
    }
    T p[3] = {T(0), T(0), T(0)};
    if (periodic) {
        if (D == 3) wrap_rotate3(b, xi, p);
        else wrap_rotate2(b, xi, p);
    } else {
        for (int k = 0; k < D; ++k) p[k] = xi[k];
    }
    Ent<T> e;
    e.x = p[0]; e.y = p[1]; e.z = p[2];
    e.w = (uint32_t)i;
    xw[i] = e;
    const int c = coff + cell_of<D>(b, p, true, flags);
    home_cell[i] = c;
    atomicAdd(&cnt[c], 1);
    atomicAdd(&creal[c], 1);
    if (periodic) {
        const int nimg = D == 3 ? 27 : 9;
        for (int m = 0; m < nimg; ++m) {
            if (m == (D == 3 ? 13 : 4)) continue;
            T q[3] = {p[0], p[1], p[2]};
            for (int k = 0; k < D; ++k) q[k] = p[k] + b.shift[m][k];
            if (!in_box<D>(b, q)) continue;
            const int cj = coff + cell_of<D>(b, q, false, flags);
            atomicAdd(&cnt[cj], 1);
        }
    }
    if (flags) atomicOr(gflags, flags);
}

template <typename T, int D>
__global__ void __launch_bounds__(256) k_bin_scatter(int n, const SysDesc<T> *__restrict__ sys,
                                                     const int *__restrict__ sys_of, const Ent<T> *__restrict__ xw,
                                                     const int *__restrict__ home_cell, const int *__restrict__ cstart,
                                                     const int *__restrict__ creal, const int *__restrict__ types,
                                                     int *__restrict__ cur_real, int *__restrict__ cur_ghost,
                                                     Ent<T> *__restrict__ E, int64_t ecap, uint32_t *__restrict__ gflags) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int c = home_cell[i];
    if (c < 0) return;
    const int si = sys_of ? sys_of[i] : 0;
    const DevBox<T> &b = sys[si].box;
    const int coff = sys[si].cell_off;
    uint32_t flags = 0;
    Ent<T> e = xw[i];
    const uint32_t ty = types ? (uint32_t)types[i] : 0u;
    e.w = w_make((uint32_t)i, ty, false);
    int slot = atomicAdd(&cur_real[c], 1);
    int64_t pos = (int64_t)cstart[c] + slot;
    if (pos < ecap) E[pos] = e;
    else flags |= FLAG_OVERFLOW;
    if (b.celltype != NONPER_FLAG) {
        T p[3] = {e.x, e.y, e.z};
        const int nimg = D == 3 ? 27 : 9;
        for (int m = 0; m < nimg; ++m) {
            if (m == (D == 3 ? 13 : 4)) continue;
            T q[3] = {p[0], p[1], p[2]};
            for (int k = 0; k < D; ++k) q[k] = p[k] + b.shift[m][k];
            if (!in_box<D>(b, q)) continue;
            uint32_t fl2 = 0;
            int cj = coff + cell_of<D>(b, q, false, fl2);
            int s2 = atomicAdd(&cur_ghost[cj], 1);
            int64_t pj = (int64_t)cstart[cj] + creal[cj] + s2;
            Ent<T> g;
            g.x = q[0]; g.y = q[1]; g.z = q[2];
            g.w = w_make((uint32_t)i, ty, true);
            if (pj < ecap) E[pj] = g;
            else flags |= FLAG_OVERFLOW;
        }
    }
    if (flags) atomicOr(gflags, flags);
}

// Slot claim shared by the lanes that add to the same counter: the lanes are grouped by
// counter (one ballot per distinct counter), then every group's first lane adds the
// group's total in one wave-wide atomic instruction (all groups' atomics in flight
// together) and hands the returned base to its group.
// The claim in two halves, so that several claims can be in flight before any result is
// used: grouped_add_issue groups the lanes and issues the leaders' atomics (the result
// stays in the leader lanes), grouped_add_slot hands each group its base.
struct GroupedClaim {
    unsigned long long base;  // the atomic's result, in the group's first lane
    int leader, rank;
};
__device__ inline GroupedClaim grouped_add_issue(unsigned long long *ctr, int c, bool act, unsigned long long inc) {
    int my_leader = 0, my_rank = 0, my_size = 0;
    uint64_t todo = ballot64(act);
    while (todo) {
        const int leader = (int)__builtin_ctzll(todo);
        const int cl = __builtin_amdgcn_readlane(c, leader);
        const bool mine = act && c == cl;
        const uint64_t grp = ballot64(mine);
        if (mine) {
            my_leader = leader;
            my_rank = rank_in(grp);
            my_size = __popcll(grp);
        }
        todo &= ~grp;
    }
    GroupedClaim g;
    g.base = 0;
    if (act && my_rank == 0) g.base = atomicAdd(&ctr[c], inc * (unsigned long long)my_size);
    g.leader = my_leader;
    g.rank = my_rank;
    return g;
}
__device__ inline uint32_t grouped_add_slot(const GroupedClaim &g) {
    return (uint32_t)__shfl((int)(uint32_t)g.base, g.leader, 64) + (uint32_t)g.rank;
}
// One particle of the single-pass binning (see k_bin_bucket); b/coff are the particle's
// system, passed uniformly when every lane of the wave is in the same system so that the
// box is read through the scalar cache.
template <typename T, int D>
__device__ __forceinline__ uint32_t bin_one(const DevBox<T> &b, int coff, const T *__restrict__ x, int i, bool in,
                                   const int *__restrict__ types, unsigned long long *__restrict__ cnt64, int shift,
                                   Ent<T> *__restrict__ Eb, int bucket) {
    const bool periodic = b.celltype != NONPER_FLAG;
    T xi[3] = {T(0), T(0), T(0)};
    bool finite = true;
    if (in) {
        for (int d = 0; d < D; ++d) {
            xi[d] = x[(size_t)i * D + d];
            finite = finite && dev_finite(xi[d]);
        }
    }
    const bool live = in && finite;
    uint32_t flags = (in && !finite) ? FLAG_NAN : 0u;
    T p[3] = {T(0), T(0), T(0)};
    if (live) {
        if (periodic) {
            if (D == 3) wrap_rotate3(b, xi, p);
            else wrap_rotate2(b, xi, p);
        } else {
            for (int d = 0; d < D; ++d) p[d] = xi[d];
        }
    }
    const uint32_t ty = (live && types) ? (uint32_t)types[i] : 0u;
    const int c = live ? coff + cell_of<D>(b, p, true, flags) : 0;
    {
        const uint32_t slot = grouped_add_slot(grouped_add_issue(cnt64, c << shift, live, (1ull << 32) | 1ull));
        if (live) {
            Ent<T> e;
            e.x = p[0]; e.y = p[1]; e.z = p[2];
            e.w = w_make((uint32_t)i, ty, false);
            if (slot < (uint32_t)bucket) Eb[(size_t)c * bucket + slot] = e;
            else flags |= FLAG_OVERFLOW;
        }
    }
    if (ballot64(live && periodic) != 0) {
        // The images, IB directions at a time: the slot claims of a batch are issued
        // together and their results used after the last one (device-scope atomics take
        // microseconds; one at a time, the waves near the faces, which hold the images,
        // set the length of the whole kernel: 0.105 -> 0.094 ms at N = 1M).  Batches of the
        // wave's active directions only, found first, measured slower (0.16-0.18 ms: the
        // direction becomes a run-time index).
        constexpr int nimg = D == 3 ? 27 : 9;
        constexpr int IB = 4;
        for (int m0 = 0; m0 < nimg; m0 += IB) {
            GroupedClaim gc[IB];
            T gq[IB][3];
            int gcj[IB];
            bool gimg[IB];
#pragma unroll
            for (int u = 0; u < IB; ++u) {
                const int m = m0 + u;
                gimg[u] = false;
                gcj[u] = 0;
                gc[u].base = 0;
                gc[u].leader = 0;
                gc[u].rank = 0;
                gq[u][0] = gq[u][1] = gq[u][2] = T(0);
                if (m >= nimg || m == (D == 3 ? 13 : 4)) continue;
                for (int d = 0; d < 3; ++d) gq[u][d] = p[d];
                for (int d = 0; d < D; ++d) gq[u][d] = p[d] + b.shift[m][d];
                gimg[u] = live && periodic && in_box<D>(b, gq[u]);
                if (ballot64(gimg[u]) == 0) continue;
                gcj[u] = gimg[u] ? coff + cell_of<D>(b, gq[u], false, flags) : 0;
                gc[u] = grouped_add_issue(cnt64, gcj[u] << shift, gimg[u], 1ull);
            }
#pragma unroll
            for (int u = 0; u < IB; ++u) {
                if (ballot64(gimg[u]) == 0) continue;
                const uint32_t slot = grouped_add_slot(gc[u]);
                if (gimg[u]) {
                    Ent<T> g;
                    g.x = gq[u][0]; g.y = gq[u][1]; g.z = gq[u][2];
                    g.w = w_make((uint32_t)i, ty, true);
                    if (slot < (uint32_t)bucket) Eb[(size_t)gcj[u] * bucket + slot] = g;
                    else flags |= FLAG_OVERFLOW;
                }
            }
        }
    }
    return flags;
}

// Single-pass binning into fixed-size cell buckets: every real particle and each of its
// ghost images takes a slot of its cell from the cell's 64-bit counter word (entries in
// the low half, reals in the high half) and is written at c * bucket + slot.  Particles
// are visited in the cell order of the previous build (order[], from k_cell_sort), so a
// wave's particles mostly fall in a few cells and grouped_add claims their slots with a
// few atomics.  Replaces k_bin_count + scan + k_bin_scatter (two passes and three atomics
// per real particle) when the bucket size covers the fullest cell; a slot at or beyond
// the bucket raises FLAG_OVERFLOW and the host repeats the pass with larger buckets.
template <typename T, int D>
__global__ void __launch_bounds__(256) k_bin_bucket(const T *__restrict__ x, int n, const int *__restrict__ order,
                                                    const SysDesc<T> *__restrict__ sys, const int *__restrict__ sys_of,
                                                    const int *__restrict__ types, unsigned long long *__restrict__ cnt64, int shift,
                                                    Ent<T> *__restrict__ Eb, int bucket, uint32_t *__restrict__ gflags) {
    // every lane stays in the wave to the end: grouped_add is a wave-wide operation
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = k < n;
    const int i = in ? (order ? order[k] : k) : 0;
    const int si = (in && sys_of) ? sys_of[i] : 0;
    const int s0 = uniform_int(si);
    uint32_t flags;
    if (ballot64(si != s0) == 0) flags = bin_one<T, D>(sys[s0].box, sys[s0].cell_off, x, i, in, types, cnt64, shift, Eb, bucket);
    else flags = bin_one<T, D>(sys[si].box, sys[si].cell_off, x, i, in, types, cnt64, shift, Eb, bucket);
    if (flags) atomicOr(gflags, flags);
}

// The same pass for small systems, one thread per particle and image direction (blockIdx.y):
// the wrap is repeated for every direction, but each thread makes one claim, all of them are
// in flight at once and none waits for another of its wave.
template <typename T, int D>
__global__ void __launch_bounds__(64) k_bin_images(const T *__restrict__ x, int n, const int *__restrict__ order,
                                                   const SysDesc<T> *__restrict__ sys, const int *__restrict__ sys_of,
                                                   const int *__restrict__ types, unsigned long long *__restrict__ cnt64, int shift,
                                                   Ent<T> *__restrict__ Eb, int bucket, uint32_t *__restrict__ gflags) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int m = blockIdx.y;
    const bool real = m == (D == 3 ? 13 : 4);
    const int i = order ? order[k] : k;
    const int si = sys_of ? sys_of[i] : 0;
    const DevBox<T> &b = sys[si].box;
    const int coff = sys[si].cell_off;
    const bool periodic = b.celltype != NONPER_FLAG;
    if (!real && !periodic) return;
    T xi[3] = {T(0), T(0), T(0)}, p[3] = {T(0), T(0), T(0)};
    bool finite = true;
    for (int d = 0; d < D; ++d) {
        xi[d] = x[(size_t)i * D + d];
        finite = finite && dev_finite(xi[d]);
    }
    if (!finite) {
        if (real) atomicOr(gflags, FLAG_NAN);
        return;
    }
    if (periodic) {
        if (D == 3) wrap_rotate3(b, xi, p);
        else wrap_rotate2(b, xi, p);
    } else {
        for (int d = 0; d < D; ++d) p[d] = xi[d];
    }
    if (!real) {
        for (int d = 0; d < D; ++d) p[d] = p[d] + b.shift[m][d];
        if (!in_box<D>(b, p)) return;
    }
    uint32_t flags = 0;
    const int c = coff + cell_of<D>(b, p, real, flags);
    const uint32_t slot = (uint32_t)atomicAdd(&cnt64[(size_t)c << shift], real ? (1ull << 32) | 1ull : 1ull);
    if (slot < (uint32_t)bucket) {
        Ent<T> e;
        e.x = p[0]; e.y = p[1]; e.z = p[2];
        e.w = w_make((uint32_t)i, types ? (uint32_t)types[i] : 0u, !real);
        Eb[(size_t)c * bucket + slot] = e;
    } else {
        flags |= FLAG_OVERFLOW;
    }
    if (flags) atomicOr(gflags, flags);
}

// Largest of a block's values into *maxcnt (one atomic per block).
__device__ inline void block_max_to(int mx, int *maxcnt) {
    __shared__ int wm[4];
    for (int off = 32; off > 0; off >>= 1) mx = max(mx, __shfl_xor(mx, off, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        int m = wm[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = max(m, wm[w]);
        if (m > 0) atomicMax(maxcnt, m);
    }
}

// Largest cell count (sizes the buckets of the single-pass binning).  Grid-stride,
// 256 threads per block.
static __global__ void __launch_bounds__(256) k_count_max(int ncells, const int *__restrict__ cnt, int *__restrict__ maxcnt) {
    int mx = 0;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += gridDim.x * blockDim.x) mx = max(mx, cnt[c]);
    block_max_to(mx, maxcnt);
}

// Orders the entries of every cell by (x, w) -- x in the aligned frame, w breaking ties
// (unique per entry) -- and records where each real particle landed: real_pos[rstart[c]
// + k] = position of the k-th real of cell c, order[rstart[c] + k] = its particle index
// (the visiting order of the next binning pass), real_cell[rstart[c] + k] = c.  Cells are contiguous intervals of x along a
// row of the grid, so a whole row of cells is then ordered by x (up to rounding at the two
// cells the border rule moves reals into), which lets the sweep stop a lane's walk along a
// row as soon as it passes the end of that lane's window.  The order is also independent
// of the atomic arrival order of the scatter.  An entry has Q threads (below): they find its cell
// among those of the workgroup and its rank by counting the smaller entries of the cell.
// Ein holds the entries of cell c at cstart[c] (compact) or, when bucket > 0, at c * bucket.
// The grid covers at least cstart[ncells] entries (their count, read on the device so
// that a captured graph sorts whatever the count of its replay is, within the capacity).
// Cells that do not end within cap entries are left out (their replay reports the
// overflow raised by the scatter).
// Rout / Gout (both null or both set): the same order split into the real entries alone
// (Rout[rstart[c] + k], k-th real of cell c) and the ghost entries alone (Gout[cstart[c] -
// rstart[c] + k], k-th ghost of cell c), the two arrays the triclinic sweep walks.
// Largest k in [lo, hi) with a[k] <= v (a non-decreasing, a[lo] <= v), found by the 64
// lanes of one wave together: each round probes 64 evenly spaced points and keeps the
// stretch between the last probe at or below v and the next one, so ~log64 of the range
// rounds of dependent loads instead of log2 (called by a whole wave; every lane returns it).
__device__ inline int wave_last_le(const int *__restrict__ a, int lo, int hi, int v) {
    const int lane = (int)(threadIdx.x & 63);
    while (hi - lo > 1) {
        const int step = (int)(((long long)(hi - lo) + 63) / 64);
        const long long k = (long long)lo + (long long)(lane + 1) * step;
        const bool ok = k < hi && a[k] <= v;
        const int t = __popcll(ballot64(ok));  // probes 0 .. t-1 are at or below v
        const int nlo = lo + t * step;
        hi = (int)std::min<long long>((long long)hi, (long long)nlo + step);
        lo = nlo;
    }
    return lo;
}

// wave_last_le over a 64-bit index range (a non-decreasing, a[lo] <= v).
__device__ inline long long wave_last_le64(const int *__restrict__ a, long long lo, long long hi, long long v) {
    const int lane = (int)(threadIdx.x & 63);
    while (hi - lo > 1) {
        const long long step = (hi - lo + 63) / 64;
        const long long k = lo + (long long)(lane + 1) * step;
        const bool ok = k < hi && (long long)a[k] <= v;
        const long long nlo = lo + (long long)__popcll(ballot64(ok)) * step;  // the last probe at or below v
        hi = std::min<long long>(hi, nlo + step);
        lo = nlo;
    }
    return lo;
}

// Q threads share an entry, each counting a Q-th of its cell.
template <typename T, int Q>
__global__ void __launch_bounds__(256) k_cell_sort(int ncells, const int *__restrict__ cstart,
                                                   const int *__restrict__ rstart, const Ent<T> *__restrict__ Ein,
                                                   int bucket, int64_t cap, Ent<T> *__restrict__ Eout,
                                                   int *__restrict__ real_pos, int *__restrict__ order,
                                                   int *__restrict__ real_cell, Ent<T> *__restrict__ Rout, Ent<T> *__restrict__ Gout) {
    // The workgroup's entries belong to the cells [c0, c1]; their keys (x, w) are staged
    // in LDS once when they fit, and every thread ranks its entry against its cell there.
    constexpr int STAGE = 1024;
    constexpr int CSTAGE = 512;  // cell starts of the workgroup's cells held in LDS
    __shared__ T s_x[STAGE];
    __shared__ uint32_t s_w[STAGE];
    __shared__ int s_cs[CSTAGE];
    __shared__ int s_c0, s_c1;
    const int total = cstart[ncells];
    const int per = (int)blockDim.x / Q;  // entries of the workgroup
    const int kb = blockIdx.x * per;
    if (kb >= total) return;  // the whole workgroup
    if (threadIdx.x < 64) {  // the first wave finds the cells [c0, c1] of the workgroup's entries
        const int c0 = wave_last_le(cstart, 0, ncells, kb);
        const int c1 = wave_last_le(cstart, c0, ncells, min(kb + per, total) - 1);
        if (threadIdx.x == 0) {
            s_c0 = c0;
            s_c1 = c1;
        }
    }
    __syncthreads();
    const int c0 = s_c0, c1 = s_c1;
    // cstart[c0 .. c1 + 1] in LDS when they fit: the cell of an entry is then found there
    const bool cs_staged = c1 + 2 - c0 <= CSTAGE;
    if (cs_staged)
        for (int t = threadIdx.x; t < c1 + 2 - c0; t += blockDim.x) s_cs[t] = cstart[c0 + t];
    __syncthreads();
    // the last cell in [c0, c1] starting at or before kk
    auto cell_of_entry = [&](int kk) -> int {
        if (!cs_staged) return last_le(cstart, c0, c1 + 1, kk);
        int lo = 0, hi = c1 + 1 - c0;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (s_cs[mid] <= kk) lo = mid;
            else hi = mid;
        }
        return c0 + lo;
    };
    const int base = cstart[c0];
    const bool staged = cstart[c1 + 1] - base <= STAGE;
    if (staged) {
        for (int t = threadIdx.x; t < cstart[c1 + 1] - base; t += blockDim.x) {
            const int kk = base + t;
            const int cc = cell_of_entry(kk);
            const int s0c = cstart[cc];
            const int nc = cstart[cc + 1] - s0c;
            // the same limits as the ranking below (capacity, bucket)
            if ((int64_t)s0c + nc > cap || (bucket > 0 && kk - s0c >= bucket)) continue;
            const Ent<T> f = Ein[bucket > 0 ? (size_t)cc * bucket + (kk - s0c) : (size_t)kk];
            s_x[t] = f.x;
            s_w[t] = ent_w(f);
        }
    }
    __syncthreads();
    const int part = threadIdx.x & (Q - 1);
    const int k = kb + (int)threadIdx.x / Q;
    if (k >= total) return;
    const int c = cell_of_entry(k);  // the last cell starting at or before k: never empty
    const int s0 = cstart[c];
    int n = cstart[c + 1] - s0;
    if ((int64_t)s0 + n > cap) return;
    if (bucket > 0 && n > bucket) {  // the cell outgrew its bucket (the build is redone): stay inside it
        n = bucket;
        if (k - s0 >= n) return;
    }
    const Ent<T> *src = Ein + (bucket > 0 ? (size_t)c * bucket : (size_t)s0);
    const Ent<T> e = src[k - s0];
    const uint32_t we = ent_w(e);
    int rank = 0, rrank = 0;
    if (staged) {
        const int o = s0 - base;
        for (int m = part; m < n; m += Q) {
            const T fx = s_x[o + m];
            const uint32_t wf = s_w[o + m];
            const bool less = (fx < e.x) || (fx == e.x && wf < we);
            rank += less ? 1 : 0;
            rrank += (less && !w_ghost(wf)) ? 1 : 0;
        }
    } else {
        for (int m = part; m < n; m += Q) {
            const Ent<T> f = src[m];
            const uint32_t wf = ent_w(f);
            const bool less = (f.x < e.x) || (f.x == e.x && wf < we);
            rank += less ? 1 : 0;
            rrank += (less && !w_ghost(wf)) ? 1 : 0;
        }
    }
    for (int off = 1; off < Q; off <<= 1) {  // (the Q threads of an entry stay together)
        rank += __shfl_xor(rank, off, 64);
        rrank += __shfl_xor(rrank, off, 64);
    }
    if (part != 0) return;
    Eout[s0 + rank] = e;
    const int r0 = rstart[c];
    if (!w_ghost(we)) {
        real_pos[r0 + rrank] = s0 + rank;
        order[r0 + rrank] = (int)w_idx(we);
        real_cell[r0 + rrank] = c;
        if (Rout) Rout[r0 + rrank] = e;
    } else if (Gout) {
        Gout[(s0 - r0) + (rank - rrank)] = e;
    }
}

// Zeroes up to 8 int arrays in one launch (grid-stride).
struct FillList {
    int *p[8];
    int n[8];
    int count;
};
static __global__ void k_fill_multi(FillList f) {
    const int stride = gridDim.x * blockDim.x;
    for (int k = 0; k < f.count; ++k)
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < f.n[k]; i += stride) f.p[k][i] = 0;
}

// Copies up to 4 word arrays one after another to dst (pinned host memory: one launch in
// place of a copy per array, each of which costs a launch and a flush of its own).
struct ReadList {
    const uint32_t *p[4];
    int n[4];
    int count;
};
static __global__ void __launch_bounds__(256) k_read_back(ReadList r, uint32_t *dst) {
    for (int k = 0; k < r.count; ++k) {
        for (int i = threadIdx.x; i < r.n[k]; i += 256) dst[i] = r.p[k][i];
        dst += r.n[k];
    }
}

// Limits of the coordinates x (nx particles) and y (ny): each workgroup writes the lowest and the
// highest of each axis and whether a coordinate is NaN; the host takes the extremes over the
// workgroups.  Bound by its launch, or for many by the read of the positions (first build of an open
// box of 5e4 at float64: 239 us, 912 with the positions copied to the host and searched there).
constexpr int LIMITS_BLOCKS = 120;
template <typename T>
struct Limits {
    T lo[3], hi[3];
    T nan, unused;
};
template <typename T>
__global__ void __launch_bounds__(256) k_limits(const T *__restrict__ x, long long nx, const T *__restrict__ y, long long ny,
                                                int dim, Limits<T> *out) {
    __shared__ Limits<T> s[4];
    Limits<T> l;
    l.nan = l.unused = T(0);
#pragma unroll
    for (int k = 0; k < 3; ++k) { l.lo[k] = T(INFINITY); l.hi[k] = -T(INFINITY); }
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < nx + ny; i += (long long)gridDim.x * 256) {
        const T *p = i < nx ? x + i * dim : y + (i - nx) * dim;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (k >= dim) break;
            const T v = p[k];
            if (v != v) l.nan = T(1);
            if (v < l.lo[k]) l.lo[k] = v;
            if (v > l.hi[k]) l.hi[k] = v;
        }
    }
    auto take = [](Limits<T> &a, const Limits<T> &b) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (b.lo[k] < a.lo[k]) a.lo[k] = b.lo[k];
            if (b.hi[k] > a.hi[k]) a.hi[k] = b.hi[k];
        }
        if (b.nan > a.nan) a.nan = b.nan;
    };
    for (int off = 32; off > 0; off >>= 1) {
        Limits<T> o;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            o.lo[k] = __shfl_xor(l.lo[k], off, 64);
            o.hi[k] = __shfl_xor(l.hi[k], off, 64);
        }
        o.nan = __shfl_xor(l.nan, off, 64);
        take(l, o);
    }
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; ++k) take(l, s[k]);
        out[blockIdx.x] = l;
    }
}

// p[i] = i.
static __global__ void k_iota(int *__restrict__ p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

static __global__ void k_fill_int(int *__restrict__ p, int n, int v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------------------------------
// single-pass scans
// ------------------------------------------------------------------------------
//
// Exclusive scans of two counts per element, produced on the fly by Prod::get(i, a, b),
// in one launch: each workgroup takes a tile of SCAN_THREADS * Prod::ITEMS elements in the order it
// started (a ticket counter), publishes the tile's sums, then walks back over the
// preceding tiles' published words until it meets a tile that published its inclusive
// prefix ("decoupled look-back").  A tile only waits on tiles that started before it and
// publish without waiting, so the walk ends; it is also bounded, and a walk that hits the
// bound raises *err (the result is then invalid and the caller reports it).  The last
// workgroup to finish clears the status words and counters, so the state is ready for the
// next launch, also inside a captured graph.  out_a[n] / out_b[n] receive the totals.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;
constexpr unsigned long long SCAN_AGG = 1ull << 62, SCAN_PRE = 2ull << 62;
constexpr unsigned int SCAN_SPIN_LIMIT = 1u << 24;

struct ScanState {
    unsigned long long *status;  // one word per tile: flag (2 bits) | a (31 bits) | b (31 bits)
    unsigned int *ticket;
    unsigned int *done;
};

// Tiles of a scan over n elements (the most any producer needs: it sizes the scan state);
// a producer with Prod::ITEMS elements per thread launches scan_tiles_for<Prod>(n).
inline long long scan_tiles(long long n) { return n / SCAN_TILE + 1; }
template <typename Prod>
inline long long scan_tiles_for(long long n) { return n / ((long long)SCAN_THREADS * Prod::ITEMS) + 1; }

__device__ inline unsigned long long scan_pack(int a, int b) {
    return ((unsigned long long)(unsigned)a << 31) | (unsigned long long)(unsigned)b;
}

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
// IT values from or to consecutive addresses, 16-byte aligned, IT a multiple of 4
template <int IT>
__device__ inline void load_all(const int *__restrict__ p, int (&v)[IT]) {
#pragma unroll
    for (int k = 0; k < IT; k += 4) {
        const i32x4 t = *(const i32x4 *)(p + k);
        v[k] = t[0]; v[k + 1] = t[1]; v[k + 2] = t[2]; v[k + 3] = t[3];
    }
}
template <int IT>
__device__ inline void store_all(int *__restrict__ p, const int (&v)[IT]) {
#pragma unroll
    for (int k = 0; k < IT; k += 4) *(i32x4 *)(p + k) = i32x4{v[k], v[k + 1], v[k + 2], v[k + 3]};
}

// The value every element needs (the same for all), read once per workgroup and passed to
// Prod::get: the sum of `words` device words, `stride` apart (words 0: none), which the first
// tile also writes to *sum.
struct ScanValue {
    const unsigned long long *p;
    int words, stride;
    unsigned long long *sum;
};
template <typename Prod>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_pair(long long n, Prod prod, ScanValue uval,
                                                            int *__restrict__ out_a, int *__restrict__ out_b, int *maxa,
                                                            int *tot_a, ScanState st, unsigned int *err,
                                                            unsigned int err_bit) {
    __shared__ int s_tile, s_pa, s_pb, s_last;
    __shared__ unsigned long long s_u;
    __shared__ int s_wa[SCAN_THREADS / 64], s_wb[SCAN_THREADS / 64], s_wm[SCAN_THREADS / 64];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    if (t < 64) {
        unsigned long long v = 0;
        if (uval.words) {
            for (int k = t; k < uval.words; k += 64) v += uval.p[(long long)k * uval.stride];
            v = wave_sum(v);
        }
        if (t == 0) {
            s_tile = (int)atomicAdd(st.ticket, 1u);
            s_u = v;
            if (s_tile == 0 && uval.sum) *uval.sum = v;
        }
    }
    __syncthreads();
    const int tile = s_tile;
    const unsigned long long u = s_u;
    constexpr int IT = Prod::ITEMS;
    static_assert(IT >= SCAN_ITEMS, "scan_tiles sizes the state for SCAN_ITEMS per thread");
    const long long base = (long long)tile * (SCAN_THREADS * IT) + (long long)t * IT;
    int va[IT], vb[IT];
    int sa = 0, sb = 0, mx = 0;
    // (a thread's elements lie side by side: where all exist they are read, and below
    // written, 16 bytes at a time; one by one a wave's loads touch a line per lane each)
    const bool whole = base + IT <= n;
    if (whole) {
        prod.template get_all<IT>(base, u, va, vb);
    } else {
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            va[k] = vb[k] = 0;
            if (base + k < n) prod.get(base + k, u, va[k], vb[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < IT; ++k) {
        sa += va[k];
        sb += vb[k];
        mx = max(mx, va[k]);
    }
    // inclusive scan of the thread sums within the wave, then across the waves
    int ia = sa, ib = sb;
    for (int off = 1; off < 64; off <<= 1) {
        const int xa = __shfl_up(ia, off, 64), xb = __shfl_up(ib, off, 64);
        if (lane >= off) { ia += xa; ib += xb; }
    }
    for (int off = 32; off > 0; off >>= 1) mx = max(mx, __shfl_xor(mx, off, 64));
    if (lane == 63) { s_wa[wv] = ia; s_wb[wv] = ib; s_wm[wv] = mx; }
    __syncthreads();
    int wa = 0, wb = 0, A = 0, B = 0, M = 0;
    for (int w = 0; w < SCAN_THREADS / 64; ++w) {
        if (w < wv) { wa += s_wa[w]; wb += s_wb[w]; }
        A += s_wa[w];
        B += s_wb[w];
        M = max(M, s_wm[w]);
    }
    if (wv == 0) {
        // publish, then look back with the whole wave: lane l reads the word of tile
        // (window start - l); the nearest tile with a published prefix ends the walk
        if (lane == 0)
            __hip_atomic_store(&st.status[tile], (tile == 0 ? SCAN_PRE : SCAN_AGG) | scan_pack(A, B), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        int pa = 0, pb = 0;
        int kb = tile - 1;
        unsigned int spins = 0;
        while (kb >= 0) {
            const int k = kb - lane;
            const unsigned long long v =
                k >= 0 ? __hip_atomic_load(&st.status[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : SCAN_PRE;
            const unsigned long long f = v >> 62;
            const uint64_t pre = ballot64(f == 2);
            const uint64_t pending = ballot64(f == 0);
            const int lp = pre ? __builtin_ctzll(pre) : 64;
            const uint64_t upto = lp >= 63 ? ~0ull : ((2ull << lp) - 1);
            if (pending & upto) {
                if (++spins > SCAN_SPIN_LIMIT) {
                    if (lane == 0) atomicOr(err, err_bit);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            int a = lane <= lp ? (int)((v >> 31) & 0x7fffffffu) : 0;
            int b = lane <= lp ? (int)(v & 0x7fffffffu) : 0;
            for (int off = 32; off > 0; off >>= 1) {
                a += __shfl_xor(a, off, 64);
                b += __shfl_xor(b, off, 64);
            }
            pa += a;
            pb += b;
            if (lp < 64) break;
            kb -= 64;
        }
        if (lane == 0) {
            if (tile > 0)
                __hip_atomic_store(&st.status[tile], SCAN_PRE | scan_pack(pa + A, pb + B), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            s_pa = pa;
            s_pb = pb;
            if (maxa && M > 0) atomicMax(maxa, M);
        }
    }
    __syncthreads();
    int ea = s_pa + wa + ia - sa, eb = s_pb + wb + ib - sb;
#pragma unroll
    for (int k = 0; k < IT; ++k) {  // each element's exclusive prefix in its place
        const int a = va[k], b = vb[k];
        va[k] = ea;
        vb[k] = eb;
        ea += a;
        eb += b;
    }
    if (whole) {
        if (out_a) store_all<IT>(out_a + base, va);
        if (out_b) store_all<IT>(out_b + base, vb);
    } else {
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            const long long i = base + k;
            if (i <= n) {
                if (out_a) out_a[i] = va[k];
                if (out_b) out_b[i] = vb[k];
                if (i == n && tot_a) *tot_a = va[k];
            }
        }
    }
    // the last workgroup to finish resets the state for the next launch
    __syncthreads();
    if (t == 0) {
        __threadfence();
        s_last = atomicAdd(st.done, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (s_last) {
        for (int k = t; k < (int)gridDim.x; k += SCAN_THREADS) st.status[k] = 0ull;
        if (t == 0) { *st.ticket = 0u; *st.done = 0u; }
    }
}

// Per-cell counts of the single-pass binning: entries in the low and real particles in
// the high half of each 64-bit counter (also written out as cnt / creal).
struct ProdCells {
    static constexpr int ITEMS = SCAN_ITEMS;
    const unsigned long long *cnt64;
    int shift;  // counter of cell c: cnt64[c << shift]
    int *cnt, *creal;
    __device__ void get(long long i, unsigned long long, int &a, int &b) const {
        const unsigned long long v = cnt64[i << shift];
        a = (int)(v & 0xffffffffull);
        b = (int)(v >> 32);
        cnt[i] = a;
        creal[i] = b;
    }
    template <int IT>
    __device__ void get_all(long long i, unsigned long long, int (&a)[IT], int (&b)[IT]) const {
        if (shift) {
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                const unsigned long long v = cnt64[(i + k) << shift];
                a[k] = (int)(v & 0xffffffffull);
                b[k] = (int)(v >> 32);
            }
        } else {
#pragma unroll
            for (int k = 0; k < IT; k += 2) {
                const i32x4 v = *(const i32x4 *)(cnt64 + i + k);
                a[k] = v[0]; b[k] = v[1]; a[k + 1] = v[2]; b[k + 1] = v[3];
            }
        }
        store_all<IT>(cnt + i, a);
        store_all<IT>(creal + i, b);
    }
};

// Homes of every cell where all entries of a cell that holds a real particle are homes.
template <typename T>
struct ProdHomes {
    static constexpr int ITEMS = SCAN_ITEMS;
    const int *cnt, *creal;
    const SysDesc<T> *sys;
    int nsys;
    bool parts;  // some system's cells are cut into parts
    // (a part is home to its entries if any part of its cell holds a real particle)
    __device__ void get(long long c, unsigned long long, int &a, int &b) const {
        a = b = 0;
        const int n = cnt[c];
        if (n == 0) return;
        bool real = creal[c] > 0;
        if (parts && !real) {
            int lo = 0, hi = nsys;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (sys[mid].cell_off <= (int)c) lo = mid;
                else hi = mid;
            }
            const DevBox<T> &bx = sys[lo].box;
            const int S = bx.sub, ncx = bx.nc[0], ny = bx.nc[1] * S;
            const int row = ((int)c - sys[lo].cell_off) / ncx, cx = (int)c - sys[lo].cell_off - row * ncx;
            const int y0 = row % ny / S * S, z0 = bx.dim == 3 ? row / ny / S * S : 0;
            for (int z = z0; z < z0 + (bx.dim == 3 ? S : 1); ++z)
                for (int y = y0; y < y0 + S; ++y) real = real || creal[sys[lo].cell_off + (z * ny + y) * ncx + cx] > 0;
        }
        if (real) a = n;
    }
    template <int IT>
    __device__ void get_all(long long c, unsigned long long u, int (&a)[IT], int (&b)[IT]) const {
        if (parts) {
#pragma unroll
            for (int k = 0; k < IT; ++k) get(c + k, u, a[k], b[k]);
            return;
        }
        load_all<IT>(cnt + c, a);
        load_all<IT>(creal + c, b);
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            a[k] = b[k] > 0 ? a[k] : 0;
            b[k] = 0;
        }
    }
};

// The same counts alone (hc[ncells] = 0, for a scan of ncells + 1).
template <typename T>
__global__ void __launch_bounds__(256) k_home_counts(int ncells, ProdHomes<T> prod, int *__restrict__ hc) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c > ncells) return;
    int a = 0, b = 0;
    if (c < ncells) prod.get(c, 0, a, b);
    hc[c] = a;
}

// Wave tasks of every system of a batch, of 2^shift homes each, where all entries of a cell
// that holds a real particle are homes.
template <typename T>
struct ProdSystems {
    static constexpr int ITEMS = SCAN_ITEMS;
    const SysDesc<T> *sys;
    const int *hstart;
    int nsys, ncells, shift;
    __device__ void get(long long k, unsigned long long, int &a, int &b) const {
        const int c1 = k + 1 < nsys ? sys[k + 1].cell_off : ncells;
        a = (hstart[c1] - hstart[sys[k].cell_off] + (1 << shift) - 1) >> shift;
        b = 0;
    }
    template <int IT>
    __device__ void get_all(long long i, unsigned long long u, int (&a)[IT], int (&b)[IT]) const {
#pragma unroll
        for (int k = 0; k < IT; ++k) get(i + k, u, a[k], b[k]);
    }
};

// Wave tasks of every row of cells (k_sweep): the row's homes / 64, rounded up.
template <typename T>
struct ProdRows {
    static constexpr int ITEMS = SCAN_ITEMS;
    const SysDesc<T> *sys;
    const int *rowoff;
    const int *hstart;
    int nsys;
    __device__ void get(long long r, unsigned long long, int &a, int &b) const {
        const int s = last_le(rowoff, 0, nsys + 1, (int)r);
        const int ncx = sys[s].box.nc[0];
        const int c0 = sys[s].cell_off + ((int)r - rowoff[s]) * ncx;
        a = (hstart[c0 + ncx] - hstart[c0] + 63) >> 6;
        b = 0;
    }
    template <int IT>
    __device__ void get_all(long long i, unsigned long long u, int (&a)[IT], int (&b)[IT]) const {
#pragma unroll
        for (int k = 0; k < IT; ++k) get(i + k, u, a[k], b[k]);
    }
};

// ------------------------------------------------------------------------------
// sweep skeleton
// ------------------------------------------------------------------------------

template <typename T>
struct SweepArgs {
    const int *hstart;
    const int *tstart;         // k_sweep: first wave task of each row
    const int *real_pos;       // entry position of every real particle, in cell order (real-home modes)
    const int *real_cell;      // its cell
    const int *rowoff;         // k_sweep: [nsys + 1] first global row of each system
    const int *systasks;       // [nsys + 1] first wave task of each system (null for one system)
    const SysDesc<T> *sys;
    int *task_counter;         // per-XCD counters (TaskQueue), zeroed before launch
    int ncells;                // cells over all systems
    int nrows;                 // rows over all systems
    int nsys;
    int nhomes;                // real-home modes: the particles
    uint32_t en_bytes;         // bytes of the neighbour entry array (buffer-load range)
    // MODE_A_TRIC (windowed sweep): the entries split by k_cell_sort into the real ones
    // (cell starts hstart) and the ghost ones (cell starts cstart - hstart)
    const Ent<T> *reals;
    const Ent<T> *ghosts;
    uint32_t reals_bytes, ghosts_bytes;
    // status block of a build not yet checked on the host (null when checked): a list
    // with an error or an overflow is not walked (the host rebuilds it and runs again)
    const uint32_t *bin_flags;
    long long e_cap;
    // the same of the neighbour set's build (two sets)
    const uint32_t *bin_flags_n;
    long long e_cap_n;
};

// Whether the cell list of sa may be walked (see SweepArgs::bin_flags).
__device__ inline bool build_usable(const uint32_t *flags, long long cap) {
    return !flags || (!(flags[0] & (FLAG_OVERFLOW | FLAG_NAN | FLAG_RANGE | FLAG_SCAN)) && (long long)flags[2] <= cap);
}
template <typename T>
__device__ inline bool list_usable(const SweepArgs<T> &sa) {
    return build_usable(sa.bin_flags, sa.e_cap) && build_usable(sa.bin_flags_n, sa.e_cap_n);
}

// The tasks of a persistent launch of one-wave workgroups.  Blocks are dealt to XCDs
// round-robin (block b runs on XCD b % 8), and each XCD walks its own contiguous share of
// the tasks (neighbouring rows share entries in that XCD's L2).  A wave's first task is
// given by its place in the grid; so are all of them when there are no more than
// FIXED_ROUNDS per wave, else the next ones come from the XCD's counter, each asked for
// while the one before is worked on, and a wave whose XCD has none left helps the others.
// Adds to one line queue, so each counter has its own, and a wave reads all of them at once
// before it helps: with the eight counters on one line, added to for every task and by every
// wave at its end, a sweep of 1000 particles took 0.57 ms against 0.04.
constexpr int TASK_COUNTERS = 8;
constexpr int TASK_COUNTER_STRIDE = 32;  // ints: one cache line
struct TaskQueue {
    static constexpr int FIXED_ROUNDS = 4;
    int *counters;
    int ntasks;
    int cur, step, end;  // the wave's fixed tasks
    int asked;           // lane 0: the answer to the request in flight
    bool own;            // its XCD's counter may have tasks (one is asked for)
    __device__ int share(int x) const { return (int)(((int64_t)ntasks * x) >> 3); }
    __device__ int waves(int x) const { return ((int)gridDim.x - x + 7) >> 3; }
    // the end of the fixed tasks of x's share
    __device__ int fixed(int x) const {
        const int lo = share(x), hi = share(x + 1), w = waves(x);
        return hi - lo <= FIXED_ROUNDS * w ? hi : lo + w;
    }
    __device__ int ask(int x) const {
        return threadIdx.x == 0 ? atomicAdd(&counters[x * TASK_COUNTER_STRIDE], 1) : 0;
    }
    __device__ TaskQueue(int *ctr, int n) : counters(ctr), ntasks(n), asked(0) {
        const int x = blockIdx.x & 7;
        step = waves(x);
        end = fixed(x);
        own = end < share(x + 1);
        cur = share(x) + (int)(blockIdx.x >> 3) - step;
    }
    // The next task; -1 when none is left (called by the whole wave).
    __device__ int next() {
        const int home = blockIdx.x & 7;
        cur += step;
        if (cur < end) {
            if (own) asked = ask(home);
            return cur;
        }
        if (own) {
            const int t = fixed(home) + uniform_int(asked);
            if (t < share(home + 1)) {
                asked = ask(home);
                return t;
            }
            own = false;
        }
        while (true) {
            const int y = threadIdx.x & 7;
            const int n = share(y + 1) - fixed(y);
            int v = n;
            if (n > 0) v = __hip_atomic_load(&counters[y * TASK_COUNTER_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t left = ballot64(threadIdx.x < 8 && v < n);
            if (left == 0) return -1;
            const uint64_t after = left >> home;  // the nearest XCD from its own on
            const int x = after ? home + (int)__builtin_ctzll(after) : (int)__builtin_ctzll(left);
            const int t = fixed(x) + uniform_int(ask(x));
            if (t < share(x + 1)) return t;
        }
    }
};

// Look-ahead batch of neighbour entries held in scalar registers.
template <typename T>
struct SweepBatch {
    static constexpr int value = sizeof(T) == 4 ? 8 : 4;
};
constexpr int SWEEP_PAD = 16;  // entries of padding after E (>= 2 * batch)

// E/cs: cell-sorted entries and cell starts of the home set; En/csn: those of the
// neighbour set (the same arrays for one set).
template <typename T, int MODE, int D, typename Op>
__global__ void __launch_bounds__(64) k_sweep(const Ent<T> *__restrict__ E, const int *__restrict__ cs,
                                              const Ent<T> *__restrict__ En, const int *__restrict__ csn,
                                              const SweepArgs<T> sa, const Op op) {
    __shared__ typename Op::Shared sh;
    if (!list_usable(sa)) return;
    const int lane = threadIdx.x;
    constexpr int B = SweepBatch<T>::value;
    typename Op::Wave ws;
    op.wave_init(sh, ws);
    TaskQueue tq(sa.task_counter, sa.tstart[sa.nrows]);
    for (int task = tq.next(); task >= 0; task = tq.next()) {
        const int r = last_le(sa.tstart, 0, sa.nrows + 1, task);
        const int si = uniform_int(last_le(sa.rowoff, 0, sa.nsys + 1, r));
        const SysDesc<T> &sd = sa.sys[si];
        const int ncx = sd.box.nc[0], ncy = sd.box.nc[1];
        const int L = sd.box.lcell;
        const T rc2 = sd.box.rc2;
        const int lr = r - sa.rowoff[si];
        const int chunk = task - sa.tstart[r];
        const int rowc0 = sd.cell_off + lr * ncx;
        const int hb = sa.hstart[rowc0] + chunk * 64;
        const int he = sa.hstart[rowc0 + ncx];
        const int h = hb + lane;
        const bool valid = h < he;
        const int c = last_le(sa.hstart, rowc0, rowc0 + ncx, valid ? h : hb);
        const int pos = mode_all_entries(MODE) ? cs[c] + ((valid ? h : hb) - sa.hstart[c]) : sa.real_pos[valid ? h : hb];
        const Ent<T> p = E[pos];
        const int cx = c - rowc0;
        const int cy = lr % ncy, cz = lr / ncy;
        const int nvalid = min(64, he - hb);
        const int cxmin = uniform_int(cx);
        const uint32_t wp = ent_w(p);
        const bool preal = !w_ghost(wp);
        typename Op::Lane ls;
        op.lane_init(ws, ls, p, valid);
        const int dzr = (D == 3) ? L : 0;
        for (int dz = -dzr; dz <= dzr; ++dz) {
            for (int dy = -L; dy <= L; ++dy) {
                const int base = sd.cell_off + ((cz + dz) * ncy + (cy + dy)) * ncx;
                int xlo = -L;
                const bool selfrow = (dz == 0 && dy == 0);
                if (MODE == MODE_A_ORTHO) xlo = (dy > 0 || (dy == 0 && dz > 0)) ? 0 : 1;
                int lo = csn[base + cx + xlo];
                int hi = csn[base + cx + L + 1];
                if (MODE == MODE_A_ORTHO && selfrow) lo = pos + 1;
                if (!valid) { lo = 0; hi = 0; }
                // MODE_X_ORTHO: entries of the same-index cell pair only with a real home
                int slo = 0, shi = 0;
                if (MODE == MODE_X_ORTHO && selfrow) { slo = csn[base + cx]; shi = csn[base + cx + 1]; }
                int J0 = uniform_int(csn[base + cxmin + (MODE == MODE_A_ORTHO && selfrow ? 0 : xlo)]);
                int J1 = uniform_int(__shfl(csn[base + cx + L + 1], nvalid - 1, 64));
                // Neighbour entries are wave-uniform: they are read with scalar loads in
                // batches of B, the next batch issued before the current one is used (E is
                // padded by 2*B entries, so the look-ahead never leaves the allocation).
                Ent<T> cur[B], nxt[B];
#pragma unroll
                for (int u = 0; u < B; ++u) cur[u] = En[J0 + u];
                for (int j0 = J0; j0 < J1; j0 += B) {
#pragma unroll
                    for (int u = 0; u < B; ++u) nxt[u] = En[j0 + B + u];
#pragma unroll
                    for (int u = 0; u < B; ++u) {
                        const int j = j0 + u;
                        if (j < J1) {
                            const Ent<T> &q = cur[u];
                            const uint32_t wq = ent_w(q);
                            const T dx = p.x - q.x, dy2 = p.y - q.y, dz2 = p.z - q.z;
                            T d2 = dx * dx + dy2 * dy2;
                            if (D == 3) d2 = d2 + dz2 * dz2;
                            bool ok = d2 <= rc2;
                            if (MODE == MODE_A_ORTHO) {
                                ok = ok && (j >= lo) && (j < hi) && (preal || !w_ghost(wq));
                            } else if (MODE == MODE_A_TRIC) {
                                ok = ok && (j >= lo) && (j < hi) && ((wp | 15u) < wq);  // index_i < index_j
                            } else if (MODE == MODE_X_ORTHO) {
                                const bool same = (j >= slo) && (j < shi);
                                ok = ok && (j >= lo) && (j < hi) && (preal || (!same && !w_ghost(wq)));
                            } else if (MODE == MODE_X_REAL) {
                                ok = ok && (j >= lo) && (j < hi);
                            } else {
                                ok = ok && valid && (wp != wq);
                            }
                            op.candidate(sh, ws, ls, ok, ballot64(ok), p, q, d2, j, 0);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < B; ++u) cur[u] = nxt[u];
                }
            }
        }
        op.template lane_end<1>(sh, ws, ls, p, valid, sd, si);
    }
    op.wave_end(sh, ws);
}

// ------------------------------------------------------------------------------
// windowed sweep
// ------------------------------------------------------------------------------
//
// Same modes and operators as k_sweep, but only the entries that can lie within the cutoff
// are visited.  For a home p and the row (dy, dz), let g be the distance from p to the
// row's slab in y and z; only points with |x - p.x| <= h = sqrt(rc^2 - g^2) can be within
// the cutoff.  The row being ordered by x (k_cell_sort), they are one contiguous window of
// it, whose two ends are found by bisection in the cells holding p.x - h and p.x + h.
// Which entries are visited never decides a pair -- the d2 <= rc^2 test and the mode filter
// do -- so the bounds are taken with a margin of 1e-3 cell sizes, far above the rounding of
// the quantities involved, and the two grid cells into which the border rule moves real
// particles are widened by a cell.
//
// G lanes share a home, 64 / G consecutive homes make a task: the lanes of a home
// find the windows of G * R stencil rows at once, then walk them, lane k taking
// every G-th entry from the k-th on.  With one lane per home a task was 64 homes and the
// sweep as long as its longest task (0.57 ms for 1000 particles on 16 of 4096 waves), each
// lane walked until the longest of 64 windows ended, and a load touched 30 cache lines; with
// G lanes the tasks are G times as many, the longest window is one of 64 / G and the lanes of
// a home load one run of entries (forces of 1000 particles: 0.72 -> 0.17 ms a call; list of
// 1e5: 0.79 -> 0.36; 1M, triclinic, lcell 2: list 1.90 -> 1.72, forces 1.96 -> 1.80).
//
// The windows go through LDS into a list for each home, the empty ones left out, and a home's
// lanes walk its list without regard to the other homes of the wave.  Row by row, all homes
// waited for the longest window of each row: 2.8 entries visited for each pair at lcell 2 and 86
// entries to a window, where the windows themselves hold 1.9.  What bounds the sweep is the
// number of visits: at 1M entries the data return of the vector cache was busy 94 % of the time
// with their 16-byte loads, and the vector units 70 % (list) to all (forces, histogram).  With
// the lists, 2.1 visits: list of 1M 1302 -> 1188 us, of 1e5 151 -> 119; forces of 1M 1438 -> 1338,
// 300k float64 878 -> 756; batch of 512 7.75 -> 6.82 ms; clustered histogram 51.0 -> 49.7 ms.
// The walk's next loads are issued whether or not there is a next step (past the end they stay
// within the buffer's range): issued under a condition, the compiler waits for them before the
// step in hand (list of 1M 1390 us, 300k float64 1017).

// Distance from coordinate v to the slab of grid row k (part k % sub of cell k / sub) along
// axis a (0 inside), with the border-rule widening and the margin.
template <bool PARTS, typename T>
__device__ inline T slab_gap(const DevBox<T> &b, int a, int k, T v, T margin) {
    const int sub = PARTS ? b.sub : 1;
    const int c = PARTS ? k / sub : k, part = k - c * sub;
    T lo = b.cbmin[a] + T(c) * b.cs[a], hi = lo + b.cs[a];
    if (PARTS) {
        const T width = b.cs[a] / T(sub);
        lo += T(part) * width;
        hi = lo + width;
    }
    lo -= margin;
    hi += margin;
    if (c == b.lcell && part == 0) lo -= b.cs[a];
    if (c == b.nc[a] - b.lcell - 1 && part == sub - 1) hi += b.cs[a];
    T g = lo - v;
    const T g2 = v - hi;
    g = g2 > g ? g2 : g;
    return g > T(0) ? g : T(0);
}

template <typename T>
__device__ inline int axis_cell(const DevBox<T> &b, int a, T v, T inv) {
    T f = dev_floor((v - b.cbmin[a]) * inv);
    const T top = T(b.nc[a]);
    f = f < T(-1) ? T(-1) : (f > top ? top : f);
    return (int)f;
}

// Neighbour entries through a raw buffer resource: 32-bit per-lane byte offsets, and a
// load past the end of the array returns zeros instead of touching memory (lanes whose
// window is exhausted keep loading without bounds arithmetic).
__device__ inline __amdgpu_buffer_rsrc_t entry_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
template <typename T>
__device__ inline Ent<T> load_entry(__amdgpu_buffer_rsrc_t r, uint32_t off);
template <>
__device__ inline Ent<float> load_entry<float>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(Ent<float>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
template <>
__device__ inline Ent<double> load_entry<double>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    struct Two { __attribute__((ext_vector_type(4))) unsigned a, b; };
    Two t;
    t.a = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    t.b = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16u, 0, 0);
    return __builtin_bit_cast(Ent<double>, t);
}

template <typename T>
__device__ inline T load_entry_x(__amdgpu_buffer_rsrc_t r, uint32_t off);
template <>
__device__ inline float load_entry_x<float>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
template <>
__device__ inline double load_entry_x<double>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}

template <typename T>
__device__ inline T window_sqrt(T v);
template <>
__device__ inline float window_sqrt<float>(float v) { return __builtin_amdgcn_sqrtf(v); }
template <>
__device__ inline double window_sqrt<double>(double v) { return __builtin_sqrt(v); }

// U: entries each lane tests per step (and as many in flight): the group width of the
// sweep's tile, a launch-shape knob of the autotuner.  Two keep the neighbour list at 96
// registers, five waves to a SIMD (with 4, walking row by row: list of 1M 1561 us against 1473,
// forces 1520 against 1433, clustered histogram 58.7 ms against 52.6); a step of 2 G entries
// shares the bookkeeping of the walk, at 5 % more visits.
constexpr int SWEEP_GROUP = 2;
// A run of entries that a home's lanes walk: the byte of its first, and how many more; and the
// mark after a home's last one.
struct alignas(8) Window {
    uint32_t first;
    int count;
};
constexpr int WINDOWS_END = -(1 << 30);
// PARTS: the cells are cut into parts (DevBox::sub > 1; a template parameter so that the kernel
// for whole cells carries no registers for it).  Five waves to a SIMD are asked for at float32
// (the adjoint over parts: 414 us against 464 with four).
template <typename T, int MODE, int D, typename Op, int G, int U, bool PARTS>
__global__ void __launch_bounds__(64, sizeof(T) == 4 && U == SWEEP_GROUP ? 5 : 1) k_sweep_win(const Ent<T> *__restrict__ E, const int *__restrict__ cs,
                                                  const Ent<T> *__restrict__ En, const int *__restrict__ csn,
                                                  const SweepArgs<T> sa, const Op op) {
    constexpr int H = 64 / G;             // homes of a task
    constexpr int R = G >= 32 ? 1 : 2;    // rows whose windows a lane finds at a time
    // windows begin at a multiple of A entries where their row allows it, so that a load of four lanes is
    // one aligned piece of 64 bytes: forces of 1M 1202 -> 1178 us, batch of 512 6.51 -> 6.38 ms; with the
    // operators that visit a pair once (list of 1M 1194 -> 1221 us) and 8 lanes the extra visits cost more
    constexpr int A = MODE == MODE_B && G == 4 && sizeof(T) == 4 ? 4 : 1;
    constexpr int CAP = Op::WINDOWS > G * R ? Op::WINDOWS : G * R;  // rows of a list of windows
    constexpr int STRIDE = CAP + 3;       // (odd: the homes' windows in different banks)
    __shared__ typename Op::Shared sh;
    __shared__ Window windows[H * STRIDE];
    if (!list_usable(sa)) return;
    const int lane = threadIdx.x;
    const int sub = lane & (G - 1), g0 = lane & ~(G - 1);
    typename Op::Wave ws;
    op.wave_init(sh, ws);
    // MODE_A_TRIC walks two arrays (the real entries, the ghost entries), the others one
    constexpr bool SPLIT = MODE == MODE_A_TRIC;
    const __amdgpu_buffer_rsrc_t rs_main = SPLIT ? entry_rsrc(sa.reals, sa.reals_bytes) : entry_rsrc(En, sa.en_bytes);
    const __amdgpu_buffer_rsrc_t rs_ghost = SPLIT ? entry_rsrc(sa.ghosts, sa.ghosts_bytes) : rs_main;
    // tasks: H consecutive homes of a system each
    const int nhomes = mode_all_entries(MODE) ? sa.hstart[sa.ncells] : sa.nhomes;
    TaskQueue tq(sa.task_counter, sa.nsys > 1 ? sa.systasks[sa.nsys] : (nhomes + H - 1) / H);
    for (int task = tq.next(); task >= 0; task = tq.next()) {
        const int si = sa.nsys > 1 ? uniform_int(wave_last_le(sa.systasks, 0, sa.nsys + 1, task)) : 0;
        const SysDesc<T> &sd = sa.sys[si];
        const DevBox<T> &bx = sd.box;
        const int S = PARTS ? bx.sub : 1;
        const int ncx = bx.nc[0], ncy = bx.nc[1] * S;  // rows of the grid along y
        const int L = bx.lcell;
        const T rc2 = bx.rc2;
        int hb = task * H, he = nhomes;
        if (sa.nsys > 1) {
            // (the homes of a system are its particles, or all entries of its real cells)
            const int h0 = mode_all_entries(MODE) ? sa.hstart[sd.cell_off] : sd.pos_off;
            hb = h0 + (task - sa.systasks[si]) * H;
            he = mode_all_entries(MODE) ? sa.hstart[sd.cell_off + ncx * grid_rows(bx)] : h0 + sd.n;
        }
        const bool valid = hb + lane / G < he;
        const int h = valid ? hb + lane / G : hb;
        int c, pos;  // the home's cell and entry
        if (mode_all_entries(MODE)) {
            c = wave_last_le(sa.hstart, 0, sa.ncells, hb);
            // the next homes lie a few cells on, or past the empty cells between two rows
            for (int k = 0; sa.hstart[c + 1] <= h; ++k) {
                if (k == 4) {
                    c = last_le(sa.hstart, c, sa.ncells, h);
                    break;
                }
                ++c;
            }
            pos = cs[c] + (h - sa.hstart[c]);
        } else {
            c = sa.real_cell[h];
            pos = sa.real_pos[h];
        }
        const Ent<T> p = E[pos];
        const int lr = (c - sd.cell_off) / ncx;  // its row of cells
        const int cx = c - sd.cell_off - lr * ncx;
        const int cy = lr % ncy, cz = lr / ncy;
        const uint32_t wp = ent_w(p);
        const uint32_t wpx = wp | 15u;  // for a real home: index_p < index_q <=> wpx < wq
        const bool preal = !w_ghost(wp);
        const uint64_t preal_mask = ballot64(preal);
        const int home = lane / G;
        const uint32_t sub_bytes = (uint32_t)sub * (uint32_t)sizeof(Ent<T>);
        const T mx = T(1e-3) * bx.cs[0], my = T(1e-3) * bx.cs[1], mz = T(1e-3) * bx.cs[2];
        const T invx = T(1) / bx.cs[0];
        // the stencil: `side` rows along y (and z) from row y0 (z0) on; qown is the number of
        // the home's own one
        const int side = S * (2 * L + 1);
        const int nrow = D == 3 ? side * side : side;
        const int yc = PARTS ? cy / S : cy, zc = D == 3 && PARTS ? cz / S : cz;  // the home's cell
        const int y0 = S * (yc - L), z0 = D == 3 ? S * (zc - L) : 0;
        const int qown = (D == 3 ? (cz - z0) * side : 0) + cy - y0;
        // MODE_X_ORTHO: whether entry j lies in the cell of the home's index (any part of it)
        auto in_own_cell = [&](int j) -> bool {
            bool in = false;
            for (int kz = 0; kz < (D == 3 ? S : 1); ++kz)
                for (int ky = 0; ky < S; ++ky) {
                    const int k = sd.cell_off + ((zc * S + kz) * ncy + yc * S + ky) * ncx + cx;
                    in = in || (j >= csn[k] && j < csn[k + 1]);
                }
            return in;
        };
        typename Op::Lane ls;
        op.lane_init(ws, ls, p, valid);
        // PASS 0: the entries of E (or, SPLIT, the real entries); PASS 1 (SPLIT only): the
        // ghost entries
        auto walk = [&](auto pass_tag) {
            constexpr int PASS = decltype(pass_tag)::value;
            const __amdgpu_buffer_rsrc_t rr = PASS == 1 ? rs_ghost : rs_main;
            auto start = [&](int k) -> int {
                if (!SPLIT) return csn[k];
                if (PASS == 0) return sa.hstart[k];
                return csn[k] - sa.hstart[k];
            };
            auto load_x = [&](int k) -> T { return load_entry_x<T>(rr, (uint32_t)k * (uint32_t)sizeof(Ent<T>)); };
            // SPLIT real entries: the half stencil that orders pairs by position (the rows
            // from the own one on, and the own row from the home on); no home's own row comes
            // before number `half`
            const int half = S * L * (D == 3 ? side + 1 : 1);
            for (int q0 = SPLIT && PASS == 0 ? half : 0; q0 < nrow; q0 += CAP) {
                const int qe = min(q0 + CAP, nrow);
                int nw = 0, steps = 0;  // the home's windows; the lane's share of their steps
                __syncthreads();
                for (int qb = q0; qb < qe; qb += G * R) {
                    // the windows of rows qb + k G + sub
                    int j0[R], j1[R], b0[R], b1[R], low[R];
                    T xb[R], xe[R];
#pragma unroll
                    for (int k = 0; k < R; ++k) {
                        const int q = qb + k * G + sub;
                        const int qz = D == 3 ? z0 + q / side : 0;
                        const int qy = y0 + (D == 3 ? q % side : q);
                        const bool own = q == qown;
                        const int row = sd.cell_off + (qz * ncy + qy) * ncx;
                        const T gz = D == 3 ? slab_gap<PARTS>(bx, 2, qz, p.z, mz) : T(0);
                        const T gy = slab_gap<PARTS>(bx, 1, qy, p.y, my);
                        const T r2 = rc2 - gy * gy - gz * gz;
                        j0[k] = j1[k] = b0[k] = b1[k] = low[k] = 0;
                        xb[k] = xe[k] = p.x;
                        if (valid && q < qe && r2 >= T(0) && !(SPLIT && PASS == 0 && q < qown)) {
                            // the cells that hold the window's ends, within the stencil
                            const T hw = window_sqrt(r2) + mx;
                            int ka = axis_cell(bx, 0, p.x - hw, invx);
                            int kb = axis_cell(bx, 0, p.x + hw, invx);
                            if (kb == L - 1) kb = L;
                            if (ka == ncx - L) ka = ncx - L - 1;
                            int xlo = -L;
                            if (MODE == MODE_A_ORTHO) {
                                // the forward cells; of the own cell the parts from the own one on
                                const int dy = (PARTS ? qy / S : qy) - yc, dz = (D == 3 && PARTS ? qz / S : qz) - zc;
                                xlo = (dy > 0 || (dy == 0 && (dz > 0 || (dz == 0 && q >= qown)))) ? 0 : 1;
                            }
                            if (SPLIT && PASS == 0 && own) xlo = 0;
                            ka = max(ka, cx + xlo);
                            kb = min(kb, cx + L);
                            if (ka <= kb) {
                                j0[k] = low[k] = start(row + ka);
                                j1[k] = start(row + ka + 1);
                                b0[k] = start(row + kb);
                                b1[k] = start(row + kb + 1);
                                xb[k] = p.x - hw - mx;
                                xe[k] = p.x + hw + mx;
                            }
                        }
                    }
                    // both ends of every window by bisection on x, all in step: the first entry
                    // of [j0, j1) at or past xb, the first of [b0, b1) past xe
                    while (true) {
                        bool open = false;
#pragma unroll
                        for (int k = 0; k < R; ++k) open = open || j0[k] < j1[k] || b0[k] < b1[k];
                        if (ballot64(open) == 0) break;
                        T va[R], vb[R];
#pragma unroll
                        for (int k = 0; k < R; ++k) {
                            va[k] = load_x((j0[k] + j1[k]) >> 1);
                            vb[k] = load_x((b0[k] + b1[k]) >> 1);
                        }
#pragma unroll
                        for (int k = 0; k < R; ++k) {
                            const int ma = (j0[k] + j1[k]) >> 1, mb = (b0[k] + b1[k]) >> 1;
                            if (j0[k] < j1[k]) {
                                if (va[k] < xb[k]) j0[k] = ma + 1;
                                else j1[k] = ma;
                            }
                            if (b0[k] < b1[k]) {
                                if (vb[k] <= xe[k]) b0[k] = mb + 1;
                                else b1[k] = mb;
                            }
                        }
                    }
#pragma unroll
                    for (int k = 0; k < R; ++k) {
                        if (qb + k * G + sub == qown) {  // the own row
                            if (MODE == MODE_A_ORTHO) low[k] = max(low[k], pos + 1);
                            if (SPLIT && PASS == 0) low[k] = max(low[k], h + 1);
                            j0[k] = max(j0[k], low[k]);
                        }
                        // (the entries before a window in its row lie outside the cutoff)
                        if (A > 1 && j0[k] < b0[k]) j0[k] = max(j0[k] & ~(A - 1), low[k]);
                        const int len = b0[k] - j0[k];
                        // (in the order of the rows, the empty ones left out)
                        const uint64_t full = (ballot64(len > 0) >> g0) & (G == 64 ? ~0ull : (1ull << G) - 1);
                        if (len > 0) {
                            windows[home * STRIDE + nw + __popcll(full & ((1ull << sub) - 1))] = Window{(uint32_t)j0[k] * (uint32_t)sizeof(Ent<T>), len - 1};
                            steps += (len + U * G - 1) / (U * G);
                        }
                        nw += __popcll(full);
                    }
                }
                if (sub == 0) windows[home * STRIDE + nw] = Window{sa.en_bytes, WINDOWS_END};
                for (int off = 1; off < G; off <<= 1) steps += __shfl_xor(steps, off, 64);
                for (int off = G; off < 64; off <<= 1) steps = max(steps, __shfl_xor(steps, off, 64));
                const int trips = uniform_int(steps);  // of the home with the most
                // the loads of these rows have arrived (the bisection waited for them)
                op.row_sync(ws);
                __syncthreads();
                // The lane's place: the next entry is at byte `at` of its home's window, of which
                // `rest` + 1 entries are left for the home's lanes; a step is a group of U entries
                // of each lane, and the next window is read ahead of its use.
                const Window *w = windows + home * STRIDE;
                Window nxt = w[0];
                w += 1;
                uint32_t at = nxt.first + sub_bytes;
                int rest = nxt.count;
                nxt = *w;
                struct Group {
                    Ent<T> e[U];
                    uint32_t at;
                    uint64_t act[U];  // the lanes with an entry
                };
                auto load = [&](Group &g) {
                    g.at = at;
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        g.e[u] = load_entry<T>(rr, at + (uint32_t)(u * G * sizeof(Ent<T>)));
                        g.act[u] = ballot64(rest >= sub + u * G);
                    }
                    const bool last = (uint32_t)rest < (uint32_t)(U * G);  // (the end mark is negative)
                    at = last ? nxt.first + sub_bytes : at + (uint32_t)(U * G * sizeof(Ent<T>));
                    rest = last ? nxt.count : rest - U * G;
                    w = last ? w + 1 : w;
                    nxt = *w;
                };
                // one group of U entries
                auto group = [&](const Group &g) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const Ent<T> &e = g.e[u];
                        const int j = (int)(g.at / (uint32_t)sizeof(Ent<T>)) + u * G;
                        const uint32_t wq = ent_w(e);
                        const T dx = p.x - e.x, dy2 = p.y - e.y, dz2 = p.z - e.z;
                        T d2 = dx * dx + dy2 * dy2;
                        if (D == 3) d2 = d2 + dz2 * dz2;
                        // the wave's mask of the pairs, from the ballots of the single
                        // comparisons; the lanes' flags are read back from it
                        uint64_t m = g.act[u] & ballot64(d2 <= rc2);
                        if (MODE == MODE_A_ORTHO) {
                            if (preal_mask != ~0ull) m &= preal_mask | ballot64(!w_ghost(wq));
                        } else if (MODE == MODE_A_TRIC) {
                            if (PASS == 1) m &= ballot64(wpx < wq);
                        } else if (MODE == MODE_X_ORTHO) {
                            // entries of the same-index cell pair only with a real home
                            if (preal_mask != ~0ull) m &= preal_mask | ballot64(!in_own_cell(j) && !w_ghost(wq));
                        } else if (MODE == MODE_B) {
                            m &= ballot64(wp != wq);
                        }
                        const bool ok = inverse_ballot(m);
                        op.candidate(sh, ws, ls, ok, m, p, e, d2, j, PASS);
                    }
                };
                // two buffers used in turn (no register copies): while one group is tested
                // the next one is in flight
                Group ga, gb;
                load(ga);
                for (int t = 0; t < trips; t += 2) {
                    load(gb);
                    group(ga);
                    if (t + 1 >= trips) break;
                    load(ga);
                    group(gb);
                }
            }
        };
        walk(std::integral_constant<int, 0>{});
        // SPLIT: each pair of real particles from the one earlier in the cell order; each
        // pair with a ghost image from the home of the lower index (the reference's rule),
        // over the full stencil
        if (SPLIT) walk(std::integral_constant<int, 1>{});
        op.template lane_end<G>(sh, ws, ls, p, valid, sd, si);
    }
    op.wave_end(sh, ws);
}

// ------------------------------------------------------------------------------
// operators
// ------------------------------------------------------------------------------

// Neighbour list (push_pair!, internals/neighborlist.jl:67-76).  Hits are staged in
// LDS and written out in coalesced blocks.  Output space is handed out in chunks of CH
// slots: a wave owns one chunk at a time and requests the next one with a single
// device-scope atomic issued well before it is needed, so the atomic's latency is hidden
// and there are ~P/CH atomics instead of one per flush.  The atomics are spread over
// NL_COUNTERS counters on separate cache lines (one address serialises them, ~13 ns
// each): counter k hands out the chunks k, k + K, k + 2K, ..., and a wave takes its
// successive requests from successive counters, so the counters advance evenly.  Slots at
// or beyond the caller's capacity go to a library-owned spill area (a slot past it sets
// an overflow word).  Partially used chunks and chunks never handed out below the pair
// count leave holes; k_scan_pair<ProdHoles> / k_nl_fill move entries from beyond the pair count into
// them, so the final list is dense (its order is unspecified, as in the reference).
// Slots of a chunk in a long list; short lists take smaller ones.  A flush of ~450 pairs then
// mostly lies in one chunk, and chunks are asked for a quarter as often as with 512 slots (1M
// float32: the sweep 1341 us against 1511, with 5M entries to move at the end against 2.4M;
// 4096: 1319 us, but 20 us more of moving).
constexpr int NL_CHUNK = 2048;
constexpr int NL_COUNTERS = 64;
constexpr int NL_COUNTER_STRIDE = 16;  // u64 words between counters (128 B)

template <typename T>
using vec4 = T __attribute__((ext_vector_type(4)));

template <typename T>
struct NLOut {
    int32_t *oi, *oj;
    T *od;
    int32_t *si, *sj;
    T *sd;
    long long cap, scap;
    unsigned int *overflow;  // set when a slot lies beyond the spill area (its pair is dropped)
    __device__ void put(long long s, int i, int j, T d) const {
        const bool u = s < cap;
        const long long q = u ? s : s - cap;
        int32_t *pi = u ? oi : si;
        int32_t *pj = u ? oj : sj;
        T *pd = u ? od : sd;
        if (u || q < scap) {
            __builtin_nontemporal_store(i, pi + q);
            __builtin_nontemporal_store(j, pj + q);
            __builtin_nontemporal_store(d, pd + q);
        } else {
            atomicOr(overflow, 1u);
        }
    }
    // The wave's staged pairs li/lj/ld2[0, m) (li: indices, lj: entry words) into the
    // consecutive slots [s, s + m) (s and m wave-uniform): the run lies in the caller's arrays or in the spill area as a
    // whole, so the destination is chosen once per run; only a run across the end of
    // either takes the per-slot path.  ordered: each pair as (lower index, higher index).
    // The list is far larger than the caches and not read again by the sweep, so it is
    // written with streaming (non-temporal) stores.
    __device__ void put_run(long long s, int m, const int *li, const int *lj, const T *ld2, bool ordered) const {
        int32_t *pi, *pj;
        T *pd;
        if (s + m <= cap) {
            pi = oi + s; pj = oj + s; pd = od + s;
        } else if (s >= cap && s - cap + m <= scap) {
            pi = si + (s - cap); pj = sj + (s - cap); pd = sd + (s - cap);
        } else {
            for (int t = threadIdx.x; t < m; t += 64) {
                int a = li[t], b = (int)w_idx((uint32_t)lj[t]);
                if (ordered) {
                    const int lo = min(a, b);
                    b = max(a, b);
                    a = lo;
                }
                put(s + t, a, b, dev_sqrt_rn(ld2[t]));
            }
            return;
        }
        // Four consecutive slots per lane and store where the slot and the three arrays
        // allow 16-byte stores: a wave's store instruction then carries 256 values, not
        // 64 (a quarter of the store instructions).  The staged arrays are 16-byte aligned
        // in LDS at every run start (runs start at multiples of 32 slots there).
        const bool wide = ((s & 3) == 0) && ((((uintptr_t)pi) | ((uintptr_t)pj) | ((uintptr_t)pd)) & 15) == 0;
        const int m4 = wide ? (m & ~3) : 0;
        // (the indices, then the distances: fewer registers held at once, as this runs in
        // the middle of the sweep's loop)
        for (int t = 4 * (int)threadIdx.x; t < m4; t += 256) {
            i32x4 a4 = *(const i32x4 *)(li + t);
            i32x4 b4 = *(const i32x4 *)(lj + t);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int a = a4[e], b = (int)w_idx((uint32_t)b4[e]);
                a4[e] = ordered ? min(a, b) : a;
                b4[e] = ordered ? max(a, b) : b;
            }
            __builtin_nontemporal_store(a4, (i32x4 *)(pi + t));
            __builtin_nontemporal_store(b4, (i32x4 *)(pj + t));
            asm volatile("" ::: "memory");
            vec4<T> d4 = *(const vec4<T> *)(ld2 + t);
            bool tiny = false;
#pragma unroll
            for (int e = 0; e < 4; ++e) tiny = tiny || !(d4[e] >= T(SQRT_FAST_MIN));
            const bool fast = sizeof(T) == 4 && ballot64(tiny) == 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) d4[e] = fast ? sqrt_short(d4[e]) : dev_sqrt_rn(d4[e]);
            __builtin_nontemporal_store(d4, (vec4<T> *)(pd + t));
        }
        for (int t = m4 + threadIdx.x; t < m; t += 64) {
            int a = li[t], b = (int)w_idx((uint32_t)lj[t]);
            if (ordered) {
                const int lo = min(a, b);
                b = max(a, b);
                a = lo;
            }
            const T d2 = ld2[t];
            T d;
            if constexpr (sizeof(T) == 4) {  // the short form unless a lane's d2 is tiny (or 0)
                if (ballot64(!(d2 >= SQRT_FAST_MIN)) == 0) d = sqrt_rn_above_tiny(d2);
                else d = dev_sqrt_rn(d2);
            } else {
                d = dev_sqrt_rn(d2);
            }
            __builtin_nontemporal_store(a, pi + t);
            __builtin_nontemporal_store(b, pj + t);
            __builtin_nontemporal_store(d, pd + t);
        }
    }
    // the float32 short square root where the caller has checked d2 >= SQRT_FAST_MIN
    // (float64 always takes the full one)
    __device__ static T sqrt_short(T d2) {
        if constexpr (sizeof(T) == 4) return sqrt_rn_above_tiny(d2);
        else return dev_sqrt_rn(d2);
    }
    __device__ void get(long long s, int &i, int &j, T &d) const {
        const bool u = s < cap;
        const long long q = u ? s : s - cap;
        const int32_t *pi = u ? oi : si;
        const int32_t *pj = u ? oj : sj;
        const T *pd = u ? od : sd;
        i = pi[q]; j = pj[q]; d = pd[q];
    }
};

__device__ inline unsigned long long uniform_u64(unsigned long long v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

template <typename T>
struct OpNeighborList {
    static constexpr int WINDOWS = 16;  // rows of a list of windows: with the staged pairs, LDS for five waves to a SIMD
    static constexpr int S = 512;
    static constexpr int PREFETCH = 256;
    // 16-byte aligned: a flush reads four slots per lane with 16-byte LDS loads
    struct alignas(16) Shared {
        int i[S];
        int j[S];
        T d2[S];
    };
    struct Lane {};
    struct Wave {  // wave-uniform state carried across tasks
        int staged;  // hits staged in LDS
        int cur_used;
        long long cur;
        unsigned long long nxt_raw;  // lane 0 holds the pending atomic result
        unsigned long long written;
        int nxt_k;                   // counter of the pending request
        int req;                     // requests made so far
        bool have_nxt;
        bool nxt_ready;              // the pending request's chunk is known (nxt_val)
        long long nxt_val;
    };
    NLOut<T> out;
    unsigned long long *chunk_counter;  // NL_COUNTERS counters, NL_COUNTER_STRIDE words apart
    unsigned long long *total;  // NL_COUNTERS counts, NL_COUNTER_STRIDE words apart, whose sum is the pair count
    int *chunk_used;
    long long max_chunks;
    int chunk;    // slots of a chunk (a multiple of 32)
    int ordered;  // write each pair as (lower index, higher index)

    __device__ void request(Wave &w) const {
        const int k = (int)((blockIdx.x + (unsigned)w.req) % NL_COUNTERS);
        w.nxt_raw = threadIdx.x == 0 ? atomicAdd(&chunk_counter[k * NL_COUNTER_STRIDE], 1ull) : 0ull;
        w.nxt_k = k;
        w.req += 1;
        w.have_nxt = true;
        w.nxt_ready = false;
    }
    __device__ long long granted(const Wave &w) const {
        if (w.nxt_ready) return w.nxt_val;
        return (long long)uniform_u64(w.nxt_raw) * NL_COUNTERS + w.nxt_k;
    }
    // Called by the sweep once the loads that start a row have arrived: vector memory
    // operations complete in issue order, so a pending request issued before them is
    // complete as well, and reading its result here costs no wait of its own.
    __device__ void row_sync(Wave &w) const {
        if (w.have_nxt && !w.nxt_ready) {
            w.nxt_val = (long long)uniform_u64(w.nxt_raw) * NL_COUNTERS + w.nxt_k;
            w.nxt_ready = true;
        }
    }
    __device__ void wave_init(Shared &, Wave &w) const {
        w.staged = 0;
        w.cur = -1;
        w.cur_used = chunk;
        w.written = 0;
        w.nxt_raw = 0;
        w.nxt_k = 0;
        w.req = 0;
        w.have_nxt = false;  // the first chunk is requested at the first flush
        w.nxt_ready = false;
        w.nxt_val = 0;
    }
    __device__ void lane_init(Wave &, Lane &, const Ent<T> &, bool) const {}
    __device__ void retire(const Wave &w, int used) const {
        if (w.cur >= 0 && w.cur < max_chunks && threadIdx.x == 0) chunk_used[w.cur] = used;
    }
    // Writes the first n staged pairs, rounded down to a multiple of 32 unless all: chunks
    // hold 64 to 2048 slots, so every run then starts and ends on whole cache lines
    // of each output array.  The pairs left over (fewer than 32) move to the front of the
    // staging arrays; returns their count.
    __device__ int flush(Shared &sh, Wave &w, int n, bool all) const {
        const int r = all ? 0 : (n & 31);
        n -= r;
        __syncthreads();
        int k = 0;
        while (k < n) {
            if (w.cur_used == chunk) {
                retire(w, chunk);
                if (!w.have_nxt) request(w);
                w.cur = granted(w);
                w.cur_used = 0;
                w.have_nxt = false;
            }
            const int m = min(n - k, chunk - w.cur_used);
            const long long base = w.cur * chunk + w.cur_used;
            out.put_run(base, m, sh.i + k, sh.j + k, sh.d2 + k, ordered != 0);
            w.cur_used += m;
            k += m;
        }
        w.written += (unsigned long long)n;
        // the next chunk is requested when few slots remain: a request left unused when the
        // wave ends leaves a chunk of holes for k_nl_fill, so it is made as late as still hides
        // its latency
        if (!w.have_nxt && !all && w.cur_used > chunk - min(chunk / 2, PREFETCH)) request(w);
        __syncthreads();
        if (r > 0) {  // n >= 32 > r here: the source and destination do not overlap
            const int t = threadIdx.x;
            int a = 0, b = 0;
            T d = T(0);
            if (t < r) { a = sh.i[n + t]; b = sh.j[n + t]; d = sh.d2[n + t]; }
            __syncthreads();
            if (t < r) { sh.i[t] = a; sh.j[t] = b; sh.d2[t] = d; }
            __syncthreads();
        }
        return r;
    }
    __device__ void candidate(Shared &sh, Wave &w, Lane &, bool ok, uint64_t m, const Ent<T> &p, const Ent<T> &q,
                              T d2, int, int) const {
        if (ok) {
            const int k = w.staged + rank_in(m);
            sh.i[k] = (int)w_idx(ent_w(p));
            sh.j[k] = (int)ent_w(q);  // the entry word: its index is taken at the flush
            sh.d2[k] = d2;
        }
        w.staged += __popcll(m);
        // (rarely true: the flush is laid out off the candidate path)
        if (__builtin_expect(w.staged > S - 64, 0)) {
            w.staged = flush(sh, w, w.staged, false);
        }
    }
    template <int G>
    __device__ void lane_end(Shared &, Wave &, Lane &, const Ent<T> &, bool, const SysDesc<T> &, int) const {}
    __device__ void wave_end(Shared &sh, Wave &w) const {
        if (w.staged > 0) flush(sh, w, w.staged, true);
        if (w.cur >= 0) retire(w, w.cur_used);
        if (w.have_nxt) {
            const long long nx = granted(w);
            if (nx < max_chunks && threadIdx.x == 0) chunk_used[nx] = 0;
        }
        // (adds to one word queue, ~15 ns each, as the counters of the chunks; for a list of 20000
        // particles one word for all waves took as long: they do not end together)
        if (threadIdx.x == 0 && w.written) atomicAdd(&total[(blockIdx.x % NL_COUNTERS) * NL_COUNTER_STRIDE], w.written);
    }
};

// Per chunk of the neighbour-list output: holes below the pair count P (the uniform
// value) and entries at or beyond P (movers); none when P exceeds the capacity.
struct ProdHoles {
    static constexpr int ITEMS = 8;
    const int *used;
    long long cap;
    int chunk;
    __device__ void get(long long c, unsigned long long total, int &a, int &b) const { count(c, used[c], total, a, b); }
    template <int IT>
    __device__ void get_all(long long c, unsigned long long total, int (&a)[IT], int (&b)[IT]) const {
        int u[IT];
        load_all<IT>(used + c, u);
#pragma unroll
        for (int k = 0; k < IT; ++k) count(c + k, u[k], total, a[k], b[k]);
    }
    __device__ void count(long long c, int n, unsigned long long total, int &a, int &b) const {
        const long long P = (long long)total;
        a = 0;
        b = 0;
        if (P > cap) return;
        const long long start = c * chunk, vend = start + n;
        if (vend < P) a = (int)(min(start + chunk, P) - vend);
        if (vend > P) b = (int)(vend - max(start, P));
    }
};

// The chunk of element k of a scan st (non-decreasing, st[nchunks] = the total) for the
// wave's elements [kw, klast] (kw, klast wave-uniform, kw <= k <= klast < st[nchunks]);
// c: a chunk at or before kw's, moved on to it.  A search only past the end of a chunk.
__device__ inline long long chunk_of_wave(const int *__restrict__ st, long long nchunks, long long &c, long long kw,
                                          long long k, long long klast) {
    long long nxt = (long long)uniform_int(st[c + 1]);  // the first element past chunk c
    if (nxt <= kw) {
        c = wave_last_le64(st, c + 1, nchunks, kw);
        nxt = (long long)uniform_int(st[c + 1]);
    }
    long long mine = c, at = c;
    while (nxt <= klast) {  // at rises on every pass, and st[nchunks] > klast
        at = wave_last_le64(st, at + 1, nchunks, nxt);
        if (k >= nxt) mine = at;
        nxt = (long long)uniform_int(st[at + 1]);
    }
    return mine;
}

// Moves the entries at or beyond the pair count P (the movers) into the holes below it:
// hole k (in the order of hstart) takes mover k (in the order of mstart).  Each wave
// moves runs of up to 256 consecutive entries (64 where there are few): the chunks of a run's
// first entry are searched for, the next ones are mostly the same (long lists: holes of ~1000
// slots; 1M: 54 us for 5M moves, 90 with a search for every 64).
template <typename T>
__global__ void __launch_bounds__(256) k_nl_fill(long long nchunks, int chunk, const int *__restrict__ used,
                                                 const int *__restrict__ hstart, const int *__restrict__ mstart,
                                                 const unsigned long long *__restrict__ total, NLOut<T> out) {
    const long long H = hstart[nchunks];
    const long long P = (long long)*total;
    const int lane = threadIdx.x & 63;
    const long long threads = (long long)gridDim.x * blockDim.x;
    const int runs = (int)min(4ll, H / threads + 1);
    const long long stride = threads * runs;
    for (long long kr = (long long)uniform_u64((unsigned long long)(((long long)blockIdx.x * blockDim.x + (threadIdx.x - lane)) * runs));
         kr < H; kr += stride) {
        long long cm0 = 0, ch0 = 0;
        for (int r = 0; r < runs; ++r) {
            const long long kw = kr + 64 * r;
            if (kw >= H) break;
            const long long k = kw + lane;
            const long long klast = min(kw + 63, H - 1);
            const long long cm = chunk_of_wave(mstart, nchunks, cm0, kw, k, klast);
            const long long ch = chunk_of_wave(hstart, nchunks, ch0, kw, k, klast);
            if (k >= H) continue;
            const long long src = max(cm * chunk, P) + (k - mstart[cm]);
            const long long dst = ch * chunk + used[ch] + (k - hstart[ch]);
            if (src < 0 || dst < 0 || src >= out.cap + out.scap) continue;  // only after a failed scan
            int i, j;
            T d;
            out.get(src, i, j, d);
            out.put(dst, i, j, d);
        }
    }
}

// Pair-potential parameters for the device: pair tables of eps_ij and sigma_ij^2 (LB
// mixing) and the form constants of u = eps_ij [s^6 - c s^3], s = sigma_ij^2/(d2 + a):
// soft-core a = 1, c = 1; Lennard-Jones (r_min form) a = 0, c = 2.
template <typename T>
struct SoftParams {
    T eps[64];
    T sig2[64];
    T isig[64];  // 1 / sigma of the pair (the adjoint's dE/dsigma takes e * w / sigma)
    T eps_t[8];
    T a, c, c3;  // c3 = 3c
    int ntypes;  // 0 = untyped (table entry 0)
};

constexpr int ACC_SLOTS = 16;
constexpr int ACC_STRIDE = 16;  // doubles: one cache line

// Energy (+ forces, + parameter adjoint) of a pair potential; in mode B the lanes of a home
// own one real particle and take u/2 per visit.
template <typename T, bool FORCES, bool ADJ, bool TYPED>
struct OpSoftCore {
    static constexpr int WINDOWS = 32;  // rows of a list of windows
    struct Shared {
        double gde[8];
        double gds[8];
        T eps[64], sig2[64], isig[64];  // pair tables, read with a per-lane index
    };
    struct Lane {
        T fx, fy, fz;
        T e;
        T aeps, asig;
        int ti;
    };
    SoftParams<T> prm;
    T *forces;            // n*D, input frame
    // The sums of all waves: energies per system; per-type gradients, deps then dsig (ADJ).
    // Of one system the waves add to ACC_SLOTS copies, ACC_STRIDE doubles apart, that the
    // host sums: adds to one address queue at ~13 ns each, and every wave makes one.
    double *energy, *grad;
    int nsys;
    double escale;        // weight of a home's pair energies: 1/2 when every pair is seen twice
    int dim;

    struct Wave {
        T e0, s20, is0;   // the untyped pair parameters, in registers for the whole sweep
        double e;         // the lane's energy over the tasks of system si
        int si;
    };
    __device__ void wave_init(Shared &sh, Wave &w) const {
        w.e0 = prm.eps[0];
        w.s20 = prm.sig2[0];
        w.is0 = prm.isig[0];
        w.e = 0;
        w.si = 0;
        if (threadIdx.x < 8) { sh.gde[threadIdx.x] = 0; sh.gds[threadIdx.x] = 0; }
        sh.eps[threadIdx.x] = prm.eps[threadIdx.x];
        sh.sig2[threadIdx.x] = prm.sig2[threadIdx.x];
        sh.isig[threadIdx.x] = prm.isig[threadIdx.x];
        __syncthreads();
    }
    __device__ void add_energy(Wave &w) const {
        const double e = wave_sum(w.e);
        if (threadIdx.x == 0 && e != 0.0)
            atomicAdd(&energy[nsys > 1 ? w.si : (int)(blockIdx.x % ACC_SLOTS) * ACC_STRIDE], e);
        w.e = 0;
    }
    __device__ void lane_init(Wave &, Lane &l, const Ent<T> &p, bool) const {
        l.fx = l.fy = l.fz = T(0);
        l.e = T(0);
        l.aeps = l.asig = T(0);
        l.ti = TYPED ? (int)w_type(ent_w(p)) : 0;
    }
    __device__ void candidate(Shared &sh, Wave &ws, Lane &l, bool ok, uint64_t, const Ent<T> &p, const Ent<T> &q,
                              T d2, int, int) const {
        if (!ok) return;
        // the pair's parameters: from the LDS tables when typed, else the wave's registers
        // (a template parameter: tested here, the choice cost four instructions of forty; forces of
        // 1M 1338 -> 1212 us, batch of 512 6.82 -> 6.44 ms)
        T e = ws.e0, s2 = ws.s20, is = ws.is0;
        if (TYPED) {
            const int t = l.ti * 8 + (int)w_type(ent_w(q));
            e = sh.eps[t];
            s2 = sh.sig2[t];
            if (ADJ) is = sh.isig[t];
        }
        const T inv = fast_rcp(d2 + prm.a);
        const T s = s2 * inv;
        const T s3 = s * s * s;
        const T s6 = s3 * s3;
        l.e += e * (s6 - prm.c * s3);
        const T w = T(6) * s6 - prm.c3 * s3;
        if (FORCES) {
            const T g = T(2) * e * w * inv;
            l.fx = fma(g, p.x - q.x, l.fx);
            l.fy = fma(g, p.y - q.y, l.fy);
            l.fz = fma(g, p.z - q.z, l.fz);
        }
        if (ADJ) {
            l.aeps += (s6 - prm.c * s3) * e;
            l.asig += e * w * is;
        }
    }
    __device__ void row_sync(Wave &) const {}
    // (the lanes of homes past the row's end hold zeros)
    template <int G>
    __device__ void lane_end(Shared &sh, Wave &w, Lane &l, const Ent<T> &p, bool valid, const SysDesc<T> &sd,
                             int si) const {
        if (si != w.si) {
            add_energy(w);
            w.si = si;
        }
        w.e += valid ? escale * (double)l.e : 0.0;
        if (!FORCES && !ADJ) return;
        double ae = (double)l.aeps, as = (double)l.asig;
        for (int off = 1; off < G; off <<= 1) {
            if (FORCES) {
                l.fx += __shfl_xor(l.fx, off, 64);
                l.fy += __shfl_xor(l.fy, off, 64);
                l.fz += __shfl_xor(l.fz, off, 64);
            }
            if (ADJ) {
                ae += __shfl_xor(ae, off, 64);
                as += __shfl_xor(as, off, 64);
            }
        }
        if (valid && (threadIdx.x & (G - 1)) == 0) {
            const uint32_t i = w_idx(ent_w(p));
            if (FORCES) {
                T f[3] = {l.fx, l.fy, l.fz};
                if (sd.box.celltype == 1) {
                    const T *invrot = sd.invrot;
                    T g[3];
                    for (int r = 0; r < 3; ++r) g[r] = (invrot[r] * f[0] + invrot[r + 3] * f[1]) + invrot[r + 6] * f[2];
                    for (int r = 0; r < 3; ++r) f[r] = g[r];
                }
                for (int k = 0; k < dim; ++k) forces[(size_t)i * dim + k] = ADJ ? -f[k] : f[k];
            }
            if (ADJ) {
                atomicAdd(&sh.gde[l.ti], ae / (2.0 * (double)prm.eps_t[l.ti]));
                atomicAdd(&sh.gds[l.ti], as);
            }
        }
    }
    __device__ void wave_end(Shared &sh, Wave &w) const {
        add_energy(w);
        __syncthreads();
        if (ADJ && threadIdx.x < 8 && (threadIdx.x < (prm.ntypes ? prm.ntypes : 1))) {
            double *g = grad + (blockIdx.x % ACC_SLOTS) * ACC_STRIDE;
            atomicAdd(&g[threadIdx.x], sh.gde[threadIdx.x]);
            atomicAdd(&g[8 + threadIdx.x], sh.gds[threadIdx.x]);
        }
    }
};

// The rotation of a triclinic cell into its aligned frame (identity when tric == 0).
template <typename T>
struct OpRot {
    T m[9];
    int tric;
};

// Copies of a histogram's sums that the waves add to: thousands of waves each add to every
// bin, and adds to one cache line queue.
constexpr int HIST_COPIES = 32;
// The sums over the copies into the first copy.
static __global__ void __launch_bounds__(256) k_hist_sum(int nbins, unsigned long long *counts, double *vsum) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nbins) return;
    unsigned long long c = 0;
    double v = 0;
    for (int s = 0; s < HIST_COPIES; ++s) {
        c += counts[s * nbins + k];
        if (vsum) v += vsum[s * nbins + k];
    }
    counts[k] = c;
    if (vsum) vsum[k] = v;
}

// Distance histogram (+ radial velocity sums), LDS-privatised per workgroup.
template <typename T>
struct OpHistogram {
    static constexpr int WINDOWS = 16;  // (as for the neighbour list)
    static constexpr int MAXB = 512;
    struct Shared {
        unsigned int cnt[MAXB];
        double vs[MAXB];
    };
    struct Lane {
        T vx, vy, vz;
    };
    int nbins;
    T width;
    T inv_width;  // 1 / width, rounded (the bin computation corrects for its rounding)
    const T *vel;       // n*D input frame, may be null (velocities of the home set)
    // velocities of the neighbour entries, in the aligned frame, in the order of the entry
    // arrays the sweep walks (vq1: the ghost entries of the triclinic split; see
    // k_entry_velocities), so a pair reads the one next to the entry just tested
    const vec4<T> *vq0, *vq1;
    T rot[9];           // maps input-frame velocities to the aligned frame
    int tric;
    int dim;
    // HIST_COPIES copies of the counts, then of the velocity sums (see k_hist_sum)
    unsigned long long *counts;
    double *vsum;

    struct Wave {};
    __device__ void wave_init(Shared &sh, Wave &) const {
        for (int k = threadIdx.x; k < nbins; k += 64) { sh.cnt[k] = 0; sh.vs[k] = 0; }
        __syncthreads();
    }
    __device__ void rotv(const T *v, T *o) const {
        if (tric) {
            for (int r = 0; r < 3; ++r) o[r] = (rot[r] * v[0] + rot[r + 3] * v[1]) + rot[r + 6] * v[2];
        } else {
            o[0] = v[0]; o[1] = v[1]; o[2] = v[2];
        }
    }
    __device__ void lane_init(Wave &, Lane &l, const Ent<T> &p, bool valid) const {
        l.vx = l.vy = l.vz = T(0);
        if (vel && valid) {
            const uint32_t i = w_idx(ent_w(p));
            T v[3] = {T(0), T(0), T(0)}, o[3];
            for (int k = 0; k < dim; ++k) v[k] = vel[(size_t)i * dim + k];
            rotv(v, o);
            l.vx = o[0]; l.vy = o[1]; l.vz = o[2];
        }
    }
    __device__ void candidate(Shared &sh, Wave &, Lane &l, bool ok, uint64_t, const Ent<T> &p, const Ent<T> &q,
                              T d2, int jq, int pass) const {
        if (!ok) return;
        if constexpr (sizeof(T) == 4) {
            // The clustered histogram is bound by instructions and by the cache's data return:
            // one estimate of 1 / d serves root and quotient, and 12 bytes of a velocity are
            // read, not 16 (sweep of 4M: 49.2 -> 43.8 ms).  The terms' error against 64 bits
            // is that of the rounded root and division (0.5 units in the last place, + 2^-20).
            if (ballot64(!(d2 >= SQRT_FAST_MIN)) == 0) {
                // d within 0.5 + 2^-20 ulp of the root, from the estimate of 1 / d
                const float rd = __builtin_amdgcn_rsqf(d2);
                const float s = d2 * rd;
                const float d = fmaf(fmaf(-s, s, d2), 0.5f * rd, s);
                // floor(d / width), d and the quotient correctly rounded: d * (1 / width) lies
                // within 2.5 * 2^-23 of that quotient, so its floor is the same unless an integer
                // is within 4 * 2^-23 of the product; then (rarely) root and division themselves
                const float qa = d * inv_width;
                const float fl = dev_floor(qa);
                int b = (int)fl;
                if (fabsf((qa - fl) - 0.5f) >= fmaf(qa, -0x1p-21f, 0.5f)) {
                    const float bf = dev_floor(dev_div_rn(dev_sqrt_rn(d2), width));
                    b = bf > T(nbins - 1) ? nbins - 1 : (int)bf;
                }
                b = min(b, nbins - 1);
                atomicAdd(&sh.cnt[b], 1u);
                if (vel) {
                    const float t = radial(l, p, q, jq, pass);
                    // t / d: one correction of t * (1 / d), which an infinite product passes by
                    const float q0 = t * rd;
                    const float q1 = fmaf(fmaf(-q0, d, t), rd, q0);
                    atomicAdd(&sh.vs[b], (double)(fabsf(q0) < INFINITY ? q1 : q0));
                }
                return;
            }
        }
        const T d = dev_sqrt_rn(d2);
        const T bf = dev_floor(dev_div_rn(d, width));
        const int b = bf > T(nbins - 1) ? nbins - 1 : (int)bf;
        atomicAdd(&sh.cnt[b], 1u);
        if (vel && d > T(0)) atomicAdd(&sh.vs[b], (double)(radial(l, p, q, jq, pass) / d));
    }
    // (v_home - v_neighbour) . (x_home - x_neighbour)
    __device__ T radial(const Lane &l, const Ent<T> &p, const Ent<T> &q, int jq, int pass) const {
        const T *o = (const T *)((pass ? vq1 : vq0) + jq);
        return (l.vx - o[0]) * (p.x - q.x) + (l.vy - o[1]) * (p.y - q.y) + (l.vz - o[2]) * (p.z - q.z);
    }
    __device__ void row_sync(Wave &) const {}
    template <int G>
    __device__ void lane_end(Shared &, Wave &, Lane &, const Ent<T> &, bool, const SysDesc<T> &, int) const {}
    __device__ void wave_end(Shared &sh, Wave &) const {
        __syncthreads();
        const int at = (int)(blockIdx.x % HIST_COPIES) * nbins;
        for (int k = threadIdx.x; k < nbins; k += 64) {
            if (sh.cnt[k]) atomicAdd(&counts[at + k], (unsigned long long)sh.cnt[k]);
            if (vel && sh.vs[k] != 0.0) atomicAdd(&vsum[at + k], sh.vs[k]);
        }
    }
};

// The neighbour velocities of a histogram sweep in the order of an entry array: out[k] =
// R v[w_idx(ents[k])] for the first total_a[0] - total_b[0] entries (counts read on the
// device, so that a build whose count the host has not read is covered), R the rotation
// into the aligned frame (triclinic).  Skipped for a list the sweep will not walk.
template <typename T>
__global__ void __launch_bounds__(256) k_entry_velocities(const Ent<T> *__restrict__ ents, const int *__restrict__ total_a,
                                                          const int *__restrict__ total_b, long long cap, const T *__restrict__ vel,
                                                          long long nvel, int dim, OpRot<T> rot, vec4<T> *__restrict__ out,
                                                          const uint32_t *__restrict__ bin_flags, long long e_cap) {
    if (!build_usable(bin_flags, e_cap)) return;
    const long long n = min((long long)total_a[0] - (total_b ? (long long)total_b[0] : 0ll), cap);
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x) {
        const long long i = (long long)w_idx(ent_w(ents[k]));
        T v[3] = {T(0), T(0), T(0)};
        if (i < nvel)
            for (int c = 0; c < dim; ++c) v[c] = vel[i * dim + c];
        vec4<T> o;
        if (rot.tric) {
            for (int r = 0; r < 3; ++r) o[r] = (rot.m[r] * v[0] + rot.m[r + 3] * v[1]) + rot.m[r + 6] * v[2];
        } else {
            o[0] = v[0]; o[1] = v[1]; o[2] = v[2];
        }
        o[3] = T(0);
        out[k] = o;
    }
}

// Minimum distance: every lane keeps its best (d2, a, b) over its wave's tasks; the wave's
// best is written to an array, and k_mindist_best takes the best of those.
template <typename T>
struct MinDistBest {
    T d2;
    int a, b;
};
template <typename T>
struct OpMinDist {
    static constexpr int WINDOWS = 32;  // rows of a list of windows
    struct Shared {};
    struct Lane {};
    using Wave = MinDistBest<T>;
    MinDistBest<T> *best;  // [gridDim.x]
    int cross;   // two sets: keep (home, neighbour) order instead of (min, max)

    __device__ static bool better(T d2, int a, int b, T e2, int ea, int eb) {
        return d2 < e2 || (d2 == e2 && (a < ea || (a == ea && b < eb)));
    }
    __device__ static void take(Wave &w, T d2, int a, int b) {
        if (better(d2, a, b, w.d2, w.a, w.b)) { w.d2 = d2; w.a = a; w.b = b; }
    }
    __device__ static void reduce(Wave &w) {
        for (int off = 32; off > 0; off >>= 1) {
            const T d2 = __shfl_xor(w.d2, off, 64);
            const int a = __shfl_xor(w.a, off, 64), b = __shfl_xor(w.b, off, 64);
            take(w, d2, a, b);
        }
    }
    __device__ static void clear(Wave &w) {
        w.d2 = T(INFINITY);
        w.a = w.b = 0x7fffffff;
    }
    __device__ void wave_init(Shared &, Wave &w) const { clear(w); }
    __device__ void lane_init(Wave &, Lane &, const Ent<T> &, bool) const {}
    __device__ void candidate(Shared &, Wave &w, Lane &, bool ok, uint64_t, const Ent<T> &p, const Ent<T> &q,
                              T d2, int, int) const {
        if (!ok) return;
        const int i = (int)w_idx(ent_w(p)), j = (int)w_idx(ent_w(q));
        take(w, d2, (cross || i < j) ? i : j, (cross || i < j) ? j : i);
    }
    __device__ void row_sync(Wave &) const {}
    template <int G>
    __device__ void lane_end(Shared &, Wave &, Lane &, const Ent<T> &, bool, const SysDesc<T> &, int) const {}
    __device__ void wave_end(Shared &, Wave &w) const {
        reduce(w);
        if (threadIdx.x == 0) best[blockIdx.x] = w;
    }
};

// The best of the waves' results into best[0] (one workgroup of 256 threads).
template <typename T>
__global__ void __launch_bounds__(256) k_mindist_best(MinDistBest<T> *best, int n) {
    using Op = OpMinDist<T>;
    __shared__ MinDistBest<T> s[4];
    MinDistBest<T> w;
    Op::clear(w);
    for (int k = threadIdx.x; k < n; k += 256) Op::take(w, best[k].d2, best[k].a, best[k].b);
    Op::reduce(w);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; ++k) Op::take(w, s[k].d2, s[k].a, s[k].b);
        best[0] = w;
    }
}

}  // namespace clm
