/*
 * clm_hip.h -- C ABI of the MI355X (gfx950) cell-list pairwise engine.
 *
 * Plain C types only: opaque context, pointers, sizes, int status codes.
 * Indices are 0-based int32.  Matrices are column-major dim x dim with the
 * columns holding the lattice vectors (the reference's convention).
 * Every entry point names the reference interface it replaces
 * (paths relative to the CellListMap.jl source tree).
 *
 * Threading: one context = one HIP stream; a context must not be used from two
 * host threads at once.  Calls return after their device work has finished
 * unless stated otherwise.
 *
 * Ownership: host buffers are caller-owned and only touched during the call.
 * Device buffers passed with on_device=1 are caller-owned device pointers that
 * must stay valid until the call returns.  All scratch device memory is owned
 * by the context and grows monotonically (InPlaceNeighborList semantics,
 * src/API/neighborlist.jl:12-15, src/API/updating.jl:18-25).
 */
#ifndef CLM_HIP_H
#define CLM_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct clm_ctx clm_ctx;

/* Status codes.  ARG/DIM/CELL/NAN map to the reference's ArgumentError /
 * DimensionMismatch (src/internals/Box.jl:192-194,243; src/internals/CellOperations.jl:6-21;
 * src/internals/CellLists.jl:740-751). */
typedef enum {
    CLM_OK = 0,
    CLM_ERR_ARG = 1,        /* invalid argument (lcell < 1, bad dtype, NULL pointer, ...) */
    CLM_ERR_DIM = 2,        /* dimension mismatch */
    CLM_ERR_CELL = 3,       /* unit cell check failed: a plane distance <= 2*cutoff */
    CLM_ERR_NAN = 4,        /* NaN or Inf coordinates */
    CLM_ERR_CAPACITY = 5,   /* output buffer too small; the required size is returned */
    CLM_ERR_HIP = 6,        /* HIP runtime error (see clm_last_error) */
    CLM_ERR_STATE = 7,      /* call order (no box / no positions yet) */
    CLM_ERR_RANGE = 8       /* a particle maps outside the computing grid (reference: BoundsError) */
} clm_status;

typedef enum { CLM_F32 = 0, CLM_F64 = 1 } clm_dtype;
typedef enum { CLM_ORTHORHOMBIC = 0, CLM_TRICLINIC = 1, CLM_NONPERIODIC = 2 } clm_celltype;

/* Box geometry as built by the library (values of the working precision). */
typedef struct {
    int dim, celltype, lcell;
    int nc[3];                  /* computing cells per dimension (Box.nc) */
    double cutoff, cutoff_sqr;
    double input[9];            /* input unit cell (column-major 3x3 storage) */
    double aligned[9];          /* aligned unit cell */
    double rotation[9], inv_rotation[9];
    double cell_size[3];
    double cbmin[3], cbmax[3];  /* computing box */
    double origin[3];
} clm_box_info;

/* Pair potential of the energy/force operators, u(d2) = eps_ij [s^6 - c s^3]:
 *   form CLM_POT_SOFTCORE: s = sigma_ij^2/(d2+1), c = 1 (the soft-core potential);
 *   form CLM_POT_LJ:       s = sigma_ij^2/d2,     c = 2, i.e. eps[(sigma/d)^12 - 2(sigma/d)^6],
 *     the Lennard-Jones closure of test/applications/namd/ParticleSystem_vs_NAMD.jl:13-19.
 * ntypes = 0: a single (eps[0], sigma[0]) for every pair.  ntypes > 0: per-type
 * eps/sigma with Lorentz-Berthelot mixing, particle types from clm_set_types. */
typedef enum { CLM_POT_SOFTCORE = 0, CLM_POT_LJ = 1 } clm_potential_form;
typedef struct {
    int ntypes;
    double eps[8];
    double sigma[8];
    int form;
} clm_softcore;

/* ---- context ---------------------------------------------------------- */

/* No reference counterpart (the reference has no device state). */
clm_status clm_create(clm_ctx **ctx, int device, int dtype, int dim);
clm_status clm_destroy(clm_ctx *ctx);
const char *clm_last_error(const clm_ctx *ctx);
/* Launch on an existing HIP stream (hipStream_t passed as void*); NULL = the context's own. */
clm_status clm_set_stream(clm_ctx *ctx, void *stream);
/* The stream the context launches on (to order a caller's own device work against it). */
clm_status clm_get_stream(clm_ctx *ctx, void **stream);
/* Orders the context's stream and `other` (a hipStream_t passed as void*): with both = 1,
 * work queued on either stream after the call starts after the work queued on both
 * before it; with both = 0 only `other` waits for the context's earlier work; with
 * both = 2 only the context's stream waits for the work queued on `other`.  No
 * reference counterpart: plumbing for callers whose buffers another stream writes. */
clm_status clm_join_stream(clm_ctx *ctx, void *other, int both);
/* Library version string. */
const char *clm_version(void);

/* ---- geometry ----------------------------------------------------------- */

/* Box(unitcell, cutoff; lcell) / update_box: src/internals/Box.jl:191-270,330-335,395-423.
 * cell: dim*dim column-major (ORTHORHOMBIC takes the diagonal).  NONPERIODIC: cell is
 * ignored and the box is rebuilt from limits(x) at each cell-list update
 * (Box.jl:374-377; src/internals/ParticleSystem.jl:158-164). */
clm_status clm_set_box(clm_ctx *ctx, const double *cell, int celltype, double cutoff, int lcell);
clm_status clm_get_box(clm_ctx *ctx, clm_box_info *out);
/* Box of system k of a batch (k = 0 for a single system). */
clm_status clm_get_system_box(clm_ctx *ctx, int k, clm_box_info *out);
/* Host-only box construction (no device needed): the same arithmetic as clm_set_box. */
clm_status clm_box_compute(int dtype, int dim, const double *cell, int celltype, double cutoff, int lcell,
                           const double *origin, clm_box_info *out);

/* A batch of nsys independent periodic systems in one context (no reference
 * counterpart: the reference handles one system per ParticleSystem).  System k has
 * n[k] particles, unit cell cells[k*dim*dim ...] (column-major), cutoff cutoffs[k] and
 * lcell lcells[k]; all systems share the cell type.  Positions are then given as the
 * concatenation of all systems (system 0 first); energies are reported per system by
 * clm_energy_forces_batch and clm_graph_launch.  Replaces the per-system loop over
 * ParticleSystem + pairwise! (src/API/ParticleSystem.jl:142-174, src/API/pairwise.jl:48-63). */
clm_status clm_set_systems(clm_ctx *ctx, int nsys, const int64_t *n, const double *cells, int celltype,
                           const double *cutoffs, const int *lcells);

/* ---- particles ---------------------------------------------------------- */

/* update!(sys; xpositions=x): src/API/updating.jl:79-113,165-187 (copies, marks dirty).
 * x: n*dim values of the context dtype, AoS (the memory of Vector{SVector{dim,T}}). */
clm_status clm_set_positions(clm_ctx *ctx, const void *x, int64_t n, int on_device);
/* Per-particle int32 types in [0, ntypes) for typed soft-core (no reference counterpart). */
clm_status clm_set_types(clm_ctx *ctx, const int32_t *types, int64_t n, int on_device);
/* Per-particle velocities (n*dim, context dtype) for the radial-velocity histogram, which is refused
 * (CLM_ERR_STATE) while there are more particles than velocities. */
clm_status clm_set_velocities(clm_ctx *ctx, const void *v, int64_t n, int on_device);

/* Second set of particles: ParticleSystem(xpositions=..., ypositions=...) and
 * update!(sys; ypositions=y) (src/API/ParticleSystem.jl:142-174, src/API/updating.jl:
 * 165-187; CellListPair, src/internals/CellLists.jl:590-605).  After this call the
 * context is a two-set system: the pair operators visit every (i in x, j in y) pair
 * within the cutoff once (src/internals/cross.jl:81-130), i indexing x and j y; a
 * non-periodic box covers both sets (limits(x, y)).  Single system only. */
clm_status clm_set_positions_y(clm_ctx *ctx, const void *y, int64_t n, int on_device);
/* Back to one set (the y positions are kept, but no longer used). */
clm_status clm_clear_positions_y(clm_ctx *ctx);
/* Types / velocities of the second set (as clm_set_types / clm_set_velocities). */
clm_status clm_set_types_y(clm_ctx *ctx, const int32_t *types, int64_t n, int on_device);
clm_status clm_set_velocities_y(clm_ctx *ctx, const void *v, int64_t n, int on_device);

/* UpdateCellList!(x, box, cl): src/internals/CellLists.jl:644-662,727-927.
 * Operators call it lazily when positions or box changed (UpdateParticleSystem!). */
clm_status clm_update_cell_list(clm_ctx *ctx);
/* CellList fields (src/internals/CellLists.jl:115-137): out = {n_particles incl. images,
 * n_cells_with_real_particles, n_cells_with_particles, number_of_cells}. */
clm_status clm_cell_list_info(clm_ctx *ctx, int64_t *out4);

/* ---- device pair operators (stand-ins for pairwise!(f, sys) with fixed f) -- */

/* neighborlist!(system) / push_pair!: src/API/neighborlist.jl:217-231,
 * src/internals/neighborlist.jl:67-76.  Writes (i[k], j[k], d[k]) for every pair
 * within the cutoff, d in the context dtype, order unspecified.  If the pair count
 * exceeds capacity, *npairs holds the required count, CLM_ERR_CAPACITY is returned
 * and the array contents are unspecified (call again with a larger capacity).
 * At most 2^31-1 pairs per call.  Two-set context: i indexes x, j indexes y
 * (neighborlist(; xpositions, ypositions), src/API/neighborlist.jl:292-312). */
clm_status clm_neighborlist(clm_ctx *ctx, int32_t *i, int32_t *j, void *d, int64_t capacity,
                            int64_t *npairs, int on_device);

/* pairwise!(f, sys) with f = soft-core energy and forces (F_i = -dE/dx_i, n*dim,
 * context dtype, input frame).  forces may be NULL (energy only).  energy is
 * accumulated in double.  Replaces the user closure of
 * docs/src/ParticleSystem/examples.md:60-106 / test/examples/gravitational_force.jl:37-46.
 * Two-set context: the energy of the x-y pairs; forces holds (nx + ny)*dim values,
 * the rows of x first, then those of y. */
clm_status clm_energy_forces(clm_ctx *ctx, const clm_softcore *p, double *energy, void *forces,
                             int on_device, int64_t *npairs);

/* Soft-core energy per system of a batch (energies[nsys]) and forces of all particles. */
clm_status clm_energy_forces_batch(clm_ctx *ctx, const clm_softcore *p, double *energies, void *forces,
                                   int on_device);

/* Energy and its adjoint in one sweep: dE/dx (n*dim, context dtype), dE/deps and
 * dE/dsigma per type (double, p->ntypes entries, or 1 when untyped).  Positions
 * are re-read, no pair data is stored.  No reference counterpart (the reference
 * differentiates closures with ForwardDiff, test/examples/generic_types.jl:25-44). */
clm_status clm_energy_adjoint(clm_ctx *ctx, const clm_softcore *p, double *energy, void *dedx,
                              double *deps, double *dsigma, int on_device);

/* Distance histogram (test/examples/distance_histogram.jl:22-26) with bins of width
 * `width` starting at 0 (bin = floor(d/width), the d == cutoff edge in the last
 * bin), counts exact; with velocities set and vsum != NULL, also the sum per bin
 * of dot(v_i - v_j, x_i - x_j)/d (test/examples/pairwise_velocities.jl:17-24). */
clm_status clm_histogram(clm_ctx *ctx, int nbins, double width, int64_t *counts, double *vsum);

/* Minimum distance over pairs within the cutoff (test/examples/nearest_neighbor.jl:9-16):
 * lexicographic minimum of (d, min(i,j), max(i,j)) -- of (d, i, j) with i in x and
 * j in y for a two-set context; i = j = -1, d = +inf if none. */
clm_status clm_min_distance(clm_ctx *ctx, int64_t *i, int64_t *j, double *d);

/* ---- captured pipeline ----------------------------------------------------- */

/* Capture UpdateCellList! + energy/forces of the context (single system or batch) into
 * a HIP graph; forces: device array (n*dim) or NULL for a context-owned one, which must
 * outlive the graph.  The cell list is built first if needed; it sizes the cell buckets
 * of the one-pass binning the graph records and the entry buffer (1/8 headroom).  No
 * reference counterpart. */
clm_status clm_graph_capture_energy_forces(clm_ctx *ctx, const clm_softcore *p, void *forces);
/* Replay the captured graph on the current positions; energies[nsys] (host, may be NULL).
 * CLM_ERR_CAPACITY when a cell outgrew its bucket or the entries the captured capacity
 * (the replay's sweep skipped the list), CLM_ERR_NAN for a NaN among the positions (skipped too;
 * the next replay, on good ones, is a full one); CLM_ERR_STATE when the box, the particle count
 * or a buffer the graph uses changed since the capture (an eager build that grew its
 * buffers, clm_set_box, clm_set_systems, new positions of another size, new types):
 * nothing is launched.  Capture again after CLM_ERR_CAPACITY and CLM_ERR_STATE. */
clm_status clm_graph_launch(clm_ctx *ctx, double *energies);

/* Sweep launch shape: one-wave workgroups per CU of the persistent sweep (0 = as many
 * as fit).  Set by the autotuner; no reference counterpart (nbatches plays this role,
 * src/internals/CellLists.jl:178-273). */
clm_status clm_set_tuning(clm_ctx *ctx, int waves_per_cu);
/* Sweep kernel: 0 = every lane walks the union of its wave's stencil ranges (wave-uniform
 * neighbour loads); 1 = the lanes of a particle walk its window of each stencil row,
 * bounded by the cutoff sphere (per-lane loads; the default).  Same pairs and results either way;
 * an autotuner knob with no reference counterpart. */
clm_status clm_set_sweep_variant(clm_ctx *ctx, int variant);
/* Group width of the windowed sweep's tile: neighbour entries each lane tests per step
 * (and keeps in flight): 0 (the default, which is 2), 2, 4 or 8 (float64: 8 means
 * the default; below 20000 particles all mean it); it applies to the sweep that visits every pair from both sides (energy and
 * forces, the adjoint).  An autotuner knob with no reference counterpart. */
clm_status clm_set_sweep_group(clm_ctx *ctx, int group);

/* ---- allocation-free entry point ------------------------------------------ */

/* Soft-core energy and forces of one periodic system in one call that allocates no
 * memory: no reference counterpart.  It is for callers that cannot allocate (code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc): the variant of
 * clm_energy_forces (untyped parameters) whose cell list, counters and task tables live in
 * a fixed 64 MiB scratch array of the library on each GPU, about 0.5M particles at float32
 * (fewer at float64 or with many ghost images); a larger system returns CLM_ERR_CAPACITY
 * with nothing left running.  x: device positions (n x dim of the dtype, the caller's);
 * forces: device output (n x dim) or NULL; energy: host.  The call runs on `stream` (NULL:
 * the null stream) on the current device and returns after synchronising it.  Calls that
 * overlap on one GPU race on the shared scratch: serialise them.  clm_last_error(NULL)
 * holds the last call's message. */
clm_status clm_energy_forces_noalloc(int dtype, int dim, const void *x, int64_t n, const double *cell, int celltype,
                                     double cutoff, int lcell, const clm_softcore *p, double *energy, void *forces,
                                     void *stream);

/* ---- measurement ----------------------------------------------------------- */

/* Per-kernel HIP-event timing on the context stream (no reference counterpart;
 * the reference has ProgressMeter only, src/internals/self.jl:55,91). */
clm_status clm_profile_enable(clm_ctx *ctx, int enable);
/* Accumulated milliseconds and launch count of kernel `name` since enabling. */
clm_status clm_profile_get(clm_ctx *ctx, const char *name, double *total_ms, int64_t *count);
clm_status clm_profile_reset(clm_ctx *ctx);

#ifdef __cplusplus
}
#endif

#endif /* CLM_HIP_H */
