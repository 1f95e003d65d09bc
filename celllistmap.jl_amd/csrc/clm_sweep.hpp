// clm_sweep.hpp -- launches of the sweep kernels (defined in clm_sweep.hip, which is
// compiled once per operator family and precision).
#pragma once

#include "clm_kernels.hpp"

namespace clm {

// What a launch of a sweep depends on besides its arguments.
struct SweepShape {
    int dim;
    int variant;       // 0 = union rows (k_sweep), 1 = windows (k_sweep_win)
    int lanes;         // lanes per home of k_sweep_win (4, 8, or 32 with whole cells)
    bool parts;        // the grid's cells are cut into parts (DevBox::sub)
    int group;         // entries per lane per step of k_sweep_win in mode B (0: the default, SWEEP_GROUP)
    int waves_per_cu;  // limit of the persistent grid; 0 = as many as fit
    int num_cus;
};

// Homes of one wave task.
inline int task_homes(int variant, int lanes) { return variant == 1 ? 64 / lanes : 64; }

// The persistent grid of a sweep kernel: as many one-wave workgroups as fit (or the tuned number).
template <typename T, int MODE, typename Op>
int sweep_grid(const SweepShape &sh);

template <typename T, int MODE, typename Op>
void sweep_launch(const SweepShape &sh, int grid, hipStream_t stream, const Ent<T> *E, const int *cs, const Ent<T> *En,
                  const int *csn, const SweepArgs<T> &sa, const Op &op);

}  // namespace clm
