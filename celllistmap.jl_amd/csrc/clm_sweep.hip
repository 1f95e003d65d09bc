// clm_sweep.hip -- the sweep kernels of one precision (CLM_SWEEP_T) and operator family
// (CLM_SWEEP_OPS: 1 neighbour list, 2 pair potential, 3 histogram and minimum distance, 4 pair
// potential of typed particles):
// compiled once for each, so that the instantiations build side by side.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "clm_sweep.hpp"

namespace clm {

namespace {

template <typename T, typename Op>
using SweepKernel = void (*)(const Ent<T> *, const int *, const Ent<T> *, const int *, const SweepArgs<T>, const Op);

template <typename T, int MODE, typename Op, int G, bool PARTS>
SweepKernel<T, Op> windowed(const SweepShape &sh) {
    constexpr int U = SWEEP_GROUP;
    if (sh.dim == 2) return k_sweep_win<T, MODE, 2, Op, G, U, PARTS>;
    if constexpr (MODE == MODE_B && G <= 8) {
        if (sh.group == 4) return k_sweep_win<T, MODE, 3, Op, G, 4, PARTS>;
        if constexpr (sizeof(T) == 4)
            if (sh.group == 8) return k_sweep_win<T, MODE, 3, Op, G, 8, PARTS>;
    }
    return k_sweep_win<T, MODE, 3, Op, G, U, PARTS>;
}

template <typename T, int MODE, typename Op>
SweepKernel<T, Op> sweep_kernel(const SweepShape &sh) {
    if (sh.variant == 0) {
        if (sh.dim == 2) return k_sweep<T, MODE, 2, Op>;
        return k_sweep<T, MODE, 3, Op>;
    }
    if (sh.lanes == 32) return windowed<T, MODE, Op, 32, false>(sh);  // (small systems: whole cells)
    if (sh.parts) return sh.lanes == 4 ? windowed<T, MODE, Op, 4, true>(sh) : windowed<T, MODE, Op, 8, true>(sh);
    return sh.lanes == 4 ? windowed<T, MODE, Op, 4, false>(sh) : windowed<T, MODE, Op, 8, false>(sh);
}

}  // namespace

template <typename T, int MODE, typename Op>
int sweep_grid(const SweepShape &sh) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, sweep_kernel<T, MODE, Op>(sh), 64, 0) != hipSuccess || per_cu <= 0)
        per_cu = 16;
    per_cu = std::min(per_cu, 32);
    if (sh.waves_per_cu > 0) per_cu = std::min(per_cu, sh.waves_per_cu);
    return std::max(64, sh.num_cus * per_cu);
}

template <typename T, int MODE, typename Op>
void sweep_launch(const SweepShape &sh, int grid, hipStream_t stream, const Ent<T> *E, const int *cs, const Ent<T> *En,
                  const int *csn, const SweepArgs<T> &sa, const Op &op) {
    hipLaunchKernelGGL((sweep_kernel<T, MODE, Op>(sh)), dim3(grid), dim3(64), 0, stream, E, cs, En, csn, sa, op);
}

#define SWEEP(MODE, ...)                                                                                              \
    template int sweep_grid<CLM_SWEEP_T, MODE, __VA_ARGS__>(const SweepShape &);                                     \
    template void sweep_launch<CLM_SWEEP_T, MODE, __VA_ARGS__>(const SweepShape &, int, hipStream_t,                  \
                                                               const Ent<CLM_SWEEP_T> *, const int *,                 \
                                                               const Ent<CLM_SWEEP_T> *, const int *,                 \
                                                               const SweepArgs<CLM_SWEEP_T> &, const __VA_ARGS__ &);
// the sweeps that visit every pair once
#define SWEEP_ONCE(...)                  \
    SWEEP(MODE_A_ORTHO, __VA_ARGS__)     \
    SWEEP(MODE_A_TRIC, __VA_ARGS__)      \
    SWEEP(MODE_X_ORTHO, __VA_ARGS__)     \
    SWEEP(MODE_X_REAL, __VA_ARGS__)

#if CLM_SWEEP_OPS == 1
SWEEP_ONCE(OpNeighborList<CLM_SWEEP_T>)
#elif CLM_SWEEP_OPS == 2 || CLM_SWEEP_OPS == 4
#define SWEEP_POTENTIAL(TYPED)                                       \
    SWEEP(MODE_A_ORTHO, OpSoftCore<CLM_SWEEP_T, false, false, TYPED>) \
    SWEEP(MODE_A_TRIC, OpSoftCore<CLM_SWEEP_T, false, false, TYPED>)  \
    SWEEP(MODE_X_REAL, OpSoftCore<CLM_SWEEP_T, false, false, TYPED>)  \
    SWEEP(MODE_B, OpSoftCore<CLM_SWEEP_T, true, false, TYPED>)        \
    SWEEP(MODE_X_REAL, OpSoftCore<CLM_SWEEP_T, true, false, TYPED>)   \
    SWEEP(MODE_B, OpSoftCore<CLM_SWEEP_T, true, true, TYPED>)
SWEEP_POTENTIAL(CLM_SWEEP_OPS == 4)
#else
SWEEP_ONCE(OpHistogram<CLM_SWEEP_T>)
SWEEP_ONCE(OpMinDist<CLM_SWEEP_T>)
#endif

}  // namespace clm
