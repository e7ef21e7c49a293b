// kbg_sweep_n64.hip -- FP64 instantiations of the sweep of small launches (k_sweep1d_narrow)
#include "kbg_sweep.h"

namespace kbg {

hipError_t launch_sweep1d_narrow64(int nf, int wg_waves, int rows, const Solve1D* d_solves, const WorkItem* d_items, int nitems,
                                   int par, double* d_rpart, int nstep, hipStream_t st) {
    if (nf == 1) return launch_sweep_narrow_t<double, 1>(wg_waves, rows, d_solves, d_items, nitems, par, d_rpart, nstep, st);
    return launch_sweep_narrow_t<double, 2>(wg_waves, rows, d_solves, d_items, nitems, par, d_rpart, nstep, st);
}

hipError_t sweep_narrow_attr64() {
    const hipError_t e = sweep_narrow_attr_t<double, 1>();
    return e != hipSuccess ? e : sweep_narrow_attr_t<double, 2>();
}

}  // namespace kbg
