// vmc_rrw_f64.hip -- multi-wavefront register-resident kernels, FP64.
#include "vmc_rrw_impl.hpp"

namespace vmc {
bool rrw_launch_f64(const DevSys &d, const DevState &st, unsigned grid, int n_sweeps,
                   unsigned long long s0, int flags, int bs, hipStream_t stream, KernelTimer &timer,
                   const ReinvLaunch &reinv, double *inv64) {
    return rrw_launch<double>(d, st, grid, n_sweeps, s0, flags, bs, stream, timer, reinv, inv64);
}
bool rrw_batch_step_f64(const DevSys &shape, const BatchItem *items, int n_items, unsigned grid,
                       const unsigned long long *sweep_ctr, int flags, int bs, bool reinv, hipStream_t stream,
                       const BatchItem *items_refresh, const BatchItem *items_m64, size_t energy_lds) {
    return rrw_batch_step<double>(shape, items, n_items, grid, sweep_ctr, flags, bs, reinv, stream, items_refresh,
                               items_m64, energy_lds);
}
bool rrw_given_f64(const DevSys &d, const DevState &st, unsigned grid, const SweepGiven &given,
                   hipStream_t stream, const ReinvLaunch &reinv) {
    return rrw_given<double>(d, st, grid, given, stream, reinv);
}
}  // namespace vmc
