// vmc_rrw_impl.hpp -- launchers of the multi-wavefront register-resident
// kernels, shared by vmc_rrw_f32.hip / vmc_rrw_f64.hip.
#pragma once

#include "vmc_rr_launch.hpp"
#include "vmc_sweep_rrw.hpp"

namespace vmc {

// Sweeps, each followed by the re-inversion of the walkers due for it and,
// with MEASURE, the local energy.  In mixed precision (inv64 set) a
// measured sweep re-inverts every walker with an FP64 result in inv64 and
// takes the FP64 local energy from it.  False, before any launch, for a
// measured sweep whose local energy does not fit its LDS.
template <typename Real, int NU, int ND, int WPS>
bool rrw_launch_g(const DevSys &d, const DevState &st, unsigned grid, int n_sweeps,
                  unsigned long long s0, int flags, int bs, hipStream_t stream, KernelTimer &timer,
                  const ReinvLaunch &reinv, double *inv64) {
    constexpr int NT = RRW<Real, NU, ND, WPS>::NT;
    const bool measure = flags & VMC_SWEEP_MEASURE;
    const bool exact = measure && inv64;
    if (measure && !measure64_fits(d)) return false;
    DevState st_refresh = st, st64 = st;
    st_refresh.inv64 = inv64;
    st64.inv = inv64;
    for (int i = 0; i < n_sweeps; ++i) {
        const unsigned long long si = s0 + (unsigned long long)i;
        hipEvent_t ev = nullptr;
        bool timed = timer.begin(stream, ev);
        hipLaunchKernelGGL((k_sweep_rrw<Real, NU, ND, WPS>), dim3(grid), dim3(NT), 0, stream, d, st, si,
                           flags);
        if (timed) timer.end(stream, ev, kTimeSweep);
        if (d.reinv_k > 0 || exact) {
            timed = timer.begin(stream, ev);
            reinv.launch(d, exact ? st_refresh : st, grid, stream);
            if (timed) timer.end(stream, ev, kTimeReinv);
        }
        if (measure) {
            timed = timer.begin(stream, ev);
            if (!measure64(d, exact ? st64 : st, grid, bs, nullptr, stream)) return false;
            if (timed) timer.end(stream, ev, kTimeMeasure);
        }
    }
    return true;
}

// f.template operator()<NU, ND, WPS>() of the system's instantiation; false
// when there is none.
template <typename Real, typename F>
bool rrw_dispatch(const DevSys &d, F &&f) {
    if (!rrw_supported_sizes(d.ndet, d.n_up, d.n_dn, d.ng, (int)sizeof(Real))) return false;
    if (d.ndet == 2) {
        if (d.n_up == 33) return f.template operator()<33, 33, 1>();
        if (d.n_up == 57) return f.template operator()<57, 57, 1>();
        if (d.n_up == 81) return f.template operator()<81, 81, 2>();
        if constexpr (sizeof(Real) == 4) {
            if (d.n_up == 123) return f.template operator()<123, 123, 2>();
            return f.template operator()<147, 147, 3>();
        }
    } else {
        if (d.n_up == 33) return f.template operator()<33, 0, 1>();
        if (d.n_up == 57) return f.template operator()<57, 0, 1>();
        if (d.n_up == 81) return f.template operator()<81, 0, 2>();
        if constexpr (sizeof(Real) == 4) {
            if (d.n_up == 123) return f.template operator()<123, 0, 2>();
            return f.template operator()<147, 0, 3>();
        }
    }
    return false;
}

template <typename Real>
bool rrw_launch(const DevSys &d, const DevState &st, unsigned grid, int n_sweeps,
                unsigned long long s0, int flags, int bs, hipStream_t stream, KernelTimer &timer,
                const ReinvLaunch &reinv, double *inv64) {
    return rrw_dispatch<Real>(d, [&]<int NU, int ND, int WPS>() {
        return rrw_launch_g<Real, NU, ND, WPS>(d, st, grid, n_sweeps, s0, flags, bs, stream, timer, reinv, inv64);
    });
}

// One sweep with the caller's moves (each recorded), then the re-inversion
// as after a sweep.
template <typename Real>
bool rrw_given(const DevSys &d, const DevState &st, unsigned grid, const SweepGiven &given, hipStream_t stream,
               const ReinvLaunch &reinv) {
    return rrw_dispatch<Real>(d, [&]<int NU, int ND, int WPS>() {
        constexpr int NT = RRW<Real, NU, ND, WPS>::NT;
        hipLaunchKernelGGL((k_sweep_rrw_given<Real, NU, ND, WPS>), dim3(grid), dim3(NT), 0, stream, d, st, 0,
                           given);
        if (d.reinv_k > 0) reinv.launch(d, st, grid, stream);
        return true;
    });
}

template <typename Real>
bool rrw_batch_step(const DevSys &shape, const BatchItem *items, int n_items, unsigned grid,
                    const unsigned long long *ctr, int flags, int bs, bool reinv, hipStream_t stream,
                    const BatchItem *items_refresh, const BatchItem *items_m64, size_t energy_lds) {
    return rrw_dispatch<Real>(shape, [&]<int NU, int ND, int WPS>() {
        constexpr int NT = RRW<Real, NU, ND, WPS>::NT;
        const bool measure = flags & VMC_SWEEP_MEASURE;
        hipLaunchKernelGGL((k_sweep_rrw_b<Real, NU, ND, WPS>), dim3(grid), dim3(NT), 0, stream, items,
                           n_items, ctr, flags);
        if (measure && items_m64) {
            reinv_batch_launch(shape, items_refresh, n_items, grid, stream, (int)sizeof(Real));
            return measure64_batch(shape.N, energy_lds, items_m64, n_items, grid, bs, stream);
        }
        if (reinv) reinv_batch_launch(shape, items, n_items, grid, stream, (int)sizeof(Real));
        return !measure || measure64_batch(shape.N, energy_lds, items, n_items, grid, bs, stream);
    });
}

}  // namespace vmc
