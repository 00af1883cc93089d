// vmc_init.hip -- the FP64 inverses of given positions for determinants of up
// to 160 electrons: log_abs_det's LU and n solves (slater_plane_wave.cpp:
// 202-318) as one Gauss-Jordan elimination in registers.
//
// One workgroup per walker and determinant.  A = D^T (A[m][i] = phi_m(r_i));
// four adjacent lanes own row m, lane q of them the columns 4 j + q.  Step c
// picks the largest |A[r][c]| of the rows not yet used (the reference's
// partial pivoting and its tolerance 1e-12, matrix.hpp:35-39) and exchanges
// that row's variable with column c in place, without moving any row; after n
// steps row p_c, column j hold the inverse's element (c, p_j).  Columns are
// taken four at a time from the first register of each lane, the registers
// then rotate by one, so every register index is a constant.
//
// What bounds it: the chain of n steps, each a workgroup maximum, two barriers
// and the broadcast of the pivot row through LDS: 61 us for 1024 walkers at 33
// per spin, 525 us for 1000 at 81, 1.28 ms for 1024 at 123 and 2.13 at 147; one
// wavefront per walker with the matrix in memory took 435 us at 33 and 42.6 ms at
// 147.  Above 128 a lane's row begins to spill (36 B of scratch per lane), above
// 160 it is left to the kernel in memory.
// FP64 inverses only: the elimination rounds in another order than k_init's, which
// moves about one FP32 element in a million by its last place, and an FP32 chain
// turns that into another accept decision now and then.
#include "../../include/vmc_hip.h"
#include "vmc_device.hpp"
#include "vmc_rr_launch.hpp"
#include "vmc_walker.hpp"

#include <hip/hip_runtime.h>

#include <type_traits>

namespace vmc {

namespace {

// Start positions: with draw Philox draws (tag INIT, counter {i, walker, 0}),
// else with aos set the caller's [w][i][3] taken into the ensemble's
// [w][3][i], else those in place.
__global__ __launch_bounds__(256) void k_place(DevSys s, DevState st, int draw, const double *aos) {
    const int N = s.N;
    const size_t total = (size_t)st.W * N;
    for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (size_t)gridDim.x * blockDim.x) {
        const int w = (int)(g / N), i = (int)(g - (size_t)w * N);
        double *gp = st.pos + (size_t)w * 3 * N + i;
        if (!draw) {
            for (int c = 0; c < 3 && aos; ++c) gp[c * N] = aos[3 * g + c];
        } else {
            const uint4 r = philox4x32_10(make_uint4((uint32_t)i, (uint32_t)w, 0u, kTagInit), s.key0, s.key1);
            gp[0] = u01(r.x) * s.L;
            gp[N] = u01(r.y) * s.L;
            gp[2 * N] = u01(r.z) * s.L;
        }
        if (i == 0) {
            st.flags[w] = 0;
            st.since[w] = 0;
            st.logdet[2 * w + 1] = 0.0;
        }
    }
}

// Largest of the wave's rows (four lanes of a row hold the same value), in
// every lane.
__device__ __forceinline__ double in_wave_max(double v) {
    const auto ror = [](double x, auto ctrl) {
        constexpr int kCtrl = decltype(ctrl)::value;
        union { double d; int i[2]; } u;
        u.d = x;
        u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], kCtrl, 0xF, 0xF, true);
        u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], kCtrl, 0xF, 0xF, true);
        return u.d;
    };
    v = fmax(v, ror(v, std::integral_constant<int, 0x124>{}));  // row_ror:4
    v = fmax(v, ror(v, std::integral_constant<int, 0x128>{}));  // row_ror:8
    const auto lane_value = [&](int l) {
        union { double d; int i[2]; } u;
        u.d = v;
        u.i[0] = __builtin_amdgcn_readlane(u.i[0], l);
        u.i[1] = __builtin_amdgcn_readlane(u.i[1], l);
        return u.d;
    };
    return fmax(fmax(lane_value(0), lane_value(16)), fmax(lane_value(32), lane_value(48)));
}

// Lane q's value of each group of four lanes, in all four.
template <int q>
__device__ __forceinline__ double in_quad(double v) {
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], q * 0x55, 0xF, 0xF, true);
    u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], q * 0x55, 0xF, 0xF, true);
    return u.d;
}

// C: columns of a lane, n <= 4 C rows and columns, 16 C threads.
template <int C>
__global__ __launch_bounds__(16 * C < 64 ? 64 : 16 * C) void k_invert(DevSys s, DevState st) {
    constexpr int NT = 16 * C < 64 ? 64 : 16 * C;
    constexpr int NW = NT / kWave;
    extern __shared__ __align__(16) double2 in_pw[];  // [axis][power][n]
    __shared__ double prow[4][C + 2];                 // the pivot row, by lane of a row
    __shared__ double wmax[2][NW];
    __shared__ int wrow[2][NW];
    __shared__ int order[4 * C];                      // p_c
    const int w = blockIdx.x / s.ndet, d = blockIdx.x - w * s.ndet;
    const int n = s.n[d], first = s.first[d];
    const int t = threadIdx.x, wave = wave_uniform(t >> 6), lane = t & (kWave - 1);
    const int row = t >> 2, q = t & 3;
    const double *gp = st.pos + (size_t)w * 3 * s.N + first;
    const int K1 = s.kmax + 1;
    for (int i = t; i < 3 * n; i += NT) {
        const int ax = i / n, e = i - ax * n;
        double f = gp[ax * s.N + e] * s.inv_L;
        f -= rint(f);
        double sn, cs;
        sincos_2pi<double>(f, &sn, &cs);
        double2 p = make_double2(1.0, 0.0);
        for (int m = 0; m < K1; ++m) {
            in_pw[(ax * K1 + m) * n + e] = p;
            p = make_double2(p.x * cs - p.y * sn, p.x * sn + p.y * cs);
        }
    }
    const int4 o = s.orb[d * s.nmax + (row < n ? row : 0)];
    const int ay = o.y < 0 ? -o.y : o.y, az = o.z < 0 ? -o.z : o.z;
    const double sy = o.y < 0 ? -1.0 : 1.0, sz = o.z < 0 ? -1.0 : 1.0;
    __syncthreads();
    double T[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const int i = 4 * j + q;
        T[j] = 0.0;
        if (i < n && row < n) {
            const double2 X = in_pw[o.x * n + i];
            double2 Y = in_pw[(K1 + ay) * n + i], Z = in_pw[(2 * K1 + az) * n + i];
            Y.y *= sy;
            Z.y *= sz;
            const double re = X.x * Y.x - X.y * Y.y, im = X.x * Y.y + X.y * Y.x;
            T[j] = o.w ? re * Z.y + im * Z.x : re * Z.x - im * Z.y;
        }
    }
    bool used = row >= n;
    bool singular = false;
    int mine = 0;  // the step that took this row
    double ldm = 1.0;
    int lde = 0;
    // Exchange of column c = 4 g + kq (lane kq's first register) with its
    // pivot row.
    const auto step = [&]<int kq>(int c) {
        const double v = in_quad<kq>(T[0]);
        const double a = used ? -1.0 : fabs(v);
        const double m = in_wave_max(a);
        const int buf = c & 1;
        if (lane == 0) {
            wmax[buf][wave] = m;
            wrow[buf][wave] = wave * 16;
        }
        const unsigned long long at = __ballot(a == m);
        if (lane == 0) wrow[buf][wave] += (at ? (int)__builtin_ctzll(at) : 0) >> 2;
        __syncthreads();
        double best = wmax[buf][0];
        int p = wrow[buf][0];
#pragma unroll
        for (int i = 1; i < NW; ++i)
            if (wmax[buf][i] > best) {
                best = wmax[buf][i];
                p = wrow[buf][i];
            }
        if (!(best >= 1e-12)) {
            singular = true;
            return;
        }
        if (row == p) {
#pragma unroll
            for (int j = 0; j < C; ++j) prow[q][j] = T[j];
            used = true;
            mine = c;
        }
        if (t == 0) order[c] = p;
        __syncthreads();
        const double piv = prow[kq][0], pinv = 1.0 / piv;
        const double f = row == p ? 1.0 - pinv : v * pinv;
#pragma unroll
        for (int j = 0; j < C; ++j) T[j] = fma(-f, prow[q][j], T[j]);
        if (q == kq) T[0] = row == p ? pinv : -f;
        int e;
        ldm = frexp(ldm * fabs(piv), &e);
        lde += e;
    };
    const int groups = (n + 3) / 4;
#pragma unroll 1
    for (int g = 0; g < groups; ++g) {
        const int c = 4 * g;
        step.template operator()<0>(c);
        if (singular) break;
        if (c + 1 < n) step.template operator()<1>(c + 1);
        if (singular) break;
        if (c + 2 < n) step.template operator()<2>(c + 2);
        if (singular) break;
        if (c + 3 < n) step.template operator()<3>(c + 3);
        if (singular) break;
        const double head = T[0];
#pragma unroll
        for (int j = 0; j + 1 < C; ++j) T[j] = T[j + 1];
        T[C - 1] = head;
    }
    if (singular) {
        if (t == 0) atomicOr(st.flags + w, kFlagSingular);
        return;
    }
    double *inv = static_cast<double *>(st.inv) + (size_t)w * s.ninv + s.inv_off[d] + (size_t)mine * n;
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const int col = 4 * (j + groups < C ? j + groups : j + groups - C) + q;
        if (row < n && col < n) inv[order[col]] = T[j];
    }
    if (t == 0) st.logdet[2 * w + d] = log(ldm) + (double)lde * 0.69314718055994531;
}

bool invert_launch(const DevSys &d, const DevState &st, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(st.W) * static_cast<unsigned>(d.ndet));
    const size_t lds = sizeof(double2) * 3 * static_cast<size_t>(d.kmax + 1) * static_cast<size_t>(d.nmax);
    const auto run = [&]<int C>() {
        hipLaunchKernelGGL((k_invert<C>), grid, dim3(16 * C < 64 ? 64 : 16 * C), lds, stream, d, st);
        return true;
    };
    const int n = d.nmax;
    if (n <= 8) return run.template operator()<2>();
    if (n <= 16) return run.template operator()<4>();
    if (n <= 32) return run.template operator()<8>();
    if (n <= 48) return run.template operator()<12>();
    if (n <= 64) return run.template operator()<16>();
    if (n <= 96) return run.template operator()<24>();
    if (n <= 128) return run.template operator()<32>();
    if (n <= 160) return run.template operator()<40>();
    return false;
}

}  // namespace

bool init_fast(const DevSys &d, const DevState &st, int draw, const double *aos, hipStream_t stream) {
    if (d.nmax > kInitFastMax) return false;
    const size_t total = static_cast<size_t>(st.W) * static_cast<size_t>(d.N);
    const unsigned grid = static_cast<unsigned>(total / 256 + 1 < 4096 ? total / 256 + 1 : 4096);
    hipLaunchKernelGGL(k_place, dim3(grid), dim3(256), 0, stream, d, st, draw, aos);
    return invert_launch(d, st, stream);
}

}  // namespace vmc
