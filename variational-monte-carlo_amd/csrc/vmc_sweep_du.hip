// vmc_sweep_du.hip -- FP64 sweep with delayed (Woodbury) inverse updates, a
// block of up to 32 moves per determinant at a time.
//
// One workgroup per walker; the transposed inverse invT of each determinant
// stays in the walker's HBM block.  Every proposal of a sweep is known before
// the sweep starts (each electron moves once), so a block of consecutive
// movers is prepared as matrix work and decided afterwards:
//   - T[k][q] = phi'_q . invT[k] for the block's movers q and their inverse
//     rows k, on the FP64 matrix cores.  The ratio of the first move is T[0][0];
//     each accepted move a updates the block's rows by
//       T[k] -= (T[k][a] / R_a) T[a],  T[a] /= R_a,
//     the row operations of Sherman-Morrison (slater_plane_wave.cpp:367-423)
//     on the 32 columns that later moves of the block read, so R_q = T[q][q]
//     (slater_plane_wave.cpp:351-365) when q's turn comes.  One wavefront holds
//     T in registers, one row per lane, both determinants in its two halves,
//     and the dead column of each mover collects the row operations
//     themselves: after the block it holds Cinv of the accepted movers.
//   - The Jastrow change of every mover against the block's starting
//     positions, by all wavefronts, and for each pair of movers (p, a) the
//     correction X[a][p] that p's change takes when a is accepted first.
//   - The chain of decisions is then a wavefront's: two lane reads, the accept
//     test, one row of X, one row broadcast and 31 FMAs per pair of moves.
//   - A flush applies the m <= 16 accepted moves to all n rows of invT on the
//     matrix cores, 16 rows per wavefront at a time:
//       Z = Phi'_acc invT[rows]^T, Y = Cinv Z, invT[rows] -= Y^T P_acc,
//     each row read once and written once (P_acc: the accepted movers' old rows,
//     copied to LDS first; the movers' own rows become Cinv^T P_acc).
// A block ends early when 16 moves are accepted in one determinant or when
// the product of its accepted ratios exceeds a limit (du_growth_limit).
//
// What bounds it (N = 294, 1024 walkers, 1.77 ms a sweep): FP64 VALU work (43 %
// of the cycles, the pair terms above all) and FP64 MFMA issue (24 %) of two
// resident workgroups; alone on its CU a walker takes 0.51 ms, of which the
// decisions are a fifth, the flushes a third and T beside the pair terms 30 %.
// Against one inverse row read, five barriers and an 8-entry window solved by
// serial lane reads per move: 7.84 -> 1.77 ms a sweep at N = 294 and 3.88 -> 1.12
// at N = 246 (1024 walkers); against the generic kernel 0.075 -> 0.050 ms at 19 + 7
// electrons (777 walkers, several sweeps a launch; 0.078 one at a time) and 138
// -> 4.3 at 485 (8 walkers).  20 to 112 B of spill per lane at 128 registers.
//
// The chain is the generic kernel's (vmc_hip.hip sweep_walker): the same
// Philox draws, sweep order and FP64 accept test, so the FP64 trajectory
// follows the oracle twin move for move.
#include "../../include/vmc_hip.h"
#include "vmc_device.hpp"
#include "vmc_rr_launch.hpp"
#include "vmc_walker.hpp"

#include <hip/hip_runtime.h>

namespace vmc {

typedef double du_v4d __attribute__((ext_vector_type(4)));
// Four consecutive doubles at an 8-byte boundary (rows of odd length).
typedef double du_v4u __attribute__((ext_vector_type(4), aligned(8)));

constexpr int kG = 8;  // decisions per unrolled group
constexpr int kDuMaxAcc = 16;  // accepted moves per determinant between flushes: one MFMA tile
// A flush forms invT as the difference of terms that grow with the product of
// the accepted ratios since the last one, from its lowest point on (the
// determinant's growth G): it loses G^2 roundings where one accepted move after
// another loses G, and walkers leaving a near-singular start accept ratios of 5
// and far more.  A block therefore ends above a growth of 4, and of 16 for equal
// spins above 64 and one determinant above 96; log2 in 1/256.  Stored inverse
// against an 80-bit one, max|error| / max|inverse|, mean over walkers after one
// sweep from uniform starts and after 36, in 1e-15: rank-1 updates of every
// accepted move -> limit 4 (limit 16)
//   10 + 10  4.8 -> 5.6 (19) and 1.2 -> 1.2 (1.4)    33 + 27  15 -> 22 (64) and 3.8 -> 5.3 (7.0)
//   13 + 13  5.9 -> 7.9 (73) and 1.5 -> 1.8 (2.0)    50 + 50  20 -> 27 (39) and 8.6 -> 9.1 (16)
//   19 + 7   5.4 -> 7.3 (15) and 1.5 -> 1.9 (2.2)    161      200 -> 210 (2300) and 70 -> 56 (210)
// the largest of 512 walkers at 13 + 13 1.0e-12 -> 1.1e-12 (5.2e-11); windows of 8
// accepted moves -> limit 16: 70 + 70 440 -> 62 and 600 -> 24, 123 + 123 160 -> 100 and
// 1000 -> 48, 147 230 -> 83 and 3400 -> 53.  Limit 4 against 16 costs 8 % of a sweep
// at 19 + 7, 24 % at 50 + 50 and 21 % at 485, more where each sweep is a launch of
// its own, as long as its slowest walker.
template <int TH, bool kTwo>
__device__ __forceinline__ int du_growth_limit(const DevSys &s) {
    const bool wide = kTwo ? TH >= 6 : TH >= 8 && s.ndet == 1;
    return wide ? 4 * 256 : 2 * 256;
}
// A move that would pass the limit by this factor (a walker leaving a node, by
// a ratio of 1e3 and more) waits for the flush of those before it and is then
// alone in its block, where the flush is a rank-1 update.
constexpr int kDuFar = 4 * 256;

// Dynamic LDS of a walker, in doubles from its start.  TH > 0: rows of up to
// 16 TH columns, so every offset but those of the arrays
// over electrons and orbitals is a constant.
template <int NB, int TH, bool kTwo, int NW>
struct DuLds {
    static constexpr int ND = kTwo ? 2 : 1;
    static constexpr int kSlots = kTwo ? 64 : 32;  // movers of a block
    static constexpr int NB16 = (NB + 15) / 16 * 16;
    // Powers 0 .. K1 - 1 of an axis phasor: the largest component of the
    // orbitals is 1 up to 16 per spin, 2 up to 64, 3 up to 160 and 5 up to 512.
    static constexpr int K1 = TH == 0 ? 6 : TH <= 1 ? 2 : TH <= 4 ? 3 : 4;
    static constexpr int prop = 0;
    static constexpr int cinv = prop + 4 * kSlots;
    static constexpr int ctl = cinv + 2 * kDuMaxAcc * (kDuMaxAcc + 1);  // 48 ints
    static constexpr int book = ctl + 24;
    static constexpr int pw = book + 6;
    // Phi' and P of the flush, or X, T and the wavefronts' Jastrow sums of the
    // block's decisions.
    static constexpr int big = pw + 3 * K1 * kSlots * 2;
    static constexpr int part = big + ND * NB * kSlots + ND * NB16 * 32;
    static constexpr int kBlock = part - big + (kTwo ? NW : 2 * NW) * kSlots;
    int pitch;  // LDS row pitch (16-byte steps, rows spread over the banks)
    int px, orb, total;
    __host__ __device__ DuLds(int N, int n, int norb) {
        pitch = TH > 0 ? 16 * TH + 2 : (n + 15) / 16 * 16 + 2;
        const int flush = 2 * kDuMaxAcc * pitch;
        px = big + (flush > kBlock ? flush : kBlock);
        orb = px + 3 * ((N + 1) & ~1);
        total = orb + (norb + 1) / 2;
    }
};

// book: step width, log|det| of both determinants, accepted moves of the launch
// and of the sweep, accepted moves since the last re-inversion (kept here, not
// in registers through every phase).
// ctl ints: [0..1] accepted masks, [2] moves decided, [4 + 16 h + i] slot (row
// in the block) of determinant h's i-th accepted mover.

__device__ __forceinline__ double du_readlane(double v, int l) {
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_readlane(u.i[0], l);
    u.i[1] = __builtin_amdgcn_readlane(u.i[1], l);
    return u.d;
}

// The thread index as a value of its own in each phase, so that a phase's
// addresses are formed there and not carried in registers through the others.
__device__ __forceinline__ int du_thread() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// LDS traffic between lanes of one wavefront: the LDS serves a wavefront's
// accesses in order, so only the compiler has to keep them in order.
__device__ __forceinline__ void du_wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Metropolis test u < R^2 exp(2 dJ) (simulation.cpp:125-131) of every lane's
// values, as lane masks: `yes`, and `near` where the hardware exp2 does not
// decide it (u within 1e-5 of the threshold, or |dJ| beyond its range) and the
// FP64 exp has to.
__device__ __forceinline__ void du_test(double R, double dj, double ua, unsigned long long &yes,
                                        unsigned long long &near) {
    const double approx = R * R * (double)__builtin_amdgcn_exp2f((float)(2.0 * dj * 1.4426950408889634));
    yes = __ballot(ua < approx);
    near = __ballot(!(fabs(ua - approx) > 1e-5 * approx) || !(fabs(dj) < 40.0));
}
// Bit `l` of the test's outcome.
__device__ __forceinline__ int du_decide(double R, double dj, double ua, int l) {
    unsigned long long yes, near;
    du_test(R, dj, ua, yes, near);
    if ((near >> l) & 1ull) yes = __ballot(ua < R * R * exp(2.0 * dj));
    return (int)((yes >> l) & 1ull);
}

// log2 |R| of lane l in 1/256, from the exponent and the leading mantissa bits
// (at most 0.09 low).
__device__ __forceinline__ int du_log2(double R, int l) {
    return ((__builtin_amdgcn_readlane(__double2hiint(R), l) & 0x7fffffff) >> 12) - (1023 << 8);
}

// Factor of the mover's row in a row's update: the row's entry in the mover's
// column over R, and 1 - 1/R for the mover's own row.  Both sides are formed
// (a branch costs more).
__device__ __forceinline__ double du_factor(bool pivot, double t, double ir) {
    double own = 1.0 - ir, other = t * ir;
    asm volatile("" : "+v"(own), "+v"(other));
    return pivot ? own : other;
}

// T[q] -= f T_l[q] for every column, T_l the row of lane l (lane reads into
// scalar registers: no LDS round trip on the chain).
template <int NB>
__device__ __forceinline__ void du_row_op(double (&T)[NB], double f, int l) {
#pragma unroll
    for (int q0 = 0; q0 < NB; q0 += 8) {
        // (eight lane reads, then their uses: a use right behind its read waits)
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = du_readlane(T[q0 + q], l);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) T[q0 + q] = fma(-f, v[q], T[q0 + q]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Orbital o (packed, du_pack) of the mover in `slot` from the axis powers.
__device__ __forceinline__ int du_pack(int4 o) {
    const int y = o.y < 0 ? -o.y : o.y, z = o.z < 0 ? -o.z : o.z;
    return o.x | (y << 8) | (z << 16) | (o.y < 0 ? 1 << 24 : 0) | (o.z < 0 ? 1 << 25 : 0) | (o.w ? 1 << 26 : 0);
}
template <int kSlots, int K1>
__device__ __forceinline__ double du_orbital(const double2 *pw, int slot, int o) {
    const double2 X = pw[(o & 255) * kSlots + slot];
    double2 Y = pw[(K1 + ((o >> 8) & 255)) * kSlots + slot];
    double2 Z = pw[(2 * K1 + ((o >> 16) & 255)) * kSlots + slot];
    Y.y = (o & (1 << 24)) ? -Y.y : Y.y;
    Z.y = (o & (1 << 25)) ? -Z.y : Z.y;
    const double re = X.x * Y.x - X.y * Y.y, im = X.x * Y.y + X.y * Y.x;
    return (o & (1 << 26)) ? re * Z.y + im * Z.x : re * Z.x - im * Z.y;
}

// Length of the minimum image of a separation in units of L: sqrt(x) from
// v_rsq_f64 (2^-24 relative) y and one third-order step: with h = x y and
// e = 1 - h y, sqrt(x) = h (1 + e/2 + 3/8 e^2) to e^3 = 2^-70.
__device__ __forceinline__ double du_dist(double dx, double dy, double dz) {
    dx -= rint(dx);
    dy -= rint(dy);
    dz -= rint(dz);
    const double x = fmax(fma(dz, dz, fma(dy, dy, dx * dx)), 1e-280);
    const double y = __builtin_amdgcn_rsq(x), h = x * y, e = fma(-h, y, 1.0);
    return fma(h * e, fma(e, 0.375, 0.5), h);
}

// (u(rn) - u(ro)) / (a L) of the Pade pair function r / (1 + b r), distances in
// units of L and bl = b L: over the common denominator (one reciprocal, from
// v_rcp_f64 and a third-order step, and no cancellation).
__device__ __forceinline__ double du_pade_diff(double rn, double ro, double bl) {
    const double d = fma(bl, rn, 1.0) * fma(bl, ro, 1.0);
    const double y = __builtin_amdgcn_rcp(d), e = fma(-d, y, 1.0);
    return (rn - ro) * fma(y, fma(e, e, e), y);
}

// This sweep's proposals of the block's movers (vmc_hip.hip sweep_walker):
// Philox tags MOVE and ACCP, counter {electron, walker, sweep}; or the
// caller's moves.  One wavefront, one lane per mover.
template <bool kTwo>
__device__ __forceinline__ void du_propose(const DevSys &s, double *prop, const double *gp, const SweepGiven &given, int w,
                           uint32_t sweep, double sigma, int hb, int q0, int cnt, int lane) {
    asm volatile("" : "+v"(lane));
    const int r = lane & 31, h = kTwo ? lane >> 5 : hb;
    if (r >= cnt || (!kTwo && lane >= 32)) return;
    const int e = s.first[h] + q0 + r, slot = kTwo ? lane : r;
    constexpr int kSlots = kTwo ? 64 : 32;
    if (given.prop) {
        const size_t g = (size_t)w * s.N + e;
        for (int c = 0; c < 3; ++c) prop[c * kSlots + slot] = given.prop[3 * g + c];
        prop[3 * kSlots + slot] = given.u[g];
        return;
    }
    const uint4 rm = philox4x32_10(make_uint4((uint32_t)e, (uint32_t)w, sweep, kTagMove), s.key0, s.key1);
    const uint4 ra = philox4x32_10(make_uint4((uint32_t)e, (uint32_t)w, sweep, kTagAccept), s.key0, s.key1);
    double d[3];
    if (s.move_kind == 1) {
        const double rho0 = sqrt(-2.0 * log(u01(rm.x)));
        const double rho1 = sqrt(-2.0 * log(u01(rm.z)));
        double s0, c0, s1, c1;
        sincospi(2.0 * u01(rm.y), &s0, &c0);
        sincospi(2.0 * u01(rm.w), &s1, &c1);
        d[0] = rho0 * c0;
        d[1] = rho0 * s0;
        d[2] = rho1 * c1;
    } else {
        d[0] = 2.0 * u01(rm.x) - 1.0;
        d[1] = 2.0 * u01(rm.y) - 1.0;
        d[2] = 2.0 * u01(rm.z) - 1.0;
    }
    for (int c = 0; c < 3; ++c) {
        const double x = gp[c * s.N + e] + sigma * d[c];
        prop[c * kSlots + slot] = x - s.L * floor(x * s.inv_L);
    }
    prop[3 * kSlots + slot] = u01(ra.x);
}

// Applies determinant h's m accepted moves to its inverse inv (n x n, row k =
// invT[k][.]).  TH: 16-column tiles of a row tile held in registers between
// its read and its write; 0 reads the row tile twice (n > 160).  Called by
// every thread.
template <int NB, int TH, bool kTwo, int NW>
__device__ __forceinline__ void du_flush(const DuLds<NB, TH, kTwo, NW> &l, double *sm, double *inv, int n, int h,
                                         int q0, int m, const int *orb) {
    using Lay = DuLds<NB, TH, kTwo, NW>;
    const int t = du_thread(), wave = wave_uniform(t >> 6), lane = t & (kWave - 1);
    const int *list = reinterpret_cast<const int *>(sm + Lay::ctl) + 4 + 16 * h;
    const double2 *pw = reinterpret_cast<const double2 *>(sm + Lay::pw);
    double *phi = sm + Lay::big, *prow = phi + kDuMaxAcc * l.pitch;
    const int r = lane & 15, g = lane >> 4;
    const int T = TH > 0 ? TH : (n + 15) / 16, TF = n / 16;  // column tiles, whole ones
    const int R = (n + 15) / 16;                               // row tiles
    // Tiles that lie within the row's n columns: with equal spins n is the n
    // that chose TH, so the first TH - 2 are known to; the smaller of two
    // unequal determinants may have any number fewer.
    const auto whole = [&](int jt) { return (kTwo && jt < TH - 2) || jt < TF; };
    const auto load = [&](const double *row, int jt) {
        du_v4d c = {0.0, 0.0, 0.0, 0.0};
        if (whole(jt)) {
            const du_v4u u = *reinterpret_cast<const du_v4u *>(row + 16 * jt);
            c = u;
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (16 * jt + 4 * g + q < n) c[q] = row[16 * jt + q];
        }
        return c;
    };
    const auto row_of = [&](int kt) {
        const int k = 16 * kt + r;
        return inv + (size_t)(k < n ? k : n - 1) * n + 4 * g;
    };
    // The first row tile is on its way while the movers' rows are gathered.
    constexpr int TR = TH > 0 ? TH : 1;
    du_v4d c[TR];
    if (TH > 0 && wave < R) {
        const double *row = row_of(wave);
#pragma unroll
        for (int jt = 0; jt < TR; ++jt) c[jt] = load(row, jt);
    }
    // The accepted movers' new orbital rows and old inverse rows (rows past m
    // and columns past n keep finite values that meet zeros).
    for (int a = wave; a < m; a += NW) {
        const int rs = list[a], slot = kTwo ? h * 32 + rs : rs;
        const double *src = inv + (size_t)(q0 + rs) * n;
        for (int j = lane; j < l.pitch - 2; j += kWave) {
            const bool in = j < n;
            prow[a * l.pitch + j] = in ? src[j] : 0.0;
            phi[a * l.pitch + j] = in ? du_orbital<Lay::kSlots, Lay::K1>(pw, slot, orb[j]) : 0.0;
        }
    }
    __syncthreads();
    const double *cinv = sm + Lay::cinv + h * kDuMaxAcc * (kDuMaxAcc + 1);
    const double *phr = phi + r * l.pitch + 4 * g;
    // Column 16 jt + 4 (r & 3) + (r >> 2) is what output row r of the update
    // stands for: register q of group g then holds column 16 jt + 4 g + q, so
    // a lane's four values are consecutive in memory.
    const double *pr = prow + g * l.pitch + 4 * (r & 3) + (r >> 2);
    // A mover's own row k is Cinv's column times P: Z of its column is -e_k and
    // the row itself is left out (C's column times Cinv is e_k, so that the row
    // would meet itself and leave 1/R of it, R roundings worse).
    int own[4];  // the row of mover 4 q + g
#pragma unroll
    for (int q = 0; q < 4; ++q) own[q] = 4 * q + g < m ? q0 + list[4 * q + g] : -1;
    const unsigned movers = (unsigned)reinterpret_cast<const int *>(sm + Lay::ctl)[h];
    for (int kt = wave; kt < R; kt += NW) {
        const int k = 16 * kt + r;
        double *row = row_of(kt);
        du_v4d z = {0.0, 0.0, 0.0, 0.0}, y = {0.0, 0.0, 0.0, 0.0};
        const auto store = [&](int jt, const du_v4d &c) {
            if (k >= n) return;
            if (whole(jt)) {
                *reinterpret_cast<du_v4u *>(row + 16 * jt) = c;
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (16 * jt + 4 * g + q < n) row[16 * jt + q] = c[q];
            }
        };
        const auto dot = [&](int jt, const du_v4d &c) {
            const du_v4d a = *reinterpret_cast<const du_v4u *>(phr + 16 * jt);
#pragma unroll
            for (int q = 0; q < 4; ++q) z = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], c[q], z, 0, 0, 0);
        };
        const auto update = [&](int jt, du_v4d &c) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[4 * q * l.pitch + 16 * jt], y[q], c, 0, 0, 0);
        };
        const bool moved = (unsigned)(k - q0) < 32u && ((movers >> (k - q0)) & 1u);
        const auto solve = [&]() {
#pragma unroll
            for (int q = 0; q < 4; ++q) z[q] = moved ? (own[q] == k ? -1.0 : 0.0) : z[q];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                y = __builtin_amdgcn_mfma_f64_16x16x4f64(cinv[r * (kDuMaxAcc + 1) + 4 * q + g], z[q], y, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) y[q] = -y[q];
        };
        if constexpr (TH > 0) {
#pragma unroll
            for (int jt = 0; jt < TH; ++jt) {
                dot(jt, c[jt]);
                if (jt % 2) __builtin_amdgcn_sched_barrier(0);
            }
            solve();
            if (__any(moved)) {
#pragma unroll
                for (int jt = 0; jt < TH; ++jt)
#pragma unroll
                    for (int q = 0; q < 4; ++q) c[jt][q] = moved ? 0.0 : c[jt][q];
            }
#pragma unroll
            for (int jt = 0; jt < TH; ++jt) {
                update(jt, c[jt]);
                if (jt % 2) __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int jt = 0; jt < TH; ++jt) store(jt, c[jt]);
            __builtin_amdgcn_sched_barrier(0);
            if (kt + NW < R) {
                const double *next = row_of(kt + NW);
#pragma unroll
                for (int jt = 0; jt < TH; ++jt) c[jt] = load(next, jt);
            }
        } else {
            // The next column tile is on its way while this one is used.
            du_v4d cc = load(row, 0);
#pragma unroll 1
            for (int jt = 0; jt < T; ++jt) {
                const du_v4d nx = load(row, jt + 1 < T ? jt + 1 : jt);
                dot(jt, cc);
                cc = nx;
            }
            solve();
            cc = load(row, 0);
#pragma unroll 1
            for (int jt = 0; jt < T; ++jt) {
                const du_v4d nx = load(row, jt + 1 < T ? jt + 1 : jt);
#pragma unroll
                for (int q = 0; q < 4; ++q) cc[q] = moved ? 0.0 : cc[q];
                update(jt, cc);
                store(jt, cc);
                cc = nx;
            }
        }
    }
    __syncthreads();
}

// kTwo: equal spins, the block's movers are up q0.., down q0.. in turn; else
// the block's movers are of one determinant.
template <int NB, int TH, bool kTwo, int NW>
__device__ void du_sweep_walker(const DevSys &s, const DevState &st, int w, int n_sweeps,
                                unsigned long long sweep0, int flags, const SweepGiven &given) {
    extern __shared__ __align__(16) double sm[];
    constexpr int NT = NW * kWave;
    constexpr int kSlots = kTwo ? 64 : 32;
    constexpr int ND = kTwo ? 2 : 1;
    constexpr int NB16 = (NB + 15) / 16 * 16;
    constexpr int kSub = kTwo ? NW : 2 * NW;  // subsets of the electrons in the pair sums
    const int t = threadIdx.x, wave = wave_uniform(t >> 6), lane = t & (kWave - 1);
    const int N = s.N, NP = (N + 1) & ~1;
    const int norb = kTwo ? s.nmax : s.n[0] + (s.ndet == 2 ? s.n[1] : 0);
    using Lay = DuLds<NB, TH, kTwo, NW>;
    const Lay l(N, s.nmax, norb);
    double *px = sm + l.px, *py = px + NP, *pz = py + NP;
    double *prop = sm + Lay::prop;
    double *X = sm + Lay::big;                        // [ND NB][kSlots]
    double *Ts = X + ND * NB * kSlots;             // [ND][NB16][32]
    double2 *pw = reinterpret_cast<double2 *>(sm + Lay::pw);
    double *part = sm + Lay::part;
    int *orbs = reinterpret_cast<int *>(sm + l.orb);
    int *ctl = reinterpret_cast<int *>(sm + Lay::ctl);
    double *invw = reinterpret_cast<double *>(st.inv) + (size_t)w * s.ninv;
    double *gp = st.pos + (size_t)w * 3 * N;
    for (int i = t; i < l.orb; i += NT) sm[i] = 0.0;
    for (int j = t; j < norb; j += NT) {
        const int d = !kTwo && j >= s.n[0] ? 1 : 0;
        orbs[j] = du_pack(s.orb[d * s.nmax + (d ? j - s.n[0] : j)]);
    }
    __syncthreads();
    for (int i = t; i < N; i += NT) {
        px[i] = gp[i] * s.inv_L;
        py[i] = gp[N + i] * s.inv_L;
        pz[i] = gp[2 * N + i] * s.inv_L;
    }
    double *book = sm + Lay::book;
    if (t == 0) {
        const int since = st.since[w];
        book[0] = st.sigma[w];
        book[1] = st.logdet[2 * w + 0];
        book[2] = st.logdet[2 * w + 1];
        book[3] = 0.0;
        book[4] = 0.0;
        book[5] = s.reinv_k > 0 && since >= s.reinv_k ? 0.0 : (double)since;  // re-inverted after the last sweep
    }
    __syncthreads();

    for (int sw = 0; sw < n_sweeps; ++sw) {
        const uint32_t sweep = (uint32_t)(sweep0 + (unsigned long long)sw);
        for (int hb = 0; hb < (kTwo ? 1 : s.ndet); ++hb) {
            const int n = s.n[hb];
            if (wave == NW - 1) du_propose<kTwo>(s, prop, gp, given, w, sweep, book[0], hb, 0, n < NB ? n : NB, lane);
            __syncthreads();
            int cnt = 0;
            for (int q0 = 0; q0 < n;) {
                cnt = n - q0 < NB ? n - q0 : NB;
                // Axis phasor powers of the block's proposals.
                for (int i = du_thread(); i < 3 * kSlots; i += NT) {
                    const int ax = i / kSlots, slot = i - ax * kSlots;
                    if ((slot & 31) >= cnt) continue;
                    double f = prop[ax * kSlots + slot] * s.inv_L;
                    f -= rint(f);
                    double sn, cs;
                    sincos_2pi<double>(f, &sn, &cs);
                    double2 p = make_double2(1.0, 0.0);
                    for (int k = 0; k < Lay::K1; ++k) {
                        pw[(ax * Lay::K1 + k) * kSlots + slot] = p;
                        p = make_double2(p.x * cs - p.y * sn, p.x * sn + p.y * cs);
                    }
                }
                __syncthreads();
                // T of the block on the first ND MT wavefronts, 16 movers
                // each; the other wavefronts start with the pair terms, of
                // which these take a share that evens the two (a column tile
                // of T costs about 1.4 electrons' pair terms).
                constexpr int MT = NB16 / 16, NTask = ND * MT;
                {
                    const int t = du_thread(), wave = wave_uniform(t >> 6), lane = t & (kWave - 1);
                    const int r = lane & 15, g = lane >> 4;
                    const int P16 = (n + 15) / 16;
                    for (int task = wave; task < NTask; task += NW) {
                        const int h = task / MT, mt = task % MT;
                        if (16 * mt >= cnt) continue;
                        const int hd = kTwo ? h : hb;
                        const int slot = (kTwo ? h * 32 : 0) + 16 * mt + r;
                        const int *orb = orbs + (!kTwo && hb ? s.n[0] : 0) + 4 * g;
                        const double *row[MT];
#pragma unroll
                        for (int kt = 0; kt < MT; ++kt) {
                            const int k = q0 + 16 * kt + r;
                            row[kt] = invw + s.inv_off[hd] + (size_t)(k < n ? k : n - 1) * n + 4 * g;
                        }
                        const auto load = [&](int kt, int jt) {
                            du_v4d c;
                            if (16 * jt + 16 <= n) {
                                const du_v4u u = *reinterpret_cast<const du_v4u *>(row[kt] + 16 * jt);
                                c = u;
                            } else {
#pragma unroll
                                for (int q = 0; q < 4; ++q)
                                    c[q] = 16 * jt + 4 * g + q < n ? row[kt][16 * jt + q] : 0.0;
                            }
                            return c;
                        };
                        du_v4d z[MT], c0[MT], c1[MT];
#pragma unroll
                        for (int kt = 0; kt < MT; ++kt) {
                            z[kt] = du_v4d{0.0, 0.0, 0.0, 0.0};
                            c0[kt] = load(kt, 0);
                            c1[kt] = load(kt, P16 > 1 ? 1 : 0);
                        }
                        const auto orbitals = [&](int jt, double (&av)[4]) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const int j = 16 * jt + 4 * g + q;
                                av[q] = du_orbital<kSlots, Lay::K1>(pw, slot, orb[j < n ? 16 * jt + q : -4 * g]);
                            }
                        };
                        double av[4];
                        orbitals(0, av);
#pragma unroll 1
                        for (int jt = 0; jt < P16; ++jt) {
                            double an[4];
                            orbitals(jt + 1 < P16 ? jt + 1 : jt, an);
#pragma unroll
                            for (int q = 0; q < 4; ++q)
#pragma unroll
                                for (int kt = 0; kt < MT; ++kt)
                                    z[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[q], c0[kt][q], z[kt], 0, 0, 0);
#pragma unroll
                            for (int kt = 0; kt < MT; ++kt) {
                                c0[kt] = c1[kt];
                                c1[kt] = load(kt, jt + 2 < P16 ? jt + 2 : P16 - 1);
                            }
#pragma unroll
                            for (int q = 0; q < 4; ++q) av[q] = an[q];
                        }
#pragma unroll
                        for (int kt = 0; kt < MT; ++kt)
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                Ts[(h * NB16 + 16 * mt + 4 * q + g) * 32 + 16 * kt + r] = z[kt][q];
                    }
                }
                // Jastrow change of the lane's mover against the electrons of
                // the wavefront's share, at the block's starting positions,
                // and the corrections by the movers among them.
                {
                    const int t = du_thread(), wave = wave_uniform(t >> 6), lane = t & (kWave - 1);
                    const double inv_L = s.inv_L, bl = s.b * s.L;
                    const int r = lane & 31, slot = kTwo ? lane : r;
                    const int h = kTwo ? lane >> 5 : hb;
                    const int half = kTwo ? 0 : lane >> 5;
                    const int e = s.first[h] + q0 + (r < cnt ? r : 0);
                    const double xo = px[e], yo = py[e], zo = pz[e];
                    const double xn = prop[slot] * inv_L, yn = prop[kSlots + slot] * inv_L,
                                 zn = prop[2 * kSlots + slot] * inv_L;
                    // u at the lane's mover's new place less u at its old one,
                    // against the point (x, y, z).
                    const double a0 = (h == 0 ? s.a_same : s.a_anti) * s.L, a1 = (h == 1 ? s.a_same : s.a_anti) * s.L;
                    const auto change = [&](double x, double y, double z, double a) {
                        const double rn = du_dist(xn - x, yn - y, zn - z);
                        const double ro = du_dist(xo - x, yo - y, zo - z);
                        return a * du_pade_diff(rn, ro, bl);
                    };
                    // Electrons come in rounds of V: four to a wavefront, `few`
                    // to one with a tile of T.
                    int few = 4;
                    if constexpr (NTask < NW) {
                        const int tc = 14 * ((n + 15) / 16) / (kTwo ? 10 : 20);
                        const int J = (N + ND * cnt) / (kTwo ? 1 : 2);
                        const int y = (J + NTask * tc) / NW;
                        few = y > tc ? (4 * (y - tc) + y / 2) / y : 0;
                    }
                    const int tw = wave < NTask ? wave : NTask;
                    const int share = NTask < NW && wave < NTask ? few : 4;
                    const int first = NTask < NW ? tw * few + (wave - tw) * 4 : wave * 4;
                    const int V = NTask < NW ? NTask * few + (NW - NTask) * 4 : NW * 4;
                    double acc = 0.0;
                    // The block's movers: at their old places for the mover's
                    // own change, and what it changes by when they move first.
                    const int nm = ND * cnt;
#pragma unroll 1
                    for (int v0 = 0; v0 * (kTwo ? 1 : 2) < nm; v0 += V)
#pragma unroll 1
                        for (int v = 0; v < share; ++v) {
                            const int jj = kTwo ? v0 + first + v : 2 * (v0 + first + v) + half;
                            const int j = jj < nm ? jj : 0;
                            const int hj = kTwo && j >= cnt ? 1 : 0, jl = j - (hj ? cnt : 0);
                            const int js = hj * 32 + jl, ej = s.first[kTwo ? hj : hb] + q0 + jl;
                            const double a = (kTwo ? hj : hb) ? a1 : a0;
                            const double d = change(px[ej], py[ej], pz[ej], a);
                            const double dn = change(prop[js] * inv_L, prop[kSlots + js] * inv_L,
                                                     prop[2 * kSlots + js] * inv_L, a);
                            if (jj < nm) X[(hj * NB + jl) * kSlots + slot] = dn - d;
                            acc += jj < nm && ej != e ? d : 0.0;
                        }
                    // The other electrons, two at a time (past the last one
                    // with a weight of zero).
                    const int no = N - nm;
                    for (int v0 = 0; v0 * (kTwo ? 1 : 2) < no; v0 += V)
#pragma unroll 1
                        for (int v = 0; v < share; v += 2) {
                            double d[2];
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const int jj = kTwo ? v0 + first + v + u : 2 * (v0 + first + v + u) + half;
                                const bool in = v + u < share && jj < no;
                                int j = in ? jj : 0;
                                j += j >= s.first[hb] + q0 ? cnt : 0;
                                if constexpr (kTwo) j += j >= s.first[1] + q0 ? cnt : 0;
                                j = j < N ? j : 0;
                                d[u] = change(px[j], py[j], pz[j], spin_of(s, j) ? a1 : a0);
                                d[u] = in ? d[u] : 0.0;
                            }
                            acc += d[0] + d[1];
                        }
                    part[(kTwo ? wave : 2 * wave + half) * kSlots + slot] = acc;
                }
                __syncthreads();
                if (wave == 0) {
                    const int lane = du_thread() & (kWave - 1);
                    const int r = lane & 31, h = kTwo ? lane >> 5 : 0, slot = kTwo ? lane : r;
                    double T[NB];
#pragma unroll
                    for (int q = 0; q < NB; ++q) T[q] = Ts[(h * NB16 + q) * 32 + r];
                    double dj = 0.0;
#pragma unroll
                    for (int i = 0; i < kSub; ++i) dj += part[i * kSlots + slot];
                    const double ua = prop[3 * kSlots + slot];
                    unsigned mask[2] = {0u, 0u};
                    // log2 of the accepted ratios' product since its lowest point, in 1/256
                    int grow[2] = {0, 0};
                    const int limit = du_growth_limit<TH, kTwo>(s);
                    // Growth after a move of log2 ratio lg, and whether the move is to
                    // wait for the flush of those accepted before it.
                    const auto grown = [&](int hh, int lg) { return (grow[hh] > 0 ? grow[hh] : 0) + lg; };
                    const auto waits = [&](int hh, int lg) { return mask[hh] && grown(hh, lg) > limit + kDuFar; };
                    double rec_r = 1.0, rec_j = 0.0;
                    int steps = cnt;
                    // Eight columns at a time by their registers, then the
                    // columns move on by eight: after all groups column a's
                    // row operations sit in T[a].
#pragma unroll 1
                    for (int i0 = 0; i0 < NB; i0 += kG) {
#pragma unroll
                        for (int k = 0; k < kG; ++k) {
                            const int i = i0 + k;
                            if (i >= steps) break;
                            const double R = T[k], irl = rcp_nr(R);
                            const bool pivot = r == i;
                            const int au = du_decide(R, dj, ua, i);
                            // (from within the limit only a ratio above kDuFar gets there)
                            const unsigned long long far =
                                __ballot(fabs(R) >= 16.0) & ((kTwo ? 0x100000001ull : 1ull) << i);
                            if (far && ((au && waits(0, du_log2(R, i))) || (kTwo && waits(1, du_log2(R, 32 + i))))) {
                                steps = i;
                                break;
                            }
                            rec_r = pivot ? R : rec_r;
                            rec_j = pivot && h == 0 ? dj : rec_j;
                            double f = 0.0;
                            if (au) {
                                mask[0] |= 1u << i;
                                grow[0] = grown(0, du_log2(R, i));
                                dj += X[i * kSlots + slot];
                                const double ir = du_readlane(irl, i);
                                f = kTwo && h ? 0.0 : du_factor(pivot, R, ir);
                                du_row_op<NB>(T, f, i);
                            }
                            if constexpr (kTwo) {
                                const int ad = du_decide(R, dj, ua, 32 + i);
                                rec_j = pivot && h == 1 ? dj : rec_j;
                                if (ad) {
                                    mask[1] |= 1u << i;
                                    grow[1] = grown(1, du_log2(R, 32 + i));
                                    dj += X[(NB + i) * kSlots + slot];
                                    const double ir = du_readlane(irl, 32 + i);
                                    const double fd = h ? du_factor(pivot, R, ir) : 0.0;
                                    du_row_op<NB>(T, fd, 32 + i);
                                    f = h ? fd : f;
                                }
                            }
                            // The mover's column is done: it takes the row
                            // operations' own column (1/R itself for the mover:
                            // 1 - f has lost R roundings, which the flush
                            // multiplies by rows that are R times too large).
                            T[k] = pivot ? (f != 0.0 ? irl : 1.0) : -f;
                            const int full = (int)(__popc(mask[0]) >= kDuMaxAcc) | (int)(__popc(mask[1]) >= kDuMaxAcc) |
                                             (int)(grow[0] > limit) | (int)(grow[1] > limit);
                            steps = full ? i + 1 : steps;
                        }
                        double head[kG];
#pragma unroll
                        for (int k = 0; k < kG; ++k) head[k] = T[k];
#pragma unroll
                        for (int k = 0; k + kG < NB; ++k) T[k] = T[k + kG];
#pragma unroll
                        for (int k = 0; k < kG; ++k) T[NB - kG + k] = head[k];
                    }
                    const unsigned mh = mask[h];
                    const bool mine = ((mh >> r) & 1u) && (kTwo || lane < 32);
                    const int pb = __popc(mh & ((1u << r) - 1u));
                    for (int i = lane; i < ND * kDuMaxAcc * (kDuMaxAcc + 1); i += kWave) sm[Lay::cinv + i] = 0.0;
                    du_wave_fence();
#pragma unroll
                    for (int hh = 0; hh < ND; ++hh) {
                        double *ci = sm + Lay::cinv + hh * kDuMaxAcc * (kDuMaxAcc + 1) + pb;
                        const bool put = mine && (!kTwo || h == hh);
#pragma unroll
                        for (int q = 0; q < NB; ++q) {
                            if ((mask[hh] >> q) & 1u) {
                                if (put) *ci = T[q];
                                ci += kDuMaxAcc + 1;
                            }
                        }
                    }
                    const int e = s.first[kTwo ? h : hb] + q0 + r;
                    if (mine) {
                        ctl[4 + 16 * h + pb] = r;
                        const double x = prop[slot], y = prop[kSlots + slot], z = prop[2 * kSlots + slot];
                        gp[e] = x;
                        gp[N + e] = y;
                        gp[2 * N + e] = z;
                        px[e] = x * s.inv_L;
                        py[e] = y * s.inv_L;
                        pz[e] = z * s.inv_L;
                    }
                    if (lane == 0) {
                        ctl[0] = (int)mask[0];
                        ctl[1] = (int)mask[1];
                        ctl[2] = steps;
                    }
                    if (given.trace && r < steps && (kTwo || lane < 32)) {
                        double *tr = given.trace + ((size_t)w * N + e) * kTraceCount;
                        tr[0] = rec_r;
                        tr[1] = rec_j;
                        tr[2] = mine ? 1.0 : 0.0;
                    }
                    const double lg = mine ? log(fabs(rec_r)) : 0.0;
                    const double l0 = wave_sum(!kTwo || h == 0 ? lg : 0.0), l1 = kTwo ? wave_sum(h == 1 ? lg : 0.0) : 0.0;
                    if (lane == 0) {
                        const double na = (double)(__popc(mask[0]) + __popc(mask[1]));
                        book[1 + hb] += l0;
                        if (kTwo) book[2] += l1;
                        book[3] += na;
                        book[4] += na;
                        book[5] += na;
                    }
                }
                __syncthreads();
                const int m0 = __popc((unsigned)ctl[0]), m1 = __popc((unsigned)ctl[1]);
                const int next = q0 + ctl[2];
                // The next block's proposals, beside the flush.
                if (wave == NW - 1 && next < n)
                    du_propose<kTwo>(s, prop, gp, given, w, sweep, book[0], hb, next, n - next < NB ? n - next : NB, lane);
#pragma unroll 1
                for (int h = 0; h < ND; ++h) {
                    const int m = h ? m1 : m0, d = kTwo ? h : hb;
                    if (m > 0)
                        du_flush<NB, TH, kTwo, NW>(l, sm, invw + s.inv_off[d], n, h, q0, m,
                                                   orbs + (!kTwo && hb ? s.n[0] : 0));
                }
                __syncthreads();
                q0 = next;
            }
        }
        if (t == 0) {
            if (flags & VMC_SWEEP_ADAPT) {
                const double sigma = book[0] * exp(0.25 * (book[4] / (double)N - 0.5));
                book[0] = sigma > 0.5 * s.L ? 0.5 * s.L : sigma;
            }
            book[4] = 0.0;
        }
        __syncthreads();
    }
    if (t == 0) {
        double *ws = st.stats + (size_t)w * kStatCount;
        ws[6] += book[3];
        ws[7] += (double)N * (double)n_sweeps;
        st.sigma[w] = book[0];
        st.since[w] = (int)book[5];
        st.flags[w] = st.flags[w] & ~kFlagJrowValid;  // this kernel keeps no row sums
        st.logdet[2 * w + 0] = book[1];
        st.logdet[2 * w + 1] = book[2];
    }
}

// Four wavefronts per SIMD: two resident walkers of eight wavefronts, so one
// walker's decisions overlap with the other's matrix work.  (Five wavefronts
// at 147 per spin, two row tiles each and 168 registers, took 2.52 ms against
// 1.70; six at 81, 0.84 against 0.60.)
template <int NB, int TH, bool kTwo, int NW>
__global__ __launch_bounds__(NW * kWave, 4) void k_sweep_du(DevSys s, DevState st, int n_sweeps,
                                                            unsigned long long sweep0, int flags, SweepGiven given) {
    du_sweep_walker<NB, TH, kTwo, NW>(s, st, blockIdx.x, n_sweeps, sweep0, flags, given);
}

namespace {

constexpr size_t kDuLdsLimit = 160 * 1024;

// Calls f.template operator()<NB, TH, kTwo, NW>() with the instantiation of a
// size: a block of 32 moves per determinant (16 up to 16 per spin), the row
// tile in registers up to 160 per spin (beyond, 16 rows of n doubles exceed a
// wavefront's registers).  Wavefronts per walker: four where a row tile
// has at most four column tiles, eight to 160, sixteen above, where few
// walkers have to fill the chip.
template <bool kTwo, typename F>
auto du_dispatch(int n, F f) {
    if (n <= 16) return f.template operator()<16, 1, kTwo, 4>();
    if (n <= 32) return f.template operator()<32, 2, kTwo, 4>();
    if (n <= 48) return f.template operator()<32, 3, kTwo, 4>();
    if (n <= 64) return f.template operator()<32, 4, kTwo, 4>();
    if (n <= 96) return f.template operator()<32, 6, kTwo, 8>();
    if (n <= 128) return f.template operator()<32, 8, kTwo, 8>();
    if (n <= 160) return f.template operator()<32, 10, kTwo, 8>();
    return f.template operator()<32, 0, kTwo, 16>();
}

bool du_two(const DevSys &d) { return d.ndet == 2 && d.n_up == d.n_dn; }

size_t du_lds(const DevSys &d) {
    const int norb = du_two(d) ? d.nmax : d.n[0] + (d.ndet == 2 ? d.n[1] : 0);
    const auto size = [&]<int NB, int TH, bool kTwo, int NW>() {
        using Lay = DuLds<NB, TH, kTwo, NW>;
        return d.kmax < Lay::K1 ? sizeof(double) * (size_t)Lay(d.N, d.nmax, norb).total : ~size_t(0);
    };
    return du_two(d) ? du_dispatch<true>(d.nmax, size) : du_dispatch<false>(d.nmax, size);
}

}  // namespace

bool du_fits(const DevSys &d) { return du_lds(d) <= kDuLdsLimit; }

bool du_launch(const DevSys &d, const DevState &st, unsigned grid, int n_sweeps, unsigned long long s0, int flags,
               const SweepGiven &given, hipStream_t stream) {
    if (!du_fits(d)) return false;
    const size_t lds = du_lds(d);
    const auto run = [&]<int NB, int TH, bool kTwo, int NW>() {
        const auto k = k_sweep_du<NB, TH, kTwo, NW>;
        // (up to the limit: the same from every thread, whatever its system)
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)kDuLdsLimit) != hipSuccess)
            return false;
        hipLaunchKernelGGL(k, dim3(grid), dim3(NW * kWave), lds, stream, d, st, n_sweeps, s0, flags, given);
        return true;
    };
    return du_two(d) ? du_dispatch<true>(d.nmax, run) : du_dispatch<false>(d.nmax, run);
}

}  // namespace vmc
