// vmc_sweep_rrw.hpp -- register-resident sweep for spins of 33 to 192
// electrons: one to three wavefronts per spin.
//
// The workgroup of a walker holds WPS wavefronts per determinant; thread
// (wave v, lane l) owns row r = (v mod WPS) * 64 + l of spin h = v / WPS:
// that electron's position, its Jastrow row sum U and its row of the spin's
// transposed inverse in registers.  A move of electron p (spin hp) is three
// phases with one workgroup barrier, between B and C:
//   A  every thread forms its new pair term against the proposal (DPP wave
//      sum -> LDS);
//   B  spin hp's rows form s_k = sum_m phi_m invT[k][m]: each of its
//      wavefronts forms the orbital row for itself from the staged powers of the
//      axis phasors and broadcasts it within the FMA (DPP); the mover publishes
//      R = s_p, its U, old position and inverse row;
//   C  every thread takes the same accept decision from the same LDS values;
//      on accept spin hp's rows apply Sherman-Morrison (one FMA per element,
//      the other spin's wavefronts skip it on a wave-uniform branch) and every
//      thread updates its U.
// What bounds it: the move's chain and VALU instructions (506 instead of 589
// in the FP32 loop at 57 per spin).  With the orbital row through LDS, a
// second barrier where a spin spans wavefronts, powers selected per move and, in FP64,
// IEEE roots and divisions: FP64 sweeps 202 -> 163 us at 57 per spin and 113 ->
// 87 at 33 (tens of walkers), FP32 285 -> 273 at 57 (2048 walkers) and, 1000
// walkers and more in a batch, 1878 -> 1657 at 81 per spin and 821 -> 744 at 33.
// Same chain as the one-wavefront kernel (the reference's
// src/simulation/simulation.cpp:80-156 with per-sweep electron order and
// Philox draws), same HBM layout, so ensembles switch kernels freely.
#pragma once

#include "vmc_sweep_rr.hpp"

namespace vmc {

__device__ __forceinline__ float fma_r(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_r(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename Real, int NU, int ND, int WPS>
struct RRWShared {
    static constexpr int N = NU + ND;
    static constexpr int NMAX = NU > ND ? NU : ND;
    static constexpr int NWAVE = (ND > 0 ? 2 : 1) * WPS;
    static constexpr int kMaxC = rr::max_component<NMAX>();
    // Axis-phasor entries of one electron's proposal: 1, X .. X^kMaxC, Y .., Z ..
    static constexpr int kPow = 1 + 3 * kMaxC;
    double pos[3][N];               // at the start of the sweep
    alignas(16) double prop[N][4];  // this sweep's proposals x, y, z and accept uniforms
    alignas(16) sf::Pair<Real> pow[N][kPow];
    // Rows padded to 16 bytes, so that a row picked at run time still moves
    // with 16-byte LDS reads.
    static constexpr int kRowPad = (NMAX + 3) / 4 * 4;
    alignas(16) Real row[2][kRowPad];   // inverse row of the (up) mover (by move parity)
    alignas(16) Real row2[2][kRowPad];  // inverse row of the down mover of a paired move
    double jred[2][NWAVE];   // per-wave new Jastrow pair sums (by move parity)
    double jred2[2][NWAVE];  // the same for the down proposal of a paired move
    alignas(16) double mv[2][8];   // (up) mover: R, U, x, y, z (by move parity)
    alignas(16) double mv2[2][8];  // down mover of a paired move
    double stat[kStatCount];
    double misc[4];      // sigma, log|det| up, log|det| down
};

template <typename Real, int NU, int ND, int WPS>
struct RRW {
    static constexpr int N = NU + ND;
    static constexpr int NMAX = NU > ND ? NU : ND;
    static constexpr int NWAVE = (ND > 0 ? 2 : 1) * WPS;
    static constexpr int NT = NWAVE * kWave;
    using Sh = RRWShared<Real, NU, ND, WPS>;
    static_assert(ND == 0 || ND == NU, "polarised or equal spins");
    static_assert(NMAX <= WPS * kWave, "rows per spin exceed the spin's wavefronts");
    static constexpr int kMaxC = Sh::kMaxC;
    static constexpr int kGroups = (NMAX + kWave - 1) / kWave;  // orbitals of a lane
    // Sizes whose sweep moves an up and a down electron per pass (move_pair):
    // measured faster there; at 81 and 123 per spin in FP32 (and 33, 57 in
    // FP64) the paired pass's registers cost more than it saves.
    static constexpr bool kPaired = ND == NU && (sizeof(Real) == 4 ? (NMAX == 33 || NMAX == 57 || NMAX == 147)
                                                                  : NMAX == 81);
    static_assert(kMaxC <= 3, "orbital phasors use powers up to 3");

    // Orbital m: its entries in Sh::pow (x | y << 4 | z << 8), the signs of its
    // y and z components (bits 31 and 30) and its type (bit 12).
    __device__ static int packed_orbital(const DevSys &s, int m) {
        const int4 o = s.orb[m < NU ? m : 0];
        const int ay = o.y < 0 ? -o.y : o.y, az = o.z < 0 ? -o.z : o.z;
        const int x = o.x, y = ay ? kMaxC + ay : 0, z = az ? 2 * kMaxC + az : 0;
        return x | (y << 4) | (z << 8) | (o.w << 12) | (o.y < 0 ? (int)0x80000000 : 0) | (o.z < 0 ? 0x40000000 : 0);
    }
    __device__ static float flip(float v, int sign) { return __int_as_float(__float_as_int(v) ^ (sign & (int)0x80000000)); }
    __device__ static double flip(double v, int sign) {
        return __longlong_as_double(__double_as_longlong(v) ^ ((long long)(sign & (int)0x80000000) << 32));
    }
    // Packed orbital ob at proposal p.
    __device__ static Real orbital(const Sh &sh, int ob, int p) {
        const sf::Pair<Real> *t = sh.pow[p];
        const sf::Pair<Real> X = t[ob & 15], Y = t[(ob >> 4) & 15], Z = t[(ob >> 8) & 15];
        // (which products are rounded and which fused is part of the FP32
        // chain, so it is written out)
        const Real yi = flip(Y.im, ob), zi = flip(Z.im, ob << 1);
        const Real re = fma_r(X.re, Y.re, -(X.im * yi));
        const Real im = kMaxC <= 2 ? fma_r(X.im, Y.re, X.re * yi) : fma_r(X.re, yi, X.im * Y.re);
        return ob & 0x1000 ? fma_r(im, Z.re, re * zi) : fma_r(re, Z.re, -(im * zi));
    }
    // s_k = sum_m phi_m(proposal p) invT[k][m] for the thread's row k: every
    // wavefront forms the whole orbital row, lane l orbitals l, 64 + l, ...,
    // and the FMA itself broadcasts them from its row of 16 lanes; even and
    // odd m in two sums.
    __device__ static Real ratio_row(const Sh &sh, const int (&ob)[kGroups], int p, const Real (&inv)[NMAX]) {
        Real s0 = (Real)0, s1 = (Real)0;
        const auto group = [&]<int g>() {
            constexpr int m0 = g * kWave;
            Real v[4];
            rr::spread_rows16(orbital(sh, ob[g], p), v);
            rr::dot_row16<NMAX, m0>(s0, s1, v[0], inv);
            if constexpr (NMAX > m0 + 16) rr::dot_row16<NMAX, m0 + 16>(s0, s1, v[1], inv);
            if constexpr (NMAX > m0 + 32) rr::dot_row16<NMAX, m0 + 32>(s0, s1, v[2], inv);
            if constexpr (NMAX > m0 + 48) rr::dot_row16<NMAX, m0 + 48>(s0, s1, v[3], inv);
        };
        group.template operator()<0>();
        if constexpr (kGroups > 1) group.template operator()<1>();
        if constexpr (kGroups > 2) group.template operator()<2>();
        return s0 + s1;
    }

    struct Thread {
        int v, lane, h, r, nh, e;
        bool has_e;
        __device__ Thread() {
            const int t = threadIdx.x;
            v = t >> 6;
            lane = t & (kWave - 1);
            h = ND > 0 ? v / WPS : 0;
            r = (v % WPS) * kWave + lane;
            nh = h ? ND : NU;
            has_e = r < nh;
            e = h ? NU + r : r;
        }
    };

    __device__ static void load(const DevSys &s, const DevState &st, int w, Sh &sh, const Thread &T,
                                Real (&inv)[NMAX], double &x, double &y, double &z) {
        const Real *blk = reinterpret_cast<const Real *>(st.inv) + (size_t)w * s.ninv;
#pragma unroll
        for (int m = 0; m < NMAX; ++m)
            inv[m] = (T.has_e && m < T.nh) ? blk[(T.h ? NU * NU : 0) + T.r * T.nh + m] : (Real)0;
        load_pos(s, st, w, sh, T, x, y, z);
    }

    // The thread's electron position, also into the LDS mirror.
    __device__ static void load_pos(const DevSys &, const DevState &st, int w, Sh &sh, const Thread &T,
                                    double &x, double &y, double &z) {
        const double *gp = st.pos + (size_t)w * 3 * N;
        x = T.has_e ? gp[T.e] : 0.0;
        y = T.has_e ? gp[N + T.e] : 0.0;
        z = T.has_e ? gp[2 * N + T.e] : 0.0;
        if (T.has_e) {
            sh.pos[0][T.e] = x;
            sh.pos[1][T.e] = y;
            sh.pos[2][T.e] = z;
        }
    }

    // Jastrow row sum of the thread's electron against every other.
    __device__ static double jastrow_row(const RRConst<Real> &c, const Sh &sh, const Thread &T,
                                         double x, double y, double z) {
        double U = 0.0;
        if (!T.has_e) return U;
        for (int j = 0; j < N; ++j) {
            if (j == T.e) continue;
            const Real dx = c.mi_r(x, sh.pos[0][j]);
            const Real dy = c.mi_r(y, sh.pos[1][j]);
            const Real dz = c.mi_r(z, sh.pos[2][j]);
            const Real rr_ = wsqrt<Real>(dx * dx + dy * dy + dz * dz);
            const Real a = ((ND > 0 && j >= NU) ? 1 : 0) == T.h ? c.a_same : c.a_anti;
            U += (double)(a * rr_ * wrcp<Real>((Real)1 + c.b * rr_));
        }
        return U;
    }

    // The moves of up electron i and then down electron i (the sweep order
    // of equal spins) in one pass: each spin's wavefronts form their orbital
    // row and ratios at their spin's proposal, and every thread forms its pair
    // terms with both proposals.  The down move then takes the up move's
    // outcome into its Jastrow change (the pair terms of the up electron with
    // the down electron, formed as the threads form them).  Same decisions
    // and updates as two calls of move.  Returns the accepted moves.
    __device__ static int move_pair(const RRConst<Real> &c, Sh &sh, const Thread &T, Real (&inv)[NMAX],
                                    double &x, double &y, double &z, double &U, const int (&ob)[kGroups], int i, int par,
                                    LogDetTrack &ldt, double *rec) {
        static_assert(ND == NU, "paired moves need equal spins");
        const int pu = i, pd = NU + i;
        const double xu = sh.prop[pu][0], yu = sh.prop[pu][1], zu = sh.prop[pu][2];
        const double xd = sh.prop[pd][0], yd = sh.prop[pd][1], zd = sh.prop[pd][2];
        // Phase A.
        Real un_u = (Real)0, un_d = (Real)0;
        if (T.has_e && T.e != pu) un_u = pair_with(c, x, y, z, xu, yu, zu, T.h == 0 ? c.a_same : c.a_anti);
        if (T.has_e && T.e != pd) un_d = pair_with(c, x, y, z, xd, yd, zd, T.h == 1 ? c.a_same : c.a_anti);
        if constexpr (sizeof(Real) == 8) {
            double wu, wd;
            rr::wave_totals(un_u, un_d, wu, wd);
            if (T.lane == 0) {
                sh.jred[par][T.v] = wu;
                sh.jred2[par][T.v] = wd;
            }
        } else {
            const Real wu = rr::wave_total(un_u), wd = rr::wave_total(un_d);
            if (T.lane == 0) {
                sh.jred[par][T.v] = (double)wu;
                sh.jred2[par][T.v] = (double)wd;
            }
        }
        // Phase B: every thread's s_k with its spin's orbital row; the two
        // movers publish their values and rows.
        const Real sk = ratio_row(sh, ob, T.h ? pd : pu, inv);
        if (T.r == i) {
            double *mvp = T.h ? sh.mv2[par] : sh.mv[par];
            Real *rowp = T.h ? sh.row2[par] : sh.row[par];
            mvp[0] = (double)sk;
            mvp[1] = U;
            mvp[2] = x;
            mvp[3] = y;
            mvp[4] = z;
#pragma unroll
            for (int m = 0; m < NMAX; ++m) rowp[m] = inv[m];
        }
        __syncthreads();
        double jn_u = 0.0, jn_d = 0.0;
#pragma unroll
        for (int v = 0; v < NWAVE; ++v) {
            jn_u += sh.jred[par][v];
            jn_d += sh.jred2[par][v];
        }
        // Phase C, up move.
        const double Ru = sh.mv[par][0];
        const double uxo = sh.mv[par][2], uyo = sh.mv[par][3], uzo = sh.mv[par][4];
        const double dj_u = jn_u - sh.mv[par][1];
        const int acc_u = accept_test(Ru, dj_u, sh.prop[pu][3]);
        double Ud = sh.mv2[par][1];
        if (acc_u) {
            ldt.add(0, Ru);
            if (T.h == 0) {
                const Real inv_ratio = wrcp<Real>((Real)Ru);
                Real f = (T.r == i) ? (Real)1 - inv_ratio : sk * inv_ratio;
                f = T.has_e ? f : (Real)0;
#pragma unroll
                for (int m = 0; m < NMAX; ++m) inv[m] -= sh.row[par][m] * f;
            }
            if (T.has_e && T.e != pu)
                U += (double)un_u - (double)pair_with(c, x, y, z, uxo, uyo, uzo, T.h == 0 ? c.a_same : c.a_anti);
            if (T.has_e && T.e == pu) {
                U = jn_u;
                x = xu;
                y = yu;
                z = zu;
            }
            // The down mover's row sum after this update, and the down
            // proposal's pair with the up electron where it now is: the up
            // electron's new and old place with the down mover and with the
            // down proposal, one of the four pairs in each lane of four.
            const double *up = T.lane & 1 ? &sh.mv[par][2] : &sh.prop[pu][0];
            const double *dn = T.lane & 2 ? &sh.prop[pd][0] : &sh.mv2[par][2];
            const Real four = pair_with(c, dn[0], dn[1], dn[2], up[0], up[1], up[2], c.a_anti);
            Ud += (double)rr::readlane(four, 0) - (double)rr::readlane(four, 1);
            const Real ud_new = rr::readlane(four, 2), ud_old = rr::readlane(four, 3);
            jn_d += (double)ud_new - (double)ud_old;
            if (T.has_e && T.e == pu) un_d = ud_new;
        }
        // Phase C, down move.
        const double Rd = sh.mv2[par][0];
        const double dj_d = jn_d - Ud;
        const int acc_d = accept_test(Rd, dj_d, sh.prop[pd][3]);
        if (rec && threadIdx.x == 0) {
            double *ru = rec + kTraceCount * pu, *rd = rec + kTraceCount * pd;
            ru[0] = Ru;
            ru[1] = dj_u;
            ru[2] = (double)acc_u;
            rd[0] = Rd;
            rd[1] = dj_d;
            rd[2] = (double)acc_d;
        }
        if (acc_d) {
            ldt.add(1, Rd);
            if (T.h == 1) {
                const Real inv_ratio = wrcp<Real>((Real)Rd);
                Real f = (T.r == i) ? (Real)1 - inv_ratio : sk * inv_ratio;
                f = T.has_e ? f : (Real)0;
#pragma unroll
                for (int m = 0; m < NMAX; ++m) inv[m] -= sh.row2[par][m] * f;
            }
            const double dxo = sh.mv2[par][2], dyo = sh.mv2[par][3], dzo = sh.mv2[par][4];
            if (T.has_e && T.e != pd)
                U += (double)un_d - (double)pair_with(c, x, y, z, dxo, dyo, dzo, T.h == 1 ? c.a_same : c.a_anti);
            if (T.has_e && T.e == pd) {
                U = jn_d;
                x = xd;
                y = yd;
                z = zd;
            }
        }
        return acc_u + acc_d;
    }

    // One move of electron p, the sweep's move number par (mod 2) selecting
    // the LDS buffers phase C reads.  Returns 1 if accepted (uniform).
    __device__ static int move(const RRConst<Real> &c, Sh &sh, const Thread &T, Real (&inv)[NMAX],
                               double &x, double &y, double &z, double &U, const int (&ob)[kGroups], int p, int par,
                               LogDetTrack &ldt, double *rec) {
        const int hp = (ND > 0 && p >= NU) ? 1 : 0;
        const int rp = hp ? p - NU : p;
        // Phase A.
        const double xn = sh.prop[p][0], yn = sh.prop[p][1], zn = sh.prop[p][2];
        const Real apair = T.h == hp ? c.a_same : c.a_anti;
        Real un = (Real)0;
        if (T.has_e && T.e != p) un = pair_with(c, x, y, z, xn, yn, zn, apair);
        {
            const Real ws = rr::wave_total(un);
            if (T.lane == 0) sh.jred[par][T.v] = (double)ws;
        }
        // Each of the mover's wavefronts forms the orbital row for itself, so
        // one workgroup barrier serves a move.  The mover's values and the
        // pair sums that phase C reads alternate between two buffers by move
        // parity, so a wavefront already in the next move's phase A or B
        // cannot overwrite what a slower one still reads.
        // Phase B.
        Real sk = (Real)0;
        if (T.h == hp) {
            sk = ratio_row(sh, ob, p, inv);
            if (T.r == rp) {
                sh.mv[par][0] = (double)sk;
                sh.mv[par][1] = U;
                sh.mv[par][2] = x;
                sh.mv[par][3] = y;
                sh.mv[par][4] = z;
#pragma unroll
                for (int m = 0; m < NMAX; ++m) sh.row[par][m] = inv[m];
            }
        }
        __syncthreads();
        double jn = 0.0;
#pragma unroll
        for (int i = 0; i < NWAVE; ++i) jn += sh.jred[par][i];
        // Phase C: the same decision in every thread (simulation.cpp:125-131),
        // exact FP64 exponential within 1e-5 of the threshold.
        const double R = sh.mv[par][0];
        const double dj = jn - sh.mv[par][1];
        const double ua = sh.prop[p][3];
        const int acc = accept_test(R, dj, ua);
        if (rec && threadIdx.x == 0) {
            double *q = rec + kTraceCount * p;
            q[0] = R;
            q[1] = dj;
            q[2] = (double)acc;
        }
        if (!acc) return 0;
        ldt.add(hp, R);
        if (T.h == hp) {
            const Real inv_ratio = wrcp<Real>((Real)R);
            Real f = (T.r == rp) ? (Real)1 - inv_ratio : sk * inv_ratio;
            f = T.has_e ? f : (Real)0;
#pragma unroll
            for (int m = 0; m < NMAX; ++m) inv[m] -= sh.row[par][m] * f;
        }
        if (T.has_e && T.e != p)
            U += (double)un - (double)pair_with(c, x, y, z, sh.mv[par][2], sh.mv[par][3], sh.mv[par][4], apair);
        if (T.has_e && T.e == p) {
            U = jn;
            x = xn;
            y = yn;
            z = zn;
        }
        return 1;
    }
};

// Proposal q (in [0, L)) of electron e, its axis phasors' powers and accept
// uniform ua into the electron's slots.
template <typename Real, typename Sh>
__device__ __forceinline__ void rrw_stage_proposal(const DevSys &s, const double (&q)[3], double ua, int e, Sh &sh) {
    sf::Pair<Real> *t = sh.pow[e];
    t[0] = {(Real)1, (Real)0};
    for (int k = 0; k < 3; ++k) {
        sh.prop[e][k] = q[k];
        const rr::Cx<Real> a = rr::axis_phasor<Real>(q[k], s.inv_L);
        t[1 + k * Sh::kMaxC] = {a.re, a.im};
        if constexpr (Sh::kMaxC >= 2) {
            const Real c = a.re * a.im;
            const rr::Cx<Real> a2{fma_r(a.re, a.re, -(a.im * a.im)), c + c};
            t[2 + k * Sh::kMaxC] = {a2.re, a2.im};
            if constexpr (Sh::kMaxC >= 3)
                t[3 + k * Sh::kMaxC] = {fma_r(a.re, a2.re, -(a.im * a2.im)), fma_r(a.re, a2.im, a.im * a2.re)};
        }
    }
    sh.prop[e][3] = ua;
}

// Philox draws of one electron for this sweep into its proposal slots.
template <typename Real, typename Sh>
__device__ __forceinline__ void rrw_proposal(const DevSys &s, double sigma, double x0, double y0, double z0, int e,
                                             int w, uint32_t sweep, Sh &sh) {
    const uint4 rm = philox4x32_10(make_uint4((uint32_t)e, (uint32_t)w, sweep, kTagMove), s.key0, s.key1);
    const uint4 ra = philox4x32_10(make_uint4((uint32_t)e, (uint32_t)w, sweep, kTagAccept), s.key0, s.key1);
    double dx, dy, dz;
    if (s.move_kind == 1) {
        const double rho0 = sqrt(-2.0 * log(u01(rm.x)));
        const double rho1 = sqrt(-2.0 * log(u01(rm.z)));
        double s0, c0, s1, c1;
        sincospi(2.0 * u01(rm.y), &s0, &c0);
        sincospi(2.0 * u01(rm.w), &s1, &c1);
        dx = rho0 * c0;
        dy = rho0 * s0;
        dz = rho1 * c1;
    } else {
        dx = 2.0 * u01(rm.x) - 1.0;
        dy = 2.0 * u01(rm.y) - 1.0;
        dz = 2.0 * u01(rm.z) - 1.0;
    }
    const double x = x0 + sigma * dx, y = y0 + sigma * dy, z = z0 + sigma * dz;
    const double q[3] = {x - s.L * floor(x * s.inv_L), y - s.L * floor(y * s.inv_L),
                         z - s.L * floor(z * s.inv_L)};
    rrw_stage_proposal<Real>(s, q, u01(ra.x), e, sh);
}

// kGiven: the moves come from the caller (SweepGiven) instead of Philox and
// each move's ratio, Jastrow change and decision are recorded.
template <typename Real, int NU, int ND, int WPS, bool kGiven = false>
__device__ __forceinline__ void sweep_rrw_body(const DevSys &s, const DevState &st, int w,
                                               unsigned long long sweep0, int flags,
                                               SweepGiven given = SweepGiven{}) {
    using K = RRW<Real, NU, ND, WPS>;
    constexpr int N = K::N;
    constexpr int NMAX = K::NMAX;
    __shared__ typename K::Sh sh;
    const RRConst<Real> cst(s);
    const typename K::Thread T;
    Real inv[NMAX];
    double x, y, z;
    K::load(s, st, w, sh, T, inv, x, y, z);
    if (threadIdx.x < kStatCount) sh.stat[threadIdx.x] = st.stats[(size_t)w * kStatCount + threadIdx.x];
    if (threadIdx.x == 0) {
        sh.misc[0] = st.sigma[w];
        sh.misc[1] = st.logdet[2 * w + 0];
        sh.misc[2] = st.logdet[2 * w + 1];
    }
    __syncthreads();
    const int wflags = st.flags[w];
    double U;
    if (!(wflags & kFlagJrowValid) || ((uint32_t)sweep0 % kJrowRefresh) == 0)
        U = K::jastrow_row(cst, sh, T, x, y, z);
    else
        U = T.has_e ? st.jrow[(size_t)w * N + T.e] : 0.0;
    int ob[K::kGroups];
#pragma unroll
    for (int g = 0; g < K::kGroups; ++g) ob[g] = K::packed_orbital(s, g * kWave + T.lane);
    double *rec = nullptr;
    if constexpr (kGiven) {
        if (T.has_e) {
            const size_t q = (size_t)w * N + T.e;
            const double p3[3] = {given.prop[3 * q], given.prop[3 * q + 1], given.prop[3 * q + 2]};
            rrw_stage_proposal<Real>(s, p3, given.u[q], T.e, sh);
        }
        rec = given.trace + (size_t)w * N * kTraceCount;
    } else {
        if (T.has_e)
            rrw_proposal<Real>(s, sh.misc[0], x, y, z, T.e, w, (uint32_t)sweep0, sh);
    }
    __syncthreads();
    int acc = 0;
    LogDetTrack ldt;
    if constexpr (K::kPaired) {
#pragma unroll 1
        for (int i = 0; i < NU; ++i) acc += K::move_pair(cst, sh, T, inv, x, y, z, U, ob, i, i & 1, ldt, rec);
    } else if constexpr (ND > 0 && sizeof(Real) == 8) {
        // The sweep order up i, down i as two calls with constant spin and
        // buffer parity (the move's addressing then folds; in FP32 at 81 and
        // 123 per spin the doubled loop body measured slower).
#pragma unroll 1
        for (int i = 0; i < NU; ++i) {
            acc += K::move(cst, sh, T, inv, x, y, z, U, ob, i, 0, ldt, rec);
            acc += K::move(cst, sh, T, inv, x, y, z, U, ob, NU + i, 1, ldt, rec);
        }
    } else {
#pragma unroll 1
        for (int t = 0; t < N; ++t)
            acc += K::move(cst, sh, T, inv, x, y, z, U, ob, sweep_visit(NU, ND, t), t & 1, ldt, rec);
    }
    __syncthreads();
    if (flags & VMC_SWEEP_ADAPT) {
        const double f = exp(0.25 * ((double)acc / (double)N - 0.5));
        if (threadIdx.x == 0) {
            const double sigma = sh.misc[0] * f;
            sh.misc[0] = sigma > 0.5 * s.L ? 0.5 * s.L : sigma;
        }
    }
    Real *blk = reinterpret_cast<Real *>(st.inv) + (size_t)w * s.ninv;
    if (T.has_e) {
#pragma unroll
        for (int m = 0; m < NMAX; ++m)
            if (m < T.nh) blk[(T.h ? NU * NU : 0) + T.r * T.nh + m] = inv[m];
        double *gq = st.pos + (size_t)w * 3 * N;
        gq[T.e] = x;
        gq[N + T.e] = y;
        gq[2 * N + T.e] = z;
        st.jrow[(size_t)w * N + T.e] = U;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        sh.stat[6] += (double)acc;
        sh.stat[7] += (double)N;
        st.sigma[w] = sh.misc[0];
        // (a count at K was re-inverted after the last sweep)
        st.since[w] = (s.reinv_k > 0 && st.since[w] >= s.reinv_k ? 0 : st.since[w]) + acc;
        st.flags[w] = wflags | kFlagJrowValid;
        st.logdet[2 * w + 0] = ldt.fold(0, sh.misc[1]);
        if (ND > 0) st.logdet[2 * w + 1] = ldt.fold(1, sh.misc[2]);
    }
    __syncthreads();
    if (threadIdx.x < kStatCount) st.stats[(size_t)w * kStatCount + threadIdx.x] = sh.stat[threadIdx.x];
}

// Waves per SIMD the sweep kernel is compiled for.  57 + 57 and 81 + 81 in
// FP32 take four (at most 128 VGPRs, 56 and 68 B of spill per lane; 84 and 68 in
// a batch): eight and four walkers per CU, so 2048 and 1024 walkers are resident
// at once.  123 + 123 takes three (168 VGPRs, 76 B of spill, 128 in a batch), FP64
// 57 + 57 as well (168, 32 B); 147 + 147 stays at two (244 VGPRs; three would spill
// 144 B of its inverse row per lane and run at half speed).
template <typename Real, int NU, int ND, int WPS>
constexpr int rrw_sweep_waves() {
    return (sizeof(Real) == 4 && ((NU == 57 && ND == 57) || (NU == 81 && ND == 81))) ? 4
           : (NU == 123 && ND == 123) || (sizeof(Real) == 8 && NU == 57 && ND == 57) ? 3 : 1;
}

template <typename Real, int NU, int ND, int WPS>
VMC_FMAC64 __global__ __launch_bounds__((ND > 0 ? 2 : 1) * WPS * 64, (rrw_sweep_waves<Real, NU, ND, WPS>())) void k_sweep_rrw(DevSys s, DevState st,
                                                                          unsigned long long sweep0,
                                                                          int flags) {
    sweep_rrw_body<Real, NU, ND, WPS>(s, st, blockIdx.x, sweep0, flags);
}

// The sweep with the caller's moves, each recorded (parity checks of the
// timed move code).
template <typename Real, int NU, int ND, int WPS>
VMC_FMAC64 __global__ __launch_bounds__((ND > 0 ? 2 : 1) * WPS * 64, (rrw_sweep_waves<Real, NU, ND, WPS>())) void k_sweep_rrw_given(
    DevSys s, DevState st, int flags, SweepGiven given) {
    sweep_rrw_body<Real, NU, ND, WPS, true>(s, st, blockIdx.x, 0, flags, given);
}

// Batch forms over a group of systems of one size (as k_sweep_rr_b).
template <typename Real, int NU, int ND, int WPS>
VMC_FMAC64 __global__ __launch_bounds__((ND > 0 ? 2 : 1) * WPS * 64, (rrw_sweep_waves<Real, NU, ND, WPS>())) void k_sweep_rrw_b(
    const BatchItem *__restrict__ items, int n_items, const unsigned long long *__restrict__ sweep_ctr,
    int flags) {
    const BatchItem &it = items[batch_find(items, n_items, blockIdx.x)];
    sweep_rrw_body<Real, NU, ND, WPS>(it.s, it.st, blockIdx.x - it.walker_begin, *sweep_ctr, flags);
}

}  // namespace vmc
