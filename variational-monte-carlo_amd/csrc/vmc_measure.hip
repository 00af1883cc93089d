// vmc_measure.hip -- the FP64 local energy from FP64 inverses in memory, six
// electrons and more (energy_tracking.cpp:253-382 with the Jastrow and Slater
// derivatives of jastrow_pade.cpp:57-138, slater_plane_wave.cpp:425-499).
//
// One workgroup per walker, 2 to 8 wavefronts by the number of electrons alone
// (a walker's result is the same in every launch).  Coordinates are kept in
// units of L.
//   - Pair terms: a thread owns one electron and one of S interleaved slices of
//     its partners (e + k) mod N, k = 1 .. N - 1: the Jastrow gradient and
//     Laplacian of its own side, and for k <= N/2 the pair's real-space Ewald
//     term.  Both sides of a pair
//     form its distance; in exchange no lane waits for another.
//   - Structure factor: with X, Y, Z the axis phasors,
//       S(mx, my, +-a) = sum_j (X^mx Y^my)_j (Z^a)_j^(conj)
//     is a matrix product over the electrons: rows the real and imaginary
//     parts of eight columns (mx, my), columns those of eight powers of Z, on
//     the FP64 matrix cores.  The four real products serve both signs of a.
//   - Slater terms: 16 electrons x 4 lanes per wavefront; a lane takes four
//     consecutive elements of its electron's inverse row per step (coalesced:
//     the four lanes read 128 B of a row), the phasors of their two wave
//     vectors as products of axis powers from LDS.
// The axis powers of 64 electrons at a time are staged in LDS for both.
//
// What bounds it: FP64 VALU issue (53 % of the cycles at N = 294), about 90
// instructions for a pair with its Ewald term and 50 without, at four walkers
// a CU.  Against the kernels that it replaced (one thread per G vector or
// column, inverse rows read an element at a time, barriers every few pair
// steps; and a sincospi per orbital and per G vector at sizes without an
// instantiation), per launch: N = 294, 1024 walkers 577 -> 319 us; N = 162,
// 1024 219 -> 115; N = 114, 2048 170 -> 122; N = 66, 1024 52 -> 39; N = 186, 512
// 290 -> 89; 19 + 7 electrons, 777 51 -> 19; 485 electrons, 8 walkers 876 -> 260.
#include "../../include/vmc_hip.h"
#include "vmc_device.hpp"
#include "vmc_rr_launch.hpp"
#include "vmc_walker.hpp"

#include <hip/hip_runtime.h>

namespace vmc {

namespace {

typedef double ms_v4d __attribute__((ext_vector_type(4)));
typedef double ms_v4u __attribute__((ext_vector_type(4), aligned(8)));

constexpr int kMsChunk = 64;      // electrons whose axis powers are staged at once
constexpr int kMsPitch = 68;      // their pitch: rows of powers start 16 banks apart
constexpr int kMsTiles = 3;       // structure-factor tiles a wavefront accumulates at once
constexpr int kMsMaxThreads = 512;

// Threads per walker: four wavefronts leave room for four walkers on a CU at
// 128 registers (1024 walkers at 147 per spin at once); above 384 electrons the
// walkers are few and eight finish one sooner.
__host__ __device__ inline int ms_threads(int N) { return N <= 40 ? 128 : N <= 384 ? 256 : kMsMaxThreads; }

struct MsLds {
    int pos, grad, ktab, kidx, work, red, total;  // doubles from the start
    __host__ __device__ MsLds(int N, int n0, int n1, int pmax) {
        const int nt = ms_threads(N);
        int o = 0;
        pos = o; o += 3 * N;              // x, y, z
        grad = o; o += 4 * N;             // per electron: Jastrow gradient and Laplacian
        const int pairs = n0 / 2 + n1 / 2;
        o = (o + 1) & ~1;
        ktab = o; o += 2 * pairs;         // per wave vector: n and |n|^2 (floats)
        kidx = o; o += (pairs + 1) / 2;   // the same packed
        o = (o + 1) & ~1;
        work = o;                         // partial pair sums, or the axis powers
        const int items = 4 * nt, powers = 3 * (pmax + 1) * kMsPitch * 2;
        o += items > powers ? items : powers;
        red = o; o += 4 * 8;
        total = o;
    }
};

// The local energy of walker w by the workgroup's first ms_threads(N) threads
// (the others only meet the barriers).  kParts: the parts and J into
// parts[w][kPartCount], the statistics untouched; else into the statistics.
template <bool kParts>
__device__ __forceinline__ void ms_walker(const DevSys &s, const DevState &st, int w, double *parts, int block_size, double *sm) {
    const int N = s.N, nt = ms_threads(N), nw = nt / kWave;
    const int t = threadIdx.x, wave = wave_uniform(t >> 6), lane = t & (kWave - 1);
    const MsLds l(N, s.n[0], s.ndet == 2 ? s.n[1] : 0, s.pmax);
    double *px = sm + l.pos, *py = px + N, *pz = py + N;
    double *grad = sm + l.grad;
    float4 *ktab = reinterpret_cast<float4 *>(sm + l.ktab);
    int *kidx = reinterpret_cast<int *>(sm + l.kidx);
    double *work = sm + l.work, *red = sm + l.red;
    const double *gp = st.pos + (size_t)w * 3 * N;
    const bool on = t < nt;
    for (int i = t; i < 3 * N && on; i += nt) px[i] = gp[i] * s.inv_L;
    // Wave vector p of determinant d is that of its orbitals 2p + 1 (cos) and
    // 2p + 2 (sin); orbital 0 is the constant.
    const int pairs0 = s.n[0] / 2;
    for (int p = t; p < pairs0 + (s.ndet == 2 ? s.n[1] / 2 : 0) && on; p += nt) {
        const int d = p >= pairs0 ? 1 : 0, q = p - (d ? pairs0 : 0);
        const int4 o = s.orb[d * s.nmax + 2 * q + 1];
        ktab[p] = make_float4((float)o.x, (float)o.y, (float)o.z, (float)(o.x * o.x + o.y * o.y + o.z * o.z));
        const int y = o.y < 0 ? -o.y : o.y, z = o.z < 0 ? -o.z : o.z;
        kidx[p] = o.x | (y << 8) | (z << 16) | (o.y < 0 ? 1 << 24 : 0) | (o.z < 0 ? 1 << 25 : 0);
    }
    __syncthreads();

    // ---------------------------------------------------------- pair terms
    double vreal = 0.0, jas = 0.0;
    {
        const double L = s.L, bl = s.b * L, m2b = -2.0 * s.b, two_il = 2.0 * s.inv_L, al = s.alpha * L;
        const double tiny = 1e-24 * s.inv_L * s.inv_L;
        // Exact erfc inside a cutoff its fit covers: the fit for every pair.
        const bool fit = s.erfc_kind == 1 && s.use_cut && s.alpha * s.rcut <= (double)kErfcFitMax;
        const double rc = s.use_cut ? s.rcut * s.inv_L : 1e300;
        // Passes of E electrons in S slices each, item = thread: as many
        // electrons as there are threads, then the rest in as many slices as
        // fit, or one slice more of fewer electrons where the two passes that
        // this makes are the shorter (162 electrons on 256 threads: 128 in 2
        // slices and 34 in 7 take 0.64 of 162 in one; a thread adds up the
        // slices of an electron, so there are at most 8 in the second).
        for (int e0 = 0, E = 0, S = 1; e0 < N; e0 += E) {
            const int rest = N - e0;
            S = 1;
            E = nt;
            if (rest < nt) {
                E = rest;
                S = nt / rest;
                const int E2 = nt / (S + 1), S2 = E2 < rest ? nt / (rest - E2) : 0;
                if (S2 > 0 && S2 <= 8 && S * (S + 1 + S2) < (S + 1) * S2) {
                    E = E2;
                    ++S;
                }
            }
            const int sl = t / E, e = e0 + t - sl * E;
            const bool act = on && sl < S;
            double gx = 0.0, gy = 0.0, gz = 0.0, lap = 0.0, uj = 0.0, vr = 0.0;
            if (act) {
                const double x = px[e], y = py[e], z = pz[e];
                // Partners of the other spin: j in [base, base + len).
                const int h = spin_of(s, e);
                const int base = h ? 0 : s.n_up, len = h ? s.n_up : N - s.n_up;
                double rmin = 1.0;
                const auto sums_zero = [&]() { gx = gy = gz = lap = uj = vr = 0.0; };
                // One partner; kEwald 0: derivatives only, 1: with the fitted
                // erfc, 2: with any erfc.  kSafe: a pair closer than 1e-12
                // (energy_tracking.cpp:132,139) counts as r = 0 with 1/r = 1
                // and no derivative; otherwise rmin shows that there was none.
                const auto pair = [&]<int kEwald, bool kSafe>(int k, double weight) {
                    // (e + k) mod N: the smaller of both as unsigned numbers
                    const unsigned ju = (unsigned)(e + k), jw = ju - (unsigned)N;
                    const int j = (int)(ju < jw ? ju : jw);
                    double dx = x - px[j], dy = y - py[j], dz = z - pz[j];
                    dx -= rint(dx);
                    dy -= rint(dy);
                    dz -= rint(dz);
                    const double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
                    const bool zero = kSafe && !(r2 >= tiny);
                    const double q2 = kSafe ? (zero ? 1.0 : r2) : fmax(r2, tiny);
                    if (!kSafe) rmin = fmin(rmin, r2);
                    // 1/rho from v_rsq_f64 and 1/(1 + b r) from v_rcp_f64 (2^-24
                    // relative), each with one third-order step
                    double yi = __builtin_amdgcn_rsq(q2);
                    const double ee = fma(-q2 * yi, yi, 1.0);
                    yi = fma(yi * ee, fma(ee, 0.375, 0.5), yi);
                    const double rho = kSafe && zero ? 0.0 : q2 * yi;
                    const double d = fma(bl, rho, 1.0);
                    double den = __builtin_amdgcn_rcp(d);
                    const double ed = fma(-d, den, 1.0);
                    den = fma(den, fma(ed, ed, ed), den);
                    const double aj = (unsigned)(j - base) < (unsigned)len ? s.a_anti : s.a_same;
                    const double ad = aj * den, d1 = kSafe && zero ? 0.0 : ad * den;
                    const double gf = d1 * yi;
                    gx = fma(gf, dx, gx);
                    gy = fma(gf, dy, gy);
                    gz = fma(gf, dz, gz);
                    lap = fma(d1, fma(m2b, den, two_il * yi), lap);
                    if (kParts) uj = fma(ad, L * rho, uj);
                    if constexpr (kEwald == 1) {
                        const double v = erfc_fit64(al * rho) * yi;
                        vr = fma(rho < rc ? weight : 0.0, v, vr);
                    } else if constexpr (kEwald == 2) {
                        if (rho < rc)
                            vr = fma(weight, erfc_r<double>(al * rho, s.erfc_kind) * (kSafe && zero ? L : yi), vr);
                    }
                };
                // k up to half way carry the pair's Ewald term (half of it
                // where both ends meet the pair).
                const int k0 = 1 + sl;
                const auto all = [&]<int kEwald, bool kSafe>() {
                    int k = k0;
#pragma unroll 2
                    for (; 2 * k < N; k += S) pair.template operator()<kEwald, kSafe>(k, 1.0);
                    if (2 * k == N) {
                        pair.template operator()<kEwald, kSafe>(k, 0.5);
                        k += S;
                    }
#pragma unroll 2
                    for (; k < N; k += S) pair.template operator()<0, kSafe>(k, 0.0);
                };
                if (fit) all.template operator()<1, false>();
                else all.template operator()<2, false>();
                if (rmin < tiny) {
                    sums_zero();
                    all.template operator()<2, true>();
                }
                vr *= s.inv_L;
            }
            vreal += vr;
            if (kParts) jas += uj;
            if (S > 1) {
                if (act) {
                    work[t] = gx;
                    work[nt + t] = gy;
                    work[2 * nt + t] = gz;
                    work[3 * nt + t] = lap;
                }
                __syncthreads();
                if (t < E) {
                    for (int c = 0; c < 4; ++c) {
                        double v = work[c * nt + t];
                        for (int i = 1; i < S; ++i) v += work[c * nt + i * E + t];
                        grad[c * N + e0 + t] = v;
                    }
                }
                __syncthreads();
            } else if (act) {
                grad[e] = gx;
                grad[N + e] = gy;
                grad[2 * N + e] = gz;
                grad[3 * N + e] = lap;
            }
        }
    }

    // ------------------------------- Slater terms and the structure factor
    double kin = 0.0, vq = 0.0;
    double2 *pw = reinterpret_cast<double2 *>(work);  // [axis][power][kMsPitch]
    const int P1 = s.pmax + 1;
    const int ntask = s.sf_tiles * s.sf_nz8;
    const int r = lane & 15, g = lane >> 4;
    for (int t0 = 0; t0 == 0 || t0 < ntask; t0 += nw * kMsTiles) {
        int xo[kMsTiles], yo[kMsTiles], zo[kMsTiles];
        double ys[kMsTiles];
        ms_v4d acc[kMsTiles];
#pragma unroll
        for (int i = 0; i < kMsTiles; ++i) {
            const int task = t0 + wave + nw * i;
            const bool in = wave < nw && task < ntask;
            const int2 c = in ? s.sf_col[(task / s.sf_nz8) * 8 + (r & 7)] : make_int2(0, 0);
            const int zt = in ? task % s.sf_nz8 : 0;
            const int za = zt * 8 + (r & 7);
            xo[i] = c.x * kMsPitch + g;
            yo[i] = (P1 + (c.y < 0 ? -c.y : c.y)) * kMsPitch + g;
            zo[i] = (2 * P1 + (za < P1 ? za : 0)) * kMsPitch + g;
            ys[i] = c.y < 0 ? -1.0 : 1.0;
            acc[i] = ms_v4d{0.0, 0.0, 0.0, 0.0};
        }
        for (int c0 = 0; c0 < N; c0 += kMsChunk) {
            __syncthreads();
            for (int i = t; i < 3 * kMsChunk && on; i += nt) {
                const int ax = i / kMsChunk, slot = i - ax * kMsChunk, e = c0 + slot;
                double sn = 0.0, cs = 0.0;
                if (e < N) {
                    double f = px[ax * N + e];
                    f -= rint(f);
                    sincos_2pi<double>(f, &sn, &cs);
                }
                // (an empty slot's powers are zero: it adds nothing)
                double2 p = make_double2(e < N ? 1.0 : 0.0, 0.0);
                for (int m = 0; m < P1; ++m) {
                    pw[(ax * P1 + m) * kMsPitch + slot] = p;
                    p = make_double2(p.x * cs - p.y * sn, p.x * sn + p.y * cs);
                }
            }
            __syncthreads();
            if (wave < nw) {
                const int cnt = N - c0 < kMsChunk ? N - c0 : kMsChunk;
                const int steps = (cnt + 3) / 4;
#pragma unroll
                for (int i = 0; i < kMsTiles; ++i) {
                    if (t0 + wave + nw * i >= ntask) break;
                    // rows r < 8: Re X^mx Y^my of column r; r >= 8: Im of column r - 8
#pragma unroll 4
                    for (int k = 0; k < steps; ++k) {
                        const double2 X = pw[xo[i] + 4 * k], Y = pw[yo[i] + 4 * k], Z = pw[zo[i] + 4 * k];
                        const double yi = Y.y * ys[i];
                        const double a = r < 8 ? fma(X.x, Y.x, -X.y * yi) : fma(X.x, yi, X.y * Y.x);
                        acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, r < 8 ? Z.x : Z.y, acc[i], 0, 0, 0);
                    }
                }
                for (int gi = wave; t0 == 0 && 16 * gi < cnt; gi += nw) {
                    const int slot = 16 * gi + r, e = c0 + slot < N ? c0 + slot : N - 1;
                    const int h = spin_of(s, e), n = s.n[h];
                    const double *row = reinterpret_cast<const double *>(st.inv) + (size_t)w * s.ninv + s.inv_off[h] +
                                        (size_t)(e - s.first[h]) * n + 1 + 4 * g;
                    const int p0 = (h ? pairs0 : 0) + 2 * g;
                    double sx = 0.0, sy = 0.0, sz = 0.0, sl = 0.0;
                    // columns m + 4 g .. m + 4 g + 3 of the row from 1 on
                    const auto load = [&](int m) {
                        ms_v4d c = {0.0, 0.0, 0.0, 0.0};
                        if (m + 16 < n) {
                            const ms_v4u u = *reinterpret_cast<const ms_v4u *>(row + m);
                            c = u;
                        } else {
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                if (1 + m + 4 * g + q < n) c[q] = row[m + q];
                        }
                        return c;
                    };
                    ms_v4d c1 = load(0), c2 = load(16);
                    for (int m = 0; m + 1 < n; m += 16) {
                        const ms_v4d c = c1;
                        c1 = c2;
                        c2 = load(m + 32);
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            // (past the last wave vector the weights are zero)
                            const int q = m / 2 + 2 * g + u;
                            const int p = 2 * q + 1 < n ? p0 + m / 2 + u : p0 - 2 * g;
                            const int o = n > 1 ? kidx[p] : 0;
                            const double2 X = pw[(o & 255) * kMsPitch + slot];
                            double2 Y = pw[(P1 + ((o >> 8) & 255)) * kMsPitch + slot];
                            double2 Z = pw[(2 * P1 + ((o >> 16) & 255)) * kMsPitch + slot];
                            Y.y = (o & (1 << 24)) ? -Y.y : Y.y;
                            Z.y = (o & (1 << 25)) ? -Z.y : Z.y;
                            const double xr = fma(X.x, Y.x, -X.y * Y.y), xi = fma(X.x, Y.y, X.y * Y.x);
                            const double re = fma(xr, Z.x, -xi * Z.y), im = fma(xr, Z.y, xi * Z.x);
                            const double wc = c[2 * u], ws = c[2 * u + 1];
                            const double gs = fma(ws, re, -wc * im);
                            const float4 kv = ktab[p];
                            sx = fma(gs, (double)kv.x, sx);
                            sy = fma(gs, (double)kv.y, sy);
                            sz = fma(gs, (double)kv.z, sz);
                            sl = fma(-fma(wc, re, ws * im), (double)kv.w, sl);
                        }
                    }
                    sx += __shfl_xor(sx, 16, kWave);
                    sy += __shfl_xor(sy, 16, kWave);
                    sz += __shfl_xor(sz, 16, kWave);
                    sl += __shfl_xor(sl, 16, kWave);
                    sx += __shfl_xor(sx, 32, kWave);
                    sy += __shfl_xor(sy, 32, kWave);
                    sz += __shfl_xor(sz, 32, kWave);
                    sl += __shfl_xor(sl, 32, kWave);
                    if (g == 0 && c0 + slot < N) {
                        const double ku = s.kunit;
                        sx *= ku;
                        sy *= ku;
                        sz *= ku;
                        sl *= ku * ku;
                        const double tx = sx + grad[e], ty = sy + grad[N + e], tz = sz + grad[2 * N + e];
                        kin += sl - (sx * sx + sy * sy + sz * sz) + grad[3 * N + e] + tx * tx + ty * ty + tz * tz;
                    }
                }
            }
        }
        // sum_G w_G |S_G|^2: lanes r < 8 hold the products with Re Z^a, lanes
        // r + 8 those with Im Z^a; registers 0, 1 the real, 2, 3 the imaginary
        // parts of columns g and 4 + g.
#pragma unroll
        for (int i = 0; i < kMsTiles; ++i) {
            const int task = t0 + wave + nw * i;
            double o[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q] = __shfl_xor(acc[i][q], 8, kWave);
            if (wave < nw && task < ntask && r < 8) {
                const int tile = task / s.sf_nz8, za = (task % s.sf_nz8) * 8 + r;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const double *wt = s.sf_w + (((size_t)tile * 8 + 4 * c + g) * (8 * s.sf_nz8) + za) * 2;
                    const double rr = acc[i][c], ri = o[c], ir = acc[i][2 + c], ii = o[2 + c];
                    const double pr = rr - ii, pi = ri + ir, mr = rr + ii, mi = ir - ri;
                    vq += wt[0] * (pr * pr + pi * pi) + wt[1] * (mr * mr + mi * mi);
                }
            }
        }
    }
    kin = wave_sum(kin);
    vreal = wave_sum(vreal);
    vq = wave_sum(vq);
    if (kParts) jas = wave_sum(jas);
    if (lane == 0 && wave < nw) {
        red[wave] = kin;
        red[8 + wave] = vreal;
        red[16 + wave] = vq;
        red[24 + wave] = jas;
    }
    __syncthreads();
    if (t != 0) return;
    double sum[4];
    for (int c = 0; c < 4; ++c) {
        sum[c] = red[8 * c];
        for (int i = 1; i < nw; ++i) sum[c] += red[8 * c + i];
    }
    Measured m;
    m.kinetic = -0.5 * sum[0];
    m.vreal = sum[1];
    m.vrecip = __dmul_rn(s.pref, sum[2]);
    m.e_local = m.kinetic + m.vreal + m.vrecip + s.e_const;
    if constexpr (kParts) {
        double *q = parts + (size_t)w * kPartCount;
        q[0] = m.kinetic;
        q[1] = m.vreal;
        q[2] = m.vrecip;
        q[3] = m.e_local;
        q[4] = st.logdet[2 * w + 0];
        q[5] = s.ndet == 2 ? st.logdet[2 * w + 1] : 0.0;
        q[6] = 0.5 * sum[3];
    } else {
        accumulate_measure(st.stats + (size_t)w * kStatCount, m, s.e_const, block_size);
    }
}

template <bool kParts>
__global__ __launch_bounds__(kMsMaxThreads, 4) void k_measure64(DevSys s, DevState st, double *parts,
                                                                int block_size) {
    extern __shared__ __align__(16) double sm[];
    ms_walker<kParts>(s, st, blockIdx.x, parts, block_size, sm);
}

// A batch group, its systems of one size or of several: one workgroup per
// walker of the group.  The walkers of a system that does not fit are
// k_measure_batch64's: the launch's LDS and threads are those of the others.
__global__ __launch_bounds__(kMsMaxThreads, 4) void k_measure64_b(const BatchItem *__restrict__ items, int n_items,
                                                                  int block_size) {
    extern __shared__ __align__(16) double sm[];
    const BatchItem &it = items[batch_find(items, n_items, blockIdx.x)];
    if (it.generic_energy) return;
    ms_walker<false>(it.s, it.st, blockIdx.x - it.walker_begin, nullptr, block_size, sm);
}

}  // namespace

size_t measure64_lds(const DevSys &d) {
    return sizeof(double) * (size_t)MsLds(d.N, d.n[0], d.ndet == 2 ? d.n[1] : 0, d.pmax).total;
}

// A system past the LDS limit, by its number of electrons or the reach of its
// reciprocal sum, keeps the generic local energy; so do the smallest, for which
// two wavefronts per walker and a staging pass cost more than they share out
// (one call, generic -> here: 1 + 0 electrons, 16384 walkers 157 -> 327 us, 2 + 2
// 201 -> 249, 3 + 2 217 -> 238, 3 + 3 232 -> 240, 6 + 0 240 -> 239, 5 + 5 301 ->
// 236; 2 + 1, one walker 34 -> 38, 6 + 0 40 -> 37).
constexpr int kMsMinN = 6;
bool measure64_fits(const DevSys &d) { return d.N >= kMsMinN && measure64_lds(d) <= kMeasure64LdsLimit; }

// Dynamic LDS above 64 KB has to be asked for, kernel by kernel; always up to
// the limit, so that two threads with systems of different sizes ask for the
// same.
static bool ms_allow(const void *kernel, size_t lds) {
    return lds <= 64 * 1024 || hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)kMeasure64LdsLimit) == hipSuccess;
}

bool measure64(const DevSys &d, const DevState &st64, unsigned grid, int bs, double *parts, hipStream_t stream) {
    if (!measure64_fits(d)) return false;
    const size_t lds = measure64_lds(d);
    if (!ms_allow(parts ? reinterpret_cast<const void *>(k_measure64<true>)
                        : reinterpret_cast<const void *>(k_measure64<false>), lds))
        return false;
    const dim3 block(static_cast<unsigned>(ms_threads(d.N)));
    if (parts)
        hipLaunchKernelGGL(k_measure64<true>, dim3(grid), block, lds, stream, d, st64, parts, bs);
    else
        hipLaunchKernelGGL(k_measure64<false>, dim3(grid), block, lds, stream, d, st64, parts, bs);
    return true;
}

bool measure64_batch(int max_n, size_t lds, const BatchItem *items_m64, int n_items, unsigned grid, int bs,
                     hipStream_t stream) {
    if (!ms_allow(reinterpret_cast<const void *>(k_measure64_b), lds)) return false;
    hipLaunchKernelGGL(k_measure64_b, dim3(grid), dim3(static_cast<unsigned>(ms_threads(max_n))), lds, stream,
                       items_m64, n_items, bs);
    return true;
}

}  // namespace vmc
