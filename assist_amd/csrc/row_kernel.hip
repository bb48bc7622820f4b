// The integration kernel with 16 lanes (one DPP row) per system, four systems per wave.
//
// ias15_kernel (kernels.hip) gives every vector of a system one lane, which then carries three
// components of the IAS15 state, and evaluates a system's 28 ephemeris slots and 27 bodies on 8
// lanes in four rounds.  A trip of its loop issues about 2 600 vector instructions for the 8 systems
// of a wave, and as many for a wave that holds a single one, which is what bounds single orbits,
// small batches and the tail of uneven ones.  Here a trip is shorter:
//
//   * one component of one vector per lane (lane 4 q + c of the row: component c of the vectors q
//     and q + 4), with b and g in registers: predictor, corrector and step end run on one component
//     of one or two vectors instead of three components;
//   * two rounds of bodies (slots 0-15 and 16-27) instead of four;
//   * the ephemeris of a step, which depends on times alone, is evaluated once per step attempt
//     for its start and its seven substeps together, by all 64 lanes of the wave (slot 8 r + i and
//     time k on lane 8 i + k of round r: four rounds, and the lanes of one slot mostly read the same
//     record), with the composed positions, the Sun's velocity and the EIH sums that no particle
//     enters, and kept in LDS for every trip of the attempt.
//
// Every operation on a system's data is the one that ias15_kernel does, with the same operands in
// the same order (the sums over bodies run in the order of its 8 lanes: slots l, l + 8, l + 16,
// l + 24, then the butterfly over l), so the results are equal bit for bit.
//
// What bounds it: a wave's instruction issue and dependencies on one trip (about 1 200 vector
// instructions in FP64 with variational vectors, 800 without), the same for one to four systems in the
// wave.  Two waves per SIMD overlap theirs, and the ephemeris tables leave LDS for six waves per CU.
// Measured on an MI355X against the 8-lane kernel: one system, FP64, 1.95 us per evaluation (4.67)
// alone and 3.3 us (5.5) with 6 vectors; 4,096 x 7 vectors over 3,650 d 37 ms (61); 262,144 x 7 over
// 365 d in the mixed form 107 ms (143); 65,536 uneven real-only spans up to 10,000 d 152 ms (297).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_types.h"
#include "force_model.h"
#include "ias15_device.h"
#include "kernels.h"

namespace assist_gpu {

// A system's ephemeris of one step attempt in LDS: for each of 8 times (the step's start, then
// its substeps 1-7) the barycentric positions of the 27 bodies (au, 81 words), the Sun's velocity
// (81-83), sum_k GM_k / r_sk (84) and the Sun's Newtonian acceleration (85-87).
constexpr int kRowSunVel = 81, kRowS1 = 84, kRowAj = 85;
static_assert(kRowSlice == 88, "27 bodies, the Sun's velocity and the four EIH sums");

#if defined(__HIP_DEVICE_COMPILE__)
enum : int { kDppRowRor8 = 0x128, kDppRowBcast = 0x150 };
template <int I, typename T>
__device__ __forceinline__ T row_bcast(T v) { return dpp<kDppRowBcast + I>(v); }
template <typename T>
__device__ __forceinline__ T row_swap8(T v) { return dpp<kDppRowRor8>(v); }
template <int J, typename T>
__device__ __forceinline__ T quad_bcast(T v) { return dpp<dpp_quad(J, J, J, J)>(v); }
__device__ __forceinline__ int row_bcast0_i(int v) { return dpp_i<kDppRowBcast>(v); }
// Butterfly over the 8 lanes of each half row (all of them end with the half's total), then the
// upper half's total on every lane of the row.
template <typename T>
__device__ __forceinline__ T upper_sum(T v) {
    v += dpp<kDppXor1>(v);
    v += dpp<kDppXor2>(v);
    v += dpp<kDppHalfMirror>(v);
    return row_bcast<8>(v);
}
__device__ __forceinline__ double row_max(double v) {
    v = fmax(v, dpp<kDppXor1>(v));
    v = fmax(v, dpp<kDppXor2>(v));
    v = fmax(v, dpp<kDppHalfMirror>(v));
    return fmax(v, row_swap8(v));
}
__device__ __forceinline__ double readlane_d(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}
#else
// (the host pass only type-checks the kernels)
template <int I, typename T> __device__ T row_bcast(T v);
template <typename T> __device__ T row_swap8(T v);
template <int J, typename T> __device__ T quad_bcast(T v);
__device__ int row_bcast0_i(int v);
template <typename T> __device__ T upper_sum(T v);
__device__ double row_max(double v);
__device__ double readlane_d(double v, int l);
#endif

// Sum over the bodies of -p d (a point mass's pull p = GM / r^3 along d), in the order of the
// 8-lane kernel: lane l takes slots l, l + 8, l + 16 and l + 24 in turn.  Here slots i and 16 + i
// are on lane i of the row (operands 0 and 1), so the running sum crosses between the row's halves
// three times and the upper half's butterfly ends it.
template <typename T>
__device__ __forceinline__ T sum_pull(T p0, T d0, T p1, T d1) {
    T a = fma(-p0, d0, T(0));
    a = row_swap8(a);
    a = fma(-p0, d0, a);
    a = row_swap8(a);
    a = fma(-p1, d1, a);
    a = row_swap8(a);
    a = fma(-p1, d1, a);
    return upper_sum(a);
}
// The same for the Jacobian's g e.
template <typename T>
__device__ __forceinline__ T sum_jac(T g0, T e0, T g1, T e1) {
    T a = fma(g0, e0, T(0));
    a = row_swap8(a);
    a = fma(g0, e0, a);
    a = row_swap8(a);
    a = fma(g1, e1, a);
    a = row_swap8(a);
    a = fma(g1, e1, a);
    return upper_sum(a);
}

// x^2 + y^2 + z^2 with the rounding of the 8-lane kernel's rounds: its second round (slots 8-15,
// `second`) rounds x^2 first, the others y^2.
template <typename T>
__device__ __forceinline__ T norm2(bool second, T x, T y, T z) {
    const T u = second ? y : x, w = second ? x : y;
    return fma(z, z, fma(u, u, w * w));
}

// The ephemeris of one step attempt (times t and t + dts h_1..h_7) into `T`, by all 64 lanes of a
// wave; t, dts and T are uniform.
__device__ __forceinline__ void row_ephemeris(const DevEphem& E, const double* h, double t, double dts, bool eih, double* T) {
    const int wl = __lane_id();
    const int i = wl >> 3, k = wl & 7;
    const double te = k == 0 ? t : fma(dts, h[k], t);
    const int short_from = __builtin_amdgcn_readfirstlane(E.short_from);
    const double inv_au = E.inv_au, inv_au_ast = E.inv_au_ast;
    double* const S = T + k * kRowSlice;
    double sun[3];
    double s1 = 0.0, aj[3] = {0.0, 0.0, 0.0};
    auto newton = [&](int b, bool second, const double pk[3]) {
        const double GM = E.GM[b];
        const double sx = sun[0] - pk[0], sy = sun[1] - pk[1], sz = sun[2] - pk[2];
        const double q2 = norm2(second, sx, sy, sz);
        const double iq = inv_sqrt(q2);
        s1 = fma(GM, iq, s1);
        const double f = GM * (iq * iq * iq);
        aj[0] = fma(-f, sx, aj[0]);
        aj[1] = fma(-f, sy, aj[1]);
        aj[2] = fma(-f, sz, aj[2]);
    };
    {
        // slots 0-7: the Sun with its velocity, Mercury, Venus, the EMB, the Earth and Moon
        // relative to it, Mars, Jupiter
        const ChebOut<double> o = cheb_eval<double, true>(E.slot[i], te);
        double p[3] = {o.x, o.y, o.z};
        const bool em = (i == kSlotEarth || i == kSlotMoon);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double emb = __shfl(p[c], 8 * kSlotEMB + k, 64);
            p[c] = (em ? p[c] + emb : p[c]) * inv_au;
            sun[c] = __shfl(p[c], k, 64);
        }
        const int b = i < 3 ? i : i - 1;
        if (i != kSlotEMB) {
#pragma unroll
            for (int c = 0; c < 3; c++) S[3 * b + c] = p[c];
        }
        if (i == 0) {
            S[kRowSunVel] = o.vx * inv_au;
            S[kRowSunVel + 1] = o.vy * inv_au;
            S[kRowSunVel + 2] = o.vz * inv_au;
        } else if (eih && i != kSlotEMB) {
            newton(b, false, p);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    {
        // slots 8-15: Saturn, Uranus, Neptune, Pluto, then asteroids
        const int s = 8 + i;
        const ChebOut<double> o = (short_from <= 8) ? cheb_eval<double, false, false, kCoefShort>(E.slot[s], te)
                                                    : cheb_eval<double, false>(E.slot[s], te);
        const bool ast = s >= kFirstAsteroidSlot;
        const double q[3] = {o.x, o.y, o.z};
        double p[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            p[c] = ast ? fma(q[c], inv_au_ast, sun[c]) : q[c] * inv_au;
            S[3 * (s - 1) + c] = p[c];
        }
        if (eih && !ast) newton(s - 1, true, p);
    }
    if (eih) {
        // the sums over the planets, in the order of 8 lanes (slots l and l + 8 above, then the
        // butterfly over l)
#pragma unroll
        for (int m = 8; m <= 32; m <<= 1) {
            s1 += __shfl_xor(s1, m, 64);
#pragma unroll
            for (int c = 0; c < 3; c++) aj[c] += __shfl_xor(aj[c], m, 64);
        }
        if (i == 0) {
            S[kRowS1] = s1;
#pragma unroll
            for (int c = 0; c < 3; c++) S[kRowAj + c] = aj[c];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int r = 2; r < 4; r++) {
        const int s = 8 * r + i;
        if (s < kNumSlots) {
            const ChebOut<double> o = (short_from <= 16) ? cheb_eval<double, false, false, kCoefShort>(E.slot[s], te)
                                                         : cheb_eval<double, false>(E.slot[s], te);
            S[3 * (s - 1)] = fma(o.x, inv_au_ast, sun[0]);
            S[3 * (s - 1) + 1] = fma(o.y, inv_au_ast, sun[1]);
            S[3 * (s - 1) + 2] = fma(o.z, inv_au_ast, sun[2]);
        }
    }
}

// Force models with kernels of their own: without Marsden parameters (kModelGravity) the kernel has no
// use for that term's powers and needs fewer registers, and in FP64 the default forces (every term but
// the two other GR forms) are a compile-time constant, with and without Marsden parameters: without
// their branches the terms are one block to the compiler's scheduler.  The mixed form reads the flags
// at run time (see its terms below).
enum : int { kModelAny = 0, kModelStd = 1, kModelGravity = 2 };
constexpr int kStdForces = 0x7F;
constexpr bool row_fixed_forces(bool mixed, int model) { return !mixed && model != kModelAny; }
// Waves per SIMD.
constexpr int row_waves(bool mixed, bool jacobian, int model) {
    return (jacobian && !mixed && model != kModelGravity) ? 1 : 2;
}

// One body's point mass on one lane: the operands of the sums above.
template <typename TS>
struct BodyOps {
    double p, d[3];   // pull and direction, FP64
    TS pt, f[3];      // the same in TS (the asteroids of the mixed form)
    TS g, e[6];       // Jacobian: GM and xx yy zz xy yz xz
};

// Acceleration of the real particle and row c of its Jacobian, as force_eval, on the row's 16 lanes;
// `S` is the evaluation's time in the ephemeris table.
template <bool Mixed, bool Jacobian, int Model>
__device__ __forceinline__ void row_force_eval(const DevEphem& E, const ForceOpts& O, const double* S, int lane, double t,
                                               const double xr[3], const double vr[3], const double A[3], bool ng,
                                               bool need_jac, int c, EvalResult<double>& out,
                                               JacRow<typename TermScalar<double, Mixed>::type>& Jrow) {
    using TS = typename TermScalar<double, Mixed>::type;
    constexpr bool kFixed = row_fixed_forces(Mixed, Model);
    const int forces = kFixed ? kStdForces : O.forces;
    out.status = (t >= O.t_lo && t <= O.t_hi) ? kOk : kCoverage;
    const bool eih = kFixed || ((forces & F_GR_EIH) && O.gr_eih_sources > 0);
    const int nbody = kNumPlanets + E.n_ast;
    // GM / r and the pull of this lane's planet (zeros without one)
    double gmir = 0.0, gm_pl = 0.0, ir_pl = 0.0, a_pl[3] = {0.0, 0.0, 0.0};
    auto body = [&](int s, bool planets, BodyOps<TS>& o) {
        const int b = s < 3 ? s : s - 1;
        const bool used = s != kSlotEMB && b < nbody;
        const int bl = used ? b : 0;
        double GM = E.GM[bl];
        const bool allowed = used && ((b == 0) ? (forces & F_SUN) : (b < kNumPlanets ? (forces & F_PLANETS) : (forces & F_ASTEROIDS)));
        double dx = xr[0] - S[3 * bl], dy = xr[1] - S[3 * bl + 1], dz = xr[2] - S[3 * bl + 2];
        // (a lane without a body adds exact zeros)
        if (!used) { GM = 0.0; dx = 1.0; dy = dz = 0.0; }
        o.p = 0.0;
        o.d[0] = dx; o.d[1] = dy; o.d[2] = dz;
        const TS g = TS(GM);
        o.g = g;
        const bool second = s >= 8 && s < 16;
        const double r2 = norm2(second, dx, dy, dz);
        if constexpr (Mixed) {
            const TS fx = TS(dx), fy = TS(dy), fz = TS(dz);
            o.pt = TS(0);
            o.f[0] = fx; o.f[1] = fy; o.f[2] = fz;
            if (b >= kNumPlanets && r2 > kFp32MinDist * kFp32MinDist) {
                const TS ir = inv_sqrt(norm2(second, fx, fy, fz));
                const TS ir2 = ir * ir;
                const TS r3inv = ir2 * ir;
                const TS pref = TS(GM) * r3inv;
                o.pt = allowed ? pref : TS(0);
                if constexpr (Jacobian) {
                    const TS r5 = TS(3) * r3inv * ir2;
                    o.e[0] = fx * fx * r5 - r3inv; o.e[1] = fy * fy * r5 - r3inv; o.e[2] = fz * fz * r5 - r3inv;
                    o.e[3] = fx * fy * r5; o.e[4] = fy * fz * r5; o.e[5] = fx * fz * r5;
                }
                return;
            }
        }
        const double ir = inv_sqrt(r2);
        const double ir2 = ir * ir;
        const double r3inv = ir2 * ir;
        const double pref = GM * r3inv;
        o.p = allowed ? pref : 0.0;
        if constexpr (Jacobian) {
            const TS r3t = TS(r3inv);
            const TS r5 = TS(3.0 * r3inv * ir2);
            const TS fx = TS(dx), fy = TS(dy), fz = TS(dz);
            o.e[0] = fx * fx * r5 - r3t; o.e[1] = fy * fy * r5 - r3t; o.e[2] = fz * fz * r5 - r3t;
            o.e[3] = fx * fy * r5; o.e[4] = fy * fz * r5; o.e[5] = fx * fz * r5;
        }
        if (planets) {
            const bool pl = used && b < kNumPlanets;
            gmir = pl ? GM * ir : 0.0;
            gm_pl = pl ? GM : 0.0;
            ir_pl = pl ? ir : 0.0;
            a_pl[0] = pl ? -pref * dx : 0.0;
            a_pl[1] = pl ? -pref * dy : 0.0;
            a_pl[2] = pl ? -pref * dz : 0.0;
        }
    };
    BodyOps<TS> o0, o1;
    body(lane, true, o0);
    {
        const int s = 16 + lane;
        body(s < kNumSlots ? s : kSlotEMB, false, o1);
    }
    // sum_k GM_k / r_ik over the planets and its gradient, slots l then l + 8
    double S0 = 0.0, dS0[3] = {0.0, 0.0, 0.0};
    if (eih) {
        S0 = upper_sum(fma(gm_pl, ir_pl, row_swap8(gmir)));
#pragma unroll
        for (int c = 0; c < 3; c++) dS0[c] = upper_sum(row_swap8(a_pl[c]) + a_pl[c]);
    }
    double ad[3];
    TS adt[3] = {TS(0), TS(0), TS(0)};
    TS jd[6] = {TS(0), TS(0), TS(0), TS(0), TS(0), TS(0)};
#pragma unroll
    for (int c = 0; c < 3; c++) {
        ad[c] = sum_pull(o0.p, o0.d[c], o1.p, o1.d[c]);
        if constexpr (Mixed) adt[c] = sum_pull(o0.pt, o0.f[c], o1.pt, o1.f[c]);
    }
    if constexpr (Jacobian) {
#pragma unroll
        for (int m = 0; m < 6; m++) jd[m] = sum_jac(o0.g, o0.e[m], o1.g, o1.e[m]);
    }
    // the single-particle terms, reference order
    const double sun[3] = {S[0], S[1], S[2]}, earth[3] = {S[9], S[10], S[11]};
    const double sunv[3] = {S[kRowSunVel], S[kRowSunVel + 1], S[kRowSunVel + 2]};
    double acc[3] = {0.0, 0.0, 0.0};
    const double GMs = E.GM[0];
    // The FP64 terms compute the one row; the mixed form's all three, as the 8-lane kernel's do (and,
    // as there, behind a run-time condition: FP32 partials keep their roundings only in the same code).
    const double aj[3] = {S[kRowAj], S[kRowAj + 1], S[kRowAj + 2]};
    if constexpr (Mixed) {
        Jac<TS> J;
        jac_zero(J);
        if (Model != kModelGravity && (forces & F_NONGRAV) && ng) term_nongrav<double, TS>(O, xr, vr, sun, sunv, A, need_jac, acc, J);
        if (forces & F_EARTH_H) term_earth_J2J4<double, TS>(E, xr, earth, E.GM[3], need_jac, acc, J);
        if (forces & F_SUN_H) term_solar_J2<double, TS>(E, xr, sun, GMs, need_jac, acc, J);
        if (eih) term_eih_sun<double, TS>(E, xr, vr, sun, sunv, GMs, S0, dS0, S[kRowS1], aj, need_jac, acc, J);
        if (forces & F_GR_POTENTIAL) term_gr_potential<double, TS>(E, xr, sun, GMs, need_jac, acc, J);
        if (forces & F_GR_SIMPLE) term_gr_simple<double, TS>(E, xr, vr, sun, sunv, GMs, need_jac, acc, J);
        if constexpr (Jacobian) {
#pragma unroll
            for (int j = 0; j < 3; j++) {
                Jrow.x[j] = pick3(c, J.x[0][j], J.x[1][j], J.x[2][j]);
                Jrow.v[j] = pick3(c, J.v[0][j], J.v[1][j], J.v[2][j]);
                Jrow.A[j] = pick3(c, J.A[0][j], J.A[1][j], J.A[2][j]);
            }
        }
    } else {
        Jrow.c = c;
        jac_zero(Jrow);
        if (Model != kModelGravity && (forces & F_NONGRAV) && ng) fp64::term_nongrav(O, xr, vr, sun, sunv, A, Jacobian, acc, Jrow);
        if (forces & F_EARTH_H) fp64::term_earth_J2J4(E, xr, earth, E.GM[3], Jacobian, acc, Jrow);
        if (forces & F_SUN_H) fp64::term_solar_J2(E, xr, sun, GMs, Jacobian, acc, Jrow);
        if (eih) fp64::term_eih_sun(E, xr, vr, sun, sunv, GMs, S0, dS0, S[kRowS1], aj, Jacobian, acc, Jrow);
        if (forces & F_GR_POTENTIAL) fp64::term_gr_potential(E, xr, sun, GMs, Jacobian, acc, Jrow);
        if (forces & F_GR_SIMPLE) fp64::term_gr_simple(E, xr, vr, sun, sunv, GMs, Jacobian, acc, Jrow);
    }
    if (forces & (F_SUN | F_PLANETS | F_ASTEROIDS)) {
#pragma unroll
        for (int k = 0; k < 3; k++) acc[k] += ad[k] + double(adt[k]);
        if constexpr (Jacobian) {
            Jrow.x[0] += pick3(c, jd[0], jd[3], jd[5]);
            Jrow.x[1] += pick3(c, jd[3], jd[1], jd[4]);
            Jrow.x[2] += pick3(c, jd[5], jd[4], jd[2]);
        }
    }
    out.acc[0] = acc[0]; out.acc[1] = acc[1]; out.acc[2] = acc[2];
}

enum : int { kRowNone = 0, kRowSetup = 1, kRowFinish = 2 };
// Mixed form: a row about to evaluate the last substep of a pass waits for rows of its wave that are at
// most this many substeps behind.  Most attempts take one pass there (8 evaluations with the step's
// start), and a step's end, the prediction of the next and its ephemeris cost about as many
// instructions as 3 evaluations, which the wave issues once for all the rows that get there together:
// waiting aligns the rows for good, since a second pass (7 evaluations) leaves a row one behind.
// Measured without and with waits of at most 1 and 2: 65,536 x 7 vectors over 100 d 17.3, 14.5,
// 14.6 ms, real particles alone 10.8, 9.4, 9.4 ms (3 to 6 give no more).  The FP64 form's attempts
// take two to four passes and drift apart again: 65,536 real particles over 60 d 9.9, 9.8, 9.7 ms,
// 4,096 x 7 over 300 d 4.85, 5.1, 5.2 ms.
constexpr int kRowAlign = 2;

// NV: vectors per lane quad (1: up to 4 vectors per system, 2: up to 8).  Jacobian: the systems
// carry variational vectors.
// Late: the systems are the records that the one-lane kernel left (a.late).
template <bool Mixed, int NV, bool Jacobian, int Model, bool Late = false>
__global__ void __launch_bounds__(kRowBlock) __attribute__((amdgpu_waves_per_eu(row_waves(Mixed, Jacobian, Model), row_waves(Mixed, Jacobian, Model))))
ias15_row_kernel(IntegrateArgs args) {
    (void)args;
    KArgs ka = (KArgs)__builtin_amdgcn_kernarg_segment_ptr();
    using TS = typename TermScalar<double, Mixed>::type;
    const int wl = threadIdx.x & 63;
    const int lane = wl & 15;
    const int row = wl >> 4;
    const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int nv = ka->nvec;
    const int c = (lane & 3) < 3 ? (lane & 3) : 2;  // (the fourth lane of a quad owns nothing)
    bool own[NV];
#pragma unroll
    for (int r = 0; r < NV; r++) own[r] = (lane & 3) < 3 && (lane >> 2) + 4 * r < nv;
    // last accepted step's b and its prediction's correction e, 14 words per component (the lane is
    // laundered, so that the words' addresses are not kept in registers across the loop)
    auto scratch = [&]() {
        int l = wl;
        asm volatile("" : "+v"(l));
        return ka->scratch + (size_t)wave * 64 * (14 * NV) + l;
    };

    extern __shared__ double s_row[];
    double* const tab = s_row;
    for (int i = threadIdx.x; i < kTabWords; i += blockDim.x) {
        double v;
        if (i < kTabPX) v = cH[i - kTabH];
        else if (i < kTabPV) v = cPX[i - kTabPX];
        else if (i < kTabRRI) v = cPV[i - kTabPV];
        else if (i < kTabC) v = cRRI[i - kTabRRI];
        else if (i < kTabW) v = cC[i - kTabC];
        else if (i < kTabW + 49) {
            const int n = (i - kTabW) / 7 + 1, k = (i - kTabW) % 7;
            v = k < n - 1 ? cC[(n - 1) * (n - 2) / 2 + k] : (k == n - 1 ? 1.0 : 0.0);
        } else {
            v = 0.0;
        }
        tab[i] = v;
    }
    __shared__ DevEphem s_E;
    {
        const unsigned long long* src = (const unsigned long long*)ka->E;
        unsigned long long* dst = (unsigned long long*)&s_E;
        for (int i = threadIdx.x; i < (int)(sizeof(DevEphem) / sizeof(unsigned long long)); i += blockDim.x) dst[i] = src[i];
    }
    __syncthreads();
    const DevEphem& E = s_E;
    double* const wave_eph = s_row + kTabWords + (size_t)(threadIdx.x >> 6) * kRowWaveWords;
    double* const eph = wave_eph + row * (kRowTimes * kRowSlice);
    double* const par = wave_eph + 4 * (kRowTimes * kRowSlice) + row * 24;  // Marsden A of the system's vectors

    double x0[NV], v0[NV], csx[NV], csv[NV], a0[NV], b[NV][7], g[NV][7];
#pragma unroll
    for (int r = 0; r < NV; r++) {
        x0[r] = (c == 0) ? 2.5 : 0.0;
        v0[r] = (c == 1) ? 0.01 : 0.0;
        csx[r] = csv[r] = a0[r] = 0.0;
#pragma unroll
        for (int k = 0; k < 7; k++) b[r][k] = g[r][k] = 0.0;
    }
    double t = 0, t_end = 0, dt = 0, dts = 0, dt_last = 0, pc_err_last = 0;
    bool phase = false, need_eph = true, ng = false;
    int n = 1, it = 0, last = 0, status = 0, attempts = 0;
    long long steps = 0, evals = 0, rejected = 0;
    int cur = 0, cend = 0;
    int todo = kRowNone;  // what the row does before its next evaluation
    // first positions row by row over the grid's waves, so that a batch smaller than the grid
    // spreads over every wave
    const int nwaves = (int)((gridDim.x * blockDim.x) >> 6);
    const int q0 = row * nwaves + wave;
    auto systems = [&]() { return Late ? min(*ka->late_count, ka->late_cap) : ka->nsys; };
    auto system_at = [&](int q) { return Late ? (int)ka->late[(size_t)q * kLateWords] : (ka->order ? ka->order[q] : q); };
    bool active = q0 < systems();
    int sys = active ? system_at(q0) : 0;

    auto load = [&](int s) {
        const double* st = ka->states + (size_t)s * nv * 6;
        double sx[NV], sv[NV];
#pragma unroll
        for (int r = 0; r < NV; r++) {
            const int v = own[r] ? (lane >> 2) + 4 * r : 0;
            sx[r] = st[6 * v + c];
            sv[r] = st[6 * v + 3 + c];
        }
        double pa = 0.0, pb = 0.0;
        if (ka->params) {
            const double* pp = ka->params + (size_t)s * nv * 3;
            pa = pp[lane < 3 * nv ? lane : 0];
            pb = pp[lane + 16 < 3 * nv ? lane + 16 : 0];
        }
        const double t0s = ka->t0[s];
        const bool dense = ka->out_t != nullptr;
        const int* po = dense ? ka->out_off + s : (const int*)(ka->t0 + s);
        const int off0 = po[0], off1 = po[dense ? 1 : 0];
        const double t1s = (dense ? ka->t0 : ka->t1)[s];
        const double dtl = (ka->dt0 ? ka->dt0 : ka->t0)[s];
        const double dt0s = ka->dt0 ? fabs(dtl) : ka->io.dt_initial;
#pragma unroll
        for (int r = 0; r < NV; r++) {
            x0[r] = own[r] ? sx[r] : 0.0;
            v0[r] = own[r] ? sv[r] : 0.0;
            csx[r] = csv[r] = a0[r] = 0.0;
#pragma unroll
            for (int k = 0; k < 7; k++) b[r][k] = g[r][k] = 0.0;
        }
        ng = false;
        if (ka->params) {
            par[lane] = pa;
            if (lane < 8) par[16 + lane] = pb;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            ng = !(par[0] == 0.0 && par[1] == 0.0 && par[2] == 0.0);
        }
        t = t0s;
        if (dense) {
            cur = off0;
            cend = off1;
            t_end = (cend > cur) ? ka->out_t[cend - 1] : t;
        } else {
            t_end = t1s;
        }
        dt = dt0s;
        if (dt * (t_end - t) < 0) dt = -dt;
        dt_last = 0.0;
        phase = false;
        need_eph = true;
        status = 0;
        steps = evals = rejected = 0;
        last = 0;
    };
    // a system that the one-lane kernel left, at the step boundary of its record
    auto resume = [&](int q) {
        const double* const rec = ka->late + (size_t)q * kLateWords;
        const double tr = rec[1], dtr = rec[2], dlr = rec[3], st = rec[4], ev = rec[5], rj = rec[6];
        if (own[0]) {
            x0[0] = rec[8 + c];
            v0[0] = rec[11 + c];
            csx[0] = rec[14 + c];
            csv[0] = rec[17 + c];
        }
        double* const scr = scratch();
#pragma unroll
        for (int k = 0; k < 14; k++) scr[k * 64] = rec[20 + 3 * k + c];
        t = tr;
        dt = dtr;
        dt_last = dlr;
        steps = (long long)st;
        evals = (long long)ev;
        rejected = (long long)rj;
    };
    auto finish = [&]() {
        double* st = ka->states + (size_t)sys * nv * 6;
#pragma unroll
        for (int r = 0; r < NV; r++) {
            if (own[r]) {
                const int v = (lane >> 2) + 4 * r;
                st[6 * v + c] = x0[r];
                st[6 * v + 3 + c] = v0[r];
            }
        }
        int next = 0;
        if (lane == 0) {
            if (ka->status) ka->status[sys] = status;
            if (ka->steps) ka->steps[sys] = steps;
            if (ka->evals) ka->evals[sys] = evals;
            if (ka->rejected) ka->rejected[sys] = rejected;
            if (ka->t_out) ka->t_out[sys] = t;
            next = atomicAdd(ka->queue, 1);
        }
        next = row_bcast0_i(next);
        active = next < systems();
        if (active) {
            sys = system_at(next);
            load(sys);
            if constexpr (Late) resume(next);
        }
    };
    // Predict b of the attempt from the last accepted step and convert it to g.  Returns false
    // when the step cannot be taken.
    auto setup_attempt = [&]() -> bool {
        if (!(fabs(dts) > 0.0) || !(fabs(dts) < 1e300) || ++attempts > 64) { status = kDtUnderflow; return false; }
        const double q = dts / dt_last;
        const double* const scr = scratch();
        double amag = 0.0;
        if (ka->bw && dt_last == 0.0) {
            const double a[3] = {row_bcast<0>(a0[0]), row_bcast<1>(a0[0]), row_bcast<2>(a0[0])};
            amag = sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
        }
#pragma unroll
        for (int r = 0; r < NV; r++) {
            if (dt_last != 0.0 && own[r]) {
                if (q > 20.0) {
#pragma unroll
                    for (int k = 0; k < 7; k++) b[r][k] = 0.0;
                } else {
                    double br[7], er[7], e[7];
#pragma unroll
                    for (int k = 0; k < 7; k++) { br[k] = scr[(14 * r + k) * 64]; er[k] = scr[(14 * r + 7 + k) * 64]; }
                    predict_e(br, q, e);
#pragma unroll
                    for (int k = 0; k < 7; k++) b[r][k] = e[k] + (br[k] - er[k]);
                }
            } else if (ka->bw && r == 0 && lane < 3) {
                // learned warm start of the first step: b_k = bw_k |a0| dt^(k+1)
                const double* w = ka->bw + (size_t)sys * 21;
                double hp = dts;
#pragma unroll
                for (int k = 0; k < 7; k++) {
                    b[r][k] = w[3 * k + c] * amag * hp;
                    hp *= dts;
                }
            } else {
#pragma unroll
                for (int k = 0; k < 7; k++) b[r][k] = 0.0;
            }
            const double b0 = b[r][0], b1 = b[r][1], b2 = b[r][2], b3 = b[r][3], b4 = b[r][4], b5 = b[r][5], b6 = b[r][6];
            // (the 8-lane kernel rounds b6's product first in x and y, and b5's in z)
            const bool xy = c < 2;
            auto top = [&](double d6, double d5) { return xy ? fma(b5, d5, b6 * d6) : fma(b6, d6, b5 * d5); };
            g[r][0] = fma(b1, cD[0], fma(b2, cD[1], fma(b3, cD[3], fma(b4, cD[6], top(cD[15], cD[10]))))) + b0;
            g[r][1] = fma(b2, cD[2], fma(b3, cD[4], fma(b4, cD[7], top(cD[16], cD[11])))) + b1;
            g[r][2] = fma(b3, cD[5], fma(b4, cD[8], top(cD[17], cD[12]))) + b2;
            g[r][3] = fma(b4, cD[9], top(cD[18], cD[13])) + b3;
            g[r][4] = top(cD[19], cD[14]) + b4;
            g[r][5] = fma(b6, cD[20], b5);
            g[r][6] = b6;
        }
        it = 1;
        pc_err_last = 1e300;
        n = 1;
        phase = true;
        return true;
    };

    if (active) {
        load(sys);
        if constexpr (Late) resume(q0);
    }
    if (!active) need_eph = false;
    // A row whose queue ran dry stays in the loop while any row of its wave is active: all 64 lanes
    // take part in the ephemeris rounds.
    while (__ballot(active) != 0ULL) {
        ka = launder(ka);
        const bool eih = row_fixed_forces(Mixed, Model) || ((ka->fo.forces & F_GR_EIH) && ka->fo.gr_eih_sources > 0);
        if (todo == kRowSetup) {
            todo = setup_attempt() ? kRowNone : kRowFinish;
        }
        if (todo == kRowFinish) {
            todo = kRowNone;
            finish();
        }
        if (active && need_eph && !phase) {
            if (ka->out_t ? cur >= cend : t == t_end) {
                // zero-length span (dense output: no output times left)
                todo = kRowFinish;
            } else {
                // the step that the start's evaluation leads to: its length is known already
                const double dir = (t_end >= t) ? 1.0 : -1.0;
                dts = dt;
                last = 0;
                if (!ka->out_t && (t + dts - t_end) * dir >= 0) { dts = t_end - t; last = 1; }
                attempts = 0;
            }
        }
        {
            // (every lane of the wave gets here: a row that has nothing to evaluate helps the others)
            unsigned long long need = __ballot(active && need_eph && todo != kRowFinish) & 0x0001000100010001ULL;
            while (need != 0ULL) {
                const int src = __ffsll((unsigned long long)need) - 1;
                need &= need - 1ULL;
                row_ephemeris(E, tab + kTabH, readlane_d(t, src), readlane_d(dts, src), eih,
                              wave_eph + (src >> 4) * (kRowTimes * kRowSlice));
            }
            // (LDS operations of one wave complete in order; the fence keeps the compiler's order too)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            need_eph = false;
        }
        bool wait = false;
        if constexpr (Mixed) {
            // (a row that is waited for never waits itself, so each trip brings one nearer)
            const bool behind = active && todo != kRowFinish && phase && n < 7 && n >= 7 - kRowAlign;
            wait = __ballot(behind) != 0ULL && phase && n == 7;
        }
        if (!active || todo == kRowFinish || wait) continue;
        // ---- evaluation point of this trip ----
        double xe[NV], ve[NV], te;
        if (!phase) {
#pragma unroll
            for (int r = 0; r < NV; r++) { xe[r] = x0[r]; ve[r] = v0[r]; }
            te = t;
        } else {
            const double* px = tab + kTabPX + 8 * n;
            const double* pv = tab + kTabPV + 7 * n;
            const double dt2 = dts * dts;
            double s[9];
            s[0] = dts * tab[kTabH + n];
#pragma unroll
            for (int k = 1; k < 9; k++) s[k] = dt2 * px[k - 1];
#pragma unroll
            for (int r = 0; r < NV; r++)
                xe[r] = -csx[r] + (fma(s[0], v0[r], fma(s[1], a0[r], fma(s[2], b[r][0], fma(s[3], b[r][1], fma(s[4], b[r][2],
                        fma(s[5], b[r][3], fma(s[6], b[r][4], fma(s[8], b[r][6], s[7] * b[r][5])))))))) + x0[r]);
#pragma unroll
            for (int k = 1; k < 8; k++) s[k] = dts * pv[k - 1];
#pragma unroll
            for (int r = 0; r < NV; r++)
                ve[r] = -csv[r] + (fma(s[0], a0[r], fma(s[1], b[r][0], fma(s[2], b[r][1], fma(s[3], b[r][2], fma(s[4], b[r][3],
                        fma(s[5], b[r][4], fma(s[7], b[r][6], s[6] * b[r][5]))))))) + v0[r]);
            te = fma(dts, tab[kTabH + n], t);
        }
        // ---- force evaluation ----
        double at[NV];
        int ev_status;
        {
            const double xr[3] = {row_bcast<0>(xe[0]), row_bcast<1>(xe[0]), row_bcast<2>(xe[0])};
            const double vr[3] = {row_bcast<0>(ve[0]), row_bcast<1>(ve[0]), row_bcast<2>(ve[0])};
            EvalResult<double> R;
            JacRow<TS> J;
            const ForceOpts fo = ka->fo;
            double A[3] = {0.0, 0.0, 0.0};
            if (Model != kModelGravity && ng) {
#pragma unroll
                for (int k = 0; k < 3; k++) A[k] = par[k];
            }
            row_force_eval<Mixed, Jacobian, Model>(E, fo, eph + (phase ? n : 0) * kRowSlice, lane, te, xr, vr, A, ng, (Jacobian || Model != kModelGravity) && nv > 1, c, R, J);
            ev_status = R.status;
            const double real = pick3(c, R.acc[0], R.acc[1], R.acc[2]);
            if constexpr (Jacobian) {
                // this lane's row of the Jacobian, applied to its vectors
#pragma unroll
                for (int r = 0; r < NV; r++) {
                    const TS xt = TS(xe[r]), vt = TS(ve[r]);
                    const TS x[3] = {quad_bcast<0>(xt), quad_bcast<1>(xt), quad_bcast<2>(xt)};
                    const TS v[3] = {quad_bcast<0>(vt), quad_bcast<1>(vt), quad_bcast<2>(vt)};
                    TS s = J.x[0] * x[0] + J.x[1] * x[1] + J.x[2] * x[2];
                    s += J.v[0] * v[0] + J.v[1] * v[1] + J.v[2] * v[2];
                    if (Model != kModelGravity && ng) {
                        const double* dA = par + 3 * ((lane >> 2) + 4 * r);
                        s += J.A[0] * TS(dA[0]) + J.A[1] * TS(dA[1]) + J.A[2] * TS(dA[2]);
                    }
                    at[r] = (r == 0 && lane < 4) ? real : double(s);
                }
            } else {
                at[0] = real;
            }
        }
        evals++;
        if (ev_status != kOk) { status = ev_status; todo = kRowFinish; continue; }
        if (!phase) {
#pragma unroll
            for (int r = 0; r < NV; r++) a0[r] = at[r];
            todo = kRowSetup;
            continue;
        }
        // ---- corrector: improve g_{n-1} and b_0..b_{n-1} (as ias15_kernel, on one component) ----
        double maxak = 0.0, maxdb6 = 0.0;
        const double pc_tol = ka->io.pc_tol;
        {
            const double* rri = tab + kTabRRI + n * (n - 1) / 2;  // 1 / (h_n - h_j), j = 0..n-1
            const double* wn = tab + kTabW + 7 * (n - 1);          // b_k += wn[k] dg_{n-1}
            double rr[6], w[7];
#pragma unroll
            for (int k = 0; k < 6; k++) rr[k] = rri[k < n ? k : 0];
#pragma unroll
            for (int k = 0; k < 7; k++) w[k] = wn[k];
            const double rl = rri[n - 1];
#pragma unroll
            for (int r = 0; r < NV; r++) {
                double gold = g[r][0];
#pragma unroll
                for (int k = 1; k < 7; k++) gold = (k == n - 1) ? g[r][k] : gold;
                double val = at[r] - a0[r];
#pragma unroll
                for (int k = 0; k < 6; k++) val = (k < n - 1) ? fma(val, rr[k], -g[r][k]) : val;
                val *= rl;
                const double tmp = val - gold;
#pragma unroll
                for (int k = 0; k < 7; k++) {
                    g[r][k] = (k == n - 1) ? val : g[r][k];
                    b[r][k] = fma(tmp, w[k], b[r][k]);
                }
                // the test's vectors: all of the system's, or the real particle alone
                const bool in_test = own[r] && (pc_tol <= 0.0 || (r == 0 && lane < 3));
                if (n == 7 && in_test) {
                    const double ak = fabs(at[r]);
                    if (is_normal(ak) && ak > maxak) maxak = ak;
                    const double db = fabs(tmp);
                    if (is_normal(db) && db > maxdb6) maxdb6 = db;
                }
            }
        }
        if (n < 7) {
            n++;
            continue;
        }
        // ---- end of a predictor-corrector iteration (the tests are ias15_kernel's) ----
        const double pc_mak = row_max(maxak);
        const double pc_err = row_max(maxdb6) / pc_mak;
        const double pc_aref = ka->io.pc_aref;
        const double pc_tol1 = (pc_aref > 0.0 && pc_mak > pc_aref) ? ka->io.pc_tol1 * fmax(0.1, pc_aref / pc_mak) : ka->io.pc_tol1;
        if (!(pc_err < (pc_tol > 0.0 ? pc_tol : 1e-16)) && !(it == 1 && pc_err < pc_tol1) &&
            !(it > 2 && pc_err_last <= pc_err) && it < 12) {
            pc_err_last = pc_err;
            it++;
            n = 1;
            continue;
        }
        // ---- step-size control (real particle only) ----
        double dt_new = dts, dt_prop = dts;
        if (ka->io.epsilon > 0) {
            const double ak = fabs(at[0]), bk = fabs(b[0][6]);
            const double mak = row_max((lane < 3 && is_normal(ak)) ? ak : 0.0);
            const double mb6 = row_max((lane < 3 && is_normal(bk)) ? bk : 0.0);
            const double err = mb6 / mak;
            if (is_normal(err)) dt_new = pow(ka->io.epsilon / err, 1.0 / 7.0) * dts;
            else dt_new = dts / 0.25;
            if (fabs(dt_new) < ka->io.min_dt) dt_new = copysign(ka->io.min_dt, dt_new);
            if (fabs(dt_new / dts) < 0.25) {
                rejected++;
                dts = dt_new;
                last = 0;
                todo = kRowSetup;
                need_eph = true;
                continue;
            }
            dt_prop = dt_new;
            if (dt_new / dts > 1. / 0.25) dt_new = dts / 0.25;
        }
        // ---- accept: advance x0, v0 (Kahan) and store br, er ----
        if (ka->trace && steps >= ka->trace_skip && steps % ka->trace_every == 0) {
            int idx = 0;
            if (lane == 0) idx = atomicAdd(ka->trace_count, 1);
            idx = row_bcast0_i(idx);
            if (lane < 3 && idx < ka->trace_cap) {
                double* rec = ka->trace + (size_t)idx * kTraceWords;
                if (lane == 0) {
                    rec[0] = t;
                    rec[7] = dt_last;
                    rec[8] = dts;
                    rec[9] = dt_prop;
                }
                rec[1 + c] = x0[0];
                rec[4 + c] = v0[0];
                rec[10 + c] = a0[0];
#pragma unroll
                for (int k = 0; k < 7; k++) rec[13 + 3 * k + c] = b[0][k];
            }
        }
        if (ka->out_t) {
            // dense output: every output time in [t, t + dts) from this step's polynomial, as
            // reference src/assist.c:556-597 (assist_interpolate)
            while (cur < cend) {
                double h = (ka->out_t[cur] - t) / dts;
                if (!(h < 1.0)) break;
                if (h < 0.0) h = 0.0;
                double s[9], sv[8];
                s[0] = dts * h;
                s[1] = s[0] * s[0] / 2.;
                s[2] = s[1] * h / 3.;
                s[3] = s[2] * h / 2.;
                s[4] = 3. * s[3] * h / 5.;
                s[5] = 2. * s[4] * h / 3.;
                s[6] = 5. * s[5] * h / 7.;
                s[7] = 3. * s[6] * h / 4.;
                s[8] = 7. * s[7] * h / 9.;
                sv[0] = dts * h;
                sv[1] = sv[0] * h / 2.;
                sv[2] = 2. * sv[1] * h / 3.;
                sv[3] = 3. * sv[2] * h / 4.;
                sv[4] = 4. * sv[3] * h / 5.;
                sv[5] = 5. * sv[4] * h / 6.;
                sv[6] = 6. * sv[5] * h / 7.;
                sv[7] = 7. * sv[6] * h / 8.;
#pragma unroll
                for (int r = 0; r < NV; r++) {
                    if (!own[r]) continue;
                    double* o = ka->out_states + ((size_t)cur * nv + (lane >> 2) + 4 * r) * 6;
                    o[c] = x0[r] + (s[8] * b[r][6] + s[7] * b[r][5] + s[6] * b[r][4] + s[5] * b[r][3] + s[4] * b[r][2] +
                                    s[3] * b[r][1] + s[2] * b[r][0] + s[1] * a0[r] + s[0] * v0[r]);
                    o[3 + c] = v0[r] + sv[7] * b[r][6] + sv[6] * b[r][5] + sv[5] * b[r][4] + sv[4] * b[r][3] +
                               sv[3] * b[r][2] + sv[2] * b[r][1] + sv[1] * b[r][0] + sv[0] * a0[r];
                }
                cur++;
            }
        }
        double wx[8], wv[7];
        {
            const double dt2 = dts * dts;
#pragma unroll
            for (int k = 0; k < 8; k++) wx[k] = cPX[64 + k] * dt2;
#pragma unroll
            for (int k = 0; k < 7; k++) wv[k] = cPV[56 + k] * dts;
        }
        bool bad = false;
        double* const scr = scratch();
        const double q = (dt_last != 0.0) ? dts / dt_last : 0.0;
#pragma unroll
        for (int r = 0; r < NV; r++) {
            double bl[7];
#pragma unroll
            for (int k = 0; k < 7; k++) bl[k] = scr[(14 * r + k) * 64];
            add_cs(x0[r], csx[r], b[r][6] * wx[7]);
            add_cs(x0[r], csx[r], b[r][5] * wx[6]);
            add_cs(x0[r], csx[r], b[r][4] * wx[5]);
            add_cs(x0[r], csx[r], b[r][3] * wx[4]);
            add_cs(x0[r], csx[r], b[r][2] * wx[3]);
            add_cs(x0[r], csx[r], b[r][1] * wx[2]);
            add_cs(x0[r], csx[r], b[r][0] * wx[1]);
            add_cs(x0[r], csx[r], a0[r] * wx[0]);
            add_cs(x0[r], csx[r], v0[r] * dts);
            add_cs(v0[r], csv[r], b[r][6] * wv[6]);
            add_cs(v0[r], csv[r], b[r][5] * wv[5]);
            add_cs(v0[r], csv[r], b[r][4] * wv[4]);
            add_cs(v0[r], csv[r], b[r][3] * wv[3]);
            add_cs(v0[r], csv[r], b[r][2] * wv[2]);
            add_cs(v0[r], csv[r], b[r][1] * wv[1]);
            add_cs(v0[r], csv[r], b[r][0] * wv[0]);
            add_cs(v0[r], csv[r], a0[r] * dts);
            double e[7];
            if (dt_last != 0.0 && q <= 20.0) predict_e(bl, q, e);
            else
#pragma unroll
                for (int k = 0; k < 7; k++) e[k] = 0.0;
#pragma unroll
            for (int k = 0; k < 7; k++) { scr[(14 * r + 7 + k) * 64] = e[k]; scr[(14 * r + k) * 64] = b[r][k]; }
            if (own[r]) bad |= !(fabs(x0[r]) < 1e300) || !(fabs(v0[r]) < 1e300);
        }
        t = last ? t_end : t + dts;
        steps++;
        dt_last = dts;
        if (!(last && ka->io.epsilon <= 0)) dt = dt_new;
        if ((__ballot(bad) >> (16 * row)) & 0xFFFFULL) { status = kNonFinite; todo = kRowFinish; continue; }
        if (last || (ka->out_t && cur >= cend)) { todo = kRowFinish; continue; }
        if (steps >= ka->io.max_steps) { status = kMaxSteps; todo = kRowFinish; continue; }
        phase = false;
        need_eph = true;
    }
}

template <bool M, int NV, bool J, bool Late = false>
static const void* row_fn(int model) {
    if constexpr (!M) {
        if (model == kModelStd) return (const void*)ias15_row_kernel<M, NV, J, kModelStd, Late>;
    }
    return model == kModelGravity ? (const void*)ias15_row_kernel<M, NV, J, kModelGravity, Late>
                                  : (const void*)ias15_row_kernel<M, NV, J, kModelAny, Late>;
}

// The force model that a launch's kernel is compiled for.
static int row_model(const IntegrateArgs& a, bool mixed) {
    const bool std_forces = a.fo.forces == kStdForces && a.fo.gr_eih_sources > 0;
    if (!mixed && !std_forces) return kModelAny;
    return !a.params ? kModelGravity : (mixed ? kModelAny : kModelStd);
}

static const void* row_lookup(const IntegrateArgs& a, bool mixed, bool late = false) {
    const int m = row_model(a, mixed);
    if (late) return a.nvec != 1 ? nullptr : (mixed ? row_fn<true, 1, false, true>(m) : row_fn<false, 1, false, true>(m));
    if (a.nvec == 1) return mixed ? row_fn<true, 1, false>(m) : row_fn<false, 1, false>(m);
    static_assert(row_scratch_words(4) == 14 * 1 && row_scratch_words(8) == 14 * 2, "14 words per component and vector");
    if (a.nvec <= 4) return mixed ? row_fn<true, 1, true>(m) : row_fn<false, 1, true>(m);
    if (a.nvec <= 8) return mixed ? row_fn<true, 2, true>(m) : row_fn<false, 2, true>(m);
    return nullptr;
}

int ias15_row_waves(const IntegrateArgs& a, bool mixed) { return row_waves(mixed, a.nvec > 1, row_model(a, mixed)); }

size_t ias15_row_lds_bytes(int threads) {
    return (kTabWords + (size_t)(threads / 64) * kRowWaveWords) * sizeof(double);
}

static hipError_t launch_row(const void* f, const IntegrateArgs& a, int blocks, int threads, hipStream_t s, bool set_attributes) {
    if (!f || threads % 64 != 0 || threads > kRowBlock) return hipErrorInvalidValue;
    const size_t lds = ias15_row_lds_bytes(threads);
    hipError_t e = hipSuccess;
    if (set_attributes) {
        e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    void* params[] = {(void*)&a};
    e = hipLaunchKernel(f, dim3(blocks), dim3(threads), params, lds, s);
    if (e != hipSuccess) return e;
    return hipGetLastError();
}

hipError_t launch_ias15_row(const IntegrateArgs& a, bool mixed, int blocks, int threads, hipStream_t s, bool set_attributes) {
    return launch_row(row_lookup(a, mixed), a, blocks, threads, s, set_attributes);
}

hipError_t launch_ias15_row_late(const IntegrateArgs& a, bool mixed, int blocks, int threads, hipStream_t s, bool set_attributes) {
    return launch_row(row_lookup(a, mixed, true), a, blocks, threads, s, set_attributes);
}

hipError_t ias15_row_occupancy(const IntegrateArgs& a, bool mixed, int threads, int* blocks_per_cu, bool late) {
    const void* f = row_lookup(a, mixed, late);
    if (!f) return hipErrorInvalidValue;
    const size_t lds = ias15_row_lds_bytes(threads);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, threads, lds);
}

}  // namespace assist_gpu
