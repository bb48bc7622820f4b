// The integration kernel with one lane per system, for large batches of real particles.
//
// A force evaluation reads about 9 KB of Chebyshev records.  With a system per lane every lane reads
// records of its own times, one cache line per lane and load, and the L1 caches look up about 1.5 lines a
// clock: a kernel that evaluates one time per trip waits on those reads (81,000 clocks a trip, 20,000 of
// them issuing vector instructions).  Here a lane reads each record once for two times:
//
//   * a pass over the substeps of an attempt is four trips, of the times n = 0 and 1 (0: the step's
//     start), 2 and 3, 4 and 5, 6 and 7.  A trip walks the 28 slots once, evaluates both times from the
//     slot's record, adds the first time's pull and leaves the second time's positions in LDS (78 doubles
//     a lane, all of a CU's LDS with one wave per SIMD), from which the second evaluation reads them;
//   * where a lane's second time lies in another record (1.7 of 28 slots a trip) the wave keeps the pair
//     of lane and body in a list and evaluates 64 of those at once;
//   * every pass of every lane is the same four trips (a pass that follows another, or a rejection,
//     leaves its first evaluation unused), so the substep is the same on all lanes of a wave: the
//     corrector is straight-line code for its substep with b and g in registers, and the step's end
//     runs once for all lanes that reach it;
//   * the next slot's record is loaded while the current one's pull is added;
//   * without variational vectors no partials are compiled in, and without Marsden parameters not that
//     term either.
//
// A wave runs for as long as one of its lanes does, and a trip takes as long with one active lane as with
// 64.  In large batches a wave whose list of systems has run out therefore leaves its last ones (at most
// kLateLanes) at a step boundary to the 16-lane kernel, which takes them on from there at a tenth of the
// time per evaluation.  Each wave has its own list, so which systems these are, and every result, is the
// same in every run.  (With 32 of 64 lanes left a wave's rate falls to the 16-lane kernel's; 48 and 20
// took 2% and up to 18% longer.)
//
// What bounds it: the L1 look-ups (1.3 a clock), then the latency of a wave's own loads (25% of its
// cycles; vector instructions issue in 40%).  Measured on an MI355X against one time per trip:
// 1,048,576 systems over 365 d 221 -> 149 ms in the mixed form from the learned start, 493 -> 330 ms in
// double precision; with the last systems left to the 16-lane kernel 300,007 systems over 40 d 28.3 -> 20.9 ms
// (double precision, 37.4 on 16 lanes alone), 131,072 over 365 d 53.3 -> 24.6 ms (mixed, 35.2).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_types.h"
#include "force_model.h"
#include "ias15_device.h"
#include "kernels.h"

namespace assist_gpu {

// The ephemeris descriptor read through the scalar cache (its indexes are the same on all lanes).
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(4))) const DevEphem* KEphem;
typedef __attribute__((address_space(4))) const DevSlot* KSlot;
typedef __attribute__((address_space(1))) const double* RecPtr;
#else
typedef const DevEphem* KEphem;
typedef const DevSlot* KSlot;
typedef const double* RecPtr;
#endif

// Keeps the evaluation of v where it stands (sunk to its use, it would keep a record's coefficients in
// registers until there).
__device__ __forceinline__ void pin(double (&v)[3]) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
#else
    (void)v;
#endif
}

__device__ __forceinline__ int lane_record(KSlot S, double t) {
    const int idx = (int)((S->c_init + t) * S->inv_intlen);
    return idx < 0 ? 0 : (idx >= S->nrec ? S->nrec - 1 : idx);
}

// A record in registers: the words that a series of NP terms uses (an odd count loads one more, inside it).
struct Record {
    double c[kRecWords];
    template <int NP>
    __device__ __forceinline__ void load(KSlot S, int idx) {
        RecPtr rec = (RecPtr)S->rec + (size_t)idx * kRecWords;
#pragma unroll
        for (int k = 0; k < 2 + 3 * NP; k += 2) {
            const Pair v = {rec[k], rec[k + 1]};
            c[k] = v.x;
            c[k + 1] = v.y;
        }
    }
    // position (km) and, with Vel, velocity (km/day) at time t, as cheb_series
    template <int NP, bool Vel>
    __device__ __forceinline__ void eval(double t, double x[3], double v[3]) const {
        const double z = (c[0] + t) * c[1];
        const double z2 = 2.0 * z;
        double T0 = 1.0, T1 = z, S0 = 0.0, S1 = 1.0;
#pragma unroll
        for (int m = 0; m < 3; m++) {
            x[m] = fma(c[5 + m], z, c[2 + m]);
            if (Vel) v[m] = c[5 + m];
        }
#pragma unroll
        for (int p = 2; p < NP; p++) {
            const double T2 = fma(z2, T1, -T0);
#pragma unroll
            for (int m = 0; m < 3; m++) x[m] = fma(c[2 + 3 * p + m], T2, x[m]);
            if (Vel) {
                const double S2 = fma(z2, S1, fma(2.0, T1, -S0));
#pragma unroll
                for (int m = 0; m < 3; m++) v[m] = fma(c[2 + 3 * p + m], S2, v[m]);
                S0 = S1;
                S1 = S2;
            }
            T0 = T1;
            T1 = T2;
        }
        if (Vel) {
#pragma unroll
            for (int m = 0; m < 3; m++) v[m] *= c[1];
        }
    }
};

// Sums over the bodies of one evaluation.
template <typename TS>
struct BodySums {
    double ad[3];  // direct acceleration, FP64 bodies
    TS adt[3];     // direct acceleration, asteroids of the mixed form
    double S0;     // sum_k GM_k / r_ik over the planets
};
template <typename TS>
__device__ __forceinline__ void sums_zero(BodySums<TS>& a) {
#pragma unroll
    for (int c = 0; c < 3; c++) { a.ad[c] = 0.0; a.adt[c] = TS(0); }
    a.S0 = 0.0;
}

// Body of mass GM at pk (au): its pull on xr (force_eval's body_term without partials).
template <bool Mixed, bool Planet, typename TS>
__device__ __forceinline__ void add_body(double GM, bool allowed, bool eih, const double xr[3], const double pk[3],
                                         BodySums<TS>& a) {
    const double dx = xr[0] - pk[0], dy = xr[1] - pk[1], dz = xr[2] - pk[2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (Mixed && !Planet && r2 > kFp32MinDist * kFp32MinDist) {
        const TS fx = TS(dx), fy = TS(dy), fz = TS(dz);
        const TS q2 = fx * fx + fy * fy + fz * fz;
        const TS ir = inv_sqrt(q2);
        const TS ir2 = ir * ir;
        const TS r3inv = ir2 * ir;
        const TS pref = TS(GM) * r3inv;
        if (allowed) { a.adt[0] -= pref * fx; a.adt[1] -= pref * fy; a.adt[2] -= pref * fz; }
        return;
    }
    const double ir = inv_sqrt(r2);
    const double ir2 = ir * ir;
    const double r3inv = ir2 * ir;
    const double pref = GM * r3inv;
    if (allowed) { a.ad[0] -= pref * dx; a.ad[1] -= pref * dy; a.ad[2] -= pref * dz; }
    if (Planet && eih) a.S0 += GM * ir;
}

// What of an evaluation time's ephemeris is kept in registers: the Sun, and the EIH sums that no
// particle enters (sum_k GM_k / r_sk and the Sun's Newtonian acceleration).
struct SunState {
    double x[3], v[3], S1, aj[3];
    __device__ __forceinline__ void newton(double GM, const double pk[3]) {
        const double sx = x[0] - pk[0], sy = x[1] - pk[1], sz = x[2] - pk[2];
        const double q2 = sx * sx + sy * sy + sz * sz;
        const double iq = inv_sqrt(q2);
        S1 += GM * iq;
        const double f = GM * (iq * iq * iq);
        aj[0] -= f * sx; aj[1] -= f * sy; aj[2] -= f * sz;
    }
};

// The single-particle terms and the total acceleration.
template <bool Mixed, bool Marsden, typename TS>
__device__ __forceinline__ void add_terms(const DevEphem& E, const ForceOpts& O, const double xr[3], const double vr[3],
                                          const SunState& s, const double earth[3], const double A[3], bool ng,
                                          const BodySums<TS>& a, double acc[3]) {
    const int forces = O.forces;
    const bool eih = (forces & F_GR_EIH) && O.gr_eih_sources > 0;
    const double GMs = E.GM[0];
    const double dS0[3] = {0.0, 0.0, 0.0};  // (partials only)
    Jac<TS> J;
    acc[0] = acc[1] = acc[2] = 0.0;
    if constexpr (Mixed) {
        if (Marsden && (forces & F_NONGRAV) && ng) term_nongrav<double, TS>(O, xr, vr, s.x, s.v, A, false, acc, J);
        if (forces & F_EARTH_H) term_earth_J2J4<double, TS>(E, xr, earth, E.GM[3], false, acc, J);
        if (forces & F_SUN_H) term_solar_J2<double, TS>(E, xr, s.x, GMs, false, acc, J);
        if (eih) term_eih_sun<double, TS>(E, xr, vr, s.x, s.v, GMs, a.S0, dS0, s.S1, s.aj, false, acc, J);
        if (forces & F_GR_POTENTIAL) term_gr_potential<double, TS>(E, xr, s.x, GMs, false, acc, J);
        if (forces & F_GR_SIMPLE) term_gr_simple<double, TS>(E, xr, vr, s.x, s.v, GMs, false, acc, J);
    } else {
        if (Marsden && (forces & F_NONGRAV) && ng) fp64::term_nongrav(O, xr, vr, s.x, s.v, A, false, acc, J);
        if (forces & F_EARTH_H) fp64::term_earth_J2J4(E, xr, earth, E.GM[3], false, acc, J);
        if (forces & F_SUN_H) fp64::term_solar_J2(E, xr, s.x, GMs, false, acc, J);
        if (eih) fp64::term_eih_sun(E, xr, vr, s.x, s.v, GMs, a.S0, dS0, s.S1, s.aj, false, acc, J);
        if (forces & F_GR_POTENTIAL) fp64::term_gr_potential(E, xr, s.x, GMs, false, acc, J);
        if (forces & F_GR_SIMPLE) fp64::term_gr_simple(E, xr, vr, s.x, s.v, GMs, false, acc, J);
    }
    if (forces & (F_SUN | F_PLANETS | F_ASTEROIDS)) {
#pragma unroll
        for (int c = 0; c < 3; c++) acc[c] += a.ad[c] + double(a.adt[c]);
    }
}

// The bodies whose second time lies in another record than their first, as a wave's list of (lane,
// body) items: a ring of kListItems in LDS, emptied by all active lanes together.
constexpr int kListItems = 128;
struct LateItems {
    unsigned short* ring;
    int head, count;  // (the same on all lanes)
};

// The second time's raw positions (km) of items of the list, one per active lane.  `column` is lane 0's
// column of the position table.
__device__ __forceinline__ void late_round(const DevEphem& E, LateItems& L, double tB, double* column) {
#if defined(__HIP_DEVICE_COMPILE__)
    const unsigned long long act = __ballot(1);
    const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(act >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)act, 0u));
    const int m = min(L.count, (int)__popcll(act));
    // (LDS operations of one wave complete in order; the fences keep the compiler's order too)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int item = L.ring[(L.head + (rank < m ? rank : 0)) & (kListItems - 1)];
    const int src = item & 63, b = item >> 6;
    const double t = __shfl(tB, src, 64);
    if (rank < m) {
        const ChebOut<double> o = cheb_eval<double, false>(E.slot[b < 3 ? b : b + 1], t);
        double* p = column + (size_t)(3 * (b - 1)) * 64 + src;
        p[0] = o.x;
        p[64] = o.y;
        p[128] = o.z;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    L.head = (L.head + m) & (kListItems - 1);
    L.count -= m;
#endif
}

// Both times of the bodies [from, to): the first time's pulls into `a`, the second time's raw positions
// (km) into LDS.  `r` holds the first body's record for the first time; while a body's pull is added, the
// next one's is loaded (after the last planet the first asteroid's; the last asteroid's again, since a
// load under a condition would cost a copy of the record).  A lane whose second time lies in another
// record (about 1.7 bodies a trip) leaves that body to the list.
template <bool Mixed, bool Planet, int NP, typename TS>
__device__ __forceinline__ void walk_bodies(KEphem E, const DevEphem& El, int from, int to, double tA, double tB, bool allowed,
                                            bool eih, const double xr[3], SunState& sA, const double embA[3],
                                            double earth[3], BodySums<TS>& a, LateItems& L, double* column, int wl,
                                            Record& r) {
    auto slot = [&](int b) { return &E->slot[Planet && b < 3 ? b : b + 1]; };
#pragma unroll 1
    for (int b = from; b < to; b++) {
        const KSlot S = slot(b);
        const bool late = lane_record(S, tB) != lane_record(S, tA);
        const bool em = Planet && (b == 3 || b == 4);  // the Earth and the Moon, relative to the EMB
        const double inv_au = E->inv_au, inv_au_ast = E->inv_au_ast, GM = E->GM[b];
        double x[3], y[3], pk[3];
        r.eval<NP, false>(tA, x, nullptr);
        r.eval<NP, false>(tB, y, nullptr);
        {
            const KSlot N = slot(Planet || b + 1 < to ? b + 1 : b);
            r.load<NP>(N, lane_record(N, tA));
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            column[(3 * (b - 1) + c) * 64 + wl] = y[c];
            pk[c] = Planet ? (em ? x[c] + embA[c] : x[c]) * inv_au : fma(x[c], inv_au_ast, sA.x[c]);
        }
        if (Planet && b == 3) { earth[0] = pk[0]; earth[1] = pk[1]; earth[2] = pk[2]; }
        add_body<Mixed, Planet>(GM, allowed, eih, xr, pk, a);
        if (Planet && eih) sA.newton(GM, pk);
#if defined(__HIP_DEVICE_COMPILE__)
        const unsigned long long mask = __ballot(late);
        if (late) {
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
            L.ring[(L.head + L.count + rank) & (kListItems - 1)] = (unsigned short)(b * 64 + wl);
        }
        L.count += (int)__popcll(mask);
#endif
        while (L.count >= 64) late_round(El, L, tB, column);
    }
}

// The corrector of substep N: improves g_{N-1} and b_0..b_{N-1}; tmp: the change of b_{N-1}.
template <int N>
__device__ __forceinline__ void correct(const double at[3], const double a0[3], double (&b)[7][3], double (&g)[7][3],
                                        double tmp[3]) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
        double val = at[c] - a0[c];
#pragma unroll
        for (int k = 0; k < N - 1; k++) val = fma(val, cRRI[N * (N - 1) / 2 + k], -g[k][c]);
        val *= cRRI[N * (N - 1) / 2 + N - 1];
        tmp[c] = val - g[N - 1][c];
        g[N - 1][c] = val;
#pragma unroll
        for (int k = 0; k < N - 1; k++) b[k][c] = fma(tmp[c], cC[(N - 1) * (N - 2) / 2 + k], b[k][c]);
        b[N - 1][c] += tmp[c];
    }
}

template <bool Mixed, bool Marsden>
__global__ void __launch_bounds__(kIas15Block) __attribute__((amdgpu_waves_per_eu(1, 1)))
ias15_lane_kernel(IntegrateArgs args) {
    (void)args;
    KArgs ka = (KArgs)__builtin_amdgcn_kernarg_segment_ptr();
    using TS = typename TermScalar<double, Mixed>::type;
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    const int wl = threadIdx.x & 63;
    // b of the last accepted step and its prediction's correction e, word k of the wave's lanes together
    // (the lane is laundered, so that the words' addresses are not kept in registers across the loop)
    auto scratch = [&]() {
        int l = wl;
        asm volatile("" : "+v"(l));
        return ka->scratch + (size_t)(tid >> 6) * (64 * 42) + l;
    };
    // the second time's positions of the bodies 1-26
    extern __shared__ double s_pos[];
    double* const column = s_pos + (size_t)(threadIdx.x >> 6) * (64 * kLanePosWords);
    double* const pos = column + wl;
    __shared__ unsigned short s_ring[kIas15Block / 64][kListItems];
    __shared__ DevEphem s_E;
    {
        const unsigned long long* src = (const unsigned long long*)ka->E;
        unsigned long long* dst = (unsigned long long*)&s_E;
        for (int i = threadIdx.x; i < (int)(sizeof(DevEphem) / sizeof(unsigned long long)); i += blockDim.x) dst[i] = src[i];
    }
    __syncthreads();

    double x0[3], v0[3], csx[3], csv[3], a0[3], A[3] = {0.0, 0.0, 0.0};
    double b[7][3], g[7][3];
#pragma unroll
    for (int k = 0; k < 7; k++)
#pragma unroll
        for (int c = 0; c < 3; c++) b[k][c] = g[k][c] = 0.0;
    double t = 0, t_end = 0, dt = 0, dts = 0, dt_last = 0, pc_err_last = 0;
    int it = 0, last = 0, status = 0, attempts = 0;
    long long steps = 0, evals = 0, rejected = 0;
    // what a pass begins with: the evaluation at the step's start (a new step), the prediction (a new
    // attempt), or neither (a repeated pass)
    bool start = true, predict = true;
    bool ng = false;
    // a wave's systems are the positions wave, wave + nwaves, wave + 2 nwaves, ... of the order: which
    // systems it leaves to the 16-lane kernel does not depend on the other waves' pace
    const int nwaves = (int)((gridDim.x * blockDim.x) >> 6), wave = tid >> 6;
    auto position = [&](int k) { return (long long)k * nwaves + wave; };
    int taken = 64;  // (the same on all active lanes)
    bool active = position(wl) < ka->nsys;
    int sys = active ? (ka->order ? ka->order[position(wl)] : (int)position(wl)) : 0;

    auto load = [&](int s) {
        const double* st = ka->states + (size_t)s * 6;
        double sv[6], pa[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 6; k++) sv[k] = st[k];
        if (Marsden) {
#pragma unroll
            for (int c = 0; c < 3; c++) pa[c] = ka->params[(size_t)s * 3 + c];
        }
        const double t0s = ka->t0[s], t1s = ka->t1[s];
        const double dtl = (ka->dt0 ? ka->dt0 : ka->t0)[s];
        const double dt0s = ka->dt0 ? fabs(dtl) : ka->io.dt_initial;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            x0[c] = sv[c];
            v0[c] = sv[3 + c];
            csx[c] = csv[c] = a0[c] = 0.0;
            A[c] = pa[c];
        }
        ng = Marsden && !(A[0] == 0.0 && A[1] == 0.0 && A[2] == 0.0);
        t = t0s;
        t_end = t1s;
        dt = dt0s;
        if (dt * (t_end - t) < 0) dt = -dt;
        dt_last = 0.0;
        start = predict = true;
        status = 0;
        steps = evals = rejected = 0;
        last = 0;
    };
    auto finish = [&]() {
        double* st = ka->states + (size_t)sys * 6;
#pragma unroll
        for (int c = 0; c < 3; c++) { st[c] = x0[c]; st[3 + c] = v0[c]; }
        if (ka->status) ka->status[sys] = status;
        if (ka->steps) ka->steps[sys] = steps;
        if (ka->evals) ka->evals[sys] = evals;
        if (ka->rejected) ka->rejected[sys] = rejected;
        if (ka->t_out) ka->t_out[sys] = t;
    };
    // Lanes that are done write their system and take the wave's next ones, in the order of the lanes; all
    // active lanes call this together.  (A system with a zero-length span is done at once.)
    auto take_next = [&](bool done) {
#if defined(__HIP_DEVICE_COMPILE__)
        for (unsigned long long fin = __ballot(done); fin != 0ULL; fin = __ballot(done)) {
            if (done) {
                finish();
                const int k = taken + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(fin >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((unsigned)fin, 0u));
                const long long q = position(k);
                active = q < ka->nsys;
                done = false;
                if (active) {
                    sys = ka->order ? ka->order[q] : (int)q;
                    load(sys);
                    done = t == t_end;
                }
            }
            taken += (int)__popcll(fin);
        }
#endif
    };
    // Leaves the system, at a step boundary, to the 16-lane kernel.
    auto leave = [&]() {
        const int q = atomicAdd(ka->late_count, 1);
        if (q >= ka->late_cap) return;  // (it stays here)
        double* const rec = ka->late + (size_t)q * kLateWords;
        const double* const scr = scratch();
        rec[0] = (double)sys; rec[1] = t; rec[2] = dt; rec[3] = dt_last;
        rec[4] = (double)steps; rec[5] = (double)evals; rec[6] = (double)rejected;
#pragma unroll
        for (int c = 0; c < 3; c++) { rec[8 + c] = x0[c]; rec[11 + c] = v0[c]; rec[14 + c] = csx[c]; rec[17 + c] = csv[c]; }
        const bool stepped = dt_last != 0.0;
#pragma unroll 6
        for (int k = 0; k < 42; k++) rec[20 + k] = stepped ? scr[k * 64] : 0.0;
        active = false;
    };
    // Predict b of the attempt from the last accepted step and convert it to g.
    auto setup_attempt = [&]() {
        if (!(fabs(dts) > 0.0) || !(fabs(dts) < 1e300) || ++attempts > 64) { status = kDtUnderflow; return; }
        const double q = dts / dt_last;
        const double* const scr = scratch();
        if (dt_last != 0.0 && !(q > 20.0)) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                double br[7], er[7], e[7];
#pragma unroll
                for (int k = 0; k < 7; k++) { br[k] = scr[(3 * k + c) * 64]; er[k] = scr[(21 + 3 * k + c) * 64]; }
                predict_e(br, q, e);
#pragma unroll
                for (int k = 0; k < 7; k++) b[k][c] = e[k] + (br[k] - er[k]);
            }
        } else if (dt_last == 0.0 && ka->bw) {
            // learned warm start of the first step: b_k = bw_k |a0| dt^(k+1)
            const double* w = ka->bw + (size_t)sys * 21;
            const double amag = sqrt(a0[0] * a0[0] + a0[1] * a0[1] + a0[2] * a0[2]);
            double hp = dts;
#pragma unroll
            for (int k = 0; k < 7; k++) {
#pragma unroll
                for (int c = 0; c < 3; c++) b[k][c] = w[3 * k + c] * amag * hp;
                hp *= dts;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 7; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) b[k][c] = 0.0;
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double b0 = b[0][c], b1 = b[1][c], b2 = b[2][c], b3 = b[3][c], b4 = b[4][c], b5 = b[5][c], b6 = b[6][c];
            g[0][c] = b6 * cD[15] + b5 * cD[10] + b4 * cD[6] + b3 * cD[3] + b2 * cD[1] + b1 * cD[0] + b0;
            g[1][c] = b6 * cD[16] + b5 * cD[11] + b4 * cD[7] + b3 * cD[4] + b2 * cD[2] + b1;
            g[2][c] = b6 * cD[17] + b5 * cD[12] + b4 * cD[8] + b3 * cD[5] + b2;
            g[3][c] = b6 * cD[18] + b5 * cD[13] + b4 * cD[9] + b3;
            g[4][c] = b6 * cD[19] + b5 * cD[14] + b4;
            g[5][c] = b6 * cD[20] + b5;
            g[6][c] = b6;
        }
        it = 1;
        pc_err_last = 1e300;
        predict = false;
    };
    // State of the particle at substep n (uniform) from the step's polynomial.
    auto predict_state = [&](int n, double xe[3], double ve[3]) {
        const double dt2 = dts * dts;
        double s[9];
        s[0] = dts * cH[n];
#pragma unroll
        for (int k = 1; k < 9; k++) s[k] = dt2 * cPX[8 * n + k - 1];
#pragma unroll
        for (int c = 0; c < 3; c++)
            xe[c] = -csx[c] + ((s[8] * b[6][c] + s[7] * b[5][c] + s[6] * b[4][c] + s[5] * b[3][c] + s[4] * b[2][c] +
                                s[3] * b[1][c] + s[2] * b[0][c] + s[1] * a0[c] + s[0] * v0[c]) + x0[c]);
#pragma unroll
        for (int k = 1; k < 8; k++) s[k] = dts * cPV[7 * n + k - 1];
#pragma unroll
        for (int c = 0; c < 3; c++)
            ve[c] = -csv[c] + ((s[7] * b[6][c] + s[6] * b[5][c] + s[5] * b[4][c] + s[4] * b[3][c] + s[3] * b[2][c] +
                                s[2] * b[1][c] + s[1] * b[0][c] + s[0] * a0[c]) + v0[c]);
    };
    // An evaluation at time te counts, and ends the system outside the ephemeris' coverage.
    auto count = [&](double te, double t_lo, double t_hi) {
        if (status != 0) return;
        evals++;
        if (!(te >= t_lo && te <= t_hi)) status = kCoverage;
    };

    if (active) {
        load(sys);
        take_next(t == t_end);
    }
    while (active) {
        ka = launder(ka);
        if (start) {
            const double dir = (t_end >= t) ? 1.0 : -1.0;
            dts = dt;
            last = 0;
            if ((t + dts - t_end) * dir >= 0) { dts = t_end - t; last = 1; }
            attempts = 0;
        }
        double at[3], tmp[3];
#pragma unroll 1
        for (int p = 0; p < 4; p++) {
            const KEphem E = (KEphem)ka->E;
            const ForceOpts fo = ka->fo;
            const int forces = fo.forces;
            const bool eih = (forces & F_GR_EIH) && fo.gr_eih_sources > 0;
            const int n = 2 * p;
            const double tA = p == 0 ? t : fma(dts, cH[n], t), tB = fma(dts, cH[n + 1], t);
            double xe[3], ve[3];
            if (p == 0) {
#pragma unroll
                for (int c = 0; c < 3; c++) { xe[c] = x0[c]; ve[c] = v0[c]; }
            } else {
                predict_state(n, xe, ve);
            }
            // ---- first time, and the ephemeris of the second ----
            SunState sA, sB;
            BodySums<TS> sums;
            double embA[3], embB[3], earth[3] = {0.0, 0.0, 0.0};
            sums_zero(sums);
            Record r;
            {
                const KSlot S0 = &E->slot[0], S3 = &E->slot[kSlotEMB];
                const int sun_A = lane_record(S0, tA), sun_B = lane_record(S0, tB);
                const int emb_A = lane_record(S3, tA), emb_B = lane_record(S3, tB);
                r.load<kCoefPad>(S0, sun_A);
                r.eval<kCoefPad, true>(tA, sA.x, sA.v);
                if (sun_B != sun_A) r.load<kCoefPad>(S0, sun_B);
                r.eval<kCoefPad, true>(tB, sB.x, sB.v);
                pin(sA.x); pin(sA.v); pin(sB.x); pin(sB.v);
                r.load<kCoefPad>(S3, emb_A);
                r.eval<kCoefPad, false>(tA, embA, nullptr);
                if (emb_B != emb_A) r.load<kCoefPad>(S3, emb_B);
                r.eval<kCoefPad, false>(tB, embB, nullptr);
                pin(embA); pin(embB);
                const KSlot S1 = &E->slot[1];
                r.load<kCoefPad>(S1, lane_record(S1, tA));
                const double inv_au = E->inv_au;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    sA.x[c] *= inv_au; sA.v[c] *= inv_au;
                    sB.x[c] *= inv_au; sB.v[c] *= inv_au;
                    sA.aj[c] = sB.aj[c] = 0.0;
                }
                sA.S1 = sB.S1 = 0.0;
            }
            const int nbody = kNumPlanets + E->n_ast;
            LateItems late{s_ring[threadIdx.x >> 6], 0, 0};
            walk_bodies<Mixed, true, kCoefPad>(E, s_E, 1, kNumPlanets, tA, tB, (forces & F_PLANETS) != 0, eih, xe, sA, embA,
                                               earth, sums, late, column, wl, r);
            if (E->short_from <= kFirstAsteroidSlot)
                walk_bodies<Mixed, false, kCoefShort>(E, s_E, kNumPlanets, nbody, tA, tB, (forces & F_ASTEROIDS) != 0, eih,
                                                      xe, sA, embA, earth, sums, late, column, wl, r);
            else
                walk_bodies<Mixed, false, kCoefPad>(E, s_E, kNumPlanets, nbody, tA, tB, (forces & F_ASTEROIDS) != 0, eih, xe,
                                                    sA, embA, earth, sums, late, column, wl, r);
            while (late.count > 0) late_round(s_E, late, tB, column);
            add_body<Mixed, true>(E->GM[0], (forces & F_SUN) != 0, eih, xe, sA.x, sums);
            add_terms<Mixed, Marsden>(s_E, fo, xe, ve, sA, earth, A, ng, sums, at);
            if (p == 0) {
                if (start) {
                    count(tA, fo.t_lo, fo.t_hi);
#pragma unroll
                    for (int c = 0; c < 3; c++) a0[c] = at[c];
                    start = false;
                }
                if (predict && status == 0) setup_attempt();
            } else {
                count(tA, fo.t_lo, fo.t_hi);
                if (p == 1) correct<2>(at, a0, b, g, tmp);
                else if (p == 2) correct<4>(at, a0, b, g, tmp);
                else correct<6>(at, a0, b, g, tmp);
            }
            // ---- second time ----
            predict_state(n + 1, xe, ve);
            sums_zero(sums);
            const double inv_au = E->inv_au, inv_au_ast = E->inv_au_ast;
#pragma unroll 2
            for (int k = 1; k < kNumPlanets; k++) {
                const bool em = k == 3 || k == 4;
                double pk[3];
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const double x = pos[(3 * (k - 1) + c) * 64];
                    pk[c] = (em ? x + embB[c] : x) * inv_au;
                }
                if (k == 3) { earth[0] = pk[0]; earth[1] = pk[1]; earth[2] = pk[2]; }
                add_body<Mixed, true>(E->GM[k], (forces & F_PLANETS) != 0, eih, xe, pk, sums);
                if (eih) sB.newton(E->GM[k], pk);
            }
#pragma unroll 4
            for (int k = kNumPlanets; k < nbody; k++) {
                double pk[3];
#pragma unroll
                for (int c = 0; c < 3; c++) pk[c] = fma(pos[(3 * (k - 1) + c) * 64], inv_au_ast, sB.x[c]);
                add_body<Mixed, false>(E->GM[k], (forces & F_ASTEROIDS) != 0, eih, xe, pk, sums);
            }
            add_body<Mixed, true>(E->GM[0], (forces & F_SUN) != 0, eih, xe, sB.x, sums);
            add_terms<Mixed, Marsden>(s_E, fo, xe, ve, sB, earth, A, ng, sums, at);
            count(tB, fo.t_lo, fo.t_hi);
            if (p == 0) correct<1>(at, a0, b, g, tmp);
            else if (p == 1) correct<3>(at, a0, b, g, tmp);
            else if (p == 2) correct<5>(at, a0, b, g, tmp);
            else correct<7>(at, a0, b, g, tmp);
        }
        // (returns whether the system is done)
        auto end_pass = [&]() -> bool {
            if (status != 0) return true;
            // ---- end of a predictor-corrector iteration (the tests are ias15_kernel's) ----
            double maxak = 0.0, maxdb6 = 0.0;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double ak = fabs(at[c]);
                if (is_normal(ak) && ak > maxak) maxak = ak;
                const double db = fabs(tmp[c]);
                if (is_normal(db) && db > maxdb6) maxdb6 = db;
            }
            const double pc_tol = ka->io.pc_tol;
            const double pc_err = maxdb6 / maxak;
            const double pc_aref = ka->io.pc_aref;
            const double pc_tol1 = (pc_aref > 0.0 && maxak > pc_aref) ? ka->io.pc_tol1 * fmax(0.1, pc_aref / maxak) : ka->io.pc_tol1;
            if (!(pc_err < (pc_tol > 0.0 ? pc_tol : 1e-16)) && !(it == 1 && pc_err < pc_tol1) &&
                !(it > 2 && pc_err_last <= pc_err) && it < 12) {
                pc_err_last = pc_err;
                it++;
                return false;
            }
            // ---- step-size control ----
            double dt_new = dts, dt_prop = dts;
            if (ka->io.epsilon > 0) {
                double mb6 = 0.0;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const double bk = fabs(b[6][c]);
                    if (is_normal(bk) && bk > mb6) mb6 = bk;
                }
                const double err = mb6 / maxak;
                if (is_normal(err)) dt_new = pow(ka->io.epsilon / err, 1.0 / 7.0) * dts;
                else dt_new = dts / 0.25;
                if (fabs(dt_new) < ka->io.min_dt) dt_new = copysign(ka->io.min_dt, dt_new);
                if (fabs(dt_new / dts) < 0.25) {
                    rejected++;
                    dts = dt_new;
                    last = 0;
                    predict = true;
                    return false;
                }
                dt_prop = dt_new;
                if (dt_new / dts > 1. / 0.25) dt_new = dts / 0.25;
            }
            // ---- accept: advance x0, v0 (Kahan) and store br, er ----
            if (ka->trace && steps >= ka->trace_skip && steps % ka->trace_every == 0) {
                const int idx = atomicAdd(ka->trace_count, 1);
                if (idx < ka->trace_cap) {
                    double* rec = ka->trace + (size_t)idx * kTraceWords;
                    rec[0] = t;
                    rec[7] = dt_last;
                    rec[8] = dts;
                    rec[9] = dt_prop;
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        rec[1 + c] = x0[c]; rec[4 + c] = v0[c]; rec[10 + c] = a0[c];
#pragma unroll
                        for (int k = 0; k < 7; k++) rec[13 + 3 * k + c] = b[k][c];
                    }
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
#pragma unroll
            for (int c = 0; c < 3; c++) {
#pragma unroll
                for (int k = 6; k >= 0; k--) add_cs(x0[c], csx[c], b[k][c] * wx[k + 1]);
                add_cs(x0[c], csx[c], a0[c] * wx[0]);
                add_cs(x0[c], csx[c], v0[c] * dts);
#pragma unroll
                for (int k = 6; k >= 0; k--) add_cs(v0[c], csv[c], b[k][c] * wv[k]);
                add_cs(v0[c], csv[c], a0[c] * dts);
            }
            const double q = (dt_last != 0.0) ? dts / dt_last : 0.0;
            double* const scr = scratch();
            const bool stepped = dt_last != 0.0 && q <= 20.0;
            int bad = 0;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                double br[7], e[7];
#pragma unroll
                for (int k = 0; k < 7; k++) br[k] = scr[(3 * k + c) * 64];
                predict_e(br, q, e);
#pragma unroll
                for (int k = 0; k < 7; k++) {
                    scr[(21 + 3 * k + c) * 64] = stepped ? e[k] : 0.0;
                    scr[(3 * k + c) * 64] = b[k][c];
                }
                bad |= !(fabs(x0[c]) < 1e300) || !(fabs(v0[c]) < 1e300);
            }
            t = last ? t_end : t + dts;
            steps++;
            dt_last = dts;
            if (!(last && ka->io.epsilon <= 0)) dt = dt_new;
            start = predict = true;
            if (bad) { status = kNonFinite; return true; }
            if (last) return true;
            if (steps >= ka->io.max_steps) { status = kMaxSteps; return true; }
            return false;
        };
        take_next(end_pass());
        // (lanes run out only when the wave's systems have)
        if (ka->late && (int)__popcll(__ballot(active)) <= kLateLanes && active && start) leave();
    }
}

static const void* lane_lookup(const IntegrateArgs& a, bool mixed) {
    if (a.nvec != 1 || a.out_t || ias15_snap(a) || ext_model(a.fo)) return nullptr;
    if (a.params) return mixed ? (const void*)ias15_lane_kernel<true, true> : (const void*)ias15_lane_kernel<false, true>;
    return mixed ? (const void*)ias15_lane_kernel<true, false> : (const void*)ias15_lane_kernel<false, false>;
}

static size_t lane_lds_bytes(int threads) { return (size_t)threads * kLanePosWords * sizeof(double); }

hipError_t launch_ias15_lane(const IntegrateArgs& a, bool mixed, int blocks, int threads, hipStream_t s, bool set_attributes) {
    const void* f = lane_lookup(a, mixed);
    if (!f || threads % 64 != 0 || threads > kIas15Block) return hipErrorInvalidValue;
    const size_t lds = lane_lds_bytes(threads);
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

hipError_t ias15_lane_occupancy(const IntegrateArgs& a, bool mixed, int threads, int* blocks_per_cu) {
    const void* f = lane_lookup(a, mixed);
    if (!f) return hipErrorInvalidValue;
    const size_t lds = lane_lds_bytes(threads);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, threads, lds);
}

}  // namespace assist_gpu
