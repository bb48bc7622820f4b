// The single-particle terms in double precision, with every rounding of a value or partial that
// reaches the result spelled out (fused multiply-adds written as such, the compiler's own contraction
// off or without effect), so that kernels of different structure agree bit for bit, and with the
// partials row by row: a lane that integrates one component of a variational vector needs one row of
// the Jacobian, and computes that one alone (the 8-lane kernels, whose lanes hold whole vectors, ask
// for all three).  The values round as force_model.h's terms do in those kernels.
//
// The mixed form's terms stay those of force_model.h: a partial in FP32 that rounded differently
// anywhere would move its variational states by FP32 round-off.
//
// Included by force_model.h, after what these use of it.
#pragma once

namespace assist_gpu {

// One row of it, d a_c / d (x, v, A): what a lane that integrates component c needs.
template <typename T>
struct JacRow {
    T x[3], v[3], A[3];
    int c;
};

template <typename T>
AHD void jac_zero(JacRow<T>& J) {
#pragma unroll
    for (int j = 0; j < 3; j++) J.x[j] = J.v[j] = J.A[j] = T(0);
}

// f(i, x, v, A) for every row i that J holds (its parts as pointers to 3 values).  The terms
// write their partials with the fused multiply-adds spelled out and the compiler's own
// contraction off, so that a row has the same bits whichever kernel computes it.
template <typename T, typename F>
AHD void jac_rows(Jac<T>& J, F f) {
#pragma unroll
    for (int i = 0; i < 3; i++) f(i, J.x[i], J.v[i], J.A[i]);
}
template <typename T, typename F>
AHD void jac_rows(JacRow<T>& J, F f) {
    f(J.c, J.x, J.v, J.A);
}

template <typename T>
AHD T pick3(int i, T a, T b, T c) {
    return i == 0 ? a : (i == 1 ? b : c);
}

// a . b and a b - c d with their roundings spelled out
template <typename T>
AHD T dot3(T ax, T ay, T az, T bx, T by, T bz) {
    return fma(az, bz, fma(ax, bx, ay * by));
}
template <typename T>
AHD T diff2(T a, T b, T c, T d) {
    return fma(a, b, -(c * d));
}

namespace fp64 {

// J.x += R^T S R for a symmetric S given as (xx, yy, zz, xy, yz, xz)
template <typename JT>
AHD void add_rotated_sym(JT& J, const Rot<double>& R, double sxx, double syy, double szz, double sxy, double syz, double sxz) {
#pragma clang fp contract(off)
    const double S[3][3] = {{sxx, sxy, sxz}, {sxy, syy, syz}, {sxz, syz, szz}};
    double SR[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++)
            SR[i][j] = fma(S[i][2], R.r[2][j], fma(S[i][1], R.r[1][j], S[i][0] * R.r[0][j]));
    jac_rows(J, [&](int i, double* x, double*, double*) {
#pragma clang fp contract(off)
        const double r0 = pick3(i, R.r[0][0], R.r[0][1], R.r[0][2]);
        const double r1 = pick3(i, R.r[1][0], R.r[1][1], R.r[1][2]);
        const double r2 = pick3(i, R.r[2][0], R.r[2][1], R.r[2][2]);
#pragma unroll
        for (int j = 0; j < 3; j++) x[j] += fma(r2, SR[2][j], fma(r1, SR[1][j], r0 * SR[0][j]));
    });
}

// Earth J2/J3/J4 (reference src/forces.c:435-642).
// The Earth's pole is fixed at RA 0, Dec 90 deg (reference src/forces.c:484-490): the rotation
// has cos RA = 1, sin RA = 0, sin Dec = 1 exactly and keeps cos Dec = cos(pi/2) = 6.1e-17,
// whose residue the reference carries, so it is written out for that form (rows (0, 1, 0),
// (-1, 0, c), (c, 0, 1) with c = cos Dec).  Powers of 1/r replace the reference's divisions.
template <typename JT>
AHD void term_earth_J2J4(const DevEphem& E, const double xr[3], const double xe[3], double GM, bool need_jac, double acc[3], JT& Jt) {
    const double c = E.e_cosd;
    const double ex = xr[0] - xe[0], ey = xr[1] - xe[1], ez = xr[2] - xe[2];
    const double r2 = dot3(ex, ey, ez, ex, ey, ez);
    const double ir = inv_sqrt(r2);
    const double ir2 = ir * ir;
    const double dx = ey, dy = fma(ez, c, -ex), dz = fma(ex, c, ez);
    const double costheta2 = dz * dz * ir2;
    const double J2p = E.k_J2 * (ir2 * ir2 * ir);  // 3 J2 Re^2 / (2 r^5)
    const double J2f = fma(5.0, costheta2, -1.0);
    double rx = GM * J2p * J2f * dx;
    double ry = GM * J2p * J2f * dy;
    double rz = GM * J2p * (J2f - 2.0) * dz;
    const double ct2 = costheta2;
    const double ir5 = ir2 * ir2 * ir;
    const double J3p = E.k_J3 * ir5;            // 5 J3 Re^3 / (2 r^5)
    const double J3f = fma(-7.0, ct2, 3.0);
    const double J4p = E.k_J4 * (ir5 * ir2);   // 5 J4 Re^4 / (8 r^7)
    const double J4f = fma(-42.0, ct2, 63.0 * ct2 * ct2) + 3.0;
    const double j3x = -GM * J3p * ir2 * J3f * dx * dz;
    const double j3y = -GM * J3p * ir2 * J3f * dy * dz;
    const double j3z = -GM * J3p * (6.0 * ct2 - 7.0 * ct2 * ct2 - 0.6);
    const double j4x = GM * J4p * J4f * dx;
    const double j4y = GM * J4p * J4f * dy;
    const double j4z = GM * J4p * (J4f + 12.0 - 28.0 * ct2) * dz;
    rx += j3x; ry += j3y; rz += j3z;
    rx += j4x; ry += j4y; rz += j4z;
    acc[0] += -ry + rz * c;
    acc[1] += rx;
    acc[2] += ry * c + rz;
    if (!need_jac) return;
    {
#pragma clang fp contract(off)
        const double one = 1.0, ct4 = ct2 * ct2, ct = dz * ir;
        const double x2 = dx * dx * ir2, y2 = dy * dy * ir2;
        const double xy = dx * dy * ir2, yz = dy * dz * ir2, xz = dx * dz * ir2;
        const double k2 = GM * J2p;
        const double f2 = fma(7.0, ct2, -one);
        const double f3 = fma(35.0, ct4, fma(-30.0, ct2, 3.0));
        const double m2 = -5.0 * f2, n2 = k2 * (-5.0 * (f2 - 2.0));
        double sxx = k2 * fma(m2, x2, J2f), syy = k2 * fma(m2, y2, J2f), szz = -k2 * f3;
        double sxy = k2 * m2 * xy, syz = n2 * yz, sxz = n2 * xz;
        const double k3 = GM * J3p, k3c = k3 * ct * ir;
        const double g2 = 21.0 * fma(-3.0, ct2, one);
        const double g3 = k3 * (3.0 * fma(-21.0, ct4, fma(14.0, ct2, -one)) * ir2);
        const double g4 = fma(-63.0, ct4, fma(70.0, ct2, -15.0)) * ct * ir;
        sxx = fma(k3c, fma(g2, x2, -J3f), sxx);
        syy = fma(k3c, fma(g2, y2, -J3f), syy);
        szz = fma(k3, g4, szz);
        sxy = fma(k3c * g2, xy, sxy);
        syz = fma(g3, dy, syz);
        sxz = fma(g3, dx, sxz);
        const double k4 = GM * J4p;
        const double h2 = -21.0 * fma(33.0, ct4, fma(-18.0, ct2, one));
        const double h3 = k4 * (-21.0 * fma(33.0, ct4, fma(-30.0, ct2, 5.0)));
        const double h4 = fma(fma(231.0, ct2, -315.0), ct4, fma(105.0, ct2, -5.0));
        sxx = fma(k4, fma(h2, x2, J4f), sxx);
        syy = fma(k4, fma(h2, y2, J4f), syy);
        szz = fma(k4, -3.0 * h4, szz);
        sxy = fma(k4 * h2, xy, sxy);
        syz = fma(h3, yz, syz);
        sxz = fma(h3, xz, sxz);
        // J += R^T S R; R's columns are u0 = (0, -1, c), u1 = (1, 0, 0), u2 = (0, c, 1) and
        // (R^T S R)_ij = u_i . (S u_j)
        const double w[3][3] = {{fma(c, sxz, -sxy), fma(c, syz, -syy), fma(c, szz, -syz)},
                            {sxx, sxy, sxz},
                            {fma(c, sxy, sxz), fma(c, syy, syz), fma(c, syz, szz)}};
        jac_rows(Jt, [&](int i, double* x, double*, double*) {
#pragma clang fp contract(off)
#pragma unroll
            for (int j = 0; j < 3; j++)
                x[j] += pick3(i, fma(c, w[j][2], -w[j][1]), w[j][0], fma(c, w[j][1], w[j][2]));
        });
    }
}

// Solar J2 (reference src/forces.c:644-772).
template <typename JT>
AHD void term_solar_J2(const DevEphem& E, const double xr[3], const double xs[3], double GMs, bool need_jac, double acc[3], JT& Jt) {
    const double cosa = E.s_cosa, sina = E.s_sina, cosd = E.s_cosd, sind = E.s_sind;
    double dx = xr[0] - xs[0], dy = xr[1] - xs[1], dz = xr[2] - xs[2];
    const double r2 = dot3(dx, dy, dz, dx, dy, dz);
    const double ir = inv_sqrt(r2);
    const double ir2 = ir * ir;
    const double dxp = diff2(dy, cosa, dx, sina);
    const double dyp = fma(dz, cosd, diff2(-(dx * cosa), sind, dy * sina, sind));
    const double dzp = dot3(dx * cosa, dy * sina, dz, cosd, cosd, sind);
    dx = dxp; dy = dyp; dz = dzp;
    const double costheta2 = dz * dz * ir2;
    const double pf = E.k_sJ2 * (ir2 * ir2 * ir);  // 3 J2sun Rs^2 / (2 r^5)
    const double f1 = fma(5.0, costheta2, -1.0);
    const double rx = GMs * pf * f1 * dx;
    const double ry = GMs * pf * f1 * dy;
    const double rz = GMs * pf * (f1 - 2.0) * dz;
    acc[0] += -rx * sina - ry * cosa * sind + rz * cosa * cosd;
    acc[1] += rx * cosa - ry * sina * sind + rz * sina * cosd;
    acc[2] += +ry * cosd + rz * sind;
    if (!need_jac) return;
    {
#pragma clang fp contract(off)
        const double t2 = costheta2, gp = GMs * pf;
        const double f2 = fma(7.0, t2, -1.0);
        const double f3 = fma(35.0, t2 * t2, fma(-30.0, t2, 3.0));
        const double m2 = -5.0 * f2, n2 = gp * (-5.0 * (f2 - 2.0));
        const double sxx = gp * fma(m2, dx * dx * ir2, f1);
        const double syy = gp * fma(m2, dy * dy * ir2, f1);
        const double szz = -gp * f3;
        const double sxy = gp * m2 * (dx * dy * ir2);
        const double syz = n2 * (dy * dz * ir2);
        const double sxz = n2 * (dx * dz * ir2);
        Rot<double> R(E.s_cosa, E.s_sina, E.s_cosd, E.s_sind);
        add_rotated_sym(Jt, R, sxx, syy, szz, sxy, syz, sxz);
    }
}

// Marsden non-gravitational acceleration (reference src/forces.c:774-1057).
template <typename JT>
AHD void term_nongrav(const ForceOpts& O, const double xr[3], const double vr[3], const double xs[3], const double vs[3], const double A[3],
                      bool need_jac, double acc[3], JT& Jt) {
    const double dx = (xr[0] - xs[0]), dy = (xr[1] - xs[1]), dz = (xr[2] - xs[2]);
    const double dvx = (vr[0] - vs[0]), dvy = (vr[1] - vs[1]), dvz = (vr[2] - vs[2]);
    const double A1 = A[0], A2 = A[1], A3 = A[2];
    const double alpha = O.alpha, nk = O.nk, nm = O.nm, nn = O.nn, r0 = O.r0;
    const double r2 = dot3(dx, dy, dz, dx, dy, dz);
    const double r = sqrt(r2);
    const double x = r / r0;
    // x^-nm: for the default model's nm = 2 as 1 / x^2, within an ulp of pow and without its cost
    const double xm = (nm == 2.0) ? 1.0 / (x * x) : pow(x, -nm);
    // nk = 0 (the reference's default, src/assist.c:435): the factor (1 + x^nn)^-nk is pow(., -0),
    // exactly 1 for every argument, so leaving it out gives g bit for bit.
    const bool nk0 = nk == 0.0;
    const double g = nk0 ? alpha * xm : alpha * xm * pow(1.0 + pow(x, nn), -nk);
    const double hx = diff2(dy, dvz, dz, dvy), hy = diff2(dz, dvx, dx, dvz), hz = diff2(dx, dvy, dy, dvx);
    const double h = sqrt(dot3(hx, hy, hz, hx, hy, hz));
    const double tx = diff2(hy, dz, hz, dy), ty = diff2(hz, dx, hx, dz), tz = diff2(hx, dy, hy, dx);
    const double _t = sqrt(dot3(tx, ty, tz, tx, ty, tz));
    // (the radial, transverse and normal unit vectors through one reciprocal each)
    const double gr = A1 * g / r, gt = A2 * g / _t, gh = A3 * g / h;
    acc[0] += dot3(gr, gt, gh, dx, tx, hx);
    acc[1] += dot3(gr, gt, gh, dy, ty, hy);
    acc[2] += dot3(gr, gt, gh, dz, tz, hz);
    if (!need_jac) return;
    {
#pragma clang fp contract(off)
        const double v2 = dot3(dvx, dvy, dvz, dvx, dvy, dvz);
        const double rdotv = dot3(dx, dy, dz, dvx, dvy, dvz);
        const double vdott = dot3(dvx, dvy, dvz, tx, ty, tz);
        // dg/dr = (alpha/r0) (-nm x^(-nm-1) (1+x^nn)^-nk + x^-nm (-nk nn) x^(nn-1) (1+x^nn)^(-nk-1)).
        // With nk = +0 and nn >= +0 finite, -nk nn = -0; for 0 < x finite the other factors of the
        // second term are >= +0, so the term is -0 whenever x^-nm and x^(nn-1) are finite, and adding
        // -0 leaves the first term unchanged bit for bit.  x^(nn-1) is finite when |nn-1| (|e|+1)
        // stays below the overflow exponent, e the binary exponent of x (x in [2^(e-1), 2^e)); then
        // the three powers of the second term are skipped.
        int ex = 0;
        (void)frexp(x, &ex);
        const double e_lim = sizeof(double) == 8 ? 1000.0 : 120.0;
        const bool short_dg = nk0 && !signbit(nk) && nn >= 0.0 && !signbit(nn) && isfinite(nn) && x > 0.0 &&
                              isfinite(x) && isfinite(xm) && fabs(nn - 1.0) * (abs(ex) + 1) < e_lim;
        // x^(-nm-1): for the default model's nm = 2 as x^-2 / x
        const double xm1 = (nm == 2.0) ? xm / x : pow(x, -nm - 1.0);
        double dgdr = (alpha / r0) * (-nm * xm1);
        if (!short_dg)
            dgdr = (alpha / r0) * (-nm * xm1 * pow(1.0 + pow(x, nn), -nk) +
                                   xm * (-nk * nn) * pow(x, nn - 1.0) * pow(1.0 + pow(x, nn), -nk - 1.0));
        // The partials of A1 g u + A2 g tau + A3 g eta (u, tau, eta the radial, transverse and normal
        // unit vectors d / r, t / |t|, h / |h|) along d and the velocity, row by row:
        // of a unit vector w / |w| they are (dw - w (w . dw) / |w|^2) / |w|, with
        // t . dt/dd_j = 2 d_j (v . t) - (d . v) t_j, h . dh/dd_j = v^2 d_j - (d . v) v_j,
        // t . dt/dv_j = d^2 t_j, h . dh/dv_j = d^2 v_j - (d . v) d_j.
        const double one = 1.0, two = 2.0;
        const double ir = one / r, it = one / _t, ih = one / h;
        const double d[3] = {dx, dy, dz}, v[3] = {dvx, dvy, dvz};
        const double u[3] = {dx * ir, dy * ir, dz * ir};
        const double tau[3] = {tx * it, ty * it, tz * it};
        const double eta[3] = {hx * ih, hy * ih, hz * ih};
        const double tv[3] = {tx, ty, tz};
        const double gr_ = A1 * (g * ir), gt_ = A2 * (g * it), gh_ = A3 * (g * ih);
        double dg[3], sx[3], hx_[3], hv_[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            dg[j] = dgdr * u[j];
            sx[j] = it * diff2(two * d[j], vdott, rdotv, tv[j]);
            hx_[j] = ih * diff2(v2, d[j], rdotv, v[j]);
            hv_[j] = ih * diff2(r2, v[j], rdotv, d[j]);
        }
        jac_rows(Jt, [&](int i, double* jx, double* jv, double* jA) {
#pragma clang fp contract(off)
            const double di = pick3(i, dx, dy, dz), vi = pick3(i, dvx, dvy, dvz);
            const double ui = pick3(i, u[0], u[1], u[2]), taui = pick3(i, tau[0], tau[1], tau[2]), etai = pick3(i, eta[0], eta[1], eta[2]);
            // row i of dh/dd (the cross product with v) and of -dh/dv (with d)
            const double ev[3] = {pick3(i, 0.0, -dvz, dvy), pick3(i, dvz, 0.0, -dvx), pick3(i, -dvy, dvx, 0.0)};
            const double ed[3] = {pick3(i, 0.0, -dz, dy), pick3(i, dz, 0.0, -dx), pick3(i, -dy, dx, 0.0)};
            const double k = fma(A3, etai, fma(A2, taui, A1 * ui));  // the term along dg/dr
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const double dr = fma(-ui, u[j], i == j ? one : 0.0);
                const double dt = diff2(two * d[j], vi, di, v[j]) - (i == j ? rdotv : 0.0);
                jx[j] += fma(dg[j], k, fma(gr_, dr, fma(gt_, fma(-taui, sx[j], dt), gh_ * fma(-etai, hx_[j], ev[j]))));
                const double dtv = (i == j ? r2 : 0.0) - d[j] * di;
                jv[j] += fma(gt_, fma(-taui, (r2 * it) * tv[j], dtv), gh_ * fma(-etai, hv_[j], -ed[j]));
            }
            jA[0] += g * ui;
            jA[1] += g * taui;
            jA[2] += g * etai;
        });
    }
}

// EIH GR with the Sun as the only source (reference src/forces.c:1288-1983, beta = gamma = 1),
// given the group-summed planet sums: S0 = sum_k GM_k / r_ik, dS0 = -sum_k GM_k d_ik / r_ik^3
// (k over the 11 planetary bodies), S1 = sum_{k != Sun} GM_k / r_sk and the Sun's Newtonian
// acceleration aj from the same bodies.  In double.
template <typename JT>
AHD void term_eih_sun(const DevEphem& E, const double xr[3], const double vr[3], const double xs[3], const double vs[3], double GMs, double S0,
                      const double dS0[3], double S1, const double aj[3], bool need_jac, double acc[3], JT& J) {
    const double oc2 = E.over_c_squared;
    const double dxij = (xr[0] - xs[0]), dyij = (xr[1] - xs[1]), dzij = (xr[2] - xs[2]);
    const double vx = vr[0], vy = vr[1], vz = vr[2];
    const double vxj = vs[0], vyj = vs[1], vzj = vs[2];
    const double GMj = GMs;
    const double rij2 = dot3(dxij, dyij, dzij, dxij, dyij, dzij);
    const double ir = inv_sqrt(rij2);
    const double ir2 = ir * ir;
    const double ir3 = ir2 * ir;
    const double prefacij = GMj * ir3;
    const double vi2 = dot3(vx, vy, vz, vx, vy, vz);
    const double vj2 = dot3(vxj, vyj, vzj, vxj, vyj, vzj);
    const double vidotvj = dot3(vx, vy, vz, vxj, vyj, vzj);
    const double rijdotvj = dot3(dxij, dyij, dzij, vxj, vyj, vzj);
    const double t5 = -1.5 * oc2 * (rijdotvj * rijdotvj);
    const double fx = diff2(4.0, vx, 3.0, vxj), fy = diff2(4.0, vy, 3.0, vyj), fz = diff2(4.0, vz, 3.0, vzj);
    const double f = dot3(dxij, dyij, dzij, fx, fy, fz);
    const double pf = prefacij * f;
    const double rel[3] = {vx - vxj, vy - vyj, vz - vzj};
    const double axj = aj[0], ayj = aj[1], azj = aj[2];
    const double da = dot3(dxij, dyij, dzij, axj, ayj, azj);
    const double t8 = GMj * ir * 3.5;
    // terms 0 to 6 of the reference's bracket
    const double factor = fma(da, -0.5 * oc2, fma(ir2, t5, fma(vidotvj, -4.0 * oc2, fma(vj2, 2.0 * oc2,
                      fma(vi2, oc2, diff2(S0, -4.0 * oc2, S1, oc2))))));
    const double dij[3] = {dxij, dyij, dzij};
    const double ajv[3] = {axj, ayj, azj};
#pragma unroll
    for (int c = 0; c < 3; c++) acc[c] += fma(-(prefacij * dij[c]), factor, fma(t8 * ajv[c], oc2, pf * rel[c] * oc2));
    if (!need_jac) return;
    {
#pragma clang fp contract(off)
        const double pv = GMj * ir3;
        const double g5 = -3.0 * GMj * (ir3 * ir2);
        const double t5f = -3.0 * oc2 * rijdotvj * ir, t5g = rijdotvj * ir3;
        const double m4 = -4.0 * oc2, t6f = -0.5 * oc2;
        const double vj[3] = {vxj, vyj, vzj};
        const double vi[3] = {vx, vy, vz};
        const double fv[3] = {fx, fy, fz};
        double dpref[3], dpf[3], pfv[3], p4d[3], dfx[3], dfv[3];
#pragma unroll
        for (int q = 0; q < 3; q++) {
            dpref[q] = g5 * dij[q];
            dpf[q] = dpref[q] * f;
            pfv[q] = pv * fv[q];
            p4d[q] = pv * (4.0 * dij[q]);
            dfx[q] = fma(dS0[q], m4, fma(t5f, fma(vj[q], ir, -(t5g * dij[q])), t6f * ajv[q]));
            dfv[q] = fma(2.0 * oc2, vi[q], m4 * vj[q]);
        }
        const double pf7 = pv * f;
        jac_rows(J, [&](int c, double* jx, double* jv, double*) {
#pragma clang fp contract(off)
            const double dc = pick3(c, dij[0], dij[1], dij[2]);
            const double rc = pick3(c, rel[0], rel[1], rel[2]);
            const double e8 = -3.5 * (GMj * ir3) * pick3(c, ajv[0], ajv[1], ajv[2]);
            const double pdc = pv * dc;
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const double d7x = fma(dpf[q], rc, pfv[q] * rc);
                double d7v = p4d[q] * rc;
                double v = -fma(dpref[q] * dc, factor, pdc * dfx[q]);
                if (q == c) {
                    d7v += pf7;
                    v = fma(-pv, factor, v);
                }
                jx[q] += v + oc2 * fma(e8, dij[q], d7x);
                jv[q] += fma(-pdc, dfv[q], d7v * oc2);
            }
        });
    }
}

// GR potential form (reference src/forces.c:1059-1161), Sun only.
template <typename JT>
AHD void term_gr_potential(const DevEphem& E, const double xr[3], const double xs[3], double GMs, bool need_jac, double acc[3], JT& J) {
    const double px = (xr[0] - xs[0]), py = (xr[1] - xs[1]), pz = (xr[2] - xs[2]);
    const double r2 = dot3(px, py, pz, px, py, pz);
    const double r = sqrt(r2);
    const double G = GMs;
    const double prefac = -6.0 * G * G / (E.c_squared * r2 * r2);
    acc[0] += (prefac * px);
    acc[1] += (prefac * py);
    acc[2] += (prefac * pz);
    if (!need_jac) return;
    const double u[3] = {px / r, py / r, pz / r};
    jac_rows(J, [&](int i, double* x, double*, double*) {
#pragma clang fp contract(off)
        const double m = -4.0 * prefac * pick3(i, u[0], u[1], u[2]);
#pragma unroll
        for (int j = 0; j < 3; j++) x[j] += fma(m, u[j], i == j ? prefac : 0.0);
    });
}

// GR simple form (reference src/forces.c:1163-1286), Sun only.
template <typename JT>
AHD void term_gr_simple(const DevEphem& E, const double xr[3], const double vr[3], const double xs[3], const double vs[3], double GMs,
                        bool need_jac, double acc[3], JT& J) {
    const double p[3] = {(xr[0] - xs[0]), (xr[1] - xs[1]), (xr[2] - xs[2])};
    const double pv[3] = {(vr[0] - vs[0]), (vr[1] - vs[1]), (vr[2] - vs[2])};
    const double G = GMs;
    const double v2 = dot3(pv[0], pv[1], pv[2], pv[0], pv[1], pv[2]);
    const double r = sqrt(dot3(p[0], p[1], p[2], p[0], p[1], p[2]));
    const double A = 4.0 * G / r - v2;
    const double B = 4.0 * dot3(p[0], p[1], p[2], pv[0], pv[1], pv[2]);
    const double prefac = G / (r * r * r * E.c_squared);
#pragma unroll
    for (int c = 0; c < 3; c++) acc[c] += (prefac * fma(B, pv[c], A * p[c]));
    if (!need_jac) return;
    {
#pragma clang fp contract(off)
        const double dpdr = -3.0 * prefac / r;
        const double g2 = 4.0 * G / (r * r);
        double u[3];
#pragma unroll
        for (int j = 0; j < 3; j++) u[j] = p[j] / r;
        jac_rows(J, [&](int i, double* x, double* v, double*) {
#pragma clang fp contract(off)
            const double pi = pick3(i, p[0], p[1], p[2]), vi = pick3(i, pv[0], pv[1], pv[2]);
            const double Fi = dpdr * fma(A, pi, B * vi);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const double m = fma(4.0 * pv[j], vi, fma(-(pi * u[j]), g2, i == j ? A : 0.0));
                x[j] += fma(u[j], Fi, prefac * m);
                v[j] += prefac * fma(-2.0 * pv[j], pi, fma(4.0 * p[j], vi, i == j ? B : 0.0));
            }
        });
    }
}

}  // namespace fp64
}  // namespace assist_gpu
