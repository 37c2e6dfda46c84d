// Reverse-mode (vector-Jacobian) arithmetic of fvm_math.hpp, derived by hand
// line by line from the forward code.  Every *_vjp function ADDS the adjoint
// of its inputs into the output arrays (so outputs may alias).
//
// Conventions match torch autograd, which the oracle uses: d|x|/dx = sign(x)
// with sign(0) = 0; a switch passes the adjoint to the branch it selected;
// max(a, b) with a == b passes half to each.
#pragma once
#include "fvm_math.hpp"

namespace adfvm {

template <typename T> ADFVM_HD T sgn(T x) { return x > T(0) ? T(1) : (x < T(0) ? T(-1) : T(0)); }

// d mu / dT
template <typename T> ADFVM_HD T viscosity_dT(const Phys<T>& ph, T Tf) {
    if (ph.muModel == 0) return T(0);
    T s = fsqrt(Tf);
    T d = Tf + ph.muTs;
    // mu = A*(T*sqrt(T))/(T+Ts)
    return ph.muA * (T(1.5) * s * d - Tf * s) / (d * d);
}

// primitive(q) -> w ; qb += (dw/dq)^T wb.
// The chain rule through e = E - |U|^2/2 gives for rho the terms
//   pb*(g-1)*e - eb*E/rho - sum_i Ub_i U_i/rho,  eb = Tb/Cv + pb*(g-1)*rho,
// whose p parts cancel down to pb*(g-1)|U|^2/2 (e ~ 1e3 |U|^2 at low Mach);
// they are summed in that cancelled form, which FP32 evaluates accurately:
//   rhob = (g-1)/2 |U|^2 pb + (|U|^2/2 - e) Tb/(Cv rho) - (U.wbU)/rho
template <typename T> ADFVM_HD void primitive_vjp(const Phys<T>& ph, const T* q, const T* wb, T* qb) {
    T rho = q[0];
    T U[3] = {q[1] / rho, q[2] / rho, q[3] / rho};
    T E = q[4] / rho;
    T U2 = U[0] * U[0] + U[1] * U[1] + U[2] * U[2];
    T e = E - T(0.5) * U2;
    T gm1 = ph.gamma - T(1);
    T Tb = wb[3] * ph.invCv;                 // adjoint of e through T
    T pb = wb[4];
    // eb = Tb + pb*gm1*rho ; qb4 = eb/rho
    qb[4] += Tb / rho + pb * gm1;
    for (int i = 0; i < 3; i++) qb[1 + i] += wb[i] / rho - (Tb / rho + pb * gm1) * U[i];
    T UwU = U[0] * wb[0] + U[1] * wb[1] + U[2] * wb[2];
    qb[0] += T(0.5) * gm1 * U2 * pb + (T(0.5) * U2 - e) * Tb / rho - UwU / rho;
}

// The same at a state given by its primitive values w (e = Cv T,
// rho = p/((g-1) e)).
template <typename T> ADFVM_HD void primitive_vjp_at(const Phys<T>& ph, const T* w, const T* wb, T* qb) {
    const T gm1 = ph.gamma - T(1);
    const T e = ph.Cv * w[3];
    const T rho = w[4] / (gm1 * e);
    const T U2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
    const T Tb = wb[3] * ph.invCv;
    const T pb = wb[4];
    const T eb = Tb / rho + pb * gm1;
    qb[4] += eb;
    for (int i = 0; i < 3; i++) qb[1 + i] += wb[i] / rho - eb * w[i];
    const T UwU = w[0] * wb[0] + w[1] * wb[1] + w[2] * wb[2];
    qb[0] += T(0.5) * gm1 * U2 * pb + (T(0.5) * U2 - e) * Tb / rho - UwU / rho;
}

// conservative(w) -> q ; wb += (dq/dw)^T qb
template <typename T> ADFVM_HD void conservative_vjp(const Phys<T>& ph, const T* w, const T* qb, T* wb) {
    T gm1 = ph.gamma - T(1);
    T e = ph.Cv * w[3];
    T rho = w[4] / (e * gm1);
    T U2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
    T rhob = qb[0] + qb[4] * (e + T(0.5) * U2);
    T eb = qb[4] * rho;
    for (int i = 0; i < 3; i++) {
        rhob += qb[1 + i] * w[i];
        wb[i] += qb[1 + i] * rho + qb[4] * rho * w[i];
    }
    wb[4] += rhob / (e * gm1);
    eb += -rhob * rho / e;
    wb[3] += eb * ph.Cv;
}

// Which value each of reconstruct()'s five results is, two bits each: 0 the
// reconstructed value, 1 clamped to the cell's own value, 2 to the other
// cell's.  Kept in place of the inputs, so that these need not stay in
// registers until the reverse of the reconstruction.
template <typename T>
ADFVM_HD int reconstruct_taken(const T* wC, const T* gC, const T* wD, T lw, const T* qw) {
    int taken = 0;
    for (int i = 0; i < 5; i++) {
        const T* g = gC + 3 * i;
        T v = wC[i] + (wD[i] - wC[i]) * lw + (qw[0] * g[0] + qw[1] * g[1] + qw[2] * g[2]);
        const bool up = wC[i] < wD[i];
        const T lo = up ? wC[i] : wD[i], hi = up ? wD[i] : wC[i];
        // out = v < lo ? lo : (v > hi ? hi : v), as in reconstruct()
        if (v < lo) taken |= (up ? 1 : 2) << (2 * i);
        else if (v > hi) taken |= (up ? 2 : 1) << (2 * i);
    }
    return taken;
}

// reconstruct (one side): out = clamp(wC + (wD-wC)*lw + qw.g); the adjoint
// follows the selected value
template <typename T>
ADFVM_HD void reconstruct_vjp(T lw, const T* qw, const T* ob, int taken, T* wCb, T* gCb, T* wDb) {
    if (taken == 0) {
        for (int i = 0; i < 5; i++) {
            const T d = ob[i] * lw;
            wCb[i] += ob[i] - d;
            wDb[i] += d;
            for (int k = 0; k < 3; k++) gCb[3 * i + k] += ob[i] * qw[k];
        }
        return;
    }
    for (int i = 0; i < 5; i++) {
        const int which = (taken >> (2 * i)) & 3;
        const T b = which == 0 ? ob[i] : T(0), d = b * lw;
        wCb[i] += which == 1 ? ob[i] : b - d;
        wDb[i] += which == 2 ? ob[i] : d;
        for (int k = 0; k < 3; k++) gCb[3 * i + k] += b * qw[k];
    }
}

// One side of a Roe face from its primitive values: total enthalpy h =
// g/(g-1) p/rho + |U|^2/2 = g Cv T + |U|^2/2, R = (g-1) Cv.
template <typename T> struct RoeSide {
    T Un, iRT, rho, h, s;        // U.n, 1/(R T), density, total enthalpy, sqrt(rho)
    T c, Ue;                     // sound speed and U.n as the entropy fix compares them
};
// FP32: density p/(R T) and sound speed sqrt(g R T) by the one reciprocal.
ADFVM_HD void roe_density(const Phys<float>& ph, const float* w, RoeSide<float>& o) {
    const float RT = (ph.gamma - 1.0f) * ph.Cv * w[3];
    o.iRT = recip(RT);
    o.rho = w[4] * o.iRT;
    o.c = fsqrt(ph.gamma * RT);
    o.Ue = o.Un;
}
// Otherwise in the reference's own terms (riemann.py:31-58: c = sqrt(g p/rho),
// U.n as (rho U.n)/rho): where a side's value equals the other's up to
// rounding, as in a field of uniform temperature, the sign that rounding
// gives the difference decides the branch of the adjoint.
template <typename T> ADFVM_HD void roe_density(const Phys<T>& ph, const T* w, RoeSide<T>& o) {
    o.iRT = recip((ph.gamma - T(1)) * ph.Cv * w[3]);
    o.rho = w[4] / (ph.Cv * w[3] * (ph.gamma - T(1)));
    o.c = fsqrt(ph.gamma * w[4] / o.rho);
    o.Ue = o.rho * o.Un / o.rho;
}
template <typename T> ADFVM_HD void roe_side(const Phys<T>& ph, const T* w, const T* n, RoeSide<T>& o) {
    o.Un = w[0] * n[0] + w[1] * n[1] + w[2] * n[2];
    roe_density(ph, w, o);
    o.h = ph.gamma * ph.Cv * w[3] + T(0.5) * (w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    o.s = fsqrt(o.rho);
}

// The Roe averages, jumps and dissipation of a face (riemann.eulerRoe,
// adFVM/riemann.py:21-70).  stabilise(eps) = eps + SMALL for eps >= 0 (adpy's
// definition is not in the reference).
template <typename T> struct RoeFace {
    T idv, a, b;                 // 1/(sL + sR) and the sides' weights sL, sR over their sum
    T U[3], h, q, c, ic, Un;     // averages: velocity, enthalpy, |U|^2/2, sound speed, 1/c, normal velocity
    T drho, drhoU[3], drhoE;
    T ieps, r1, r2, r3;          // 1/eps; eigenvalues over eps
    bool f1, f2, f3;             // eigenvalues inside the entropy fix
    T l1;                        // fixed |Un|
    T m2, m3;                    // (l2 - l3)/2, (l2 + l3)/2 - l1
    T x, y;                      // pressure jump over c, -rho U.n jump
    T k6, s6, s7;                // m3 x - m2 y; s6 = k6/c; s7 = m3 y - m2 x
};
template <typename T>
ADFVM_HD void roe_face(const Phys<T>& ph, const T* wL, const RoeSide<T>& L, const T* wR, const RoeSide<T>& R,
                       const T* n, RoeFace<T>& o) {
    const T gm1 = ph.gamma - T(1);
    o.idv = recip(L.s + R.s);
    o.a = L.s * o.idv;
    o.b = R.s * o.idv;
    for (int i = 0; i < 3; i++) o.U[i] = wL[i] * o.a + wR[i] * o.b;
    o.h = L.h * o.a + R.h * o.b;
    o.q = T(0.5) * (o.U[0] * o.U[0] + o.U[1] * o.U[1] + o.U[2] * o.U[2]);
    o.c = fsqrt(gm1 * (o.h - o.q));
    o.ic = recip(o.c);
    o.Un = o.U[0] * n[0] + o.U[1] * n[1] + o.U[2] * n[2];
    o.drho = R.rho - L.rho;
    for (int i = 0; i < 3; i++) o.drhoU[i] = R.rho * wR[i] - L.rho * wL[i];
    o.drhoE = (R.h * R.rho - wR[4]) - (L.h * L.rho - wL[4]);
    const T lam1 = fabs_(o.Un), lam2 = fabs_(o.Un + o.c), lam3 = fabs_(o.Un - o.c);
    T eps = T(0.5) * fabs_(L.Ue - R.Ue);
    eps += T(0.5) * fabs_(L.c - R.c);
    eps = eps + ph.small;
    o.ieps = recip(eps);
    const T e2 = T(2) * eps;
    o.f1 = lam1 < e2; o.f2 = lam2 < e2; o.f3 = lam3 < e2;
    o.r1 = lam1 * o.ieps; o.r2 = lam2 * o.ieps; o.r3 = lam3 * o.ieps;
    o.l1 = o.f1 ? T(0.25) * lam1 * o.r1 + eps : lam1;
    const T l2 = o.f2 ? T(0.25) * lam2 * o.r2 + eps : lam2;
    const T l3 = o.f3 ? T(0.25) * lam3 * o.r3 + eps : lam3;
    o.m2 = T(0.5) * (l2 - l3);
    o.m3 = T(0.5) * (l2 + l3) - o.l1;
    o.x = gm1 * (o.q * o.drho - (o.U[0] * o.drhoU[0] + o.U[1] * o.drhoU[1] + o.U[2] * o.drhoU[2]) + o.drhoE) * o.ic;
    o.y = o.Un * o.drho - (o.drhoU[0] * n[0] + o.drhoU[1] * n[1] + o.drhoU[2] * n[2]);
    o.k6 = o.m3 * o.x - o.m2 * o.y;
    o.s6 = o.k6 * o.ic;
    o.s7 = o.m3 * o.y - o.m2 * o.x;
}

// Reverse of one side's derived values: adds the adjoints of U, T, p from
// those of Un, rho, h and c (s goes through rho).
template <typename T>
ADFVM_HD void roe_side_vjp(const Phys<T>& ph, const T* w, const T* n, const RoeSide<T>& o, T Unb, T rhob, T hb, T cb,
                           T* wb) {
    const T RiRT = (ph.gamma - T(1)) * ph.Cv * o.iRT;         // 1/T
    for (int i = 0; i < 3; i++) wb[i] += Unb * n[i] + hb * w[i];
    wb[3] += ph.gamma * ph.Cv * hb + (T(0.5) * cb * o.c - rhob * o.rho) * RiRT;
    wb[4] += rhob * o.iRT;
}

// Roe flux reverse: wLb, wRb += (dF/dw)^T Fb.  Arithmetic and registers bound
// the kernels that call it: quotients by one divisor share a reciprocal,
// h and c^2 come from T, and the reverse runs on normalised quantities, about
// half the instructions of a reverse of the forward formulas as they stand
// (interior face adjoint of a 64-cell tile in FP32: 1756 -> 996 vector
// instructions per wave, 199 -> 100 registers).
template <typename T>
ADFVM_HD void roe_flux_vjp(const Phys<T>& ph, const T* wL, const T* wR, const T* n, const T* Fb, T* wLb, T* wRb) {
    const T gm1 = ph.gamma - T(1);
    RoeSide<T> L, R;
    RoeFace<T> f;
    roe_side(ph, wL, n, L);
    roe_side(ph, wR, n, R);
    roe_face(ph, wL, L, wR, R, n, f);
    // F = (central - dissipation)/2: H the adjoint of either half
    T H[5];
    for (int i = 0; i < 5; i++) H[i] = T(0.5) * Fb[i];
    const T Hn = H[1] * n[0] + H[2] * n[1] + H[3] * n[2];
    // dissipation: l1 drho + s6, l1 drhoU + U s6 - n s7, l1 drhoE + h s6 - Un s7
    T l1b = -(H[0] * f.drho + H[1] * f.drhoU[0] + H[2] * f.drhoU[1] + H[3] * f.drhoU[2] + H[4] * f.drhoE);
    const T s6b = -(H[0] + H[1] * f.U[0] + H[2] * f.U[1] + H[3] * f.U[2] + H[4] * f.h);
    const T s7b = Hn + H[4] * f.Un;
    T drhob = -H[0] * f.l1, drhoEb = -H[4] * f.l1, hb = -H[4] * f.s6, Unb = H[4] * f.s7;
    T drhoUb[3], Ub[3];
    for (int i = 0; i < 3; i++) {
        drhoUb[i] = -H[1 + i] * f.l1;
        Ub[i] = -H[1 + i] * f.s6;
    }
    // s6 = k6 ic, k6 = m3 x - m2 y; s7 = m3 y - m2 x
    const T k6b = s6b * f.ic;
    const T m3b = k6b * f.x + s7b * f.y;
    const T m2b = -(k6b * f.y + s7b * f.x);
    const T xb = k6b * f.m3 - s7b * f.m2;
    const T yb = s7b * f.m3 - k6b * f.m2;
    // x = gm1 (q drho - U.drhoU + drhoE) ic: x's own share of the adjoint of c
    // is -xb x ic, s6's -s6b s6 ic
    T cb = -(s6b * f.s6 + xb * f.x) * f.ic;
    const T t = gm1 * xb * f.ic;
    T qb = t * f.drho;
    drhob += t * f.q;
    drhoEb += t;
    // y = Un drho - drhoU.n
    Unb += yb * f.drho;
    drhob += yb * f.Un;
    for (int i = 0; i < 3; i++) {
        Ub[i] -= t * f.drhoU[i];
        drhoUb[i] -= t * f.U[i] + yb * n[i];
    }
    // m2 = (l2 - l3)/2, m3 = (l2 + l3)/2 - l1
    l1b -= m3b;
    const T l2b = T(0.5) * (m3b + m2b), l3b = T(0.5) * (m3b - m2b);
    // entropy fix l = lam^2/(4 eps) + eps below 2 eps
    T epsb = T(0), lam1b = l1b, lam2b = l2b, lam3b = l3b;
    if (f.f1) { lam1b = T(0.5) * l1b * f.r1; epsb += l1b - l1b * (T(0.25) * f.r1 * f.r1); }
    if (f.f2) { lam2b = T(0.5) * l2b * f.r2; epsb += l2b - l2b * (T(0.25) * f.r2 * f.r2); }
    if (f.f3) { lam3b = T(0.5) * l3b * f.r3; epsb += l3b - l3b * (T(0.25) * f.r3 * f.r3); }
    const T eUn = T(0.5) * sgn(L.Ue - R.Ue) * epsb, ec = T(0.5) * sgn(L.c - R.c) * epsb;
    const T g1 = lam1b * sgn(f.Un), g2 = lam2b * sgn(f.Un + f.c), g3 = lam3b * sgn(f.Un - f.c);
    Unb += g1 + g2 + g3;
    cb += g2 - g3;
    // c^2 = gm1 (h - q), q = |U|^2/2
    const T c2b = gm1 * T(0.5) * cb * f.ic;
    hb += c2b;
    qb -= c2b;
    for (int i = 0; i < 3; i++) Ub[i] += Unb * n[i] + qb * f.U[i];
    // averages: a = sL/(sL + sR) = 1 - b
    T D = hb * (L.h - R.h);
    for (int i = 0; i < 3; i++) D += Ub[i] * (wL[i] - wR[i]);
    D = T(0.5) * D * f.idv;
    const T mL = L.rho * L.Un, mR = R.rho * R.Un;
    const T mLb = H[0] + H[1] * wL[0] + H[2] * wL[1] + H[3] * wL[2] + H[4] * L.h;
    const T mRb = H[0] + H[1] * wR[0] + H[2] * wR[1] + H[3] * wR[2] + H[4] * R.h;
    const T rhoLb = D * f.b * recip(L.s) - (drhob + drhoUb[0] * wL[0] + drhoUb[1] * wL[1] + drhoUb[2] * wL[2] +
                                            drhoEb * L.h) + mLb * L.Un;
    const T rhoRb = (drhob + drhoUb[0] * wR[0] + drhoUb[1] * wR[1] + drhoUb[2] * wR[2] + drhoEb * R.h) -
                    D * f.a * recip(R.s) + mRb * R.Un;
    for (int i = 0; i < 3; i++) {
        wLb[i] += Ub[i] * f.a - drhoUb[i] * L.rho + H[1 + i] * mL;
        wRb[i] += Ub[i] * f.b + drhoUb[i] * R.rho + H[1 + i] * mR;
    }
    wLb[4] += Hn + drhoEb;
    wRb[4] += Hn - drhoEb;
    roe_side_vjp(ph, wL, n, L, mLb * L.rho + eUn, rhoLb, hb * f.a - drhoEb * L.rho + H[4] * mL, ec, wLb);
    roe_side_vjp(ph, wR, n, R, mRb * R.rho - eUn, rhoRb, hb * f.b + drhoEb * R.rho + H[4] * mR, -ec, wRb);
}

// Lax-Friedrichs flux reverse.  Inputs used: U, p (w) and rho, rhoU, rhoE (q).
template <typename T>
ADFVM_HD void lf_flux_vjp(const Phys<T>& ph, const T* wL, const T* qL, const T* wR, const T* qR, const T* n,
                          const T* Fb, T* wLb, T* qLb, T* wRb, T* qRb) {
    const T g = ph.gamma;
    T pL = wL[4], pR = wR[4], rhoL = qL[0], rhoR = qR[0];
    T UnL = wL[0] * n[0] + wL[1] * n[1] + wL[2] * n[2];
    T UnR = wR[0] * n[0] + wR[1] * n[1] + wR[2] * n[2];
    T cL = fsqrt(g * pL / rhoL), cR = fsqrt(g * pR / rhoR);
    T aL = fabs_(UnL) + cL, aR = fabs_(UnR) + cR;
    T aF = aL > aR ? aL : aR;
    T aFb = -T(0.5) * Fb[0] * (rhoR - rhoL) - T(0.5) * Fb[4] * (qR[4] - qL[4]);
    qLb[0] += T(0.5) * Fb[0] * UnL + T(0.5) * Fb[0] * aF;
    qRb[0] += T(0.5) * Fb[0] * UnR - T(0.5) * Fb[0] * aF;
    T UnLb = T(0.5) * Fb[0] * rhoL + T(0.5) * Fb[4] * (qL[4] + pL);
    T UnRb = T(0.5) * Fb[0] * rhoR + T(0.5) * Fb[4] * (qR[4] + pR);
    for (int i = 0; i < 3; i++) {
        T b = Fb[1 + i];
        aFb += -T(0.5) * b * (qR[1 + i] - qL[1 + i]);
        UnLb += T(0.5) * b * qL[1 + i];
        UnRb += T(0.5) * b * qR[1 + i];
        qLb[1 + i] += T(0.5) * b * UnL + T(0.5) * b * aF;
        qRb[1 + i] += T(0.5) * b * UnR - T(0.5) * b * aF;
        wLb[4] += T(0.5) * b * n[i];
        wRb[4] += T(0.5) * b * n[i];
    }
    wLb[4] += T(0.5) * Fb[4] * UnL;
    wRb[4] += T(0.5) * Fb[4] * UnR;
    qLb[4] += T(0.5) * Fb[4] * UnL + T(0.5) * Fb[4] * aF;
    qRb[4] += T(0.5) * Fb[4] * UnR - T(0.5) * Fb[4] * aF;
    T aLb, aRb;
    if (aL > aR) { aLb = aFb; aRb = 0; }
    else if (aR > aL) { aLb = 0; aRb = aFb; }
    else { aLb = T(0.5) * aFb; aRb = T(0.5) * aFb; }
    UnLb += aLb * sgn(UnL);
    UnRb += aRb * sgn(UnR);
    T cLb = aLb, cRb = aRb;
    wLb[4] += cLb * g / (T(2) * cL * rhoL);
    qLb[0] += -cLb * g * pL / (T(2) * cL * rhoL * rhoL);
    wRb[4] += cRb * g / (T(2) * cR * rhoR);
    qRb[0] += -cRb * g * pR / (T(2) * cR * rhoR * rhoR);
    for (int i = 0; i < 3; i++) { wLb[i] += UnLb * n[i]; wRb[i] += UnRb * n[i]; }
}

// viscous_flux reverse: adjoint of (TL, TR, UL, UR, TF, UF, gTF0, gUF0).
template <typename T>
ADFVM_HD void viscous_flux_vjp(const Phys<T>& ph, T TL, T TR, const T* UL, const T* UR, T TF, const T* UF,
                               const T* gTF0, const T* gUF0, const T* n, T delta, const T* D, const T* Fb,
                               T* TLb, T* TRb, T* ULb, T* URb, T* TFb, T* UFb, T* gTF0b, T* gUF0b) {
    const T mu = viscosity(ph, TF);
    const T kappa = mu * (ph.Cp / ph.Pr);
    const T id = recip(delta);
    T gU[9];
    for (int i = 0; i < 3; i++) {
        T c = (UR[i] - UL[i]) * id - (gUF0[3 * i] * D[0] + gUF0[3 * i + 1] * D[1] + gUF0[3 * i + 2] * D[2]);
        for (int k = 0; k < 3; k++) gU[3 * i + k] = gUF0[3 * i + k] + c * D[k];
    }
    const T tr = T(2.0 / 3.0) * (gU[0] + gU[4] + gU[8]);
    T t2[3];                                     // sigma = mu t2
    for (int i = 0; i < 3; i++)
        t2[i] = (gU[3 * i] + gU[i]) * n[0] + (gU[3 * i + 1] + gU[3 + i]) * n[1] + (gU[3 * i + 2] + gU[6 + i]) * n[2] -
                tr * n[i];
    // reverse: F[1+i] -= sigma_i, F[4] -= q + sigma.UF
    T sb[3];                                     // adjoint of sigma
    for (int i = 0; i < 3; i++) {
        sb[i] = -Fb[1 + i] - Fb[4] * UF[i];
        UFb[i] -= Fb[4] * (mu * t2[i]);
    }
    const T qFb = -Fb[4];
    if (ph.muModel != 0) {                       // the viscosity's own adjoint, into TF
        T cT = (TR - TL) * id - (gTF0[0] * D[0] + gTF0[1] * D[1] + gTF0[2] * D[2]);
        T gTn = T(0);
        for (int k = 0; k < 3; k++) gTn += (gTF0[k] + cT * D[k]) * n[k];
        const T mub = sb[0] * t2[0] + sb[1] * t2[1] + sb[2] * t2[2] + qFb * gTn * (ph.Cp / ph.Pr);
        *TFb += mub * viscosity_dT(ph, TF);
    }
    // t2 = (gU + gU^T) n - 2/3 tr(gU) n: a symmetric adjoint B of gU, of
    // which the part along D goes to the difference across the face
    for (int i = 0; i < 3; i++) sb[i] *= mu;
    const T trb = -T(2.0 / 3.0) * (sb[0] * n[0] + sb[1] * n[1] + sb[2] * n[2]);
    T B[9];
    for (int a = 0; a < 3; a++)
        for (int b = a; b < 3; b++) B[3 * a + b] = B[3 * b + a] = sb[a] * n[b] + sb[b] * n[a] + (a == b ? trb : T(0));
    for (int i = 0; i < 3; i++) {
        const T along = B[3 * i] * D[0] + B[3 * i + 1] * D[1] + B[3 * i + 2] * D[2];
        for (int k = 0; k < 3; k++) gUF0b[3 * i + k] += B[3 * i + k] - along * D[k];
        URb[i] += along * id;
        ULb[i] -= along * id;
    }
    const T z = qFb * kappa;
    const T along = z * (n[0] * D[0] + n[1] * D[1] + n[2] * D[2]);
    for (int k = 0; k < 3; k++) gTF0b[k] += z * n[k] - along * D[k];
    *TRb += along * id;
    *TLb -= along * id;
}

template <typename T>
ADFVM_HD void riemann_vjp(const Phys<T>& ph, int which, const T* wL, const T* wR, const T* n, const T* Fb, T* wLb,
                          T* wRb) {
    if (which == 0) {
        roe_flux_vjp(ph, wL, wR, n, Fb, wLb, wRb);
    } else {
        T qL[5], qR[5], qLb[5] = {0, 0, 0, 0, 0}, qRb[5] = {0, 0, 0, 0, 0};
        conservative(ph, wL, qL);
        conservative(ph, wR, qR);
        lf_flux_vjp(ph, wL, qL, wR, qR, n, Fb, wLb, qLb, wRb, qRb);
        conservative_vjp(ph, wL, qLb, wLb);
        conservative_vjp(ph, wR, qRb, wRb);
    }
}

// Reverse of face_flux with respect to the F output (the lam output's
// adjoint is zero in the adjoint solver, apps/adjoint.py:268: dtca = 0).
// Adds into wPb[5], gPb[15], wNb[5], gNb[15] (gNb may alias gPb).
template <typename T>
ADFVM_HD void face_flux_vjp(const Phys<T>& ph, int kind, const T* wP, const T* gP, const T* wN, const T* gN,
                            const FaceGeo<T>& f, const T* Fb, T* wPb, T* gPb, T* wNb, T* gNb) {
    T TF, UF[3], gTF[3], gUF[9];
    T wLF[5], wRF[5];
    int takenL = 0, takenR = 0;
    if (kind == FACE_BOUNDARY) {
        TF = wN[3];
        for (int i = 0; i < 3; i++) UF[i] = wN[i];
        for (int k = 0; k < 3; k++) gTF[k] = gN[9 + k];
        for (int k = 0; k < 9; k++) gUF[k] = gN[k];
    } else {
        reconstruct(wP, gP, wN, f.lw0, f.qw0, wLF, ph.limit);
        if (ph.limit) takenL = reconstruct_taken(wP, gP, wN, f.lw0, f.qw0);
        if (kind == FACE_CHARACTERISTIC) {
            for (int i = 0; i < 5; i++) wRF[i] = wN[i];
            TF = wN[3];
            for (int i = 0; i < 3; i++) UF[i] = wN[i];
            for (int k = 0; k < 3; k++) gTF[k] = gN[9 + k];
            for (int k = 0; k < 9; k++) gUF[k] = gN[k];
        } else {
            reconstruct(wN, gN, wP, f.lw1, f.qw1, wRF, ph.limit);
            if (ph.limit) takenR = reconstruct_taken(wN, gN, wP, f.lw1, f.qw1);
            for (int i = 0; i < 3; i++) UF[i] = T(0.5) * (wLF[i] + wRF[i]);
            TF = T(0.5) * (wLF[3] + wRF[3]);
            for (int k = 0; k < 3; k++) gTF[k] = T(0.5) * (gP[9 + k] + gN[9 + k]);
            for (int k = 0; k < 9; k++) gUF[k] = T(0.5) * (gP[k] + gN[k]);
        }
    }
    // viscous part
    T TFb = 0, UFb[3] = {0, 0, 0}, gTFb[3] = {0, 0, 0}, gUFb[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    viscous_flux_vjp(ph, wP[3], wN[3], wP, wN, TF, UF, gTF, gUF, f.n, f.delta, f.D, Fb,
                     &wPb[3], &wNb[3], wPb, wNb, &TFb, UFb, gTFb, gUFb);
    if (kind == FACE_BOUNDARY) {
        wNb[3] += TFb;
        for (int i = 0; i < 3; i++) wNb[i] += UFb[i];
        for (int k = 0; k < 3; k++) gNb[9 + k] += gTFb[k];
        for (int k = 0; k < 9; k++) gNb[k] += gUFb[k];
        // physical flux of the ghost state
        T qR[5];
        conservative(ph, wN, qR);
        T Un = wN[0] * f.n[0] + wN[1] * f.n[1] + wN[2] * f.n[2];
        T Unb = Fb[0] * qR[0] + Fb[4] * (qR[4] + wN[4]);
        T qRb[5] = {Fb[0] * Un, 0, 0, 0, Fb[4] * Un};
        T pb = Fb[4] * Un;
        for (int i = 0; i < 3; i++) {
            Unb += Fb[1 + i] * qR[1 + i];
            qRb[1 + i] = Fb[1 + i] * Un;
            pb += Fb[1 + i] * f.n[i];
        }
        wNb[4] += pb;
        for (int i = 0; i < 3; i++) wNb[i] += Unb * f.n[i];
        conservative_vjp(ph, wN, qRb, wNb);
        return;
    }
    T wLFb[5] = {0, 0, 0, 0, 0}, wRFb[5] = {0, 0, 0, 0, 0};
    if (kind == FACE_CHARACTERISTIC) {
        wNb[3] += TFb;
        for (int i = 0; i < 3; i++) wNb[i] += UFb[i];
        for (int k = 0; k < 3; k++) gNb[9 + k] += gTFb[k];
        for (int k = 0; k < 9; k++) gNb[k] += gUFb[k];
        riemann_vjp(ph, ph.boundaryRiemann, wLF, wRF, f.n, Fb, wLFb, wRFb);
    } else {
        for (int i = 0; i < 3; i++) { wLFb[i] += T(0.5) * UFb[i]; wRFb[i] += T(0.5) * UFb[i]; }
        wLFb[3] += T(0.5) * TFb; wRFb[3] += T(0.5) * TFb;
        for (int k = 0; k < 3; k++) { gPb[9 + k] += T(0.5) * gTFb[k]; gNb[9 + k] += T(0.5) * gTFb[k]; }
        for (int k = 0; k < 9; k++) { gPb[k] += T(0.5) * gUFb[k]; gNb[k] += T(0.5) * gUFb[k]; }
        riemann_vjp(ph, ph.riemann, wLF, wRF, f.n, Fb, wLFb, wRFb);
    }
    reconstruct_vjp(f.lw0, f.qw0, wLFb, takenL, wPb, gPb, wNb);
    if (kind == FACE_CHARACTERISTIC) {
        for (int i = 0; i < 5; i++) wNb[i] += wRFb[i];
    } else {
        reconstruct_vjp(f.lw1, f.qw1, wRFb, takenR, wNb, gNb, wPb);
    }
}

}  // namespace adfvm
