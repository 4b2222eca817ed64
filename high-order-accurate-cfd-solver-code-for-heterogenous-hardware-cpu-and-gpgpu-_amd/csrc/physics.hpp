// Device physics shared by the drop-in kernels and the structured sweeps.
// T is the arithmetic type of fluxes / reconstruction / viscous terms (double for
// the plain form, float for the mixed form). gamma = 1.4 as the reference's
// literals 1.4 / 0.4 / 0.2 (Weno.cl:2292-2295, U_Q.cl:73).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace cfdx {
namespace dev {

template <typename T> __device__ __forceinline__ T sqrt_(T x);
template <> __device__ __forceinline__ double sqrt_<double>(double x) { return __builtin_sqrt(x); }
template <> __device__ __forceinline__ float sqrt_<float>(float x) { return __builtin_amdgcn_sqrtf(x); }

template <typename T> __device__ __forceinline__ T fabs_(T x) { return x < T(0) ? -x : x; }

// Reciprocal and quotient: exact IEEE division in double (the plain form's parity bar), the
// hardware reciprocal / square root (about 1 ulp) in float for the mixed form.
template <typename T> __device__ __forceinline__ T inv_(T x);
template <> __device__ __forceinline__ double inv_<double>(double x) { return 1.0 / x; }
template <> __device__ __forceinline__ float inv_<float>(float x) { return __builtin_amdgcn_rcpf(x); }
template <typename T> __device__ __forceinline__ T div_(T a, T b);
template <> __device__ __forceinline__ double div_<double>(double a, double b) { return a / b; }
template <> __device__ __forceinline__ float div_<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// Reciprocal, square root and reciprocal square root of a strictly positive normal operand (a
// density, a squared norm, a sum of positive terms): the hardware estimate (relative error below
// 6e-8 on gfx950) refined in double by one Newton-Raphson step (reciprocal: relative error below
// 2.2e-15, 0.7 ulp on average) or one Goldschmidt step and one residual correction (square root:
// within 0.5 ulp, correctly rounded for 99.98 % of operands; its reciprocal within 1.5 ulp); the
// hardware instructions in float (within 1 ulp). Measured on 2^20 log-uniform operands in
// [1e-300, 1e300]. Not for 0, inf, NaN or operands whose result is subnormal (no range scaling).
template <typename T> __device__ __forceinline__ T pinv_(T x);
template <> __device__ __forceinline__ double pinv_<double>(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, e, r);
}
template <> __device__ __forceinline__ float pinv_<float>(float x) { return __builtin_amdgcn_rcpf(x); }

// s = sqrt(x) and h = 1 / (2 sqrt(x)) by one Goldschmidt step on the rsq estimate, then one
// residual correction of s
__device__ __forceinline__ double gold_sqrt(double x, double &h)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    h = 0.5 * y;
    const double r = __builtin_fma(-g, h, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    const double d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
}
template <typename T> __device__ __forceinline__ T psqrt_(T x);
template <> __device__ __forceinline__ double psqrt_<double>(double x) { double h; return gold_sqrt(x, h); }
template <> __device__ __forceinline__ float psqrt_<float>(float x) { return __builtin_amdgcn_sqrtf(x); }
// 1 / sqrt(x)
template <typename T> __device__ __forceinline__ T prsq_(T x);
template <> __device__ __forceinline__ double prsq_<double>(double x)
{
    double h;
    const double s = gold_sqrt(x, h);
    const double r = 2.0 * h;
    return __builtin_fma(r, __builtin_fma(-s, r, 1.0), r);   // one Newton step on 1 / s
}
template <> __device__ __forceinline__ float prsq_<float>(float x) { return __builtin_amdgcn_rsqf(x); }

// Keeps the computation of x where it stands in the instruction stream: the scheduler otherwise moves
// loads up and uses down until a long kernel holds far more values than it needs (the FP64 face
// sweep: 168 registers, 128 and no spill with the pins of characteristic_states).
template <typename T>
__device__ __forceinline__ void pin_(T &x)
{
    if constexpr (std::is_arithmetic<T>::value) asm volatile("" : "+v"(x));
}

// s = sqrt(x) and r = 1 / sqrt(x) together: in double from one hardware estimate (h of the square
// root's step is half of r, refined once), in float the hardware square root and reciprocal
template <typename T> __device__ __forceinline__ T psqrt_half_(T x, T &h);
template <> __device__ __forceinline__ double psqrt_half_<double>(double x, double &h) { return gold_sqrt(x, h); }
template <typename T>
__device__ __forceinline__ void psqrt_rsq_(T x, T &s, T &r)
{
    if constexpr (std::is_same<T, float>::value) {
        s = psqrt_(x);
        r = pinv_(s);
    } else {
        T h;
        s = psqrt_half_(x, h);
        r = T(2) * h;
        r = r + r * (T(1) - s * r);
    }
}

// Conserved state Q = (rho, rho u, rho v, rho w, p/0.4 + rho |u|^2 / 2) of primitives (U_Q.cl:118-122).
// No fused multiply-adds, so every kernel that builds the RK base det * Q from the same primitives
// (the last RK stage, set_flow) gets the same bits: a state saved and restored continues exactly.
template <typename T>
__device__ __forceinline__ void prim_to_q(T rho, T u, T v, T w, T p, T (&q)[5])
{
#pragma clang fp contract(off)
    const T ke = T(0.5) * rho * (u * u + v * v + w * w);
    q[0] = rho;
    q[1] = rho * u;
    q[2] = rho * v;
    q[3] = rho * w;
    q[4] = p * T(2.5) + ke;   // p / (gamma - 1)
}

// Total enthalpy H = (E + p) / rho of primitives (U_Q.cl:73-74).
template <typename T>
__device__ __forceinline__ T enthalpy(T rho, T u, T v, T w, T p)
{
    return (p * T(3.5) + T(0.5) * rho * (u * u + v * v + w * w)) * pinv_(rho);   // (p/0.4 + ke + p) / rho
}

// The reciprocals of two positive operands: in double by one reciprocal of their product (the
// hardware estimate issues at a quarter of the rate of a multiplication).
template <typename T>
__device__ __forceinline__ void pinv2_(T x, T y, T &ix, T &iy)
{
    if constexpr (std::is_same<T, float>::value) {
        ix = pinv_(x);
        iy = pinv_(y);
    } else {
        const T r = pinv_(x * y);
        ix = r * y;
        iy = r * x;
    }
}

// Roe-average inputs (u, v, w, H) of a node from its conserved state Q and r = 1 / Q0: the face kernels
// hold the Q of the stencil points already, so the two centre nodes need no primitive loads.
template <typename T>
__device__ __forceinline__ void q_roe_inputs(const T (&q)[5], T r, T &u, T &v, T &w, T &h)
{
    u = q[1] * r;
    v = q[2] * r;
    w = q[3] * r;
    h = (T(1.4) * q[4] - T(0.2) * (q[1] * u + q[2] * v + q[3] * w)) * r;   // (E + p) / rho, p = 0.4 (E - rho |u|^2 / 2)
}

// Roe average of the face between states a and b (U_Q.cl:60-109): (u, v, w, h, rho), and 1 / rho.
template <typename T>
__device__ __forceinline__ T roe_average(T ra, T ua, T va, T wa, T ha, T rb, T ub, T vb, T wb, T hb, T (&r)[5])
{
    const T sa = psqrt_(ra), sb = psqrt_(rb);
    T is, irho;
    r[4] = sb * sa;
    pinv2_(sa + sb, r[4], is, irho);
    r[0] = (sb * ub + sa * ua) * is;
    r[1] = (sb * vb + sa * va) * is;
    r[2] = (sb * wb + sa * wa) * is;
    r[3] = (sb * hb + sa * ha) * is;
    return irho;
}

// Contravariant, det-scaled inviscid node flux along metric row m (Viscous.cl:560-611):
// D * (mx F1 + my E1 + mz G1) with F1, E1, G1 the Cartesian Euler fluxes; Ep = E + p.
template <typename T>
__device__ __forceinline__ void node_flux_e(T rho, T u, T v, T w, T p, T Ep, T mx, T my, T mz, T D, T (&f)[5])
{
    const T V = mx * u + my * v + mz * w;
    const T rV = rho * V;
    f[0] = D * rV;
    f[1] = D * (rV * u + mx * p);
    f[2] = D * (rV * v + my * p);
    f[3] = D * (rV * w + mz * p);
    f[4] = D * (Ep * V);
}
template <typename T>
__device__ __forceinline__ void node_flux(T rho, T u, T v, T w, T p, T mx, T my, T mz, T D, T (&f)[5])
{
    const T V = mx * u + my * v + mz * w;
    const T Ep = p * T(3.5) + T(0.5) * rho * (u * u + v * v + w * w);   // E + p
    const T rV = rho * V;
    f[0] = D * rV;
    f[1] = D * (rV * u + mx * p);
    f[2] = D * (rV * v + my * p);
    f[3] = D * (rV * w + mz * p);
    f[4] = D * (Ep * V);
}

// WCNS-E5 interpolation of one characteristic field W[0..5] (offsets -2..+3 from the left node) to the
// face between W[2] and W[3], Weno.cl:1056-1279, from its first differences d_m = W[m+1] - W[m]:
//   candidates (15/8, -5/4, 3/8), (3/8, 3/4, -1/8), (-1/8, 3/4, 3/8),
//   Jiang-Shu indicators, w_k = d_k / (eps + IS_k)^2, value = sum w_k q_k / sum w_k.
// pos = right-biased (d = 1/16, 5/8, 5/16), neg = left-biased (d = 5/16, 5/8, 1/16), both as eight
// times the value less the mean (W[2] + W[3]) / 2: every candidate less that mean is a combination
// of two neighbouring second differences s_k = d_{k+1} - d_k,
//   8 (pos q0 - mean) = 3 s3 - 4 s2   8 (pos q1, neg q0) = -s2   8 (pos q2, neg q1) = -s1
//   8 (neg q2 - mean) = 3 s0 - 4 s1,
// so no value of W itself is needed, the middle candidates cost nothing, and nothing large cancels.
template <typename T>
__device__ __forceinline__ void wcns_pair(const T (&d)[5], T eps4, T &pos, T &neg)
{
    // the indicators are formed four times larger, 4 IS = 13/3 s^2 + t^2, from the second
    // differences (each 13/3 s_k^2 shared by two indicators) and the first-derivative terms t; with
    // eps also taken four times larger (eps4) every (eps + IS)^2 carries the same factor 16, which
    // cancels in the weights
    const T c13 = T(13.0 / 3.0);
    const T s0 = d[1] - d[0], s1 = d[2] - d[1], s2 = d[3] - d[2], s3 = d[4] - d[3];
    // eps + 13/3 s_k^2, each shared by two indicators
    const T S0 = c13 * s0 * s0 + eps4, S1 = c13 * s1 * s1 + eps4, S2 = c13 * s2 * s2 + eps4, S3 = c13 * s3 * s3 + eps4;
    const T t0 = d[4] - T(3) * d[3];   // 3 W3 - 4 W4 + W5
    const T t1 = d[2] + d[3];          // W4 - W2
    const T t2 = T(3) * d[2] - d[1];   // W1 - 4 W2 + 3 W3
    const T u0 = d[3] - T(3) * d[2];   // 3 W2 - 4 W3 + W4
    const T u1 = d[1] + d[2];          // W3 - W1
    const T u2 = T(3) * d[1] - d[0];   // W0 - 4 W1 + 3 W2
    T a0 = S3 + t0 * t0, a1 = S2 + t1 * t1, a2 = S1 + t2 * t2;   // eps + IS, four times larger
    T b0 = S2 + u0 * u0, b1 = S1 + u1 * u1, b2 = S0 + u2 * u2;
    // w_k proportional to d_k * prod_{m != k} (eps + IS_m)^2, so each side needs one division; the
    // linear weights are taken 16 times larger (pos 1, 10, 5; neg 5, 10, 1): the factor cancels in
    // the quotients
    T np_, dp_, nn_, dn_;
    {
        a0 *= a0; a1 *= a1; a2 *= a2;
        const T e = a1 * a2, w = T(5) * a0, a22 = T(2) * a2;
        np_ = e * (T(3) * s3 - T(4) * s2) - w * (a22 * s2 + a1 * s1);
        dp_ = e + w * (a22 + a1);
    }
    {
        b0 *= b0; b1 *= b1; b2 *= b2;
        const T e = b0 * b1, w = T(5) * b2, b02 = T(2) * b0;
        nn_ = e * (T(3) * s0 - T(4) * s1) - w * (b1 * s2 + b02 * s1);
        dn_ = e + w * (b1 + b02);
    }
    if constexpr (!std::is_same<T, float>::value) {
        // one reciprocal serves both sides
        const T r = pinv_(dp_ * dn_);
        pos = np_ * (dn_ * r);
        neg = nn_ * (dp_ * r);
    } else {
        // float: the weights of smooth data are ~eps^4 ~ 1e-28, within the float range, but the
        // product of the two sides' sums (~eps^8) is not: one hardware reciprocal per side
        pos = np_ * inv_(dp_);
        neg = nn_ * inv_(dn_);
    }
}

// Characteristic reconstruction of the two interface states of one face
// (Weno.cl:336-455 eigenvectors and projection, :1056-2187 WCNS, :2188-2287 back projection).
//   q(m, c): conserved Q at offsets -2..+3 from the left node (m = 0..5)
//   roe = (u, v, w, h, rho) of the face, irho = 1 / rho; (kx, ky, kz) = the face metric row over its
//   length
//   qp / qn: right-biased / left-biased conserved states (not det-scaled)
// The five first differences of the stencil states are projected, not the six states: the
// reconstruction needs nothing else, and the interface states are the mean of the two centre
// states plus the back projection of the corrections.
template <typename T, typename GetQ>
__device__ __forceinline__ void characteristic_states(const GetQ &q, const T (&roe)[5], T irho, T kx, T ky, T kz, T eps,
                                                      T (&qp)[5], T (&qn)[5])
{
    const T u = roe[0], v = roe[1], w = roe[2], h = roe[3], rho = roe[4];
    const T q2 = u * u + v * v + w * w;
    T a, ia;
    psqrt_rsq_(T(0.4) * (h - T(0.5) * q2), a, ia);
    const T theta = kx * u + ky * v + kz * w;
    const T phi = T(0.2) * q2;
    const T iaa = ia * ia;
    const T s2 = T(0.70710678118654752440);             // 1/sqrt(2)
    const T beta = irho * ia * s2;                      // 1 / (sqrt2 rho a)
    const T g4aa = T(0.4) * iaa;
    const T one_m = T(1) - phi * iaa;
    const T cv = kz * v - ky * w, cw = kx * w - kz * u, cu = ky * u - kx * v;  // u x k

    // Projection L dq of the 5 stencil differences, written through L's structure: rows 0-2 are
    // k_c E + (1/rho) (q_mom x k - (u x k) q0)_c with E = (1 - phi/a^2) q0 + (0.4/a^2) m and
    // m = u.q_mom - q4; rows 3 and 4 are beta (phi q0 - 0.4 m) -/+ beta a (theta q0 - k.q_mom).
    const T ikx = irho * kx, iky = irho * ky, ikz = irho * kz;
    const T icu = irho * cu, icv = irho * cv, icw = irho * cw;
    const T bphi = beta * phi, b04 = beta * T(0.4), ba = irho * s2;
    T W[5][5];
    T lo[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) lo[c] = q(0, c);
#pragma unroll
    for (int m = 0; m < 5; ++m) {
        T d[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            const T hi = q(m + 1, c);
            d[c] = hi - lo[c];
            lo[c] = hi;
            pin_(lo[c]);
        }
        const T mm = u * d[1] - d[4] + v * d[2] + w * d[3];
        const T B = theta * d[0] - kx * d[1] - ky * d[2] - kz * d[3];
        const T E = one_m * d[0] + g4aa * mm;
        W[0][m] = kx * E + (ikz * d[2] - iky * d[3] - icv * d[0]);
        W[1][m] = ky * E + (ikx * d[3] - ikz * d[1] - icw * d[0]);
        W[2][m] = kz * E + (iky * d[1] - ikx * d[2] - icu * d[0]);
        const T bA = bphi * d[0] - b04 * mm;
        W[3][m] = bA - ba * B;
        W[4][m] = bA + ba * B;
#pragma unroll
        for (int c = 0; c < 5; ++c) pin_(W[c][m]);
    }
    const T eps4 = T(4) * eps;
    T xp[5], xn[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        wcns_pair(W[c], eps4, xp[c], xn[c]);
        pin_(xp[c]);
        pin_(xn[c]);
    }
    // Back projection R x of the corrections through R's structure (x carries the factor 8 of
    // wcns_pair): with x' = (x0, x1, x2), X = k.x', P = alpha (x3 + x4) and M = alpha a (x3 - x4),
    // alpha = rho / (sqrt2 a): Q0 = X + P, Q_mom = u Q0 + k M + rho (k x x'),
    // Q4 = (phi/0.4) X + H P + theta M + rho (u x k).x'
    const T k8x = T(0.125) * kx, k8y = T(0.125) * ky, k8z = T(0.125) * kz, r8 = T(0.125) * rho;
    const T rkx = r8 * kx, rky = r8 * ky, rkz = r8 * kz;
    const T rcu = r8 * cu, rcv = r8 * cv, rcw = r8 * cw;
    const T aa = r8 * s2, alpha = aa * ia;
    const T phi_g = phi * T(2.5);
    const T hh = phi_g + a * a * T(2.5);
    T qm[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) qm[c] = T(0.5) * (q(2, c) + q(3, c));
    auto back = [&](const T (&x)[5], T (&Q)[5]) {
        const T X = k8x * x[0] + k8y * x[1] + k8z * x[2];
        const T P = alpha * (x[3] + x[4]);
        const T M = aa * (x[3] - x[4]);
        const T d0 = X + P;
        Q[0] = qm[0] + d0;
        Q[1] = qm[1] + u * d0 + kx * M + rky * x[2] - rkz * x[1];
        Q[2] = qm[2] + v * d0 + ky * M + rkz * x[0] - rkx * x[2];
        Q[3] = qm[3] + w * d0 + kz * M + rkx * x[1] - rky * x[0];
        Q[4] = qm[4] + phi_g * X + hh * P + theta * M + rcv * x[0] + rcw * x[1] + rcu * x[2];
    };
    back(xp, qp);
    back(xn, qn);
}

// n . (F, E, G)(Q) and lambda_5 = n.u + c of one interface state along the unit face normal n
// (Weno.cl:2291-2507 fluxes, :2511-2581 eigenvalues, :2585-2655 contravariant form: the face's
// |k| det_f scales the LLF sum once).
// r = 1 / Q0.
template <typename T>
__device__ __forceinline__ void face_state_flux(const T (&Q)[5], T r, T kx, T ky, T kz, T (&c)[5], T &lam)
{
    const T ke = (Q[1] * Q[1] + Q[2] * Q[2] + Q[3] * Q[3]) * r;
    const T P = T(0.4) * (Q[4] - T(0.5) * ke);
    const T Un = (kx * Q[1] + ky * Q[2] + kz * Q[3]) * r;
    c[0] = Q[0] * Un;
    c[1] = Q[1] * Un + kx * P;
    c[2] = Q[2] * Un + ky * P;
    c[3] = Q[3] * Un + kz * P;
    c[4] = (T(1.4) * Q[4] - T(0.2) * ke) * Un;
    lam = Un + psqrt_(T(1.4) * P * r);
}

// LLF face flux with alpha = max(|lambda_5|) of the two interface states (Weno.cl:2859-2947):
// (kx, ky, kz) the unit face normal, dk = det_f |k| of the face metric row k.
template <typename T, typename GetQ>
__device__ __forceinline__ void face_llf(const GetQ &q, const T (&roe)[5], T irho, T kx, T ky, T kz, T dk, T eps,
                                         T (&llf)[5])
{
    T qp[5], qn[5];
    characteristic_states(q, roe, irho, kx, ky, kz, eps, qp, qn);
    T cp[5], cn[5], lp, ln, rp, rn;
    pinv2_(qp[0], qn[0], rp, rn);
    face_state_flux(qp, rp, kx, ky, kz, cp, lp);
    face_state_flux(qn, rn, kx, ky, kz, cn, ln);
    const T al = fabs_(lp) >= fabs_(ln) ? fabs_(lp) : fabs_(ln);
    const T hd = T(0.5) * dk;
#pragma unroll
    for (int c = 0; c < 5; ++c) llf[c] = hd * (cp[c] + cn[c] - al * (qp[c] - qn[c]));
}

// Explicit midpoint correction - delta2 F / 24 + 7 delta4 F / 5760 of one component from the node
// fluxes at offsets -2..+3 (Weno.cl:2951-3058).
template <typename T>
__device__ __forceinline__ T midpoint_correction(T f0, T f1, T f2, T f3, T f4, T f5)
{
    // d2 = (-5 f0 + 39 f1 - 34 f2 - 34 f3 + 39 f4 - 5 f5) / 48,
    // d4 = (f0 - 3 f1 + 2 f2 + 2 f3 - 3 f4 + f5) / 2; -d2 / 24 + 7 d4 / 5760 collects to
    // (57 (f0 + f5) - 411 (f1 + f4) + 354 (f2 + f3)) / 11520
    return T(57.0 / 11520.0) * (f0 + f5) - T(411.0 / 11520.0) * (f1 + f4) + T(354.0 / 11520.0) * (f2 + f3);
}

// LLF face flux of a face metric row (k0, k1, k2) as stored by the reference; detf the face det.
template <typename T, typename GetQ>
__device__ __forceinline__ void face_flux(const GetQ &q, const T (&roe)[5], T k0, T k1, T k2, T detf, T eps, T (&llf)[5])
{
    const T kn = sqrt_(k0 * k0 + k1 * k1 + k2 * k2), ik = inv_(kn);
    face_llf(q, roe, pinv_(roe[4]), k0 * ik, k1 * ik, k2 * ik, detf * kn, eps, llf);
}

// Viscous + SGS node fluxes (Viscous.cl:439-631, its mixed-time-scale model or the Smagorinsky
// option) of one node.
//   dU[c][d] = dU_c / d(zeta, eta, xi)_d of the det-scaled state U (Viscous.cl:285-435)
//   U[5]     = U at the node; u, v, w = the velocity at the node (Viscous.cl:146-154 reads it from
//              FLOW; the block kernel passes U_1..3 / U_0 of the same stage vector away from the
//              sides of a block)
//   m[9]     = node metrics zeta_x..xi_z; D = det
//   KS[3]    = MTS scale-similarity terms KS_x, KS_y, KS_z (Viscous.cl:493-495)
// Writes the contravariant det-scaled viscous fluxes fvis[0..2] = Fv, Ev, Gv and returns mu.
struct ViscParams {
    double mach, reyl, pr, free_t, c_mts, c_t;
    // derived on the host (uniform per launch)
    double inv_reyl;     // 1 / Re
    double kheat;        // 1.4 / (Pr Re)
    double suth;         // 110.4 / T_inf
    double suth1;        // 1 + 110.4 / T_inf
    double tfac;         // 1.4 M^2 0.4
    double kQ;           // -1 / (1.4 0.4 M^2)
    double inv_ct;       // 1 / C_T
    double cs2;          // Smagorinsky: C_s^2
    int sgs;             // 0: mixed time scale (the reference); 1: Smagorinsky
    double kheat_t;      // Smagorinsky heat flux: 1.4 / Pr
};

inline ViscParams make_visc_params(double mach, double reyl, double pr, double free_t, double c_mts, double c_t,
                                   int sgs = 0, double c_s = 0.0)
{
    ViscParams v{mach, reyl, pr, free_t, c_mts, c_t, 0, 0, 0, 0, 0, 0, 0, c_s * c_s, sgs, 1.4 / pr};
    v.inv_reyl = 1.0 / reyl;
    v.kheat = 1.4 / (pr * reyl);
    v.suth = 110.4 / free_t;
    v.suth1 = 1.0 + v.suth;
    v.tfac = 1.4 * mach * mach * 0.4;
    v.kQ = -(1.0 / (1.4 * 0.4 * mach * mach));
    v.inv_ct = 1.0 / c_t;
    return v;
}

// x^(-1/3) of a positive normal operand (a det): the float estimate 2^(-log2(x) / 3) of the
// hardware log2 and exp2, refined by one Newton step y <- y + y (1 - x y^3) / 3 in float and two
// more in double (within 1 ulp on operands in [1e-36, 1e36]; float form within 1 ulp too).
template <typename T> __device__ __forceinline__ T prcbrt_(T x);
template <> __device__ __forceinline__ float prcbrt_<float>(float x)
{
    const float y = __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(x) * (-1.0f / 3.0f));
    return __builtin_fmaf(y * (1.0f / 3.0f), __builtin_fmaf(-x * y, y * y, 1.0f), y);
}
template <> __device__ __forceinline__ double prcbrt_<double>(double x)
{
    double y = (double)prcbrt_<float>((float)x);
    y = __builtin_fma(y * (1.0 / 3.0), __builtin_fma(-x * y, y * y, 1.0), y);
    return __builtin_fma(y * (1.0 / 3.0), __builtin_fma(-x * y, y * y, 1.0), y);
}

// The smallest denominator the positive-operand reciprocal and the square root are given in the
// eddy viscosity: below it |S| or the scale-similarity magnitude is taken as zero.
template <typename T> __device__ __forceinline__ T tiny_();
template <> __device__ __forceinline__ double tiny_<double>() { return 1e-280; }
template <> __device__ __forceinline__ float tiny_<float>() { return 1e-35f; }

// U_c / U_0 of a node: velocity (0..2) and E / rho (3), with 1 / U_0.
template <typename T>
struct NodeRatios {
    T iU0, r[4];
};
template <typename T>
__device__ __forceinline__ NodeRatios<T> node_ratios(const T (&U)[5])
{
    NodeRatios<T> n;
    n.iU0 = pinv_(U[0]);
#pragma unroll
    for (int c = 0; c < 4; ++c) n.r[c] = U[1 + c] * n.iU0;
    return n;
}

// Adds the part of direction d to the Cartesian gradients G[0..3][x, y, z] of u, v, w and the internal
// energy: X_x = X_zeta zeta_x + X_eta eta_x + X_xi xi_x, one direction at a time (dU = dU_c / d(zeta,
// eta, xi)_d, (mx, my, mz) the metric row of d), so that a kernel holds twelve gradients instead of
// fifteen differences and nine metrics (k_visc in FP64: 167 VGPRs with all directions held).
template <typename T>
__device__ __forceinline__ void add_gradient(const T (&dU)[5], const NodeRatios<T> &n, T mx, T my, T mz, T (&G)[4][3])
{
    T g[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) g[c] = n.iU0 * (dU[1 + c] - n.r[c] * dU[0]);
    g[3] = g[3] - n.r[0] * g[0] - n.r[1] * g[1] - n.r[2] * g[2];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        G[c][0] += g[c] * mx;
        G[c][1] += g[c] * my;
        G[c][2] += g[c] * mz;
    }
}

// Viscous and SGS node fluxes from the Cartesian gradients. (u, v, w): the velocity in the work
// terms; sk: the magnitudes of the scale-similarity terms (square roots of KS_x, KS_y, KS_z).
template <typename T>
__device__ __forceinline__ T viscous_fluxes(const T (&G)[4][3], const T (&U)[5], const NodeRatios<T> &n, T u, T v, T w,
                                            const T (&m)[9], T D, const T (&sk)[3], const ViscParams &vp, T (&fvis)[3][5])
{
    const T ux = G[0][0], uy = G[0][1], uz = G[0][2];
    const T vx = G[1][0], vy = G[1][1], vz = G[1][2];
    const T wx = G[2][0], wy = G[2][1], wz = G[2][2];
    const T ex = G[3][0], ey = G[3][1], ez = G[3][2];
    const T C_MTS = T(vp.c_mts);

    // Viscous.cl:455-458: T = gamma M^2 (gamma-1) e, Sutherland mu with S = 110.4
    const T d_temp = T(vp.tfac) * (n.r[3] - T(0.5) * (n.r[0] * n.r[0] + n.r[1] * n.r[1] + n.r[2] * n.r[2]));
    const T st = psqrt_(d_temp);
    const T mu = (st * d_temp) * (T(vp.suth1) * pinv_(d_temp + T(vp.suth)));
    // Viscous.cl:461-476 heat flux and Stokes stresses
    const T kq = -(mu * T(vp.kheat));
    const T qx = kq * ex, qy = kq * ey, qz = kq * ez;
    const T mr = mu * T(vp.inv_reyl);
    const T sxy2 = uy + vx, syz2 = vz + wy, sxz2 = wx + uz;
    const T dv = T(2.0 / 3.0) * (ux + vy + wz);
    const T txx = mr * (T(2) * ux - dv);
    const T tyy = mr * (T(2) * vy - dv);
    const T tzz = mr * (T(2) * wz - dv);
    const T txy = mr * sxy2, txz = mr * sxz2, tyz = mr * syz2;
    // Viscous.cl:490-558 mixed-time-scale eddy viscosity, one per direction: with S_xy = sxy2 / 2,
    // |S|^2 = 2 (S_xy^2 + S_yz^2 + S_xz^2 + 2/3 (S_xx^2 + S_yy^2 + S_zz^2))
    const T off = sxy2 * sxy2 + syz2 * syz2 + sxz2 * sxz2, diag = ux * ux + vy * vy + wz * wz;
    const T DEL = prcbrt_(D);
    T eddy[3];
    if (vp.sgs == 1) {
        // Smagorinsky (no reference counterpart): nu_t = (C_s Delta)^2 |S| with Delta = det^(1/3) and
        // |S| = sqrt(2 S_ij S_ij), the same in every direction. The SGS stress below is
        // -2 U0 eddy S_ij with U0 = det rho, so eddy = nu_t / det = C_s^2 |S| det^(-1/3) = C_s^2 |S| DEL.
        const T s2 = T(2) * diag + off;
        const T e = T(vp.cs2) * DEL * (s2 > tiny_<T>() ? psqrt_(s2) : T(0));
        eddy[0] = e; eddy[1] = e; eddy[2] = e;
    } else {
        const T s2 = T(0.5) * off + T(4.0 / 3.0) * diag;
        const T dm = DEL * (s2 > tiny_<T>() ? psqrt_(s2) : T(0)) * T(vp.inv_ct);
        const T cd = C_MTS * DEL;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            // C_MTS / (1 + R / C_T) * DEL * sk with R = DEL |S| / sk, written with one division (sk = 0
            // gives R = inf and a zero eddy viscosity either way; |S| = 0 gives C_MTS DEL sk)
            const T den = sk[d] + dm;
            eddy[d] = den > tiny_<T>() ? (cd * sk[d] * sk[d]) * pinv_(den) : cd * sk[d];
        }
    }
    // SGS stresses scale with U0 = det * rho (Viscous.cl:529-535)
    const T mU = -U[0];
    const T e0 = mU * eddy[0], e1 = mU * eddy[1], e2 = mU * eddy[2];   // -2 U0 eddy S_ij = e (2 S_ij)
    const T Sxy = e0 * sxy2, Syz = e1 * syz2, Sxz = e2 * sxz2;
    const T Sxx = e0 * (T(2) * ux), Syy = e1 * (T(2) * vy), Szz = e2 * (T(2) * wz);
    T Hx, Hy, Hz;
    if (vp.sgs == 1) {
        // Smagorinsky: the molecular forms with rho nu_t (= U0 eddy) for mu / Re: heat flux
        // -1.4 rho nu_t / Pr grad e, and the work of the SGS stresses
        const T kS = T(vp.kheat_t) * e0;
        Hx = kS * ex + (u * Sxx + v * Sxy + w * Sxz);
        Hy = kS * ey + (u * Sxy + v * Syy + w * Syz);
        Hz = kS * ez + (u * Sxz + v * Syz + w * Szz);
    } else {
        // H = Q + DEL and D = 0.4 Q (Viscous.cl:549-557): 1.4 Q + (row sum) times the velocity component
        const T kQ = T(1.4) * T(vp.kQ);
        Hx = kQ * eddy[0] * ex + (Sxx + Sxy + Sxz) * u;
        Hy = kQ * eddy[1] * ey + (Sxy + Syy + Syz) * v;
        Hz = kQ * eddy[2] * ez + (Sxz + Syz + Szz) * w;
    }
    // Viscous.cl:576-595 Cartesian viscous fluxes
    const T tF[5] = {T(0), Sxx - txx, Sxy - txy, Sxz - txz, (-u * txx - v * txy - w * txz) + qx + Hx};
    const T tE[5] = {T(0), Sxy - txy, Syy - tyy, Syz - tyz, (-u * txy - v * tyy - w * tyz) + qy + Hy};
    const T tG[5] = {T(0), Sxz - txz, Syz - tyz, Szz - tzz, (-u * txz - v * tyz - w * tzz) + qz + Hz};
    // Viscous.cl:615-631 contravariant and det-scaled
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T a = D * m[3 * d], b = D * m[3 * d + 1], c3 = D * m[3 * d + 2];
        fvis[d][0] = T(0);
#pragma unroll
        for (int c = 1; c < 5; ++c) fvis[d][c] = a * tF[c] + b * tE[c] + c3 * tG[c];
    }
    return mu;
}

// One-direction derivative of Viscous.cl:285-435 (weno_form = false) or Weno.cl:2732-2856
// (weno_form = true) selected by the loc codes; f[0..6] at offsets -3..+3. Branches are
// taken in source order, a later match overwriting an earlier one; with no match the
// reference leaves the value undefined and this returns 0.
template <typename T>
__device__ __forceinline__ T loc_derivative(const T (&f)[7], int LI, int LM2, int LM1, int LP1, int LP2, bool weno_form)
{
    T d = T(0);
    if (LI > 0 && LI <= 52 && LP1 == 100) d = T(1.0 / 6.0) * (T(11) * f[3] - T(18) * f[2] + T(9) * f[1] - T(2) * f[0]);
    if (LI > 0 && LI <= 52 && LM1 == 100) d = T(1.0 / 6.0) * (T(-11) * f[3] + T(18) * f[4] - T(9) * f[5] + T(2) * f[6]);
    if (LI == 0 && LP1 > 0 && LP1 <= 52 && LP2 == 100) d = T(1.0 / 6.0) * (T(2) * f[4] + T(3) * f[3] - T(6) * f[2] + f[1]);
    if (LI == 0 && LM1 > 0 && (weno_form ? LM1 <= 52 : true) && LM2 == 100)
        d = T(1.0 / 6.0) * (T(-2) * f[2] - T(3) * f[3] + T(6) * f[4] - f[5]);
    if (LM2 != 100 && LM1 != 100 && LP2 != 100 && LP1 != 100 && (LI == 0 || (!weno_form && LI > 0)))
        d = T(1.0 / 12.0) * (T(8) * (f[4] - f[2]) - (f[5] - f[1]));
    return d;
}

}  // namespace dev
}  // namespace cfdx
