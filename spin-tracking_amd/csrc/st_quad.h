// st_quad.h -- spin kernels with four lanes per particle, for ensembles that do
// not fill the chip.
//
// What bounds a small ensemble is one lane's chain of trial steps: with one
// wave per SIMD nothing else can issue, and a lone wave issues one instruction
// in 4.3 cycles, whether or not it needs the result before it.  A
// one-lane trial is about 1,000 instructions, the segment set-up that some
// lane of a wave needs on most trips included (fast: 2.1 us on neutrons,
// 3.2 us on He-3, whose segments are short; exact 5.4 and 7.1 us; 1.6 us per
// fast trial when three waves share the SIMD).  Here a particle takes a quad
// of lanes, one spin component each (lane 3 repeats lane 0):
//   * the stage sums, two thirds of the trial's operations, run once per quad
//     instead of once per component;
//   * the components meet in the cross products and the error norm, through
//     quad-permute moves (no LDS, no waits);
//   * the tableau stays in registers for the whole launch (the one-lane kernel
//     needs them for its state; a lane of a quad holds a third of that state);
//   * the next segment record is loaded while the current one is integrated;
//   * the pulse's stage cosines are split over the quad.
// Per trial 0.86 us on neutrons and 1.3 us on He-3 (1,000 particles, fast),
// 2.4 and 3.1 us exact.  RK45: 0.51 us fast, of one lane 1.15 (and 1.40 before
// its sums were chains of FMAs); exact 1.41 and 2.92 us.
// Every value is formed by the one-lane trial's operations in its order, so
// accept/reject decisions and results are those of the one-lane kernels bit
// for bit; a quad's four lanes always agree on the control flow.
#pragma once

#include "st_adjoint.h"

namespace st {

// ---------------------------------------------------------------------------
// quad moves
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ double quad_perm(double v) {
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// the value of component c+1 / c+2 (cyclic) in the lane of component c
__device__ __forceinline__ double q_next1(double v) { return quad_perm<1 | 2 << 2 | 0 << 4 | 1 << 6>(v); }
__device__ __forceinline__ double q_next2(double v) { return quad_perm<2 | 0 << 2 | 1 << 4 | 2 << 6>(v); }
// the value of component I (lane I) in all four lanes
template <int I>
__device__ __forceinline__ double q_all(double v) {
    return quad_perm<I | I << 2 | I << 4 | I << 6>(v);
}
__device__ __forceinline__ d3 q_vec(double v) { return d3{q_all<0>(v), q_all<1>(v), q_all<2>(v)}; }

// lane I's vector in all four lanes
template <int I>
__device__ __forceinline__ d3 q_vec3(const d3& v) { return d3{q_all<I>(v.x), q_all<I>(v.y), q_all<I>(v.z)}; }

// v[c], c = 0..2
__device__ __forceinline__ double q_pick(const d3& v, uint32_t c) { return c == 0 ? v.x : (c == 1 ? v.y : v.z); }

// List position of a quad's first particle: a wave holds ppw of them (slot =
// quad % ppw), and the grid covers the list.  (Taken from a work queue, two
// requests a wave, each cost 11 ns on the queue's one address, as the work
// counters did; st_state.h.  The loops still look for a next particle, a grid
// further on: with that branch gone the compiler keeps 30 registers more and
// spills inside the trial, 16,384 He-3 2.54 and 3.36 ms.)
__device__ __forceinline__ uint32_t quad_index(uint32_t ppw) {
    return (blockIdx.x * 4u + (threadIdx.x >> 6)) * ppw + ((__lane_id() >> 2) & (ppw - 1u));
}

// The launch's arguments, one by-value kernel parameter, read through an
// opaque copy of the kernel-argument pointer: the scalar loads stay at their
// use.  Hoisted out of the lane loop, the arguments of the record and queue
// handling would take the scalar registers the trial needs for the tableau
// (60 spilled, most of them read back inside the trial).
struct QuadArgs {
    SimParams P;
    DevState D;
    PipeArgs A;
    uint32_t ppw;
};
template <typename ARGS>
__device__ __forceinline__ const ARGS& kernel_args() {
    typedef const __attribute__((address_space(4))) ARGS* cptr;
    cptr p = (cptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const ARGS*)p;
}

// ---------------------------------------------------------------------------
// the tableau in registers
// ---------------------------------------------------------------------------
#define ST_DOP_RESIDENT(X)                                                                                          \
    X(a81) X(a84) X(a85) X(a86) X(a87) X(a91) X(a94) X(a95) X(a96) X(a97) X(a98) X(a101) X(a104) X(a105) X(a106) X(a107)   \
    X(a108) X(a109) X(a111) X(a114) X(a115) X(a116) X(a117) X(a118) X(a119) X(a1110) X(a121) X(a124) X(a125)        \
    X(a126) X(a127) X(a128) X(a129) X(a1210) X(a1211) X(er1) X(er6) X(er7) X(er8) X(er9) X(er10) X(er11) X(er12)
#define ST_DOP_LITERAL(X) X(a21) X(a31) X(a32) X(a41) X(a43) X(a51) X(a53) X(a54)
#define ST_DOP_SPIN_RESIDENT(X) X(a61) X(a64) X(a65) X(a71) X(a74) X(a75) X(a76)
#define ST_DOP_SCALAR(X)                                                                                            \
    X(c2) X(c3) X(c4) X(c5) X(c6) X(c7) X(c8) X(c9) X(c10) X(c11) X(b1) X(b6) X(b7) X(b8) X(b9) X(b10) X(b11)       \
    X(b12) X(bhh1) X(bhh2) X(bhh3)
// The stage coefficients in vector registers and the nodes and weights in
// scalar ones (a product takes one scalar-register operand).  The empty
// statements make each value opaque once per launch: the compiler would
// otherwise rebuild it from literals at each use, two scalar moves that cost
// as much as the product when the wave is alone on its SIMD.  (The first
// stages' eight stay literals, fifteen in the adjoint, which carries the
// quadrature: 256 registers hold no more.)
struct DopTab {
#define X(n) double n;
    ST_DOP_RESIDENT(X)
    ST_DOP_SPIN_RESIDENT(X)
    ST_DOP_SCALAR(X)
    ST_DOP_LITERAL(X)
#undef X
};
template <bool ADJ>
__device__ __forceinline__ void dop_tab_load(DopTab& T) {
#define X(n) T.n = dop::n; asm volatile("" : "+v"(T.n));
    ST_DOP_RESIDENT(X)
#undef X
#define X(n) T.n = dop::n; if constexpr (!ADJ) asm volatile("" : "+v"(T.n));
    ST_DOP_SPIN_RESIDENT(X)
#undef X
#define X(n) T.n = dop::n; asm volatile("" : "+s"(T.n));
    ST_DOP_SCALAR(X)
#undef X
#define X(n) T.n = dop::n;
    ST_DOP_LITERAL(X)
#undef X
}

// ---------------------------------------------------------------------------
// the fast trial, one component per lane
// ---------------------------------------------------------------------------
// Field polynomial of components c+1 (a) and c+2 (b): what the cross product
// of component c needs.
struct QPoly {
    double a0, a1, a2, b0, b1, b2;
};
// Pulse of a particle: w, whether there is one at all, and its amplitude
// (gamma*a) on the lane's components a and b (adjoint: negated).
struct QPulse {
    double pw, ma, mb;
    bool on;
};

// Loop state of a segment: DopState with the lane's component of k1.
struct QDop {
    double x, xf, facold, k1, posneg;   // (posneg: exact variant)
    int32_t reject, last;
    uint32_t left;                      // trials left before nmax is exceeded
};

// What the fast DOP853 trial reads of the caller's parameters.  A scalar load
// costs a wave alone on its SIMD some 50 cycles, nine of them a fifth of a
// trial's time, and all scalar registers are taken: here each lane of a quad
// holds one of four values, and a use is a quad move of two instructions
// (64 neutrons x 0.5 s: 1.26 and 1.11 ms).  (The exact trial has no vector
// registers left for it: spilling two, it was 3 % slower.)
struct DopCtl {
    double a;         // lanes 0..3: atol, rtol, safe, hmin
    double b;         // lanes 0..2: fac1, fac2, hmax
    bool fixed;       // fixed step size
    bool plain;       // no power needed (dop_factors)
};
__device__ __forceinline__ void dop_ctl_load(DopCtl& C, const SimParams& P) {
    const uint32_t l = __lane_id() & 3u;
    C.a = l == 0 ? P.atol : l == 1 ? P.rtol : l == 2 ? P.safe : P.hmin;
    C.b = l == 0 ? P.fac1 : l == 1 ? P.fac2 : P.hmax;
    asm volatile("" : "+v"(C.a), "+v"(C.b));
    C.fixed = P.fixed != 0;
    C.plain = !P.pow_beta_on && P.expo1 == 0.125;
}
// QDop::left of a new segment: the trials before nmax is exceeded
__device__ __forceinline__ uint32_t dop_trials(const SimParams& P) { return min(P.nmax, 0xfffffffeu) + 1u; }

// y x w of the lane's component, w given by its components a and b
__device__ __forceinline__ double q_cross(double y, double wa, double wb) {
    const double ya = q_next1(y), yb = q_next2(y);
    return __builtin_fma(ya, wb, -(yb * wa));
}
__device__ __forceinline__ void q_field(double tau, const QPoly& q, double& wa, double& wb) {
#pragma clang fp contract(fast)
    wa = q.a0 + tau * (q.a1 + tau * q.a2);
    wb = q.b0 + tau * (q.b1 + tau * q.b2);
}

// Quadrature moments of the lane's component and the segment's end time
// (adjoint only; AdjQuad in st_integrators.h).
struct QQuad {
    double n0, n1, n2, t_end;
};

// dop_trial_fast_t (st_integrators.h) on a quad.  About 250 vector
// instructions and 70 quad moves without a pulse, 0.80 us alone on a SIMD.
template <bool ADJ, bool PULSE>
__device__ __forceinline__ int q_trial_fast(const SimParams& P, const DopCtl& C, const DopTab& T, QDop& D, double& y, double& h,
                                            double seg_t0, const QPoly& q, const QPulse& pl,
                                            uint32_t& nacc, uint32_t& nrej, QQuad* Q) {
#pragma clang fp contract(fast)
    if (D.left == 0) return -1;
    D.left--;
    if (D.x + 1.01 * h - D.xf > 0.0) {
        h = D.xf - D.x;
        D.last = 1;
    }
    const double hmin = q_all<3>(C.a);
    if (h < hmin && D.last != 1) h = hmin;
    const double x = D.x;
    const double tx = x - seg_t0;
    QPoly hq = q;
    if constexpr (!PULSE) hq = QPoly{h * q.a0, h * q.a1, h * q.a2, h * q.b0, h * q.b1, h * q.b2};
    // The pulse at the eleven stage offsets: lane l of the quad takes offsets
    // l, l + 4, l + 8 of the list, and each stage reads its lane's.
    double hp0 = 0.0, hp1 = 0.0, hp2 = 0.0;
    if constexpr (PULSE) {
        if (pl.on) {
            double pS, pC;
            phase_sincos(pl.pw * (ADJ ? (Q->t_end - x) : x), pS, pC);
            auto pcos = [&](double cc) -> double {
                double a = pl.pw * (cc * h), sn, cs;
                int halvings = 0;
                while (fabs(a) > 0.5 && halvings < 1100) {
                    a *= 0.5;
                    ++halvings;
                }
                small_sincos(a, sn, cs);
                for (; halvings > 0; --halvings) {
                    const double s2 = 2.0 * sn * cs;
                    cs = 1.0 - 2.0 * sn * sn;
                    sn = s2;
                }
                return __builtin_fma(pC, cs, ADJ ? pS * sn : -(pS * sn));
            };
            const uint32_t l = __lane_id() & 3u;
            hp0 = pcos(l == 0 ? T.c2 : l == 1 ? T.c3 : l == 2 ? T.c4 : T.c5);
            hp1 = pcos(l == 0 ? T.c6 : l == 1 ? T.c7 : l == 2 ? T.c8 : T.c9);
            hp2 = pcos(l == 0 ? T.c10 : l == 1 ? T.c11 : 1.0);
        }
    }
    auto stage = [&](double tau, double Y, double cosv) -> double {
        double wa, wb;
        q_field(tau, hq, wa, wb);
        if constexpr (PULSE) {
            wa = h * __builtin_fma(pl.ma, cosv, wa);
            wb = h * __builtin_fma(pl.mb, cosv, wb);
        }
        return q_cross(Y, wa, wb);
    };
#define QK(C, LANE, HP) stage(__builtin_fma(T.C, h, tx), yy, PULSE ? q_all<LANE>(HP) : 0.0)
#define QF(S, A, K) S = __builtin_fma(T.A, K, S)
    double q0 = 0.0, q1 = 0.0, q2 = 0.0;
    auto quad = [&](double b, double si, double Y) {
        if constexpr (ADJ) {
            const double w1 = b * si, w2 = w1 * si;
            q0 = q0 + b * Y;
            q1 = q1 + w1 * Y;
            q2 = q2 + w2 * Y;
        }
    };
    const double K1 = h * D.k1;
    quad(T.b1, tx, y);
    double yy = __builtin_fma(T.a21, K1, y);
    const double K2 = QK(c2, 0, hp0);
    yy = y;
    QF(yy, a31, K1); QF(yy, a32, K2);
    const double K3 = QK(c3, 1, hp0);
    yy = y;
    QF(yy, a41, K1); QF(yy, a43, K3);
    const double K4 = QK(c4, 2, hp0);
    yy = y;
    QF(yy, a51, K1); QF(yy, a53, K3); QF(yy, a54, K4);
    const double K5 = QK(c5, 3, hp0);
    yy = y;
    QF(yy, a61, K1); QF(yy, a64, K4); QF(yy, a65, K5);
    quad(T.b6, __builtin_fma(T.c6, h, tx), yy);
    const double K6 = QK(c6, 0, hp1);
    yy = y;
    QF(yy, a71, K1); QF(yy, a74, K4); QF(yy, a75, K5); QF(yy, a76, K6);
    quad(T.b7, __builtin_fma(T.c7, h, tx), yy);
    const double K7 = QK(c7, 1, hp1);
    yy = y;
    QF(yy, a81, K1); QF(yy, a84, K4); QF(yy, a85, K5); QF(yy, a86, K6); QF(yy, a87, K7);
    quad(T.b8, __builtin_fma(T.c8, h, tx), yy);
    const double K8 = QK(c8, 2, hp1);
    yy = y;
    QF(yy, a91, K1); QF(yy, a94, K4); QF(yy, a95, K5); QF(yy, a96, K6); QF(yy, a97, K7); QF(yy, a98, K8);
    quad(T.b9, __builtin_fma(T.c9, h, tx), yy);
    const double K9 = QK(c9, 3, hp1);
    yy = y;
    QF(yy, a101, K1); QF(yy, a104, K4); QF(yy, a105, K5); QF(yy, a106, K6); QF(yy, a107, K7); QF(yy, a108, K8);
    QF(yy, a109, K9);
    quad(T.b10, __builtin_fma(T.c10, h, tx), yy);
    const double K10 = QK(c10, 0, hp2);
    yy = y;
    QF(yy, a111, K1); QF(yy, a114, K4); QF(yy, a115, K5); QF(yy, a116, K6); QF(yy, a117, K7); QF(yy, a118, K8);
    QF(yy, a119, K9); QF(yy, a1110, K10);
    quad(T.b11, __builtin_fma(T.c11, h, tx), yy);
    const double K11 = QK(c11, 1, hp2);
    yy = y;
    QF(yy, a121, K1); QF(yy, a124, K4); QF(yy, a125, K5); QF(yy, a126, K6); QF(yy, a127, K7); QF(yy, a128, K8);
    QF(yy, a129, K9); QF(yy, a1210, K10); QF(yy, a1211, K11);
    quad(T.b12, tx + h, yy);
    const double c12 = PULSE ? q_all<2>(hp2) : 0.0;
    const double K12 = stage(tx + h, yy, c12);
    double bs = T.b1 * K1;
    QF(bs, b6, K6); QF(bs, b7, K7); QF(bs, b8, K8); QF(bs, b9, K9); QF(bs, b10, K10); QF(bs, b11, K11); QF(bs, b12, K12);
    double er = T.er1 * K1;
    QF(er, er6, K6); QF(er, er7, K7); QF(er, er8, K8); QF(er, er9, K9); QF(er, er10, K10); QF(er, er11, K11);
    QF(er, er12, K12);
#undef QK
#undef QF
    const double xph = x + h;
    const double y1 = y + bs;
    double e = __builtin_fma(-T.bhh1, K1, bs);
    // the derivative at the new point (used when the trial is accepted),
    // formed while the error norm's chain waits
    double na, nb;
    q_field(tx + h, q, na, nb);
    if constexpr (PULSE) {
        na = __builtin_fma(pl.ma, c12, na);
        nb = __builtin_fma(pl.mb, c12, nb);
    }
    const double is = fast_rcp(q_all<0>(C.a) + q_all<1>(C.a) * __builtin_fmax(fabs(y), fabs(y1)));
    e = __builtin_fma(-T.bhh2, K9, e);
    e = __builtin_fma(-T.bhh3, K12, e);
    const double k1n = q_cross(y1, na, nb);
    const d3 v2 = q_vec(e * is), v1 = q_vec(er * is);
    const double err2 = __builtin_fma(v2.z, v2.z, __builtin_fma(v2.y, v2.y, v2.x * v2.x));
    const double e1 = __builtin_fma(v1.z, v1.z, __builtin_fma(v1.y, v1.y, v1.x * v1.x));
    const double deno = e1 + 0.01 * err2;
    const double err = (deno <= 0.0) ? 0.0 : e1 * fast_rsq(3.0 * deno);
    double grow, shrink;
    if (C.plain) {   // dop_factors without a power
        double inv = __builtin_inf();
        if (err > 0.0) inv = fast_sqrt(fast_sqrt(fast_rsq(err)));   // err^(-1/8)
        shrink = __builtin_fmax(q_all<0>(C.b), q_all<2>(C.a) * inv);
        grow = __builtin_fmin(q_all<1>(C.b), shrink);
    } else {
        dop_factors(P, err, D.facold, grow, shrink);
        if (err <= 1.0 || C.fixed) D.facold = max_d(err, 1.0E-4);
    }
    const bool ok = err <= 1.0 || C.fixed, done = ok && D.last;
    nacc += ok;
    nrej += !ok;
    if constexpr (ADJ) {
        if (ok) {
            Q->n0 = Q->n0 + h * q0;
            Q->n1 = Q->n1 + h * q1;
            Q->n2 = Q->n2 + h * q2;
        }
    }
    D.k1 = ok ? k1n : D.k1;
    y = ok ? y1 : y;
    D.x = ok ? xph : D.x;
    double hnew = h * (ok ? grow : shrink);
    const double hmax = q_all<2>(C.b);
    hnew = ok && fabs(hnew) > hmax ? hmax : hnew;
    hnew = ok && D.reject ? min_d(fabs(hnew), fabs(h)) : hnew;
    h = done || C.fixed ? h : hnew;
    D.reject = ok ? (done ? D.reject : 0) : 1;
    D.last = ok ? D.last : 0;
    return done;
}

// ---------------------------------------------------------------------------
// the exact trial, one component per lane
// ---------------------------------------------------------------------------
// What omega_exact reads for one component, and the segment's start state of
// that component.  hg and gg: half the gravity and the gravity along the
// component (0 across it, where (0*d)*d and 0*d are the +0 the one-lane form
// adds).
struct QExact {
    double p0, v0, hg, gg;
    double G0, G1, G2, B0, Ea, Eb, gamma;
    double pa, pw;
    int32_t axis;        // the pulse's axis; -1: none on this particle
    bool mine;           // it is the lane's component
};
__device__ __forceinline__ void q_exact_load(QExact& X, const SimParams& P, const Phys& F, uint32_t c) {
    const uint32_t a = c == 2 ? 0u : c + 1, b = c == 0 ? 2u : c - 1;
    X.G0 = F.G[3 * c]; X.G1 = F.G[3 * c + 1]; X.G2 = F.G[3 * c + 2];
    X.B0 = (&F.B0x)[c];
    X.Ea = (&F.Ex)[a];
    X.Eb = (&F.Ex)[b];
    X.gamma = F.gamma;
    X.pa = F.pa;
    X.pw = F.pw;
    X.axis = F.pulse_on ? F.pulse_axis : -1;
    X.mine = X.axis == (int32_t)c;
    X.hg = P.gravity && c == 1 ? HALF_G : 0.0;
    X.gg = P.gravity && c == 1 ? G_CONST : 0.0;
}
// the pulse at time t (whole field hook, its one nonzero component)
__device__ __forceinline__ double q_pulse_exact(const QExact& X, double t) {
    double pl[3] = {0.0, 0.0, 0.0};
    st_field_pulse(t, X.pa, X.pw, X.axis, pl);
    return X.axis == 0 ? pl[0] : (X.axis == 1 ? pl[1] : pl[2]);
}
// Bloch's y x omega at time t, component c (rhs_exact, st_device.h); pulse:
// the pulse's value at t.  The gradient is the default hook's, written out:
// a handle with other hooks never comes here (fields_by_component, st_device.h).
__device__ __forceinline__ double q_rhs_exact(const QExact& X, bool gravity, double t, double t0, double y, double pulse) {
    const double d = t - t0;
    double p = X.p0 + X.v0 * d, v = X.v0;
    if (gravity) {
        p = p + (X.hg * d) * d;
        v = v + X.gg * d;
    }
    const d3 r = q_vec(p);
    const double g = r.x * X.G0 + r.y * X.G1 + r.z * X.G2;
    const double cr = q_next1(v) * X.Eb - q_next2(v) * X.Ea;
    const double B = (((X.mine ? pulse : 0.0) + X.B0) + cr * IC2) + g;
    const double w = B * X.gamma;
    return q_next1(y) * q_next2(w) - q_next2(y) * q_next1(w);
}
// dop_trial_exact (st_integrators.h) on a quad.  The pulse's cosines are
// split over the quad as in q_trial_fast.
template <bool PULSE>
__device__ __forceinline__ int q_trial_exact(const SimParams& P, const DopTab& T, QDop& D, double& y, double& h,
                                             double t0, const QExact& X, uint32_t& nacc, uint32_t& nrej) {
    if (D.left == 0) return -1;
    D.left--;
    if ((D.x + 1.01 * h - D.xf) * D.posneg > 0.0) {
        h = D.xf - D.x;
        D.last = 1;
    }
    if (h < P.hmin && D.last != 1) h = P.hmin;
    const double x = D.x, xph = x + h;
    const bool gravity = P.gravity;
    double hp0 = 0.0, hp1 = 0.0, hp2 = 0.0;
    if constexpr (PULSE) {
        if (X.axis >= 0) {
            const uint32_t l = __lane_id() & 3u;
            hp0 = q_pulse_exact(X, x + (l == 0 ? T.c2 : l == 1 ? T.c3 : l == 2 ? T.c4 : T.c5) * h);
            hp1 = q_pulse_exact(X, x + (l == 0 ? T.c6 : l == 1 ? T.c7 : l == 2 ? T.c8 : T.c9) * h);
            hp2 = q_pulse_exact(X, l == 0 ? x + T.c10 * h : l == 1 ? x + T.c11 * h : xph);
        }
    }
#define QX(TT, LANE, HP) q_rhs_exact(X, gravity, (TT), t0, yy, PULSE ? q_all<LANE>(HP) : 0.0)
    const double k1 = D.k1;
    double yy = y + k1 * (h * T.a21);
    double k2 = QX(x + T.c2 * h, 0, hp0);
    ST_CODE_ALIGN(k2);
    yy = y + h * (T.a31 * k1 + T.a32 * k2);
    double k3 = QX(x + T.c3 * h, 1, hp0);
    ST_CODE_ALIGN(k3);
    yy = y + h * (T.a41 * k1 + T.a43 * k3);
    double k4 = QX(x + T.c4 * h, 2, hp0);
    ST_CODE_ALIGN(k4);
    yy = y + h * (T.a51 * k1 + T.a53 * k3 + T.a54 * k4);
    double k5 = QX(x + T.c5 * h, 3, hp0);
    ST_CODE_ALIGN(k5);
    yy = y + h * (T.a61 * k1 + T.a64 * k4 + T.a65 * k5);
    double k6 = QX(x + T.c6 * h, 0, hp1);
    ST_CODE_ALIGN(k6);
    yy = y + h * (T.a71 * k1 + T.a74 * k4 + T.a75 * k5 + T.a76 * k6);
    double k7 = QX(x + T.c7 * h, 1, hp1);
    ST_CODE_ALIGN(k7);
    yy = y + h * (T.a81 * k1 + T.a84 * k4 + T.a85 * k5 + T.a86 * k6 + T.a87 * k7);
    double k8 = QX(x + T.c8 * h, 2, hp1);
    ST_CODE_ALIGN(k8);
    yy = y + h * (T.a91 * k1 + T.a94 * k4 + T.a95 * k5 + T.a96 * k6 + T.a97 * k7 + T.a98 * k8);
    double k9 = QX(x + T.c9 * h, 3, hp1);
    ST_CODE_ALIGN(k9);
    yy = y + h * (T.a101 * k1 + T.a104 * k4 + T.a105 * k5 + T.a106 * k6 + T.a107 * k7 + T.a108 * k8 + T.a109 * k9);
    double k10 = QX(x + T.c10 * h, 0, hp2);
    ST_CODE_ALIGN(k10);
    yy = y + h * (T.a111 * k1 + T.a114 * k4 + T.a115 * k5 + T.a116 * k6 + T.a117 * k7 + T.a118 * k8 + T.a119 * k9 + T.a1110 * k10);
    double k11 = QX(x + T.c11 * h, 1, hp2);
    ST_CODE_ALIGN(k11);
    yy = y + h * (T.a121 * k1 + T.a124 * k4 + T.a125 * k5 + T.a126 * k6 + T.a127 * k7 + T.a128 * k8 + T.a129 * k9 + T.a1210 * k10 + T.a1211 * k11);
    double k12 = QX(xph, 2, hp2);
    ST_CODE_ALIGN(k12);
#undef QX
    const double b = T.b1 * k1 + T.b6 * k6 + T.b7 * k7 + T.b8 * k8 + T.b9 * k9 + T.b10 * k10 + T.b11 * k11 + T.b12 * k12;
    const double y1 = y + h * b;
    const double sk = P.atol + P.rtol * max_d(fabs(y), fabs(y1));
    d3 e = q_vec((b - T.bhh1 * k1 - T.bhh2 * k9 - T.bhh3 * k12) / sk);
    const double err2 = 0.0 + (e.x * e.x + e.y * e.y + e.z * e.z);
    e = q_vec((T.er1 * k1 + T.er6 * k6 + T.er7 * k7 + T.er8 * k8 + T.er9 * k9 + T.er10 * k10 + T.er11 * k11 + T.er12 * k12) / sk);
    double err = 0.0 + (e.x * e.x + e.y * e.y + e.z * e.z);
    double deno = err + 0.01 * err2;
    if (deno <= 0.0) deno = 1.0;
    err = fabs(h) * err * sqrt(1.0 / (deno * 3.0));
    const double fac11 = pow(err, P.expo1);
    double fac = P.pow_beta_on ? fac11 / pow(D.facold, P.beta) : fac11 / 1.0;
    fac = max_d(P.facc2, min_d(P.facc1, fac / P.safe));
    double hnew = h / fac;
    if (err <= 1.0 || P.fixed) {
        D.facold = max_d(err, 1.0E-4);
        nacc++;
        D.k1 = q_rhs_exact(X, gravity, xph, t0, y1, PULSE ? q_all<2>(hp2) : 0.0);
        y = y1;
        D.x = xph;
        if (D.last) return 1;
        if (fabs(hnew) > P.hmax) hnew = D.posneg * P.hmax;
        if (D.reject) hnew = D.posneg * min_d(fabs(hnew), fabs(h));
        D.reject = 0;
    } else {
        nrej++;
        hnew = h / min_d(P.facc1, fac11 / P.safe);
        D.reject = 1;
        D.last = 0;
    }
    if (!P.fixed) h = hnew;
    return 0;
}

// ---------------------------------------------------------------------------
// RK45 (integratorType 1), one component per lane
// ---------------------------------------------------------------------------
#define ST_RK_RESIDENT(X)                                                                                            \
    X(A2) X(A3) X(A4) X(A6) X(B21) X(B31) X(B32) X(B41) X(B42) X(B43) X(B51) X(B52) X(B53) X(B54) X(B61) X(B62) X(B63) \
    X(B64) X(B65) X(CH1) X(CH3) X(CH4) X(CH5) X(CH6) X(CT1) X(CT3) X(CT4) X(CT5) X(CT6)
struct RkTab {
#define X(n) double n;
    ST_RK_RESIDENT(X)
#undef X
};
__device__ __forceinline__ void rk_tab_load(RkTab& T) {
#define X(n) T.n = rk::n; asm volatile("" : "+v"(T.n));
    ST_RK_RESIDENT(X)
#undef X
}
// What every trial reads besides, resident as well: the controller's series
// and limits, and the caller's step-size parameters.  Alone on its SIMD a wave
// issues an instruction in 4.3 cycles but waits some 50 for a scalar load, and
// builds a literal with two instructions; of a trial's 522 issue slots 163
// went by in waits and 97 in scalar instructions.  With these resident and
// the step control in selects in place of branches, fast trials on 1,000
// neutrons take 0.51 us (before: 0.90), exact ones 1.41 (1.63).
// (0 and 1 of the series are inline constants; e[2] is too.)
struct RkCtl {
    double l[11], e[14];             // TAYLOR_HOST[2], [3]
    double ln2_hi, ln2_lo, inv_ln2, clamp, root_half, grow, damp, accept, floor2;
    double h0, hmax, hmin, tol2, tol2x4;
    uint32_t nmax;
    bool fixed;
};
__device__ __forceinline__ void rk_ctl_load(RkCtl& C, const SimParams& P) {
    C.l[0] = C.e[0] = C.e[1] = 1.0;
    C.e[2] = 0.5;
#define ST_RK_CTL(N, ROW, K) N[K] = TAYLOR_HOST[ROW][K]; asm volatile("" : "+v"(N[K]));
    ST_RK_CTL(C.l, 2, 1) ST_RK_CTL(C.l, 2, 2) ST_RK_CTL(C.l, 2, 3) ST_RK_CTL(C.l, 2, 4) ST_RK_CTL(C.l, 2, 5)
    ST_RK_CTL(C.l, 2, 6) ST_RK_CTL(C.l, 2, 7) ST_RK_CTL(C.l, 2, 8) ST_RK_CTL(C.l, 2, 9) ST_RK_CTL(C.l, 2, 10)
    ST_RK_CTL(C.e, 3, 3) ST_RK_CTL(C.e, 3, 4) ST_RK_CTL(C.e, 3, 5) ST_RK_CTL(C.e, 3, 6) ST_RK_CTL(C.e, 3, 7)
    ST_RK_CTL(C.e, 3, 8) ST_RK_CTL(C.e, 3, 9) ST_RK_CTL(C.e, 3, 10) ST_RK_CTL(C.e, 3, 11) ST_RK_CTL(C.e, 3, 12)
    ST_RK_CTL(C.e, 3, 13)
#undef ST_RK_CTL
#define ST_RK_CTL(N, V) C.N = V; asm volatile("" : "+s"(C.N));
    ST_RK_CTL(ln2_hi, LN2_HI) ST_RK_CTL(ln2_lo, LN2_LO) ST_RK_CTL(inv_ln2, INV_LN2) ST_RK_CTL(clamp, 2000.0)
    ST_RK_CTL(root_half, 0.70710678118654752440) ST_RK_CTL(grow, 0.7 / 7.0) ST_RK_CTL(damp, -0.4 / 7.0)
    ST_RK_CTL(accept, 0.81) ST_RK_CTL(floor2, 1.0E-32)
    ST_RK_CTL(h0, P.h0) ST_RK_CTL(hmax, P.hmax) ST_RK_CTL(hmin, P.hmin)
#undef ST_RK_CTL
    C.tol2 = P.rtol * P.rtol;
    C.tol2x4 = 4.0 * C.tol2;
    asm volatile("" : "+v"(C.tol2), "+v"(C.tol2x4));
    C.nmax = P.nmax;
    C.fixed = P.fixed != 0;
}
template <int N>
__device__ __forceinline__ double q_series(const double (&c)[N], double x) {
    double a = c[N - 1];
#pragma unroll
    for (int k = N - 2; k >= 0; --k) a = __builtin_fma(x, a, c[k]);
    return a;
}
// ctl_log, ctl_exp and rk_factor_fast from the resident coefficients
__device__ __forceinline__ double q_ctl_log(const RkCtl& C, double x) {
    int e;
    double m = frexp(x, &e);
    if (m < C.root_half) {
        m *= 2.0;
        e -= 1;
    }
    const double r0 = __builtin_amdgcn_rcp(m + 1.0);
    const double sv = (m - 1.0) * __builtin_fma(r0, __builtin_fma(-(m + 1.0), r0, 1.0), r0);
    const double p = (2.0 * sv) * q_series(C.l, sv * sv);
    double l = __builtin_fma((double)e, C.ln2_hi, __builtin_fma((double)e, C.ln2_lo, p));
    if (!__builtin_amdgcn_class(x, 0x180)) l = log(x);   // not a positive finite number
    return l;
}
__device__ __forceinline__ double q_ctl_exp(const RkCtl& C, double y) {
    const double n = fmin(fmax(rint(y * C.inv_ln2), -C.clamp), C.clamp);
    const double r = __builtin_fma(-n, C.ln2_lo, __builtin_fma(-n, C.ln2_hi, y));
    return ldexp(q_series(C.e, r), (int)n);
}
__device__ __forceinline__ double q_rk_factor(const RkCtl& C, double e2_in, double& prev_lr, bool& small) {
    const double e2 = std_max(e2_in, C.floor2);
    const double lr = 0.5 * q_ctl_log(C, C.tol2 * fast_rcp(e2));
    const double q = q_ctl_exp(C, __builtin_fma(C.damp, prev_lr, C.grow * lr));
    prev_lr = lr;
    small = e2 < C.tol2x4;
    return q;
}
// RkState with the lane's component of yy1
struct QRk {
    double t, tf, lastH, prev_ratio, prev_lr, yy1;
    int32_t nstep;
    bool stop;
};
__device__ __forceinline__ void q_rk_begin(QRk& R, double t0, double t_end, double h) {
    R.t = t0;
    R.tf = t_end;
    R.stop = false;
    R.nstep = 0;
    R.lastH = h;
    R.yy1 = 0.0;
    R.prev_ratio = 1.0;
    R.prev_lr = 0.0;
}
// rk_bounds with one branch, taken at an error (h stays)
__device__ __forceinline__ int q_rk_bounds(const RkCtl& C, QRk& R, double& h) {
    R.nstep++;
    const bool over = (uint32_t)R.nstep > C.nmax, below = !C.fixed && h < C.hmin && !(h > C.hmax);
    if (over || below) return over ? -2 : -1;
    const double endDt = R.tf - R.t;
    const double hn = C.fixed ? C.h0 : (h > C.hmax ? C.hmax : h);
    R.stop = hn >= endDt;
    R.lastH = R.stop ? h : hn;
    h = R.stop ? endDt : hn;
    return 0;
}
// end of an iteration: accept or reject, next step size
__device__ __forceinline__ int q_rk_end(const RkCtl& C, QRk& R, double& y, double ws, double& h, double q_, bool small,
                                        uint32_t& nacc, uint32_t& nrej) {
    q_ = std_min(q_, 4.0);
    const bool ok = (q_ > C.accept && small) || C.fixed;
    const bool done = ok && R.stop;
    nacc += ok;
    nrej += !ok;
    y = ok ? ws : y;
    R.t = ok ? R.t + h : R.t;
    const double next = C.fixed ? h : h * q_;
    h = done ? R.lastH : next;
    R.stop = done;
    return done;
}
// rk_trial_fast (st_integrators.h) on a quad; the pulse's cosines at the six
// stage times are split over the quad.
template <bool PULSE>
__device__ __forceinline__ int q_trial_rk_fast(const RkCtl& C, const RkTab& T, QRk& R, double& y, double& h,
                                               double t0, const QPoly& q, const QPulse& pl, uint32_t& nacc,
                                               uint32_t& nrej) {
    if (const int b = q_rk_bounds(C, R, h)) return b;
    const double t = R.t, tx = t - t0;
    const QPoly hq{h * q.a0, h * q.a1, h * q.a2, h * q.b0, h * q.b1, h * q.b2};
    double hp0 = 0.0, hp1 = 0.0, ha = 0.0, hb = 0.0;
    if constexpr (PULSE) {
        if (pl.on) {
            const uint32_t l = __lane_id() & 3u;
            const double c0 = l == 1 ? T.A2 : l == 2 ? T.A3 : T.A4, c1 = l == 0 ? rk::A5 : T.A6;
            const double t0_ = __builtin_fma(c0, h, t);
            hp0 = phase_cos(pl.pw * (l == 0 ? t : t0_));
            hp1 = phase_cos(pl.pw * __builtin_fma(c1, h, t));
            ha = h * pl.ma;
            hb = h * pl.mb;
        }
    }
    auto K = [&](double tau, double yy, double cosv) -> double {
        double wa, wb;
        q_field(tau, hq, wa, wb);
        if constexpr (PULSE) {
            wa = __builtin_fma(ha, cosv, wa);
            wb = __builtin_fma(hb, cosv, wb);
        }
        return q_cross(yy, wa, wb);
    };
#define QF(S, A, K) S = __builtin_fma(T.A, K, S)
    const double K1 = K(tx, R.yy1, q_all<0>(hp0));
    double yy = y;
    QF(yy, B21, K1);
    const double K2 = K(__builtin_fma(T.A2, h, tx), yy, q_all<1>(hp0));
    yy = y;
    QF(yy, B31, K1); QF(yy, B32, K2);
    const double K3 = K(__builtin_fma(T.A3, h, tx), yy, q_all<2>(hp0));
    yy = y;
    QF(yy, B41, K1); QF(yy, B42, K2); QF(yy, B43, K3);
    const double K4 = K(__builtin_fma(T.A4, h, tx), yy, q_all<3>(hp0));
    yy = y;
    QF(yy, B51, K1); QF(yy, B52, K2); QF(yy, B53, K3); QF(yy, B54, K4);
    const double K5 = K(__builtin_fma(rk::A5, h, tx), yy, q_all<0>(hp1));
    yy = y;
    QF(yy, B61, K1); QF(yy, B62, K2); QF(yy, B63, K3); QF(yy, B64, K4); QF(yy, B65, K5);
    const double K6 = K(__builtin_fma(T.A6, h, tx), yy, q_all<1>(hp1));
    R.yy1 = yy;
    double ws = y;
    QF(ws, CH1, K1); QF(ws, CH3, K3); QF(ws, CH4, K4); QF(ws, CH5, K5); QF(ws, CH6, K6);
    double te = T.CT1 * K1;
    QF(te, CT3, K3); QF(te, CT4, K4); QF(te, CT5, K5); QF(te, CT6, K6);
#undef QF
    const d3 e = q_vec(te);
    bool small;
    const double f = q_rk_factor(C, __builtin_fma(e.z, e.z, __builtin_fma(e.y, e.y, e.x * e.x)), R.prev_lr, small);
    return q_rk_end(C, R, y, ws, h, f, small, nacc, nrej);
}
// rk_trial_exact on a quad
template <bool PULSE>
__device__ __forceinline__ int q_trial_rk_exact(const SimParams& P, const RkCtl& C, const RkTab& T, QRk& R, double& y, double& h,
                                                double t0, const QExact& X, uint32_t& nacc, uint32_t& nrej) {
    if (const int b = q_rk_bounds(C, R, h)) return b;
    const bool gravity = P.gravity;
    const double t = R.t, t2 = t + T.A2 * h, t3 = t + T.A3 * h, t4 = t + T.A4 * h, t5 = t + rk::A5 * h, t6 = t + T.A6 * h;
    double hp0 = 0.0, hp1 = 0.0;
    if constexpr (PULSE) {
        if (X.axis >= 0) {
            const uint32_t l = __lane_id() & 3u;
            hp0 = q_pulse_exact(X, l == 0 ? t : l == 1 ? t2 : l == 2 ? t3 : t4);
            hp1 = q_pulse_exact(X, l == 0 ? t5 : t6);
        }
    }
#define QX(TT, LANE, HP) q_rhs_exact(X, gravity, (TT), t0, yy, PULSE ? q_all<LANE>(HP) : 0.0)
    double yy = R.yy1;
    double k1 = QX(t, 0, hp0);
    ST_CODE_ALIGN(k1);
    yy = y + (h * T.B21) * k1;
    double k2 = QX(t2, 1, hp0);
    ST_CODE_ALIGN(k2);
    yy = y + (h * T.B31) * k1 + (h * T.B32) * k2;
    double k3 = QX(t3, 2, hp0);
    ST_CODE_ALIGN(k3);
    yy = y + (h * T.B41) * k1 + (h * T.B42) * k2 + (h * T.B43) * k3;
    double k4 = QX(t4, 3, hp0);
    ST_CODE_ALIGN(k4);
    yy = y + (h * T.B51) * k1 + (h * T.B52) * k2 + (h * T.B53) * k3 + (h * T.B54) * k4;
    double k5 = QX(t5, 0, hp1);
    ST_CODE_ALIGN(k5);
    yy = y + (h * T.B61) * k1 + (h * T.B62) * k2 + (h * T.B63) * k3 + (h * T.B64) * k4 + (h * T.B65) * k5;
    double k6 = QX(t6, 1, hp1);
    ST_CODE_ALIGN(k6);
#undef QX
    R.yy1 = yy;
    const double ws = y + h * (k1 * T.CH1 + k2 * rk::CH2 + k3 * T.CH3 + k4 * T.CH4 + k5 * T.CH5 + k6 * T.CH6);
    const double te = h * (T.CT1 * k1 + rk::CT2 * k2 + T.CT3 * k3 + T.CT4 * k4 + T.CT5 * k5 + T.CT6 * k6);
    const double tol = P.rtol;
    double error = len3(q_vec(te));
    error = std_max(error, 1.0E-16);
    const double ratio = tol / error;
    // both powers at once: lanes 0 and 1 of the quad take the first, 2 and 3 the other
    const bool low = (__lane_id() & 2u) == 0u;
    const double p = pow(low ? ratio : R.prev_ratio, low ? 0.7 / 7.0 : -0.4 / 7.0);
    const double f = q_all<0>(p) * q_all<2>(p);
    R.prev_ratio = ratio;
    return q_rk_end(C, R, y, ws, h, f, error < 2 * tol, nacc, nrej);
}

// ---------------------------------------------------------------------------
// MagnusCFET (integratorType 2, fast variant) on a quad
// ---------------------------------------------------------------------------
// The one-lane trial forms sixteen rotations one after another, each with its
// scalar loads of coefficients to wait for: 8.4 us on He-3 with a wave per
// SIMD.  On a quad each lane forms four of them, from coefficients it keeps:
//   lane 0: factors 0, 3, 6, 9 of the order-8 chain, lane 1: 1, 4, 7, 10,
//   lane 2: 2, 5, 8 and the order-6 chain's last, lane 3: that chain's 0..3.
// The products then follow the one-lane trial's order, the order-8 chain in
// lanes 0 and 1, the order-6 chain in lanes 2 and 3, each factor brought from
// its lane by quad moves.  k_spin, He-3 x 0.2 s: 4,096 particles 2.19 and
// 0.79 ms, 32,768 2.34 and 1.17 ms (65,536, past the limit: 2.25 and 2.19 ms).
struct MagTab {
    double m[4][3];          // the lane's four exponents (CFET_MOM)
    double c[8], s[8];       // the series of half_series<true>
};
__device__ __forceinline__ uint32_t mag_row(uint32_t l, uint32_t slot) {
    return l < 3 ? (l == 2 && slot == 3 ? 15u : 3 * slot + l) : 11 + slot;
}
__device__ __forceinline__ double mag_coef(uint32_t row, int k) {
#if defined(__HIP_DEVICE_COMPILE__)
    return CFET_MOM.m[row][k];
#else
    return CFET_MOM_HOST.m[row][k];
#endif
}
__device__ __forceinline__ void mag_tab_load(MagTab& T) {
    const uint32_t l = __lane_id() & 3u;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            T.m[j][k] = mag_coef(mag_row(l, j), k);
            asm volatile("" : "+v"(T.m[j][k]));
        }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        T.c[k] = TAYLOR_HOST[0][k];
        T.s[k] = TAYLOR_HOST[1][k];
        if (k > 1) asm volatile("" : "+v"(T.c[k]));   // (1 and -1/2 are inline constants)
        if (k > 0) asm volatile("" : "+v"(T.s[k]));
    }
}
// rot_quat_half from the resident series
__device__ __forceinline__ Quat q_rot_half(const MagTab& T, const d3& g) {
#pragma clang fp contract(fast)
    const double t2 = len2_fma(g);
    const bool extra = t2 >= 1.0;   // beyond one halving (cos_sinc_doubled<1, true, true>)
    int d = 1;
    double x2 = t2 * 0.25;
    if (__any(extra)) {
        int E;
        (void)frexp(t2, &E);
        d = E + 2 > 2 ? (E + 3) >> 1 : 1;
        x2 = ldexp(t2, -2 * d);
    }
    double c = q_series(T.c, x2), s = q_series(T.s, x2);
    auto twice = [&]() {
        const double s2 = s * s;
        s = s * c;
        c = 1.0 - (2.0 * x2) * s2;
        x2 *= 4.0;
    };
    const bool good = t2 > 0.0 && t2 <= 0.25 * FAST_ROT_MAX_X2;
    if (__any(extra && good))
        for (int i = good ? d : 1; i > 1; --i) twice();
    twice();
    Quat r{c, g.x * s, g.y * s, g.z * s};
    if (!good) r = rodriguez_quat(d3{-2.0 * g.x, -2.0 * g.y, -2.0 * g.z}, 1.0);
    return r;
}
// lane A's value in lanes 0 and 1, lane B's in lanes 2 and 3
template <int A, int B>
__device__ __forceinline__ Quat q_pair(const Quat& q) {
    constexpr int CTRL = A | A << 2 | B << 4 | B << 6;
    return Quat{quad_perm<CTRL>(q.w), quad_perm<CTRL>(q.x), quad_perm<CTRL>(q.y), quad_perm<CTRL>(q.z)};
}
// bounds_v2 with one branch, taken at an error (h stays)
__device__ __forceinline__ int q_bounds_v2(const RkCtl& C, QRk& R, double& h) {
    R.nstep++;
    const double endDt = R.tf - R.t;
    const bool ends = !C.fixed && h >= endDt;
    const bool over = (uint32_t)R.nstep > C.nmax, below = !C.fixed && !ends && h < C.hmin && !(h > C.hmax);
    if (over || below) return over ? -2 : -1;
    R.lastH = h;
    R.stop = C.fixed ? R.stop : ends;
    h = C.fixed ? C.h0 : ends ? endDt : (h > C.hmax ? C.hmax : h);
    return 0;
}
template <bool PULSE>
__device__ __forceinline__ int q_trial_magnus(const RkCtl& C, const MagTab& T, QRk& R, double& y, double& h, double t0,
                                              const Poly& q, uint32_t c, uint32_t& nacc, uint32_t& nrej) {
#pragma clang fp contract(fast)
    if (const int b = q_bounds_v2(C, R, h)) return b;
    const double t = R.t;
    const double tau = t - t0, h2 = h * h, h3 = h2 * h, tt = 2.0 * tau;
    const d3 u0{h * (q.w0.x + tau * (q.w1.x + tau * q.w2.x)), h * (q.w0.y + tau * (q.w1.y + tau * q.w2.y)),
                h * (q.w0.z + tau * (q.w1.z + tau * q.w2.z))};
    const d3 u1{h2 * (q.w1.x + tt * q.w2.x), h2 * (q.w1.y + tt * q.w2.y), h2 * (q.w1.z + tt * q.w2.z)};
    const d3 u2{h3 * q.w2.x, h3 * q.w2.y, h3 * q.w2.z};
    auto f = [](double x, double y, double z) -> double { return __builtin_fma(x, y, z); };
    const uint32_t l = __lane_id() & 3u;
    double hp[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if constexpr (PULSE) {
        if (q.pon) {   // h * pulse at the five nodes, four of them a lane each
            using namespace cfet;
            const double X = l == 0 ? X1 : l == 1 ? X2 : l == 2 ? X3 : X4;
            const double a = h * (q.pag * phase_cos(q.pw * (t + X * h)));
            hp[0] = q_all<0>(a); hp[1] = q_all<1>(a); hp[2] = q_all<2>(a); hp[3] = q_all<3>(a);
            hp[4] = h * (q.pag * phase_cos(q.pw * (t + X5 * h)));
        }
    }
    auto rot = [&](int j) -> Quat {
        const double* m = T.m[j];
        d3 k{f(m[2], u2.x, f(m[1], u1.x, m[0] * u0.x)), f(m[2], u2.y, f(m[1], u1.y, m[0] * u0.y)),
             f(m[2], u2.z, f(m[1], u1.z, m[0] * u0.z))};
        if constexpr (PULSE) {
            if (q.pon) {
                const uint32_t r = mag_row(l, j);
                const double pe = f(mag_coef(r, 7), hp[4],
                                    f(mag_coef(r, 6), hp[3],
                                      f(mag_coef(r, 5), hp[2], f(mag_coef(r, 4), hp[1], mag_coef(r, 3) * hp[0]))));
                k.x += q.paxis == 0 ? pe : 0.0;
                k.y += q.paxis == 1 ? pe : 0.0;
                k.z += q.paxis == 2 ? pe : 0.0;
            }
        }
        return q_rot_half(T, k);
    };
    const Quat r0 = rot(0), r1 = rot(1), r2 = rot(2), r3 = rot(3);
    // order 8 | order 6
    Quat p = q_pair<0, 3>(r0);
    {
        const Quat b = q_pair<1, 3>(Quat{l == 3 ? r1.w : r0.w, l == 3 ? r1.x : r0.x, l == 3 ? r1.y : r0.y, l == 3 ? r1.z : r0.z});
        p = q_mult_fast(b, p);       // factor 1 | 1
    }
    {
        const Quat b = q_pair<2, 3>(Quat{l == 3 ? r2.w : r0.w, l == 3 ? r2.x : r0.x, l == 3 ? r2.y : r0.y, l == 3 ? r2.z : r0.z});
        p = q_mult_fast(b, p);       // 2 | 2
    }
    {
        const Quat b = q_pair<0, 3>(Quat{l == 3 ? r3.w : r1.w, l == 3 ? r3.x : r1.x, l == 3 ? r3.y : r1.y, l == 3 ? r3.z : r1.z});
        p = q_mult_fast(b, p);       // 3 | 3
    }
    {
        const Quat b = q_pair<1, 2>(Quat{l == 2 ? r3.w : r1.w, l == 2 ? r3.x : r1.x, l == 2 ? r3.y : r1.y, l == 2 ? r3.z : r1.z});
        p = q_mult_fast(b, p);       // 4 | 4, the order-6 chain's last
    }
    Quat p8 = p;                     // (lanes 2 and 3: repeated work)
    p8 = q_mult_fast(q_pair<2, 2>(r1), p8);
    p8 = q_mult_fast(q_pair<0, 0>(r2), p8);
    p8 = q_mult_fast(q_pair<1, 1>(r2), p8);
    p8 = q_mult_fast(q_pair<2, 2>(r2), p8);
    p8 = q_mult_fast(q_pair<0, 0>(r3), p8);
    p8 = q_mult_fast(q_pair<1, 1>(r3), p8);
    const bool six = l >= 2;
    const Quat qq{six ? p.w : p8.w, six ? p.x : p8.x, six ? p.y : p8.y, six ? p.z : p8.z};
    const d3 v = qrot_fast(qq, q_vec(y));
    const d3 y8 = q_vec3<0>(v), y6 = q_vec3<2>(v);
    const d3 d{y8.x - y6.x, y8.y - y6.y, y8.z - y6.z};
    bool small;
    const double fac = q_rk_factor(C, len2_fma(d), R.prev_lr, small);
    return q_rk_end(C, R, y, q_pick(y8, c), h, fac, small, nacc, nrej);
}

// The products make_poly reads, for the lane's components a = c+1 and b = c+2.
__device__ __forceinline__ void q_pulse_load(QPulse& pl, const Phys& F, uint32_t c, double sign = 1.0) {
    const int32_t a = c == 2 ? 0 : (int32_t)c + 1, b = c == 0 ? 2 : (int32_t)c - 1;
    pl.pw = F.pw;
    pl.on = F.pulse_on != 0;
    pl.ma = (pl.on && F.pulse_axis == a) ? sign * F.gpa : 0.0;
    pl.mb = (pl.on && F.pulse_axis == b) ? sign * F.gpa : 0.0;
}
// make_poly's components a and b
__device__ __forceinline__ void q_make_poly(QPoly& q, const Phys& F, const d3& p, const d3& v, uint32_t c) {
#pragma clang fp contract(fast)
    const uint32_t a = c == 2 ? 0u : c + 1, b = c == 0 ? 2u : c - 1;
    const double vc = q_pick(v, c), va = q_next1(vc), vb = q_next2(vc);
    const double *Ga = F.gG + 3 * a, *Gb = F.gG + 3 * b;
    const double Ec = F.gE[c], Ea = F.gE[a], Eb = F.gE[b];
    // row i: gB0 + G.p + v_{i+1} gE_{i+2} - v_{i+2} gE_{i+1}
    q.a0 = F.gB0[a] + Ga[0] * p.x + Ga[1] * p.y + Ga[2] * p.z + vb * Ec - vc * Eb;
    q.b0 = F.gB0[b] + Gb[0] * p.x + Gb[1] * p.y + Gb[2] * p.z + vc * Ea - va * Ec;
    q.a1 = F.gw1[a] + Ga[0] * v.x + Ga[1] * v.y + Ga[2] * v.z;
    q.b1 = F.gw1[b] + Gb[0] * v.x + Gb[1] * v.y + Gb[2] * v.z;
    q.a2 = F.gw2[a];
    q.b2 = F.gw2[b];
}

// ---------------------------------------------------------------------------
// the spin loop on quads
// ---------------------------------------------------------------------------
// spin_body (st_pipeline.h) with a particle per quad: same records, same
// bookkeeping, lane 0 of the quad writing what is not per component.  A
// wave takes ppw particles at a time, ppw a power of two up to 16: a small
// list is spread over more waves, so that a quad rarely waits for another's
// segment set-up (1,000 He-3 x 0.2 s: 1.17 ms at 16 a wave, 0.91 ms at one).
// The quads beyond ppw repeat the first ones and write nothing: with those
// lanes masked off instead, a full compute unit ran the same instructions
// 2.5 times slower (3.7 against 1.4 ms on 1,000 neutrons x 0.5 s).
__device__ __forceinline__ void quad_block(const RunArgs& R, uint32_t pid, int32_t k, uint32_t c, double y) {
    if (R.blocks) reinterpret_cast<double*>(R.blocks + (uint64_t)k * R.block_bytes + 56 * (uint64_t)R.n)[3 * (uint64_t)pid + c] = y;
}
template <int VAR, int INTEG, bool BATCH, bool PULSE>
__device__ __forceinline__ void quad_spin() {
    auto args = []() -> const QuadArgs& { return kernel_args<QuadArgs>(); };
    const uint32_t lane = __lane_id();
    const uint32_t c = (lane & 3u) == 3u ? 0u : (lane & 3u);   // lane 3 repeats lane 0
    const uint32_t ppw = args().ppw;
    const bool first = (lane >> 2) < ppw;
    const bool lead = first && (lane & 3u) == 0u, owner = first && (lane & 3u) != 3u;
    constexpr bool DOP = INTEG == INT_DOP853, MAG = INTEG == INT_MAGNUS;
    static_assert(!MAG || VAR == VAR_FAST, "MagnusCFET on quads is the fast variant's");
    DopTab T;
    RkTab TR;
    MagTab TM;
    RkCtl C;
    DopCtl CD;
    if constexpr (DOP) {
        dop_tab_load<false>(T);
        if constexpr (VAR == VAR_FAST) dop_ctl_load(CD, args().P);
    } else {
        if constexpr (MAG) mag_tab_load(TM);
        else rk_tab_load(TR);
        rk_ctl_load(C, args().P);
    }
    // a plain handle's physics in LDS, one copy per workgroup
    __shared__ Phys shared_phys;
    if constexpr (!BATCH) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(args().A.phys);
        for (uint32_t i = threadIdx.x; i < sizeof(Phys) / 4; i += blockDim.x) reinterpret_cast<uint32_t*>(&shared_phys)[i] = src[i];
        __syncthreads();
    }
    QPulse pl;
    QExact X;
    auto physics = [&](const Phys& F) {
        if constexpr (VAR == VAR_EXACT) q_exact_load(X, args().P, F, c);
        else if constexpr (PULSE && !MAG) q_pulse_load(pl, F, c);
    };
    if constexpr (!BATCH) physics(shared_phys);
    SpinLane L;      // (S unused: the lane's component is y)
    double y = 0.0;
    QDop dop;
    QRk rk;
    QPoly q;
    Poly full;       // (MagnusCFET: all components)
    auto seg_end = [&]() { return DOP ? dop.xf : rk.tf; };
    double seg_t0 = 0.0;
    SegRec nxt;      // record L.j, loaded while record L.j - 1 is integrated
    uint32_t cur_flags = 0;
    uint32_t cnt[4] = {0, 0, 0, 0};   // accepted, rejected, segments, trips (of this launch)
    enum { S_DONE = 0, S_NEXT = 1, S_INT = 2 };
    int phase = S_DONE;
    uint32_t pos = quad_index(ppw);
    auto take = [&]() {
        const PipeArgs& A = args().A;
        const DevState& D = args().D;
        const uint32_t i = pos;
        pos += 4u * gridDim.x * ppw;
        if (i >= A.n_list) return;
        spin_load<BATCH>(D, A, A.list[i], L);
        y = q_pick(L.S, c);
        if constexpr (BATCH) physics(A.phys[L.cfg]);
        if (L.nrec > 0) nxt = load_rec(rec_at_seq(A, L.pid, 0, L.page));
        phase = S_NEXT;
    };
    take();
    // The fast RK45 trial's place within a cache line is worth up to 3 % to a
    // lone wave (8,192 neutrons, whole run: 18.8 to 19.5 ms over the sixteen
    // places of the same code); from the start of one it takes 18.87.
    if constexpr (INTEG == INT_RK45 && VAR == VAR_FAST) asm volatile(".p2align 6");
    while (phase != S_DONE) {
        cnt[3] += lead;
        if (phase == S_NEXT) {
            while (phase == S_NEXT) {
                if (L.j >= L.nrec) {
                    if (lead) {
                        cnt[0] += L.acc; cnt[1] += L.rej; cnt[2] += L.seg;
                    }
                    L.S = q_vec(y);
                    if (lead) spin_store(args().D, L);
                    phase = S_DONE;
                    take();
                    if (phase == S_DONE) break;
                    continue;
                }
                const PipeArgs& A = args().A;
                const RunArgs& R = A.R;
                const SegRec rec = nxt;
                if (L.j + 1 < L.nrec) nxt = load_rec(rec_at_seq(A, L.pid, L.j + 1, L.page));
                cur_flags = (uint32_t)rec.flags;
                if (rec.flags & R_FIRST) L.tempH = L.h;
                if (rec.flags & R_INTEGRATE) {
                    seg_t0 = L.t_spin;
                    if constexpr (VAR == VAR_EXACT) {
                        X.p0 = q_pick(d3{rec.px, rec.py, rec.pz}, c);
                        X.v0 = q_pick(d3{rec.vx, rec.vy, rec.vz}, c);
                    } else if constexpr (MAG) {
                        Seg seg;
                        seg.t0 = seg_t0;
                        seg.p0 = d3{rec.px, rec.py, rec.pz};
                        seg.v0 = d3{rec.vx, rec.vy, rec.vz};
                        full = make_poly(args().P, BATCH ? A.phys[L.cfg] : shared_phys, seg);
                        if constexpr (!PULSE) full.pon = 0;
                    } else {
                        q_make_poly(q, BATCH ? A.phys[L.cfg] : shared_phys, d3{rec.px, rec.py, rec.pz},
                                    d3{rec.vx, rec.vy, rec.vz}, c);
                    }
                    if constexpr (DOP) {
                        dop.x = seg_t0;
                        dop.xf = rec.t;
                        dop.facold = 1.0E-4;
                        dop.last = 0;
                        dop.reject = 0;
                        dop.left = dop_trials(args().P);
                        if constexpr (VAR == VAR_EXACT) {
                            dop.posneg = sign_d(1.0, rec.t - seg_t0);
                            dop.k1 = q_rhs_exact(X, args().P.gravity, seg_t0, seg_t0, y,
                                                 PULSE && X.axis >= 0 ? q_pulse_exact(X, seg_t0) : 0.0);
                        } else {
                            double wa = q.a0, wb = q.b0;
                            if constexpr (PULSE) {
                                const double cosv = pl.on ? phase_cos(pl.pw * seg_t0) : 0.0;
                                wa = __builtin_fma(pl.ma, cosv, wa);
                                wb = __builtin_fma(pl.mb, cosv, wb);
                            }
                            dop.k1 = q_cross(y, wa, wb);
                        }
                    } else {
                        q_rk_begin(rk, seg_t0, rec.t, L.tempH);
                    }
                    L.seg++;
                    if (R.trace && L.pid == R.trace_pid) {
                        const d3 S = q_vec(y);
                        if (lead)
                            ST_TRACE(R, 1, seg_t0, rec.t, d3{rec.px, rec.py, rec.pz}, d3{rec.vx, rec.vy, rec.vz}, S,
                                     L.tempH, L.acc, L.rej, (char)(rec.flags >> 8), (char)(rec.flags >> 16), 0, 0, 0);
                    }
                    phase = S_INT;
                } else {
                    if (rec.flags & R_STOP) y = __builtin_nan("");
                    if (rec.flags & R_IEND) {
                        if (owner) quad_block(R, L.pid, L.k, c, y);
                        L.k++;
                    }
                    if (!(rec.flags & R_EMPTY)) L.t_spin = rec.t;
                    L.j++;
                }
            }
        }
        if (phase == S_INT) {
            // Trials until some quad of the wave ends its segment (DOP853 with
            // more than four particles in the wave: one at a time, since some
            // quad ends its segment on most trips; He-3 at 16 a wave: 1.20
            // against 1.24 ms).
            int st;
            for (;;) {
                const SimParams& P = args().P;
                if constexpr (DOP && VAR == VAR_EXACT) st = q_trial_exact<PULSE>(P, T, dop, y, L.tempH, seg_t0, X, L.acc, L.rej);
                else if constexpr (DOP) st = q_trial_fast<false, PULSE>(P, CD, T, dop, y, L.tempH, seg_t0, q, pl, L.acc, L.rej, nullptr);
                else if constexpr (VAR == VAR_EXACT) st = q_trial_rk_exact<PULSE>(P, C, TR, rk, y, L.tempH, seg_t0, X, L.acc, L.rej);
                else if constexpr (MAG) st = q_trial_magnus<PULSE>(C, TM, rk, y, L.tempH, seg_t0, full, c, L.acc, L.rej);
                else st = q_trial_rk_fast<PULSE>(C, TR, rk, y, L.tempH, seg_t0, q, pl, L.acc, L.rej);
                if ((DOP && ppw > 4) || __any(st != 0)) break;
                cnt[3] += lead;
            }
            if (st != 0) {
                const PipeArgs& A = args().A;
                const RunArgs& R = A.R;
                if (R.trace && L.pid == R.trace_pid) {
                    const d3 S = q_vec(y);
                    if (lead)
                        ST_TRACE(R, 2, L.t_spin, seg_end(), d3{0, 0, 0}, d3{0, 0, 0}, S, L.tempH, L.acc, L.rej,
                                 (char)(cur_flags >> 8), (char)(cur_flags >> 16), st, 0, 0);
                }
                if (args().P.keep) L.h = L.tempH;
                L.t_spin = seg_end();
                if (st < 0) {
                    if (lead) {
                        const uint32_t slot = atomicAdd(A.fail_count, 1u);
                        if (slot < A.fail_cap) {
                            A.fail_list[3 * slot + 0] = L.pid;
                            A.fail_list[3 * slot + 1] = L.j;
                            A.fail_list[3 * slot + 2] = (uint32_t)st;
                        }
                    }
                    L.nrec = 0;   // (spin_body: the records after a failure)
                }
                if (st < 0 || (cur_flags & R_STOP)) y = __builtin_nan("");
                if ((cur_flags & R_IEND) && st > 0) {
                    if (owner) quad_block(R, L.pid, L.k, c, y);
                    L.k++;
                }
                L.j++;
                phase = S_NEXT;
            }
        }
    }
    unsigned long long sum[4] = {cnt[0], cnt[1], cnt[2], cnt[3]};
    flush_counters(args().A.R.work, sum);
}

template <int VAR, int INTEG, bool BATCH, bool PULSE>
__global__ __launch_bounds__(256, 2) void k_spin_quad(const QuadArgs) {
    quad_spin<VAR, INTEG, BATCH, PULSE>();
}

// ---------------------------------------------------------------------------
// the adjoint's walk back on quads (k_adj, st_adjoint.h)
// ---------------------------------------------------------------------------
struct QuadAdjArgs {
    SimParams P;
    DevState D;
    AdjArgs A;
    uint32_t ppw;
};
// The lane of component c carries u_c, its moments and its share of the
// gradient sums: u_c r_j (3), (u x v)_c and u_c.
template <bool BATCH, bool PULSE>
__global__ __launch_bounds__(256, 2) void k_adj_quad(const QuadAdjArgs) {
#pragma clang fp contract(fast)
    auto args = []() -> const QuadAdjArgs& { return kernel_args<QuadAdjArgs>(); };
    const uint32_t lane = __lane_id();
    const uint32_t c = (lane & 3u) == 3u ? 0u : (lane & 3u);
    const uint32_t ppw = args().ppw;
    const bool first = (lane >> 2) < ppw;
    const bool lead = first && (lane & 3u) == 0u, owner = first && (lane & 3u) != 3u;
    DopTab T;
    dop_tab_load<true>(T);
    DopCtl CD;
    dop_ctl_load(CD, args().P);
    __shared__ Phys shared_phys;
    // per lane: its gradient sums, and p0 and v0 of the segment being
    // integrated (registers go to the tableau)
    __shared__ double sums[5][256], pv[6][256];
    if constexpr (!BATCH) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(args().A.phys);
        for (uint32_t i = threadIdx.x; i < sizeof(Phys) / 4; i += blockDim.x) reinterpret_cast<uint32_t*>(&shared_phys)[i] = src[i];
        __syncthreads();
    }
    QPulse pl;
    if constexpr (PULSE && !BATCH) q_pulse_load(pl, shared_phys, c, -1.0);
    uint32_t pid = 0, cfg = 0;
    double u = 0.0, h = 0.0;
    int32_t kb = 0, fail = 0, j = -1;
    SegRec nxt;                 // record j, loaded while record j + 1 is integrated,
    double nxt_t0 = 0.0;        // and its start time
    QPoly q;
    QQuad Q;
    QDop dop;
    uint32_t nacc = 0, nrej = 0;
    enum { S_DONE = 0, S_NEXT = 1, S_INT = 2 };
    int phase = S_DONE;
    // record i and its start time
    auto load = [&](const AdjArgs& A, int32_t i) {
        if (i < 0) return;
        nxt = get_rec(A.recs, A.C, pid, (uint32_t)i);
        nxt_t0 = i > 0 ? get_rec(A.recs, A.C, pid, (uint32_t)(i - 1)).t : A.ck.ld(F_T, pid * 8u);
    };
    uint32_t pos = quad_index(ppw);
    auto take = [&]() {
        const AdjArgs& A = args().A;
        const uint32_t i = pos;
        pos += 4u * gridDim.x * ppw;
        if (i >= A.n_list) return;
        pid = A.list[i];
        const uint32_t o = pid * 8u;
        u = A.adj.ld(A_UX + (int)c, o);
        h = A.adj.ld(A_H, o);
        kb = (int32_t)A.adj.ld<int64_t>(A_K, o);
        fail = (int32_t)A.adj.ld<int64_t>(A_FAIL, o);
        if constexpr (BATCH) {
            const DevState& D = args().D;
            cfg = (uint32_t)*(D.template f<uint64_t>(F_CFG) + pid);
        }
        if constexpr (PULSE && BATCH) q_pulse_load(pl, A.phys[cfg], c, -1.0);
        for (int k = 0; k < 3; ++k) sums[k][threadIdx.x] = A.adj.ld(A_G0 + 3 * (int)c + k, o);
        sums[3][threadIdx.x] = A.adj.ld(A_G0 + 9 + (int)c, o);
        sums[4][threadIdx.x] = A.adj.ld(A_G0 + 12 + (int)c, o);
        j = (int32_t)A.seg_count[pid] - 1;
        load(A, j);
        phase = S_NEXT;
    };
    take();
    while (phase != S_DONE) {
        while (phase == S_NEXT) {
            const AdjArgs& A = args().A;
            if (j < 0) {
                const uint32_t o = pid * 8u;
                if (owner) {
                    A.adj.st(A_UX + (int)c, o, u);
                    for (int k = 0; k < 3; ++k) A.adj.st(A_G0 + 3 * (int)c + k, o, sums[k][threadIdx.x]);
                    A.adj.st(A_G0 + 9 + (int)c, o, sums[3][threadIdx.x]);
                    A.adj.st(A_G0 + 12 + (int)c, o, sums[4][threadIdx.x]);
                }
                if (lead) {
                    A.adj.st(A_H, o, h);
                    A.adj.st<int64_t>(A_K, o, kb);
                    A.adj.st<int64_t>(A_FAIL, o, fail);
                }
                phase = S_DONE;
                take();
                continue;
            }
            const SegRec rec = nxt;
            const double t0 = nxt_t0;
            load(A, j - 1);
            if ((rec.flags & R_IEND) && kb >= 0) {
                const double* Sk = reinterpret_cast<const double*>(A.blocks + (uint64_t)kb * A.block_bytes + 56ull * A.n) +
                                   3ull * pid;
                const double* gp = A.seeds + 3 * ((uint64_t)cfg * A.n_targets + (uint64_t)kb);
                const double gc = gp[c], Sc = Sk[c];
                u = u + __builtin_fma(q_next1(gc), q_next2(Sc), -(q_next2(gc) * q_next1(Sc)));
                --kb;
                const d3 all = q_vec(u);
                if (!(__builtin_isfinite(all.x) && __builtin_isfinite(all.y) && __builtin_isfinite(all.z))) fail = -3;
            }
            const double Ts = rec.t - t0;
            if (!(rec.flags & R_INTEGRATE) || fail || !(Ts > 0.0)) {
                --j;
                continue;
            }
            QPoly f;
            q_make_poly(f, BATCH ? A.phys[cfg] : shared_phys, d3{rec.px, rec.py, rec.pz}, d3{rec.vx, rec.vy, rec.vz}, c);
            q.a0 = -(f.a0 + Ts * (f.a1 + Ts * f.a2));
            q.b0 = -(f.b0 + Ts * (f.b1 + Ts * f.b2));
            q.a1 = f.a1 + 2.0 * Ts * f.a2;
            q.b1 = f.b1 + 2.0 * Ts * f.b2;
            q.a2 = -f.a2;
            q.b2 = -f.b2;
            pv[0][threadIdx.x] = rec.px; pv[1][threadIdx.x] = rec.py; pv[2][threadIdx.x] = rec.pz;
            pv[3][threadIdx.x] = rec.vx; pv[4][threadIdx.x] = rec.vy; pv[5][threadIdx.x] = rec.vz;
            Q.n0 = Q.n1 = Q.n2 = 0.0;
            Q.t_end = rec.t;
            dop.x = 0.0;
            dop.xf = Ts;
            dop.facold = 1.0E-4;
            dop.last = 0;
            dop.reject = 0;
            dop.left = dop_trials(args().P);
            double wa = q.a0, wb = q.b0;
            if constexpr (PULSE) {
                const double cosv = pl.on ? phase_cos(pl.pw * rec.t) : 0.0;
                wa = __builtin_fma(pl.ma, cosv, wa);
                wb = __builtin_fma(pl.mb, cosv, wb);
            }
            dop.k1 = q_cross(u, wa, wb);
            phase = S_INT;
        }
        if (phase == S_INT) {
            const int st = q_trial_fast<true, PULSE>(args().P, CD, T, dop, u, h, 0.0, q, pl, nacc, nrej, &Q);
            if (st < 0) {
                fail = st;
                --j;
                phase = S_NEXT;
            } else if (st > 0) {
                const double ay = args().P.gravity ? G_CONST : 0.0;
                const AdjMoments M = adj_moments(dop.xf, Q.n0, Q.n1, Q.n2);
                const uint32_t i = threadIdx.x;
                const d3 v{pv[3][i], pv[4][i], pv[5][i]};
                const double vc = q_pick(v, c);
                // (u x v)_c plus -int u_z tau ay dt for x, +int u_x tau ay dt for z
                const double uv = __builtin_fma(q_next1(M.m0), q_next2(vc), -(q_next2(M.m0) * q_next1(vc)));
                const double mz = q_next2(M.m1), mx = q_next1(M.m1);
                const double uva = c == 0 ? __builtin_fma(mz, -ay, uv) : (c == 2 ? __builtin_fma(mx, ay, uv) : uv);
                sums[0][i] += adj_ur(M, pv[0][i], v.x, 0.0);
                sums[1][i] += adj_ur(M, pv[1][i], v.y, 0.5 * ay);
                sums[2][i] += adj_ur(M, pv[2][i], v.z, 0.0);
                sums[3][i] += uva;
                sums[4][i] += M.m0;
                --j;
                phase = S_NEXT;
            }
        }
    }
}

}  // namespace st
