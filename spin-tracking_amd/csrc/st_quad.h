// st_quad.h -- DOP853 spin kernels with four lanes per particle, for ensembles
// that do not fill the chip.
//
// What bounds a small ensemble is one lane's chain of trial steps: with one
// wave per SIMD nothing else can issue, so every instruction of the trial,
// scalar ones included, costs its own issue slot (about 800 vector and 1,300
// scalar instructions per one-lane fast trial, most of the scalar ones moves
// of 64-bit tableau literals: 3.8 us per trial, against 1.7 us when three
// waves share the SIMD).  Here a particle takes a quad of lanes, one spin
// component each (lane 3 repeats lane 0):
//   * the stage sums, two thirds of the trial's operations, run once per quad
//     instead of once per component;
//   * the components meet in the cross products and the error norm, through
//     quad-permute moves (no LDS, no waits);
//   * the tableau stays in vector registers for the whole launch (the
//     one-lane kernel needs them for its state; a lane of a quad holds a third
//     of that state);
//   * the next segment record is loaded while the current one is integrated.
// Every value is formed by the one-lane trial's operations in its order, so
// accept/reject decisions and results are those of the one-lane kernels; a
// quad's four lanes always agree on the control flow.
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

// v[c], c = 0..2
__device__ __forceinline__ double q_pick(const d3& v, uint32_t c) { return c == 0 ? v.x : (c == 1 ? v.y : v.z); }

// Work queue of a wave whose quads hold ppw particles (slot s = quad % ppw):
// one atomic per wave, consecutive indices to the slots that ask.  All quads
// of a slot ask together (they run the same particle).
__device__ __forceinline__ uint32_t quad_acquire(uint32_t* queue, uint32_t ppw) {
    const uint64_t mask = __ballot(1);
    const uint64_t first = ppw >= 16 ? ~0ull : (1ull << (4 * ppw)) - 1ull;
    const uint64_t quads = mask & first & 0x1111111111111111ull;
    const int leader = __ffsll((unsigned long long)mask) - 1;
    const uint32_t lane = __lane_id();
    uint32_t base = 0;
    if ((int)lane == leader) base = atomicAdd(queue, (uint32_t)__popcll(quads));
    base = __shfl(base, leader);
    return base + (uint32_t)__popcll(quads & ((1ull << (4 * ((lane >> 2) % ppw))) - 1ull));
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
    X(a61) X(a64) X(a65) X(a71) X(a74) X(a75) X(a76) X(a81) X(a84) X(a85) X(a86) X(a87) X(a91) X(a94) X(a95) X(a96) X(a97) X(a98) X(a101) X(a104) X(a105) X(a106) X(a107)   \
    X(a108) X(a109) X(a111) X(a114) X(a115) X(a116) X(a117) X(a118) X(a119) X(a1110) X(a121) X(a124) X(a125)        \
    X(a126) X(a127) X(a128) X(a129) X(a1210) X(a1211) X(er1) X(er6) X(er7) X(er8) X(er9) X(er10) X(er11) X(er12)
#define ST_DOP_LITERAL(X) X(a21) X(a31) X(a32) X(a41) X(a43) X(a51) X(a53) X(a54)
#define ST_DOP_SCALAR(X)                                                                                            \
    X(c2) X(c3) X(c4) X(c5) X(c6) X(c7) X(c8) X(c9) X(c10) X(c11) X(b1) X(b6) X(b7) X(b8) X(b9) X(b10) X(b11)       \
    X(b12) X(bhh1) X(bhh2) X(bhh3)
// The stage coefficients in vector registers and the nodes and weights in
// scalar ones (a product takes one scalar-register operand).  The empty
// statements make each value opaque once per launch: the compiler would
// otherwise rebuild it from literals at each use, two scalar moves that cost
// as much as the product when the wave is alone on its SIMD.  (The first
// stages' eight stay literals: 256 registers hold no more.)
struct DopTab {
#define X(n) double n;
    ST_DOP_RESIDENT(X)
    ST_DOP_SCALAR(X)
    ST_DOP_LITERAL(X)
#undef X
};
__device__ __forceinline__ void dop_tab_load(DopTab& T) {
#define X(n) T.n = dop::n; asm volatile("" : "+v"(T.n));
    ST_DOP_RESIDENT(X)
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
    double x, xf, facold, k1;
    int32_t reject, last;
    uint32_t nstep;
};

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

// dop_trial_fast_t (st_integrators.h) on a quad.
//
// The trial is one chain: a stage's input, two quad moves, the cross product,
// and the update of the next stage's input with it, each waiting for the one
// before (an FP64 result is ready two issue slots after its instruction).
// The products of older stages and the next stage's field fill those slots:
// every stage sum is an accumulator that takes each K some stages before its
// turn, and ST_KEEP pins the order the statements are written in (left
// alone, the compiler, which schedules for registers here, issues each chain
// back to back: 7.3 cycles per instruction).
#define ST_KEEP __builtin_amdgcn_sched_barrier(0)
template <bool ADJ, bool PULSE>
__device__ __forceinline__ int q_trial_fast(const SimParams& P, const DopTab& T, QDop& D, double& y, double& h,
                                            double seg_t0, const QPoly& q, const QPulse& pl,
                                            uint32_t& nacc, uint32_t& nrej, QQuad* Q) {
#pragma clang fp contract(fast)
    if (D.nstep > P.nmax) return -1;
    if (D.x + 1.01 * h - D.xf > 0.0) {
        h = D.xf - D.x;
        D.last = 1;
    }
    if (h < P.hmin && D.last != 1) h = P.hmin;
    D.nstep++;
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
    // the stage fields: a stage's is formed in five steps while the stage
    // before it waits
    double wa, wb, na, nb, tau;
    auto pulse = [&](double p) {
        if constexpr (PULSE) {
            na = h * __builtin_fma(pl.ma, p, na);
            nb = h * __builtin_fma(pl.mb, p, nb);
        }
    };
#define QF1(C) tau = __builtin_fma((C), h, tx)
#define QF2 na = hq.a1 + tau * hq.a2
#define QF3 nb = hq.b1 + tau * hq.b2
#define QF4 na = hq.a0 + tau * na
#define QF5(LANE, HP) nb = hq.b0 + tau * nb; pulse(q_all<LANE>(HP))
#define QFMA(S, A, K) S = __builtin_fma(T.A, K, S)
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
    QF1(T.c2); QF2; QF3; QF4; QF5(0, hp0);
    quad(T.b1, tx, y);
    double ya, yb, t, yy = __builtin_fma(T.a21, K1, y);
    double s3, s4, s5, s6, s7, s8, s9, s10, s11, s12, bs, er;
    // one stage: moves | A | product | B | K | C | next input | D
#define QSTAGE(N, A, B, C, CRIT, DD)                              \
    wa = na; wb = nb;                                             \
    ya = q_next1(yy); yb = q_next2(yy); ST_KEEP;                  \
    A; ST_KEEP;                                                   \
    t = yb * wa; ST_KEEP;                                         \
    B; ST_KEEP;                                                   \
    const double K##N = __builtin_fma(ya, wb, -t); ST_KEEP;       \
    C; ST_KEEP;                                                   \
    CRIT; ST_KEEP;                                                \
    DD; ST_KEEP
    QSTAGE(2, s3 = __builtin_fma(T.a31, K1, y); QF1(T.c3), QF2; s4 = __builtin_fma(T.a41, K1, y), QF3; QF4,
           yy = __builtin_fma(T.a32, K2, s3), QF5(1, hp0); s5 = __builtin_fma(T.a51, K1, y);
           s6 = __builtin_fma(T.a61, K1, y));
    QSTAGE(3, QF1(T.c4); s7 = __builtin_fma(T.a71, K1, y), QF2; QF3, QF4; s8 = __builtin_fma(T.a81, K1, y),
           yy = __builtin_fma(T.a43, K3, s4), QF5(2, hp0); QFMA(s5, a53, K3); s9 = __builtin_fma(T.a91, K1, y));
    QSTAGE(4, QF1(T.c5); s10 = __builtin_fma(T.a101, K1, y), QF2; QF3, QF4; s11 = __builtin_fma(T.a111, K1, y),
           yy = __builtin_fma(T.a54, K4, s5), QF5(3, hp0); QFMA(s6, a64, K4); QFMA(s7, a74, K4));
    QSTAGE(5, QF1(T.c6); QFMA(s8, a84, K4), QF2; QF3, QF4; QFMA(s9, a94, K4),
           yy = __builtin_fma(T.a65, K5, s6), QF5(0, hp1); QFMA(s7, a75, K5); QFMA(s8, a85, K5));
    quad(T.b6, __builtin_fma(T.c6, h, tx), yy);
    QSTAGE(6, QF1(T.c7); QFMA(s9, a95, K5), QF2; QF3, QF4; QFMA(s10, a104, K4),
           yy = __builtin_fma(T.a76, K6, s7), QF5(1, hp1); QFMA(s8, a86, K6); QFMA(s9, a96, K6));
    quad(T.b7, __builtin_fma(T.c7, h, tx), yy);
    QSTAGE(7, QF1(T.c8); QFMA(s10, a105, K5), QF2; QF3, QF4; QFMA(s10, a106, K6),
           yy = __builtin_fma(T.a87, K7, s8), QF5(2, hp1); QFMA(s9, a97, K7); QFMA(s11, a114, K4));
    quad(T.b8, __builtin_fma(T.c8, h, tx), yy);
    QSTAGE(8, QF1(T.c9); QFMA(s10, a107, K7), QF2; QF3; QFMA(s11, a115, K5), QF4; s12 = __builtin_fma(T.a121, K1, y),
           yy = __builtin_fma(T.a98, K8, s9), QF5(3, hp1); QFMA(s10, a108, K8); QFMA(s11, a116, K6));
    quad(T.b9, __builtin_fma(T.c9, h, tx), yy);
    QSTAGE(9, QF1(T.c10); QFMA(s11, a117, K7), QF2; QF3; QFMA(s12, a124, K4), QF4; bs = T.b1 * K1; er = T.er1 * K1,
           yy = __builtin_fma(T.a109, K9, s10), QF5(0, hp2); QFMA(s11, a118, K8); QFMA(s12, a125, K5));
    quad(T.b10, __builtin_fma(T.c10, h, tx), yy);
    QSTAGE(10, QF1(T.c11); QFMA(s11, a119, K9), QF2; QF3; QFMA(s12, a126, K6), QF4; QFMA(bs, b6, K6); QFMA(er, er6, K6),
           yy = __builtin_fma(T.a1110, K10, s11), QF5(1, hp2); QFMA(s12, a127, K7); QFMA(bs, b7, K7));
    quad(T.b11, __builtin_fma(T.c11, h, tx), yy);
    QSTAGE(11, tau = tx + h; QFMA(s12, a128, K8), QF2; QF3; QFMA(s12, a129, K9), QF4; QFMA(s12, a1210, K10),
           yy = __builtin_fma(T.a1211, K11, s12), QF5(2, hp2); QFMA(er, er7, K7); QFMA(bs, b8, K8));
    quad(T.b12, tx + h, yy);
    QSTAGE(12, QFMA(er, er8, K8); QFMA(bs, b9, K9), QFMA(er, er9, K9); QFMA(bs, b10, K10),
           QFMA(er, er10, K10); QFMA(bs, b11, K11), QFMA(bs, b12, K12), QFMA(er, er11, K11); QFMA(er, er12, K12));
#undef QSTAGE
#undef QF1
#undef QF2
#undef QF3
#undef QF4
#undef QF5
    const double xph = x + h;
    const double y1 = y + bs;
    double e = __builtin_fma(-T.bhh1, K1, bs);
    // the derivative at the new point (used when the trial is accepted),
    // formed while the error norm's chain waits
    const double c12 = PULSE ? q_all<2>(hp2) : 0.0;
    q_field(tx + h, q, na, nb);
    if constexpr (PULSE) {
        na = __builtin_fma(pl.ma, c12, na);
        nb = __builtin_fma(pl.mb, c12, nb);
    }
    const double is = fast_rcp(P.atol + P.rtol * __builtin_fmax(fabs(y), fabs(y1)));
    e = __builtin_fma(-T.bhh2, K9, e);
    e = __builtin_fma(-T.bhh3, K12, e);
    const double k1n = q_cross(y1, na, nb);
    const d3 v2 = q_vec(e * is), v1 = q_vec(er * is);
    const double err2 = __builtin_fma(v2.z, v2.z, __builtin_fma(v2.y, v2.y, v2.x * v2.x));
    const double e1 = __builtin_fma(v1.z, v1.z, __builtin_fma(v1.y, v1.y, v1.x * v1.x));
#undef QFMA
    const double deno = e1 + 0.01 * err2;
    const double err = (deno <= 0.0) ? 0.0 : e1 * fast_rsq(3.0 * deno);
    double grow, shrink;
    dop_factors(P, err, D.facold, grow, shrink);
    double hnew = h * grow;
    if (err <= 1.0 || P.fixed) {
        D.facold = max_d(err, 1.0E-4);
        nacc++;
        D.k1 = k1n;
        if constexpr (ADJ) {
            Q->n0 = Q->n0 + h * q0;
            Q->n1 = Q->n1 + h * q1;
            Q->n2 = Q->n2 + h * q2;
        }
        y = y1;
        D.x = xph;
        if (D.last) return 1;
        if (fabs(hnew) > P.hmax) hnew = P.hmax;
        if (D.reject) hnew = min_d(fabs(hnew), fabs(h));
        D.reject = 0;
    } else {
        nrej++;
        hnew = h * shrink;
        D.reject = 1;
        D.last = 0;
    }
    if (!P.fixed) h = hnew;
    return 0;
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
template <bool BATCH, bool PULSE>
__device__ __forceinline__ void quad_spin_fast() {
    auto args = []() -> const QuadArgs& { return kernel_args<QuadArgs>(); };
    const uint32_t lane = __lane_id();
    const uint32_t c = (lane & 3u) == 3u ? 0u : (lane & 3u);   // lane 3 repeats lane 0
    const uint32_t ppw = args().ppw;
    const bool first = (lane >> 2) < ppw;
    const bool lead = first && (lane & 3u) == 0u, owner = first && (lane & 3u) != 3u;
    DopTab T;
    dop_tab_load(T);
    // a plain handle's physics in LDS, one copy per workgroup
    __shared__ Phys shared_phys;
    if constexpr (!BATCH) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(args().A.phys);
        for (uint32_t i = threadIdx.x; i < sizeof(Phys) / 4; i += blockDim.x) reinterpret_cast<uint32_t*>(&shared_phys)[i] = src[i];
        __syncthreads();
    }
    QPulse pl;
    if constexpr (PULSE && !BATCH) q_pulse_load(pl, shared_phys, c);
    SpinLane L;      // (S unused: the lane's component is y)
    double y = 0.0;
    QDop dop;
    QPoly q;
    double seg_t0 = 0.0;
    SegRec nxt;      // record L.j, loaded while record L.j - 1 is integrated
    uint32_t cur_flags = 0;
    uint32_t cnt[4] = {0, 0, 0, 0};   // accepted, rejected, segments, trips (of this launch)
    enum { S_DONE = 0, S_NEXT = 1, S_INT = 2 };
    int phase = S_DONE;
    const uint32_t n_list = list_len(args().A);
    auto take = [&]() {
        const PipeArgs& A = args().A;
        const DevState& D = args().D;
        const uint32_t i = quad_acquire(A.R.queue, ppw);
        if (i >= n_list) return;
        spin_load<BATCH>(D, A, A.list[i], L);
        y = q_pick(L.S, c);
        if constexpr (PULSE && BATCH) q_pulse_load(pl, A.phys[L.cfg], c);
        if (L.nrec > 0) nxt = load_rec(rec_at_seq(A, L.pid, 0, L.page));
        phase = S_NEXT;
    };
    take();
    while (phase != S_DONE) {
        if (lead) ++cnt[3];
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
                if ((rec.flags & R_INTEGRATE) && !L.stopped) {
                    seg_t0 = L.t_spin;
                    q_make_poly(q, BATCH ? A.phys[L.cfg] : shared_phys, d3{rec.px, rec.py, rec.pz}, d3{rec.vx, rec.vy, rec.vz}, c);
                    dop.x = seg_t0;
                    dop.xf = rec.t;
                    dop.facold = 1.0E-4;
                    dop.last = 0;
                    dop.reject = 0;
                    dop.nstep = 0;
                    double wa = q.a0, wb = q.b0;
                    if constexpr (PULSE) {
                        const double cosv = pl.on ? phase_cos(pl.pw * seg_t0) : 0.0;
                        wa = __builtin_fma(pl.ma, cosv, wa);
                        wb = __builtin_fma(pl.mb, cosv, wb);
                    }
                    dop.k1 = q_cross(y, wa, wb);
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
            const int st = q_trial_fast<false, PULSE>(args().P, T, dop, y, L.tempH, seg_t0, q, pl, L.acc, L.rej, nullptr);
            if (st != 0) {
                const PipeArgs& A = args().A;
                const RunArgs& R = A.R;
                if (R.trace && L.pid == R.trace_pid) {
                    const d3 S = q_vec(y);
                    if (lead)
                        ST_TRACE(R, 2, L.t_spin, dop.xf, d3{0, 0, 0}, d3{0, 0, 0}, S, L.tempH, L.acc, L.rej,
                                 (char)(cur_flags >> 8), (char)(cur_flags >> 16), st, 0, 0);
                }
                if (args().P.keep) L.h = L.tempH;
                L.t_spin = dop.xf;
                if (st < 0) {
                    if (lead) {
                        const uint32_t slot = atomicAdd(A.fail_count, 1u);
                        if (slot < A.fail_cap) {
                            A.fail_list[3 * slot + 0] = L.pid;
                            A.fail_list[3 * slot + 1] = L.j;
                            A.fail_list[3 * slot + 2] = (uint32_t)st;
                        }
                    }
                    L.stopped = true;
                }
                if (L.stopped || (cur_flags & R_STOP)) y = __builtin_nan("");
                if ((cur_flags & R_IEND) || st < 0) {
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

template <bool BATCH, bool PULSE>
__global__ __launch_bounds__(256, 2) void k_spin_quad(const QuadArgs) {
    quad_spin_fast<BATCH, PULSE>();
}

}  // namespace st
