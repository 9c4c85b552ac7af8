// st_adjoint.h -- adjoint (reverse-mode) Bloch integration along recorded
// trajectories.
//
// The forward spin obeys S' = S x omega(t), omega = gamma*(B0 + G.r +
// (1/c^2) v x E + pulse).  For a loss L that depends on the spins at the
// output times through the ensemble means, L = l(<S>(t_1), ..., <S>(t_K)),
// the adjoint lambda of one particle obeys the same equation backwards,
// lambda' = lambda x omega, and jumps by g_k = dl/d<S>(t_k) at every output
// time.  Both lambda and S are transported by the same rotation, so
// u = lambda x S obeys u' = u x omega as well, and
//
//   dL/dtheta = (1/N) sum_particles int u . (d omega / d theta) dt,
//
// with jumps u(t_k-) = u(t_k+) + g_k x S(t_k).  Only u (3 components) is
// integrated, backwards over every segment, with the DOP853 controller; the
// gradient integrals ride along as a quadrature.  omega is linear in
// theta = (G, E, B0):
//   dL/dG_ij = gamma int u_i r_j dt,  dL/dE = gamma/c^2 int u x v dt,
//   dL/dB0 = gamma int u dt,
// and along one segment r and v are polynomials in tau = t - t0, so the
// kernel only accumulates the moments int u tau^n dt (n = 0, 1, 2) per
// segment and folds them with the segment's p0, v0 and gravity.
//
// The trajectory is recomputed, not stored: the forward pipeline keeps the
// kinematic state at every chunk start (every C segments of each particle);
// the backward pass replays one chunk's kinematics (k_kin, bit-identical
// records) and integrates that chunk's records in reverse.
#pragma once

#include "st_pipeline.h"

namespace st {

// per-particle adjoint state, one 8-byte array per field (same layout rule
// as DevState)
enum AdjField : int {
    A_UX, A_UY, A_UZ,   // u = lambda x S at the current backward time
    A_H,                // carried step size
    A_K,                // interval index of the next output time going backwards
    A_FAIL,             // nonzero: a backward segment failed (integrator status)
    A_G0,               // 15 accumulators: int u_i r_j dt (9, row-major i, j),
                        // int u x v dt (3), int u dt (3)
    A_COUNT = A_G0 + 15
};
constexpr int N_GRAD = 15;

struct AdjArgs {
    const char* recs;        // records of the replayed chunk
    uint32_t C;
    const uint32_t* list;    // particles of the chunk
    uint32_t n_list;
    const uint32_t* seg_count;
    DevState ck;             // kinematic state at the chunk start (checkpoint)
    DevState adj;            // adjoint state
    const char* blocks;      // forward snapshot blocks (S at the output times)
    uint64_t block_bytes;
    uint32_t n;              // particles per block
    const double* seeds;     // g_k, 3 per output time (per configuration for batches)
    uint32_t n_targets;
    const Phys* phys;        // batched handles
    uint32_t* queue;         // work-queue head (zero at the launch)
};

__global__ __launch_bounds__(256) void k_adj_begin(const DevState A, uint32_t n, int32_t k_last, double h0) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t o = i * 8u;
    A.st(A_UX, o, 0.0); A.st(A_UY, o, 0.0); A.st(A_UZ, o, 0.0);
    A.st(A_H, o, h0);
    A.st<int64_t>(A_K, o, k_last);
    A.st<int64_t>(A_FAIL, o, 0);
    for (int f = 0; f < N_GRAD; ++f) A.st(A_G0 + f, o, 0.0);
}

// Moments of one component over a segment of length Ts: int u tau^n dt,
// n = 0, 1, 2, from the quadrature's s-moments (tau = Ts - s).
struct AdjMoments {
    double m0, m1, m2;
};
__device__ __forceinline__ AdjMoments adj_moments(double Ts, double n0, double n1, double n2) {
    return AdjMoments{n0, __builtin_fma(Ts, n0, -n1), __builtin_fma(Ts, __builtin_fma(Ts, n0, -(2.0 * n1)), n2)};
}
// int u r_j dt with r_j = p + v tau + (1/2) a tau^2 (ha = a/2)
__device__ __forceinline__ double adj_ur(const AdjMoments& M, double p, double v, double ha) {
    return __builtin_fma(ha, M.m2, __builtin_fma(v, M.m1, p * M.m0));
}

// One particle's walk back through its records, one trial step or one record
// change per loop trip: the loop of spin_body (st_pipeline.h) in reverse.  A
// lane that finishes a particle takes the next one from the queue.  (With the
// trials of a segment in a loop of their own, every lane of a wave waited at
// each record for the lane with the longest segment: 44.4 ms against 12.5 ms
// of the forward spin kernel on 8,192 neutrons x 2 s.)
// PULSE = false: the fast trial's pulse-free form (runs without a pulse term)
template <bool BATCH, bool PULSE>
__global__ __launch_bounds__(256) void k_adj(const SimParams P, const DevState D, const AdjArgs A) {
#pragma clang fp contract(fast)
    const double ay = P.gravity ? G_CONST : 0.0;
    uint32_t pid = 0, o = 0;
    d3 u{0.0, 0.0, 0.0};
    double h = 0.0, t_chunk0 = 0.0;
    int64_t kb = 0, fail = 0;
    int32_t j = -1;
    SegRec rec;
    Seg sb;
    Poly qb;
    AdjQuad Q;
    DopState dop;
    uint32_t nacc = 0, nrej = 0;
    enum { S_DONE = 0, S_NEXT = 1, S_INT = 2 };
    int phase = S_DONE;
    auto take = [&]() {
        const uint32_t i = acquire_index(A.queue);
        if (i >= A.n_list) return;
        pid = A.list[i];
        o = pid * 8u;
        u = d3{A.adj.ld(A_UX, o), A.adj.ld(A_UY, o), A.adj.ld(A_UZ, o)};
        h = A.adj.ld(A_H, o);
        kb = A.adj.ld<int64_t>(A_K, o);
        fail = A.adj.ld<int64_t>(A_FAIL, o);
        j = (int32_t)A.seg_count[pid] - 1;
        t_chunk0 = A.ck.ld(F_T, o);
        phase = S_NEXT;
    };
    take();
    while (phase != S_DONE) {
        while (phase == S_NEXT) {
            if (j < 0) {
                A.adj.st(A_UX, o, u.x); A.adj.st(A_UY, o, u.y); A.adj.st(A_UZ, o, u.z);
                A.adj.st(A_H, o, h);
                A.adj.st<int64_t>(A_K, o, kb);
                A.adj.st<int64_t>(A_FAIL, o, fail);
                phase = S_DONE;
                take();
                continue;
            }
            const Phys& F = lane_phys<BATCH>(P, D, A.phys, pid);
            rec = get_rec(A.recs, A.C, pid, (uint32_t)j);
            if ((rec.flags & R_IEND) && kb >= 0) {
                // the output time t_k closes this record: u += g_k x S(t_k)
                const double* Sk = reinterpret_cast<const double*>(A.blocks + (uint64_t)kb * A.block_bytes + 56ull * A.n) +
                                   3ull * pid;
                const uint64_t cfg = BATCH ? D.ld<uint64_t>(F_CFG, o) : 0;
                const double* gp = A.seeds + 3 * (cfg * A.n_targets + (uint64_t)kb);
                const d3 gS = cross3_fma(d3{gp[0], gp[1], gp[2]}, d3{Sk[0], Sk[1], Sk[2]});
                u = d3{u.x + gS.x, u.y + gS.y, u.z + gS.z};
                --kb;
                // a non-finite spin (a particle that failed forward) cannot be
                // integrated: flag it instead of running the controller on NaN
                if (!(__builtin_isfinite(u.x) && __builtin_isfinite(u.y) && __builtin_isfinite(u.z))) fail = -3;
            }
            const double t0 = (j > 0) ? get_rec(A.recs, A.C, pid, (uint32_t)(j - 1)).t : t_chunk0;
            const double Ts = rec.t - t0;
            if (!(rec.flags & R_INTEGRATE) || fail || !(Ts > 0.0)) {
                --j;
                continue;
            }
            sb.t0 = 0.0;
            sb.p0 = d3{rec.px, rec.py, rec.pz};
            sb.v0 = d3{rec.vx, rec.vy, rec.vz};
            // omega along the segment in tau = t - t0, then the backward field
            // -omega(t_end - s) as a polynomial in s
            const Poly q = make_poly(P, F, sb);
            qb.w0 = d3{-(q.w0.x + Ts * (q.w1.x + Ts * q.w2.x)), -(q.w0.y + Ts * (q.w1.y + Ts * q.w2.y)),
                       -(q.w0.z + Ts * (q.w1.z + Ts * q.w2.z))};
            qb.w1 = d3{q.w1.x + 2.0 * Ts * q.w2.x, q.w1.y + 2.0 * Ts * q.w2.y, q.w1.z + 2.0 * Ts * q.w2.z};
            qb.w2 = d3{-q.w2.x, -q.w2.y, -q.w2.z};
            qb.pag = q.pag;
            qb.pw = q.pw;
            qb.paxis = q.paxis;
            qb.pon = q.pon;
            Q.n0 = Q.n1 = Q.n2 = d3{0.0, 0.0, 0.0};
            Q.t_end = rec.t;
            dop.x = 0.0;
            dop.xf = Ts;
            dop.facold = 1.0E-4;
            dop.posneg = 1.0;
            dop.last = 0;
            dop.reject = 0;
            dop.nstep = 0;
            dop.k1 = poly_rhs<PULSE>(0.0, u, qb, -qb.pag, PULSE && qb.pon ? phase_cos(qb.pw * rec.t) : 0.0);
            phase = S_INT;
        }
        if (phase == S_INT) {
            const int st = dop_trial_fast_t<true, PULSE>(P, lane_phys<BATCH>(P, D, A.phys, pid), dop, u, h, sb, qb, nacc,
                                                         nrej, &Q);
            if (st < 0) {
                fail = st;
                --j;
                phase = S_NEXT;
            } else if (st > 0) {
                const double Ts = dop.xf;
                const AdjMoments mx = adj_moments(Ts, Q.n0.x, Q.n1.x, Q.n2.x), my = adj_moments(Ts, Q.n0.y, Q.n1.y, Q.n2.y),
                                 mz = adj_moments(Ts, Q.n0.z, Q.n1.z, Q.n2.z);
                // the segment's contributions (accumulated in HBM: a segment
                // spans tens of steps, and 15 sums held in registers would
                // halve the occupancy)
                double dg[N_GRAD];
                const AdjMoments Mi[3] = {mx, my, mz};
                const double p[3] = {sb.p0.x, sb.p0.y, sb.p0.z}, v[3] = {sb.v0.x, sb.v0.y, sb.v0.z};
#pragma unroll
                for (int i = 0; i < 3; ++i) {
#pragma unroll
                    for (int jj = 0; jj < 3; ++jj) dg[3 * i + jj] = adj_ur(Mi[i], p[jj], v[jj], jj == 1 ? 0.5 * ay : 0.0);
                }
                // int u x v dt with v = v0 + a tau, a = (0, ay, 0)
                const d3 uv = cross3_fma(d3{mx.m0, my.m0, mz.m0}, sb.v0);
                dg[9] = __builtin_fma(mz.m1, -ay, uv.x);
                dg[10] = uv.y;
                dg[11] = __builtin_fma(mx.m1, ay, uv.z);
                dg[12] = mx.m0;
                dg[13] = my.m0;
                dg[14] = mz.m0;
#pragma unroll
                for (int f = 0; f < N_GRAD; ++f) A.adj.st(A_G0 + f, o, A.adj.ld(A_G0 + f, o) + dg[f]);
                --j;
                phase = S_NEXT;
            }
        }
    }
}

// Per-block partial sums of the 15 accumulators (deterministic order; the
// host adds the partials in block order).  Batched handles sum per
// configuration: partial[(block * n_cfg + cfg) * 15 + f] -- blocks never
// straddle configurations because the grid is laid out per configuration.
__global__ __launch_bounds__(256) void k_adj_partials(const DevState A, const uint32_t* cfg_off, uint32_t blocks_per_cfg,
                                                      double* partial) {
    const uint32_t cfg = blockIdx.y;
    const uint32_t lo = cfg_off[cfg], hi = cfg_off[cfg + 1];
    __shared__ double red[256];
    double acc[N_GRAD];
#pragma unroll
    for (int f = 0; f < N_GRAD; ++f) acc[f] = 0.0;
    for (uint32_t i = lo + blockIdx.x * 256 + threadIdx.x; i < hi; i += blocks_per_cfg * 256) {
#pragma unroll
        for (int f = 0; f < N_GRAD; ++f) acc[f] += A.ld(A_G0 + f, i * 8u);
    }
    for (int f = 0; f < N_GRAD; ++f) {
        red[threadIdx.x] = acc[f];
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
            __syncthreads();
        }
        if (threadIdx.x == 0) partial[((uint64_t)cfg * blocks_per_cfg + blockIdx.x) * N_GRAD + f] = red[0];
        __syncthreads();
    }
}

}  // namespace st
