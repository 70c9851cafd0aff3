// Reduced camera system: unknown-level assembly and Jacobi-preconditioned CG on the device.
//
// Restates the reference's _solve_CG / _pcg (src/blast3r/inference/ba_solver.py:184-206,
// :1197-1238) on the explicit image-pair blocks produced by ba_linearize_schur:
//   S_u = P^T S_img P + diag(damping),  M = clamp(diag(A), 1e-12),
// where P maps image-level parameters [foc(cam) | tau(node) | zcf(img)] to the
// reference's unknown order [foc | tau | zcf] (ba_solver.py:119).  The CG
// iteration, its stopping test, the clamps and the best-so-far return follow
// _pcg line by line; scalars stay on the device (no host synchronisation).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include <cmath>

#include "ba_common.h"
#include "ba_error.h"

namespace ba {

#define PCG_T 256
// threads of the image-row SpMV: 8 groups of 16 lanes.  Two waves per row keep every row of a
// 1024-image system resident at once (the kernel needs ~112 VGPRs: 4 waves per SIMD).
#define PCG_ST 128
// Block partials of the update launch (nb blocks): r.r and r.z, PCG_NP per block.
#define PCG_NP 2
#define PCG_LF 16           // entries of a long inverse list each lane has in flight
#define PCG_IPF 4           // image partials of p.Ap each update thread requests at launch
enum { PT_RR = 0, PT_RZ = 1 };

// state (working precision): ST_RZ0/1 r.z after n updates and ST_BEST0/1 the best residual norm after n updates,
// both in slot n & 1; ST_BETA the beta of the current direction; ST_LEAF.. the camera-leaf damping.
// ST_LEAFMAX.. (3 words): the per-leaf maxima of |diag(A)| as bit patterns, accumulated by k_leaf_max.
enum { ST_BNORM = 0, ST_RZ0 = 1, ST_RZ1 = 2, ST_BEST0 = 3, ST_BEST1 = 4, ST_BETA = 5, ST_LEAF = 8, ST_LEAFMAX = 11 };
// istate: IS_DONE0 / IS_DONE1 "stopped before update n" in slot n & 1, IS_K iterations run,
// IS_CONV converged, IS_BESTK best iterate, IS_USEBEST the best iterate is returned.
enum { IS_DONE0 = 0, IS_DONE1 = 1, IS_K = 2, IS_CONV = 3, IS_BESTK = 4, IS_USEBEST = 5 };

// The arrays of ba_pcg_args in the working precision Real (double, or float when real32 is set).
template <typename Real>
struct PcgV {
    const Real *S_pairs, *e_img, *dg_img;
    Real *rhs, *diagA, *damp, *x, *xbest, *r, *z, *p, *y_img, *partials, *state, *S_rows, *img_part;
    __device__ __forceinline__ explicit PcgV(const ba_pcg_args& a)
        : S_pairs((const Real*)a.S_pairs), e_img((const Real*)a.e_img), dg_img((const Real*)a.dg_img),
          rhs((Real*)a.rhs), diagA((Real*)a.diagA), damp((Real*)a.damp), x((Real*)a.x), xbest((Real*)a.xbest),
          r((Real*)a.r), z((Real*)a.z), p((Real*)a.p), y_img((Real*)a.y_img), partials((Real*)a.partials),
          state((Real*)a.state), S_rows((Real*)a.S_rows), img_part((Real*)a.img_part) {}
};

// search direction of update n: p_n = z_n + beta_n p_{n-1} (ba_solver.py:1235), written as one
// fused multiply-add so that every kernel that forms it gets the same bits
template <typename Real>
__device__ __forceinline__ Real pdir(Real z, Real pold, Real beta) { return fma(beta, pold, z); }

// Sum over the 64 lanes of a wave; every lane gets the same bits (each butterfly step adds the
// same two values in either lane, and fp addition commutes).
template <typename Real>
__device__ __forceinline__ Real wave_sum(Real v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Sum over a block of NT threads in a fixed order (waves by butterfly, then the wave sums in wave
// order); every thread gets the result.  sh holds at least NT / 64 doubles.
template <int NT, typename Real>
__device__ __forceinline__ Real block_sum(Real v, Real* sh) {
    v = wave_sum(v);
    __syncthreads();                                  // sh may still be read by a previous call
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    Real t = Real(0);
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) t += sh[k];
    return t;
}

// K block sums at once with two barriers; v[k] becomes the sum of every thread's v[k], in the
// same order as block_sum.  sh holds at least K * NT / 64 doubles.
template <int NT, int K, typename Real>
__device__ __forceinline__ void block_sums(Real (&v)[K], Real* sh) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) sh[k * (NT / 64) + (threadIdx.x >> 6)] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        Real t = Real(0);
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) t += sh[k * (NT / 64) + w];
        v[k] = t;
    }
}

// Sums of r.r and r.z over the nb block partials (deterministic, identical in every block of NT
// threads); sh holds at least 2 * NT / 64 doubles.
template <int NT, typename Real>
__device__ __forceinline__ void sum_partials(const Real* __restrict__ part, int nb, Real (&rs)[2], Real* sh) {
    rs[0] = Real(0); rs[1] = Real(0);
    for (int b = threadIdx.x; b < nb; b += NT) { rs[0] += part[PCG_NP * b + PT_RR]; rs[1] += part[PCG_NP * b + PT_RZ]; }
    block_sums<NT, 2>(rs, sh);
}

// unknown-level rhs and diag(H_cc) from the image-level vectors; one wave per unknown so that
// shared unknowns (one focal pair for every image of a camera) reduce in parallel
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_unk_setup(ba_pcg_args a) {
    const PcgV<Real> av(a);
    const int lane = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x < 3)                  // k_leaf_max's accumulators
        av.state[ST_LEAFMAX + threadIdx.x] = Real(0);
    int64_t u = (int64_t)blockIdx.x * (PCG_T / 64) + (threadIdx.x >> 6);
    if (u >= a.n_u) return;
    Real e = Real(0), g = Real(0);
    for (int q = a.inv_ptr[u] + lane; q < a.inv_ptr[u + 1]; q += 64) {
        int src = a.inv_src[q];
        e += av.e_img[src];
        g += av.dg_img[src];
    }
    for (int off = 32; off > 0; off >>= 1) {
        e += __shfl_down(e, off);
        g += __shfl_down(g, off);
    }
    if (lane == 0) { av.rhs[u] = e; av.diagA[u] = g; }
}

// per-leaf damping (BlockDiagMat.dampen_, ba_solver.py:575-582) and the Jacobi preconditioner.
// leaf ids 0..2 = foc, tau, zcf; 3..5 = the same groups switched off (a zero matrix damped by
// dampen * I, ZerosMat.dampen_, ba_solver.py:510-517).
// Two launches over every block of unknowns: the per-leaf maxima (fmax within a block; across blocks
// an integer max of the bit patterns, which orders non-negative doubles as their values, so the
// result does not depend on the order; a block whose maximum is NaN contributes nothing, as fmax
// ignores NaN), then the damping and the clamped preconditioner diagonal per unknown.
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_leaf_max(ba_pcg_args a) {
    const PcgV<Real> av(a);
    __shared__ Real sh[3][PCG_T];
    Real m[3] = {Real(0), Real(0), Real(0)};
    for (int64_t u = (int64_t)blockIdx.x * PCG_T + threadIdx.x; u < a.n_u; u += (int64_t)gridDim.x * PCG_T) {
        const int l = a.leaf[u];
        if (l < 3) m[l] = fmax(m[l], fabs(av.diagA[u]));
    }
#pragma unroll
    for (int l = 0; l < 3; ++l) sh[l][threadIdx.x] = m[l];
    __syncthreads();
    for (int w = PCG_T / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
#pragma unroll
            for (int l = 0; l < 3; ++l) sh[l][threadIdx.x] = fmax(sh[l][threadIdx.x], sh[l][threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x < 3) {
        const Real mv = sh[threadIdx.x][0];
        if (!isnan(mv)) atomic_max_nonneg(av.state + ST_LEAFMAX + threadIdx.x, mv);
    }
}

template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_leaf_damp(ba_pcg_args a) {
    const PcgV<Real> av(a);
    Real lam[6];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const Real mx = av.state[ST_LEAFMAX + l];        // the bits k_leaf_max combined are the value's
        lam[l] = a.adaptive ? Real(a.dampen) * mx : Real(a.dampen);
        lam[l + 3] = Real(a.dampen);
    }
    for (int64_t u = (int64_t)blockIdx.x * PCG_T + threadIdx.x; u < a.n_u; u += (int64_t)gridDim.x * PCG_T) {
        Real dmp = lam[a.leaf[u]];
        av.damp[u] = dmp;
        Real dA = av.diagA[u] + dmp;
        av.diagA[u] = dA > Real(1e-12) ? dA : Real(1e-12);          // diagA.clamp(min=1e-12) (ba_solver.py:191-192)
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        for (int l = 0; l < 3; ++l) av.state[ST_LEAF + l] = lam[l];
    }
}

// x = 0, r = b, z = M^-1 r, p_{-1} = 0 (so that p_0 = z_0); partials of b.b and r.z
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_init(ba_pcg_args a) {
    const PcgV<Real> av(a);
    __shared__ Real sh[PCG_T];
    int64_t u = (int64_t)blockIdx.x * PCG_T + threadIdx.x;
    Real t[2] = {Real(0), Real(0)};
    if (u < a.n_u) {
        Real b = av.rhs[u];
        Real z = b / av.diagA[u];
        av.x[u] = Real(0); av.xbest[u] = Real(0); av.r[u] = b; av.z[u] = z; av.p[a.n_u + u] = Real(0);
        t[0] = b * b; t[1] = b * z;
    }
    block_sums<PCG_T, 2>(t, sh);
    if (threadIdx.x == 0) { av.partials[PCG_NP * blockIdx.x + PT_RR] = t[0]; av.partials[PCG_NP * blockIdx.x + PT_RZ] = t[1]; }
}

template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_init2(ba_pcg_args a, int nb) {
    const PcgV<Real> av(a);
    __shared__ Real sh[PCG_T];
    Real rs[2];
    sum_partials<PCG_T>(av.partials, nb, rs, sh);
    const Real bb = rs[0], rz = rs[1];
    if (threadIdx.x == 0) {
        Real bn = sqrt(bb);
        av.state[ST_BNORM] = bn > Real(1e-12) ? bn : Real(1e-12);    // torch.norm(b).clamp(min=1e-12)
        av.state[ST_RZ0] = rz;
        av.state[ST_BEST0] = INFINITY; av.state[ST_BEST1] = INFINITY;
        av.state[ST_BETA] = Real(0);
        a.istate[IS_DONE0] = a.maxiter <= 0; a.istate[IS_DONE1] = 0; a.istate[IS_K] = 0; a.istate[IS_CONV] = 0;
        a.istate[IS_BESTK] = 0;
        a.istate[IS_USEBEST] = 1;
        a.istate[6] = 0;                                       // set by a resident solve that gave up
    }
}

// Image-row copies of the pair blocks, column-major: entry q of image row i (pair p, flag tr) holds
// B = S(i, i2) with B[j][j2] at S_rows[q][j2 * d + j], so that the SpMV's lanes (one per output
// row j) read each column of a block contiguously.  S(i, i2) is S_p for tr = 0 and S_p^T for tr = 1.
// row_u[q][j2] = umap[i2][j2] (-1 past d, gw entries per block: 16 for d <= 16, else 32): the unknowns
// the block multiplies.  One wave per destination entry (its d^2 elements and gw unknowns over the
// lanes), so that the entry's indices are resolved once per wave.
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_rows_build(ba_pcg_args a, int64_t n_ent, int gw) {
    const PcgV<Real> av(a);
    const int d = a.d, dd = d * d;
    const int64_t q = (int64_t)blockIdx.x * (PCG_T / 64) + (threadIdx.x >> 6);      // destination block
    if (q >= n_ent) return;
    const int lane = threadIdx.x & 63;
    int64_t qs = q;                                    // its source entry of row_ent
    if (a.row_cap > 0) {                               // fixed capacity: row i at [i cap, (i + 1) cap)
        const int64_t i = q / a.row_cap, k = q - i * a.row_cap;
        qs = a.row_ptr[i] + k;
        if (qs >= a.row_ptr[i + 1]) {                  // past the row's end: a zero block, no unknowns
            for (int e = lane; e < dd; e += 64) av.S_rows[q * dd + e] = Real(0);
            if (lane < gw) a.row_u[q * gw + lane] = -1;
            return;
        }
    }
    const int ent = a.row_ent[qs];
    const int64_t p = ent >> 1;
    const Real* S = av.S_pairs + p * dd;
    for (int e = lane; e < dd; e += 64) {
        const int j2 = e / d, j = e - j2 * d;
        av.S_rows[q * dd + e] = (ent & 1) ? S[j2 * d + j] : S[j * d + j2];
    }
    if (lane < gw) {
        const int i2 = (ent & 1) ? a.pair_i1[p] : a.pair_i2[p];
        a.row_u[q * gw + lane] = lane < d ? a.umap[(int64_t)i2 * d + lane] : -1;
    }
}

// ----------------------------------------------------------------------------- one CG iteration
// Iteration n (n = 0 .. maxiter - 1; the reference numbers it n + 1, ba_solver.py:1216-1236) is two
// launches:
//   k_pcg_spmv(n)    the stopping decisions after update n - 1 (every block forms them from the same
//                    partial sums, so they agree without a grid barrier), the best-so-far copy, then
//                    y_img = S_img p_n with p_n formed on the fly from z and p_{n-1}, and per image
//                    row i a partial of p.Ap = sum_e p_u(e) y_e + sum_u damp_u p_u^2 (e over the
//                    image-level entries, u over the unknowns, the block of row i taking
//                    u = i, i + n_imgs, ...: A p = P^T y_img + damp p);
//   k_pcg_update(n)  alpha, A p of the block's unknowns (one thread per short inverse list, one
//                    wave per long one), x, r, z, the stored p_n, and the block partials of r.r
//                    and r.z.
// p is Real-buffered (p_n in slot n & 1).  A launch after the stopping point returns at once: the
// flag "stopped before update n" lives in IS_DONE0 + (n & 1) and is written by k_pcg_spmv(n - 1).

// y_img[i][j] = sum over the blocks of image row i of S(i, i2)[j, :] . p(i2): one workgroup of
// PCG_ST threads per image row; its PCG_ST / 16 lane groups (one lane per row j) take every
// (PCG_ST / 16)-th block of the row.  Lane j2 of a group forms p_n at the block's column unknown j2 and the group shares the
// 16 values by shuffles; the group sums are added in LDS in a fixed order.  The operands of the
// first pass, the row's own unknowns and the partial sums are requested before any of them is used.
template <int GW, typename Real>
__global__ void __launch_bounds__(PCG_ST) k_pcg_spmv(ba_pcg_args a, int n, int nb) {
    const PcgV<Real> av(a);
    __shared__ Real sh[PCG_ST];
    __shared__ Real sDamp[PCG_ST / 64];
    const int i = blockIdx.x;
    const int grp = threadIdx.x / GW, j = threadIdx.x % GW;
    const int d = a.d, dd = d * d;
    const Real* __restrict__ pold = av.p + (int64_t)((n + 1) & 1) * a.n_u;
    // operands that depend on nothing are requested first: each thread's first block partials of
    // update n - 1, the scalar state, and (threads 0..d-1) the row's own unknowns with z and p_{n-1}
    Real pr0 = Real(0), pr1 = Real(0);
    if (threadIdx.x < nb) { pr0 = av.partials[PCG_NP * threadIdx.x + PT_RR]; pr1 = av.partials[PCG_NP * threadIdx.x + PT_RZ]; }
    const Real best = av.state[ST_BEST0 + ((n - 1) & 1)], rz_old = av.state[ST_RZ0 + ((n - 1) & 1)];
    const Real bnorm = av.state[ST_BNORM];
    int uo = -1;
    Real zo = Real(0), po = Real(0);
    if (threadIdx.x < GW && j < d) {
        uo = a.umap[(int64_t)i * d + j];
        if (uo >= 0) { zo = av.z[uo]; po = pold[uo]; }
    }
    // the row's blocks: from the fixed capacity when set (no load on this chain), else from row_ptr
    const int q0 = a.row_cap > 0 ? i * a.row_cap : a.row_ptr[i];
    const int q1 = a.row_cap > 0 ? q0 + a.row_cap : a.row_ptr[i + 1];
    auto load = [&](int q, int& u, Real& zv, Real& pv, Real (&bcol)[GW]) {
        const bool live = q < q1;
        u = live ? a.row_u[(int64_t)q * GW + j] : -1;
        zv = Real(0); pv = Real(0);
        if (u >= 0) { zv = av.z[u]; pv = pold[u]; }
        const Real* B = av.S_rows + (int64_t)q * dd;
#pragma unroll
        for (int j2 = 0; j2 < GW; ++j2) bcol[j2] = (live && j < d && j2 < d) ? B[j2 * d + j] : Real(0);
    };
    auto mac = [&](int u, Real zv, Real pv, Real beta, const Real (&bcol)[GW], Real acc) {
        const Real xj = u >= 0 ? pdir(zv, pv, beta) : Real(0);
#pragma unroll
        for (int j2 = 0; j2 < GW; ++j2) acc += bcol[j2] * __shfl(xj, j2, GW);
        return acc;
    };
    int u;
    Real zv, pv, bcol[GW];
    load(q0 + grp, u, zv, pv, bcol);                 // requested before the done flag is known
    // damping term of the unknowns v = i + k n_imgs (thread k): its first operands are requested now
    const int64_t v0 = i + (int64_t)threadIdx.x * a.n_imgs;
    Real dz = Real(0), dpo = Real(0), dd0 = Real(0);
    if (v0 < a.n_u) { dz = av.z[v0]; dpo = pold[v0]; dd0 = av.damp[v0]; }
    if (a.istate[IS_DONE0 + (n & 1)]) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.istate[IS_DONE0 + ((n + 1) & 1)] = 1;
        return;
    }

    Real beta = Real(0);
    if (n >= 1) {
        // end of update n - 1 (ba_solver.py:1222-1236)
        Real rs[2] = {Real(0), Real(0)};
        if (threadIdx.x < nb) { rs[0] += pr0; rs[1] += pr1; }     // the order of sum_partials
        for (int b = threadIdx.x + PCG_ST; b < nb; b += PCG_ST) { rs[0] += av.partials[PCG_NP * b + PT_RR]; rs[1] += av.partials[PCG_NP * b + PT_RZ]; }
        block_sums<PCG_ST, 2>(rs, sh);
        const Real rr = rs[0], rz_new = rs[1];
        const Real rnorm = sqrt(rr);
        const bool improved = rnorm < best;
        const bool conv = rnorm <= Real(a.tol) * bnorm;
        const bool bad = !isfinite(rz_new);
        const bool stop = conv || bad || n >= a.maxiter;
        beta = rz_new / (rz_old > Real(1e-32) ? rz_old : Real(1e-32));
        if (improved)                                    // best_so_far = r_norm, x, k
            for (int64_t v = (int64_t)blockIdx.x * PCG_ST + threadIdx.x; v < a.n_u; v += (int64_t)gridDim.x * PCG_ST)
                av.xbest[v] = av.x[v];
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            av.state[ST_BEST0 + (n & 1)] = improved ? rnorm : best;
            if (improved) a.istate[IS_BESTK] = n;
            av.state[ST_RZ0 + (n & 1)] = rz_new;
            av.state[ST_BETA] = beta;
            a.istate[IS_K] = n;
            if (conv) { a.istate[IS_CONV] = 1; a.istate[IS_USEBEST] = 0; }
            a.istate[IS_DONE0 + ((n + 1) & 1)] = stop;
        }
        if (stop) return;
    } else if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.istate[IS_DONE0 + 1] = 0;
    }
    Real dsum = Real(0);
    {
        const Real pv0 = pdir(dz, dpo, beta);
        dsum = dd0 * pv0 * pv0;
        for (int64_t v = v0 + (int64_t)PCG_ST * a.n_imgs; v < a.n_u; v += (int64_t)PCG_ST * a.n_imgs) {
            const Real pv2 = pdir(av.z[v], pold[v], beta);
            dsum += av.damp[v] * pv2 * pv2;
        }
        dsum = wave_sum(dsum);
    }
    // the row's further blocks: each block's unknown index is requested one block ahead, so that its z,
    // p and values are requested together (the sum keeps the block order)
    auto index_of = [&](int q) { return q < q1 ? a.row_u[(int64_t)q * GW + j] : -1; };
    int un = index_of(q0 + PCG_ST / GW + grp);
    Real acc = mac(u, zv, pv, beta, bcol, Real(0));
    for (int qb = q0 + PCG_ST / GW; qb < q1; qb += PCG_ST / GW) {
        const int q = qb + grp;
        u = un;
        zv = Real(0); pv = Real(0);
        if (u >= 0) { zv = av.z[u]; pv = pold[u]; }
        const Real* B = av.S_rows + (int64_t)q * dd;
#pragma unroll
        for (int j2 = 0; j2 < GW; ++j2) bcol[j2] = (q < q1 && j < d && j2 < d) ? B[j2 * d + j] : Real(0);
        un = index_of(q + PCG_ST / GW);
        acc = mac(u, zv, pv, beta, bcol, acc);
    }
    __syncthreads();
    sh[threadIdx.x] = acc;
    if ((threadIdx.x & 63) == 0) sDamp[threadIdx.x >> 6] = dsum;
    __syncthreads();
    // y of this image row; the row's share of p.Ap: sum_e p_u(e) y_e over its entries (one wave,
    // 16 rows at most) plus the damping sum of its unknowns
    if (threadIdx.x < 64) {
        Real part = Real(0);
        if (j < d && threadIdx.x < GW) {
            Real t = Real(0);
            for (int g = 0; g < PCG_ST / GW; ++g) t += sh[GW * g + j];
            av.y_img[(int64_t)i * d + j] = t;
            if (uo >= 0) part = pdir(zo, po, beta) * t;
        }
        part = wave_sum(part);
        if (threadIdx.x == 0) {
            Real dt = Real(0);
#pragma unroll
            for (int w = 0; w < PCG_ST / 64; ++w) dt += sDamp[w];
            av.img_part[i] = part + dt;
        }
    }
}

// alpha = rz / max(p.Ap, 1e-32); x += alpha p; r -= alpha Ap; z = M^-1 r (ba_solver.py:1217-1228);
// p_n stored in slot n & 1; block partials r.r, r.z.  A p of
// unknown u is the sum of the image-level rows mapping to u plus damp[u] p_n[u]: one thread sums a
// list of at most BA_PCG_LONG_LIST entries; the block's long lists (a focal pair shared by every
// image of a camera) are summed first, one wave each, 8 entries per lane in flight, into LDS.
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_update(ba_pcg_args a, int n) {
    const PcgV<Real> av(a);
    __shared__ Real sh[2 * (PCG_T / 64)];
    __shared__ Real sLong[PCG_T];
    // requested first: the image partials of p.Ap (the first PCG_IPF of each thread) and the scalars
    Real ipf[PCG_IPF];
#pragma unroll
    for (int k = 0; k < PCG_IPF; ++k) {
        const int b = threadIdx.x + k * PCG_T;
        ipf[k] = b < a.n_imgs ? av.img_part[b] : Real(0);
    }
    const Real beta = av.state[ST_BETA], rz = av.state[ST_RZ0 + (n & 1)];
    if (a.istate[IS_DONE0 + ((n + 1) & 1)]) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t u = (int64_t)blockIdx.x * PCG_T + threadIdx.x;
    const Real* __restrict__ pold = av.p + (int64_t)((n + 1) & 1) * a.n_u;
    Real zu = Real(0), pu = Real(0), xu = Real(0), ru = Real(0), du = Real(1), dmp = Real(0), y1 = Real(0);
    int q0 = 0, q1 = 0, li = -1, s1 = -1;
    if (u < a.n_u) {                                   // operands first, then the reductions
        zu = av.z[u]; pu = pold[u]; xu = av.x[u]; ru = av.r[u]; du = av.diagA[u]; dmp = av.damp[u];
        li = a.long_idx[u];
        if (a.src1 != nullptr) {                       // a one-entry list resolved ahead
            s1 = a.src1[u];
            if (s1 >= 0) y1 = av.y_img[s1];
        }
        if (s1 < 0) { q0 = a.inv_ptr[u]; q1 = a.inv_ptr[u + 1]; }
    }
    const int lk0 = a.long_ptr[blockIdx.x], lk1 = a.long_ptr[blockIdx.x + 1];
    for (int k = lk0 + w; k < lk1; k += PCG_T / 64) {
        int b0, b1;
        if (a.long_rng != nullptr) {
            b0 = a.long_rng[2 * k]; b1 = a.long_rng[2 * k + 1];
        } else {
            const int v = a.long_u[k];
            b0 = a.inv_ptr[v]; b1 = a.inv_ptr[v + 1];
        }
        Real s = Real(0);
        for (int q = b0 + lane; q < b1; q += 64 * PCG_LF) {
            int src[PCG_LF];
#pragma unroll
            for (int t = 0; t < PCG_LF; ++t) src[t] = q + 64 * t < b1 ? a.inv_src[q + 64 * t] : -1;
#pragma unroll
            for (int t = 0; t < PCG_LF; ++t) s += src[t] >= 0 ? av.y_img[src[t]] : Real(0);
        }
        s = wave_sum(s);
        if (lane == 0) sLong[k - lk0] = s;
    }
    // the short lists: y_img is complete at launch, so these sums need nothing from the reductions
    Real ys = Real(0);
    if (s1 >= 0)
        ys = Real(0) + y1;                                 // the same sum as the one-entry loop below
    else if (li < 0)
        for (int q = q0; q < q1; ++q) ys += av.y_img[a.inv_src[q]];
    Real sums[1] = {Real(0)};
#pragma unroll
    for (int k = 0; k < PCG_IPF; ++k)
        if (threadIdx.x + k * PCG_T < a.n_imgs) sums[0] += ipf[k];
    for (int b = threadIdx.x + PCG_IPF * PCG_T; b < a.n_imgs; b += PCG_T) sums[0] += av.img_part[b];
    block_sums<PCG_T, 1>(sums, sh);                    // p.Ap (its barriers also publish sLong)
    const Real pap = sums[0];
    const Real denom = pap > Real(1e-32) ? pap : Real(1e-32);
    const Real alpha = rz / denom;
    Real t[PCG_NP] = {Real(0), Real(0)};
    if (u < a.n_u) {
        const Real pn = pdir(zu, pu, beta);
        const Real apu = (li >= 0 ? sLong[li] : ys) + dmp * pn;
        av.p[(int64_t)(n & 1) * a.n_u + u] = pn;
        const Real x = xu + alpha * pn;
        const Real r = ru - alpha * apu;
        const Real z = r / du;
        av.x[u] = x; av.r[u] = r; av.z[u] = z;
        t[PT_RR] = r * r; t[PT_RZ] = r * z;
    }
    block_sums<PCG_T, PCG_NP>(t, sh);
    if (threadIdx.x < PCG_NP) av.partials[PCG_NP * blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? t[0] : t[1];
}

// ----------------------------------------------------------------------------- large systems
// The product by pair blocks (d <= 16), for systems whose row copies would stream from memory on every
// iteration: each block of the upper triangle is read once, in place in S_pairs, and serves both S x and
// S^T x, where the row copies hold (and read) every off-diagonal block twice.  Bound by memory: at 4096 images,
// 557 k pairs, d = 13 in fp64, k_pcg_pairs moves 0.82 GB in 179 us (4.6 TB/s, a large copy reaches 4.8), with
// k_pcg_cols 21 us and k_pcg_dir 5 us, where k_pcg_spmv took 314 us for 1.5 GB; in fp32 93 us less an iteration.
// The four launches of an iteration are
//   k_pcg_dir(n)     the decisions after update n - 1 (as k_pcg_spmv forms them), p_n at image level
//   k_pcg_pairs(n)   per image row its upper blocks: y_i, and t_p = S_p^T p_i per pair
//   k_pcg_cols(n)    y_i += the t_p of the pairs whose second image is i; the row's share of p.Ap
//   k_pcg_update(n)
// Every sum runs in the order of the pair list.

#define PCG_GW 16           // lanes per block, and the stride of t and p_img: whole 64- or 128-byte rows

template <typename Real>
struct PcgPairsV {
    Real *t, *p_img;
    const int32_t* up_ptr;
    __device__ __forceinline__ explicit PcgPairsV(const ba_pcg_pairs& w)
        : t((Real*)w.t), p_img((Real*)w.p_img), up_ptr(w.up_ptr) {}
};

// up_ptr[i] = the first pair of image row i (pair_i1 ascending), i = 0 .. n_imgs
__global__ void __launch_bounds__(PCG_T) k_pcg_up_ptr(const int32_t* __restrict__ pair_i1, int64_t n_pairs, int n_imgs,
                                                      int32_t* __restrict__ up_ptr) {
    const int i = (int)(blockIdx.x * PCG_T + threadIdx.x);
    if (i > n_imgs) return;
    int64_t lo = 0, hi = n_pairs;
    while (lo < hi) {
        const int64_t m = (lo + hi) >> 1;
        if (pair_i1[m] < i) lo = m + 1; else hi = m;
    }
    up_ptr[i] = (int32_t)lo;
}

// The decisions of k_pcg_spmv(n), from the same partial sums (every block forms them alike), the best-so-far
// copy, and p_img[i][j] = p_n at entry (i, j) (0 past d and where the parameter is not an unknown).
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_dir(ba_pcg_args a, ba_pcg_pairs w, int n, int nb) {
    const PcgV<Real> av(a);
    const PcgPairsV<Real> pv(w);
    __shared__ Real sh[2 * (PCG_T / 64)];
    const int64_t e = (int64_t)blockIdx.x * PCG_T + threadIdx.x;
    const int64_t i = e / PCG_GW;
    const int j = (int)(e % PCG_GW), d = a.d;
    const Real* __restrict__ pold = av.p + (int64_t)((n + 1) & 1) * a.n_u;
    const Real best = av.state[ST_BEST0 + ((n - 1) & 1)], rz_old = av.state[ST_RZ0 + ((n - 1) & 1)];
    const Real bnorm = av.state[ST_BNORM];
    int u = -1;
    Real zv = Real(0), po = Real(0);
    if (i < a.n_imgs && j < d) {
        u = a.umap[i * d + j];
        if (u >= 0) { zv = av.z[u]; po = pold[u]; }
    }
    if (a.istate[IS_DONE0 + (n & 1)]) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.istate[IS_DONE0 + ((n + 1) & 1)] = 1;
        return;
    }
    Real beta = Real(0);
    if (n >= 1) {
        Real rs[2];
        sum_partials<PCG_T>(av.partials, nb, rs, sh);
        const Real rnorm = sqrt(rs[0]), rz_new = rs[1];
        const bool improved = rnorm < best;
        const bool conv = rnorm <= Real(a.tol) * bnorm;
        const bool bad = !isfinite(rz_new);
        const bool stop = conv || bad || n >= a.maxiter;
        beta = rz_new / (rz_old > Real(1e-32) ? rz_old : Real(1e-32));
        if (improved)
            for (int64_t v = e; v < a.n_u; v += (int64_t)gridDim.x * PCG_T) av.xbest[v] = av.x[v];
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            av.state[ST_BEST0 + (n & 1)] = improved ? rnorm : best;
            if (improved) a.istate[IS_BESTK] = n;
            av.state[ST_RZ0 + (n & 1)] = rz_new;
            av.state[ST_BETA] = beta;
            a.istate[IS_K] = n;
            if (conv) { a.istate[IS_CONV] = 1; a.istate[IS_USEBEST] = 0; }
            a.istate[IS_DONE0 + ((n + 1) & 1)] = stop;
        }
        if (stop) return;
    } else if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.istate[IS_DONE0 + 1] = 0;
    }
    if (i < a.n_imgs) pv.p_img[e] = u >= 0 ? pdir(zv, po, beta) : Real(0);
}

// One workgroup per image row i, PCG_GW lanes per block, lane c holding column c of it: y_i[r] gathers
// S[r][c] p_c per lane over the row's blocks (added over the lanes once per row), t_p[c] = sum_r S[r][c] p_i[r]
// is the lane's own, so the loop needs no shuffles.  The next block's column is requested before this block's
// products (three waves per SIMD in fp64; four, with spills, doubled the step's time).  Plain loads:
// non-temporal ones cost 12%, and turning the row order round every other iteration for the memory-side cache
// gained 0.5%.
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_pairs(ba_pcg_args a, ba_pcg_pairs w, int n) {
    const PcgV<Real> av(a);
    const PcgPairsV<Real> pv(w);
    constexpr int NG = PCG_T / PCG_GW;
    __shared__ Real sh[NG][PCG_GW];
    const int i = blockIdx.x;
    const int g = threadIdx.x / PCG_GW, c = threadIdx.x % PCG_GW;
    const int d = a.d, dd = d * d;
    if (a.istate[IS_DONE0 + ((n + 1) & 1)]) return;
    const int p0 = pv.up_ptr[i], p1 = pv.up_ptr[i + 1];
    Real xi[PCG_GW];                                      // p_n of this image (uniform over the workgroup)
#pragma unroll
    for (int r = 0; r < PCG_GW; ++r) xi[r] = pv.p_img[(int64_t)i * PCG_GW + r];
    Real acc[PCG_GW];
#pragma unroll
    for (int r = 0; r < PCG_GW; ++r) acc[r] = Real(0);
    auto load = [&](int p, Real& x, Real (&col)[PCG_GW]) {
        const bool live = p < p1;
        x = live ? pv.p_img[(int64_t)a.pair_i2[p] * PCG_GW + c] : Real(0);
        const Real* S = av.S_pairs + (int64_t)p * dd + c;
#pragma unroll
        for (int r = 0; r < PCG_GW; ++r) col[r] = (live && c < d && r < d) ? S[r * d] : Real(0);
    };
    Real x, col[PCG_GW];
    load(p0 + g, x, col);
    for (int p = p0 + g; p < p1; p += NG) {
        Real xn, coln[PCG_GW];
        load(p + NG, xn, coln);
        Real t = Real(0);
#pragma unroll
        for (int r = 0; r < PCG_GW; ++r) {
            acc[r] = fma(col[r], x, acc[r]);
            t = fma(col[r], xi[r], t);
        }
        pv.t[(int64_t)p * PCG_GW + c] = t;                // read by k_pcg_cols (never for a diagonal block)
        x = xn;
#pragma unroll
        for (int r = 0; r < PCG_GW; ++r) col[r] = coln[r];
    }
    // sum of acc[r] over the group's lanes, left in lane r: each step halves the rows a lane keeps
#pragma unroll
    for (int h = PCG_GW / 2; h >= 1; h >>= 1) {
        const bool up = (c & h) != 0;
#pragma unroll
        for (int r = 0; r < h; ++r) {
            const Real send = up ? acc[r] : acc[r + h], keep = up ? acc[r + h] : acc[r];
            acc[r] = keep + __shfl_xor(send, h, PCG_GW);
        }
    }
    sh[g][c] = acc[0];
    __syncthreads();
    if (threadIdx.x < d) {
        Real y = Real(0);
        for (int k = 0; k < NG; ++k) y += sh[k][threadIdx.x];
        av.y_img[(int64_t)i * d + threadIdx.x] = y;
    }
}

// y_i += t_p over the pairs whose second image is i (the leading, transposed entries of its row list: the
// pairs are ordered by first image), and the row's share of p.Ap: sum_e p_u(e) y_e plus the damping term of
// the unknowns u = i + k n_imgs, as in k_pcg_spmv.
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_cols(ba_pcg_args a, ba_pcg_pairs w, int n) {
    const PcgV<Real> av(a);
    const PcgPairsV<Real> pv(w);
    constexpr int NG = PCG_T / PCG_GW, NF = 4;            // entries in flight per group
    __shared__ Real sh[NG][PCG_GW];
    __shared__ Real sDamp[PCG_T / 64];
    const int i = blockIdx.x;
    const int g = threadIdx.x / PCG_GW, c = threadIdx.x % PCG_GW;
    const int d = a.d;
    const Real* __restrict__ pold = av.p + (int64_t)((n + 1) & 1) * a.n_u;
    const Real beta = av.state[ST_BETA];
    if (a.istate[IS_DONE0 + ((n + 1) & 1)]) return;
    const int q0 = a.row_ptr[i], q1 = a.row_ptr[i + 1] - (pv.up_ptr[i + 1] - pv.up_ptr[i]);
    Real y0 = Real(0), pi = Real(0);
    if (threadIdx.x < d) { y0 = av.y_img[(int64_t)i * d + c]; pi = pv.p_img[(int64_t)i * PCG_GW + c]; }
    Real acc = Real(0);
    for (int q = q0 + g; q < q1; q += NG * NF) {
        int ent[NF];
#pragma unroll
        for (int k = 0; k < NF; ++k) ent[k] = q + k * NG < q1 ? a.row_ent[q + k * NG] : -1;
#pragma unroll
        for (int k = 0; k < NF; ++k) acc += ent[k] >= 0 ? pv.t[(int64_t)(ent[k] >> 1) * PCG_GW + c] : Real(0);
    }
    Real dsum = Real(0);
    for (int64_t v = i + (int64_t)threadIdx.x * a.n_imgs; v < a.n_u; v += (int64_t)PCG_T * a.n_imgs) {
        const Real pn = pdir(av.z[v], pold[v], beta);
        dsum += av.damp[v] * pn * pn;
    }
    dsum = wave_sum(dsum);
    sh[g][c] = acc;
    if ((threadIdx.x & 63) == 0) sDamp[threadIdx.x >> 6] = dsum;
    __syncthreads();
    if (threadIdx.x < 64) {
        Real part = Real(0);
        if (threadIdx.x < d) {
            Real y = y0;
            for (int k = 0; k < NG; ++k) y += sh[k][c];
            av.y_img[(int64_t)i * d + c] = y;
            part = pi * y;
        }
        part = wave_sum(part);
        if (threadIdx.x == 0) {
#pragma unroll
            for (int k = 0; k < PCG_T / 64; ++k) part += sDamp[k];
            av.img_part[i] = part;
        }
    }
}

// ----------------------------------------------------------------------------- resident solve
// The whole loop in one cooperative launch, for systems whose image rows fit the workgroups' registers and LDS
// and that share few unknowns.  A launch sequence pays two launches per iteration, and in each the dependent
// loads of its operands; here every workgroup keeps m image rows (their blocks, the search direction at their
// column images, the state of their unknowns) for the whole solve, and an iteration costs two exchanges:
//   A  after update n - 1: each workgroup's partials of r.r and r.z, and z at its image-level entries
//   B  after the product:  each workgroup's partials of p.Ap and of A p at the shared unknowns
// Everything exchanged travels in words of eight bytes that hold 32 bits of data and the exchange's number, so
// a reader that finds the number has the data: no fence, no barrier, no second load (a word is written once per
// exchange, with a relaxed agent-scope store).  A word is overwritten only after its readers are done: what a
// workgroup publishes in A follows its reading of B from every workgroup, each of which published B after it
// had read A, and the other way round.
// Every workgroup forms the loop's scalars from the same partials in the same order, so all decide alike.
// A wait that exceeds its limit gives up: the workgroup sets istate[6] and leaves, the others follow, and the
// caller solves by the launch sequence.
// Bound by the exchanges' latency.  Per iteration, against the launch sequence (d = 13 where not said):
//   1024 images, windows of 23, fp64 (205 workgroups)   10.3 us   15.3 us
//   1024 images, the same, d = 9 (205)                   7.5 us   13.3 us
//   256 images, 47 neighbours, fp64 (128)                8.1 us   15.0 us
//   777 images, windows, fp32 (156)                      7.3 us   14.6 us
//   500 images, d = 17, fp64 (167)                       8.5 us   18.2 us
//   32 images, all pairs, fp32 (16)                      4.0 us   11.4 us
//   8 images, fp64 (1, no exchange)                      2.0 us    7.1 us
// of which (1024 images, cycles) A 6 to 7 k, B 9 k, the product 3.4 k, the updates and scalars 3 k.  While a
// workgroup's own values are under way, its other waves stay at a barrier: polling then crowds out its stores.

#define PP_T 512            // threads of a workgroup: PP_T / GW lane groups for the product
#define PP_K 4              // column entries per thread
#define PP_E 2              // own entries per lane of the first wave
#define PP_NS 2             // most shared unknowns
#define PP_G 16             // workgroups of a group whose partials its first one adds
#define PP_WG 256           // most workgroups
#define PP_LDS (158 * 1024) // dynamic LDS of a workgroup (160 KB per CU, less the static arrays)

// {data, number} words of the exchanges: a double is two of them (low half, high half), a float one
template <typename Real> struct LL;
template <>
struct LL<double> {
    static constexpr int W = 2;
    static __device__ __forceinline__ uint32_t part(double v, int h) {
        return (uint32_t)(h ? __double2hiint(v) : __double2loint(v));
    }
    static __device__ __forceinline__ double join(const uint64_t (&w)[2]) {
        return __hiloint2double((int)(uint32_t)w[1], (int)(uint32_t)w[0]);
    }
};
template <>
struct LL<float> {
    static constexpr int W = 1;
    static __device__ __forceinline__ uint32_t part(float v, int) { return __float_as_uint(v); }
    static __device__ __forceinline__ float join(const uint64_t (&w)[1]) { return __uint_as_float((uint32_t)w[0]); }
};
__device__ __forceinline__ void ll_put(uint64_t* w, uint32_t data, uint32_t ep) {
    __hip_atomic_store(w, (uint64_t)ep << 32 | data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t ll_get(const uint64_t* w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One bounded wait of a thread: polls until try_() says that all its words have arrived, or the limit (ticks
// of the 100 MHz clock) has passed; a limit of 0 gives up at once.
template <typename F>
__device__ __forceinline__ bool pp_wait(int64_t limit, F&& try_) {
    int64_t t0 = 0;
    for (unsigned k = 1;; ++k) {
        if (limit <= 0) return false;
        if (try_()) return true;
        if ((k & 63) == 0) {
            const int64_t t = (int64_t)wall_clock64();
            if (k == 64) t0 = t;
            else if (t - t0 > limit) return false;
        }
    }
}

// DPP move: lanes that have no source, or lie outside the row mask, get 0
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, true));
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp(double v) {
    const long r = __builtin_amdgcn_update_dpp(0l, __builtin_bit_cast(long, v), CTRL, ROWS, 0xf, true);
    return __builtin_bit_cast(double, r);
}
__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// Sums over the wave without LDS (all lanes active): shifts within the rows of 16 lanes, then the rows' last
// lanes into the rows above; every lane gets the total from lane 63.
template <int K, typename Real>
__device__ __forceinline__ void wave_sums(Real (&v)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] += dpp<0x111>(v[k]);              // row_shr:1
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] += dpp<0x112>(v[k]);
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] += dpp<0x114>(v[k]);
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] += dpp<0x118>(v[k]);
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] += dpp<0x142, 0xa>(v[k]);         // row_bcast:15
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] += dpp<0x143, 0xc>(v[k]);         // row_bcast:31
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = lane_value(v[k], 63);
}

// num / den with inv = 1 / den at hand: the quotient corrected by its remainder
template <typename Real>
__device__ __forceinline__ Real div_by(Real num, Real den, Real inv) {
    const Real q = num * inv;
    return fma(fma(-q, den, num), inv, q);
}

// acc += sum over the columns c of a block of B[c][row] x[c], C0 <= c < DM, x[c] in lane c - C0 of the row of
// 16 lanes (0 past d); the block's column c at the lane's row is col(c)
template <int C0, int DM, int N = C0, typename Real, typename F>
__device__ __forceinline__ void pp_cols(F&& col, Real x, Real (&acc)[2]) {
    if constexpr (N < DM && N < C0 + 16) {
        acc[N & 1] = fma(col(N), dpp<0x150 + N - C0>(x), acc[N & 1]);  // row_newbcast
        pp_cols<C0, DM, N + 1>(col, x, acc);
    }
}

// Blocks of a lane group that its lanes hold in registers (about 100 VGPRs of the 256 that two waves per SIMD
// leave each); the others lie in LDS.
constexpr int pp_regs_of(int dm, bool real32) {
    return real32 ? (dm <= 16 ? 4 : dm <= 25 ? 3 : 2) : (dm <= 9 ? 3 : dm <= 16 ? 2 : dm <= 25 ? 1 : 0);
}
template <int DM, typename Real> struct PpRegs { static constexpr int N = pp_regs_of(DM, sizeof(Real) == 4); };
// the unrolled block width: steps of about a quarter, so that little of an unrolled product is idle
static inline int pp_width(int d) { return d <= 9 ? 9 : d <= 13 ? 13 : d <= 16 ? 16 : d <= 20 ? 20 : d <= 25 ? 25 : 32; }
// An exchange of V partial sums per workgroup.  Up to 2 PP_G workgroups: each publishes its partials to
// everyone (1.1 us).  More: to the first of its group of PP_G, which adds them (relay) and publishes the group's: every
// workgroup polling the partials of 205 others took 3.5 to 4 us, two hops over few lines 2.8.  What everyone polls is
// kept in as many copies as one store instruction writes, the readers spread over them, as the readers of one line
// are served one after the other.
template <int V, typename Real>
struct PpSums {
    typedef LL<Real> L;
    static constexpr int W = L::W, VW = V * W, NC = 64 / VW;            // words of one publication; copies
    uint64_t *xm, *xg;                                                  // to the group's first; to everyone
    int nwg, wg, ng, gs;                                                // groups (padded to lines: gs)
    bool two;
    __device__ __forceinline__ PpSums(uint64_t* words, int nwg_, int wg_) : nwg(nwg_), wg(wg_) {
        two = nwg > 2 * PP_G;
        ng = two ? (nwg + PP_G - 1) / PP_G : nwg;
        gs = (ng + 15) & ~15;
        xg = words;
        xm = words + (int64_t)64 * gs;
    }
    static __host__ __device__ int64_t words_of(int nwg) {
        const int ng = nwg > 2 * PP_G ? (nwg + PP_G - 1) / PP_G : nwg;
        return 64 * (int64_t)((ng + 15) & ~15) + (int64_t)(nwg + PP_G - 1) / PP_G * PP_G * 6;   // for every V <= 3
    }
    __device__ __forceinline__ int64_t words() const { return words_of(nwg); }
    __device__ __forceinline__ Real pick(const Real (&v)[V], int s) const {
        Real r = v[0];
#pragma unroll
        for (int k = 1; k < V; ++k) r = s == k ? v[k] : r;
        return r;
    }
    // to everyone, as group g: lane l writes word l % VW of copy l / VW
    __device__ __forceinline__ void put_all(const Real (&v)[V], uint32_t ep, int lane, int g) const {
        const int c = lane % VW;
        if (lane < NC * VW) ll_put(xg + lane * gs + g, L::part(pick(v, c / W), c % W), ep);
    }
    // one wave, all lanes holding the workgroup's partials
    __device__ __forceinline__ void put(const Real (&v)[V], uint32_t ep, int lane) const {
        if (!two) put_all(v, ep, lane, wg);
        else if (lane < VW)
            ll_put(xm + ((wg / PP_G) * VW + lane) * PP_G + wg % PP_G, L::part(pick(v, lane / W), lane % W), ep);
    }
    // the group's first workgroup, one wave: lane (value, member) polls one partial; the rows of 16 lanes are
    // added and published
    __device__ __forceinline__ bool relay(int64_t limit, uint32_t ep, int lane) const {
        if (!two || wg % PP_G != 0) return true;
        const int g = wg / PP_G, s = lane / 16, k = lane % 16;
        Real x = Real(0);
        bool good = true;
        if (s < V && wg + k < nwg) {
            const uint64_t* q = xm + (g * VW + s * W) * PP_G + k;
            good = pp_wait(limit, [&]() {
                uint64_t raw[W];
                bool all = true;
#pragma unroll
                for (int h = 0; h < W; ++h) raw[h] = ll_get(q + h * PP_G);
#pragma unroll
                for (int h = 0; h < W; ++h) all = all && (uint32_t)(raw[h] >> 32) == ep;
                x = L::join(raw);
                return all;
            });
        }
        x += dpp<0x111>(x);
        x += dpp<0x112>(x);
        x += dpp<0x114>(x);
        x += dpp<0x118>(x);                                             // lane 15 of each row: its sum
        Real v[V];
#pragma unroll
        for (int q = 0; q < V; ++q) v[q] = lane_value(x, 16 * q + 15);
        put_all(v, ep, lane, g);
        return good;
    }
    // one wave: lane g gets the partials of group g (0 past the groups); wave_sums makes the sums of them
    __device__ __forceinline__ bool get(int64_t limit, uint32_t ep, int lane, Real (&v)[V]) const {
#pragma unroll
        for (int q = 0; q < V; ++q) v[q] = Real(0);
        if (lane >= ng) return true;
        const uint64_t* q = xg + (wg % NC) * VW * gs + lane;
        return pp_wait(limit, [&]() {
            uint64_t raw[V][W];
            bool all = true;
#pragma unroll
            for (int s = 0; s < V; ++s)
#pragma unroll
                for (int h = 0; h < W; ++h) raw[s][h] = ll_get(q + (s * W + h) * gs);
#pragma unroll
            for (int s = 0; s < V; ++s) {
#pragma unroll
                for (int h = 0; h < W; ++h) all = all && (uint32_t)(raw[s][h] >> 32) == ep;
                v[s] = L::join(raw[s]);
            }
            return all;
        });
    }
};

// LDS of a workgroup: the blocks of its rows that are not in registers (before they are loaded, the map from
// images to column slots), then p at its column images, the lane groups' products, the column images and the
// LDS blocks' column slots.
struct PpLds {
    size_t S, pcol, yp, col, cidx, total;
};
static __host__ __device__ inline PpLds pp_lds(int d, int gw, size_t R, int n_imgs, int max_blk, int max_col) {
    PpLds o;
    size_t at = 0;
    auto take = [&](size_t n) { const size_t r = at; at += (n + 15) & ~(size_t)15; return r; };
    const size_t sb = R * d * d * (size_t)max_blk, mb = sizeof(uint16_t) * (size_t)n_imgs;
    o.S = take(sb > mb ? sb : mb);
    o.pcol = take(R * gw * (size_t)max_col);
    o.yp = take(R * PP_T);
    o.col = take(sizeof(int) * (size_t)max_col);
    o.cidx = take(sizeof(int) * (size_t)max_blk);
    o.total = at;
    return o;
}

__global__ void __launch_bounds__(PCG_T) k_pp_clear(uint64_t* __restrict__ w, int64_t n, int32_t* __restrict__ istate) {
    const int64_t t = (int64_t)blockIdx.x * PCG_T + threadIdx.x;
    if (t < n) w[t] = 0;
    if (t < 8) istate[t] = 0;
}

__global__ void k_pp_refused(int32_t* istate) { istate[6] = 1; }

// DM: the block width the product is unrolled for (d <= DM <= GW); NS: shared unknowns exchanged.  The first
// wave owns the workgroup's entries (their x, r, z, p and the loop's partial sums); all waves poll, form the
// loop's scalars and take part in the product.  Four barriers per iteration.
template <int GW, int DM, int NS, typename Real>
__global__ void __launch_bounds__(PP_T) k_pcg_resident(ba_pcg_args a, ba_pcg_resident w) {
    typedef LL<Real> L;
    constexpr int W = L::W, NG = PP_T / GW, NW = PP_T / 64;
    extern __shared__ __align__(16) char lds[];
    __shared__ Real sA[2];
    __shared__ int sCnt[NW], sFailA, sFailB;
    const PcgV<Real> av(a);
    const int d = a.d, dd = d * d, tid = threadIdx.x, wg = blockIdx.x, nwg = gridDim.x, m = w.m;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const PpLds o = pp_lds(d, GW, sizeof(Real), a.n_imgs, w.max_blk, w.max_col);
    Real* const sS = reinterpret_cast<Real*>(lds + o.S);
    Real* const sP = reinterpret_cast<Real*>(lds + o.pcol);
    Real* const sY = reinterpret_cast<Real*>(lds + o.yp);
    int* const sCol = reinterpret_cast<int*>(lds + o.col);
    int* const sCidx = reinterpret_cast<int*>(lds + o.cidx);
    // word h of z at entry (i, j): xz[(i W + h) GW + j]
    uint64_t* const xz = w.words;
    const PpSums<2, Real> xA(w.words + (int64_t)a.n_imgs * GW * W, nwg, wg);
    const PpSums<1 + NS, Real> xB(w.words + (int64_t)a.n_imgs * GW * W + xA.words(), nwg, wg);
    const int i0 = wg * m, i1 = min(i0 + m, a.n_imgs);
    const int e0 = a.row_ptr[i0], nblk = a.row_ptr[i1] - e0;
    constexpr int NBR = PpRegs<DM, Real>::N;
    if (tid == 0) { sFailA = 0; sFailB = 0; }

    // ---- column images of the own rows: marked in a map, then numbered in image order
    uint16_t* const map = reinterpret_cast<uint16_t*>(lds + o.S);
    for (int i = tid; i < a.n_imgs; i += PP_T) map[i] = 0;
    __syncthreads();
    auto col_of = [&](int b) {
        const int ent = a.row_ent[e0 + b], p = ent >> 1;
        return (ent & 1) ? a.pair_i1[p] : a.pair_i2[p];
    };
    for (int b = tid; b < nblk; b += PP_T) map[col_of(b)] = 1;          // equal stores may meet
    for (int i = i0 + tid; i < i1; i += PP_T) map[i] = 1;               // an own image without blocks, too
    __syncthreads();
    const int per = (a.n_imgs + PP_T - 1) / PP_T, lo = min(tid * per, a.n_imgs), hi = min(lo + per, a.n_imgs);
    int cnt = 0;
    for (int i = lo; i < hi; ++i) cnt += map[i];
    int scan = cnt;                                                     // inclusive over the wave, then the waves
    for (int s = 1; s < 64; s <<= 1) {
        const int v = __shfl_up(scan, s);
        if (lane >= s) scan += v;
    }
    if (lane == 63) sCnt[wave] = scan;
    __syncthreads();
    int base = scan - cnt, ncol = 0;
    for (int k = 0; k < NW; ++k) {
        if (k < wave) base += sCnt[k];
        ncol += sCnt[k];
    }
    // max_col or max_blk of a plan for other rows or another m: the columns or (below) the LDS blocks would run past their
    // arrays; the solve is given up, by all threads alike
    if (__builtin_expect(ncol > w.max_col, 0)) {
        if (tid == 0) a.istate[6] = 1;
        return;
    }
    for (int i = lo; i < hi; ++i)
        if (map[i]) { map[i] = (uint16_t)base; sCol[base++] = i; }
    __syncthreads();
    // ---- the own entries, in the first wave: lane l holds entries l and l + 64 (entry e: image i0 + e / d,
    // parameter e % d); an unknown shared by several entries has its state at each of them, and counts once (at
    // the first entry of its list)
    int u[PP_E], sh[PP_E], oy[PP_E], op[PP_E], ow[PP_E];
    bool counts[PP_E];
    Real x[PP_E], xb_[PP_E], r[PP_E], z[PP_E], p[PP_E], dA[PP_E], iA[PP_E], dmp[PP_E];
    const int gpr = NG / m;                                             // lane groups per row
#pragma unroll
    for (int k = 0; k < PP_E; ++k) {
        const int e = lane + 64 * k, el = e / d, ej = e - el * d;
        u[k] = -1; sh[k] = -1; counts[k] = false;
        oy[k] = op[k] = ow[k] = 0;
        x[k] = xb_[k] = r[k] = z[k] = p[k] = dmp[k] = Real(0);
        dA[k] = iA[k] = Real(1);
        if (wave == 0 && e < (i1 - i0) * d) {
            u[k] = a.umap[(int64_t)(i0 + el) * d + ej];
            oy[k] = el * gpr * GW + ej;                                 // its products in sY
            op[k] = map[i0 + el] * GW + ej;                             // its place in sP
            ow[k] = ((i0 + el) * W) * GW + ej;                          // its words
            if (u[k] >= 0) {
                r[k] = av.rhs[u[k]]; dA[k] = av.diagA[u[k]]; dmp[k] = av.damp[u[k]];
                iA[k] = Real(1) / dA[k];
                z[k] = r[k] / dA[k];
                counts[k] = a.inv_src[a.inv_ptr[u[k]]] == (i0 + el) * d + ej;
                for (int s = 0; s < w.n_shared; ++s)
                    if (w.shared_u[s] == u[k]) sh[k] = s;
            }
        } else {
            op[k] = -1;
        }
    }
    // this thread's column entries of other workgroups: the word of z, its place in sP
    const int nk = (ncol * GW + PP_T - 1) / PP_T;                       // at most PP_K
    int cw[PP_K];
    Real zc[PP_K];
#pragma unroll
    for (int k = 0; k < PP_K; ++k) {
        const int q = tid + k * PP_T, c = q / GW, cj = q % GW;
        cw[k] = -1;
        zc[k] = Real(0);
        if (c < ncol) {
            const int img = sCol[c];
            if ((img < i0 || img >= i1) && cj < d) cw[k] = img * W * GW + cj;
            sP[q] = Real(0);
        }
    }
    // ---- this lane group's row: blocks part, part + gpr, ... of it, the first NBR in registers (lane = row of
    // the block), the others in LDS from slot ls on, column-major (a column's lanes read contiguously)
    const int g = tid / GW, j = tid % GW, row = g / gpr, part = g - row * gpr;
    int ls0 = 0, ls1 = 0;                                               // this row's LDS slots
    Real B[NBR + 1][DM];
    int bx[NBR + 1];                                                        // the column slots of the register blocks
    {
        int at = 0;
        for (int q = 0; q < i1 - i0; ++q) {                             // rows in order: at most 32
            const int b0 = a.row_ptr[i0 + q] - e0, len = a.row_ptr[i0 + q + 1] - e0 - b0;
            const int more = max(0, len - NBR * gpr);
            if (__builtin_expect(at + more > w.max_blk, 0)) {
                if (tid == 0) a.istate[6] = 1;
                return;
            }
            for (int t = tid; t < more; t += PP_T) sCidx[at + t] = map[col_of(b0 + NBR * gpr + t)] * GW;
            if (q == row) { ls0 = at; ls1 = at + more; }
            at += more;
        }
    }
    const int rb0 = row < i1 - i0 ? a.row_ptr[i0 + row] - e0 : 0, rb1 = row < i1 - i0 ? a.row_ptr[i0 + row + 1] - e0 : 0;
#pragma unroll
    for (int k = 0; k < NBR; ++k) {
        const int b = rb0 + part + k * gpr;
        const bool live = b < rb1;
        bx[k] = live ? map[col_of(b)] * GW : 0;
        const int ent = live ? a.row_ent[e0 + b] : 0;
        const Real* S = av.S_pairs + (int64_t)(ent >> 1) * dd;
#pragma unroll
        for (int c = 0; c < DM; ++c)
            B[k][c] = live && j < d && c < d ? ((ent & 1) ? S[c * d + j] : S[j * d + c]) : Real(0);
    }
    int nbr = 0;                                                        // register blocks of the longest row
    for (int q = 0; q < i1 - i0; ++q) nbr = max(nbr, (a.row_ptr[i0 + q + 1] - a.row_ptr[i0 + q] + gpr - 1) / gpr);
    __syncthreads();                                                    // the map is done with
    {
        int at = 0;
        for (int q = 0; q < i1 - i0; ++q) {
            const int b0 = a.row_ptr[i0 + q] - e0 + NBR * gpr, more = max(0, a.row_ptr[i0 + q + 1] - e0 - b0);
            for (int t = wave; t < more; t += NW) {                     // one wave per block
                const int ent = a.row_ent[e0 + b0 + t];
                const Real* S = av.S_pairs + (int64_t)(ent >> 1) * dd;
                for (int e = lane; e < dd; e += 64) {
                    const int c = e / d, rr = e - c * d;
                    sS[(at + t) * dd + e] = (ent & 1) ? S[c * d + rr] : S[rr * d + c];
                }
            }
            at += more;
        }
    }
    // unknowns without an entry stay 0
    for (int64_t v = (int64_t)wg * PP_T + tid; v < a.n_u; v += (int64_t)nwg * PP_T)
        if (a.inv_ptr[v] == a.inv_ptr[v + 1]) av.x[v] = Real(0);

    // Exchange A number ep (first wave): z of the own entries, the workgroup's partials of r.r and r.z.  A
    // single workgroup leaves the partials in LDS instead.
    auto publish_a = [&](uint32_t ep) {
        Real v[2] = {Real(0), Real(0)};
#pragma unroll
        for (int k = 0; k < PP_E; ++k) {
            if (op[k] >= 0 && nwg > 1) {                                // 0 where the entry is no unknown
#pragma unroll
                for (int h = 0; h < W; ++h) ll_put(xz + ow[k] + h * GW, L::part(z[k], h), ep);
            }
            if (counts[k]) { v[0] += r[k] * r[k]; v[1] += r[k] * z[k]; }
        }
        wave_sums(v);
        if (nwg > 1) xA.put(v, ep, lane);
        else if (lane == 0) { sA[0] = v[0]; sA[1] = v[1]; }
    };
    if (wave == 0) publish_a(1);

    Real bnorm = Real(1), best = INFINITY, rz_old = Real(1), inv_old = Real(1);
    int bestk = 0, conv_at = 0, n = 0;
    bool failed = false;
    for (;; ++n) {
        const uint32_t ep = (uint32_t)n + 1;
        // ---- A: the sums of the partials (second wave) and z at the column images (all)
        if (nwg > 1) {
            bool good = true;
            if (wave == 1) {
                Real v[2] = {Real(0), Real(0)};
                good = xA.relay(w.limit, ep, lane) && xA.get(w.limit, ep, lane, v);
                wave_sums(v);
                if (lane == 0) { sA[0] = v[0]; sA[1] = v[1]; }
            }
            good = pp_wait(w.limit, [&]() {
                uint64_t raw[PP_K][W];
                bool all = true;
#pragma unroll
                for (int k = 0; k < PP_K; ++k)
                    if (k < nk && cw[k] >= 0)
#pragma unroll
                        for (int h = 0; h < W; ++h) raw[k][h] = ll_get(xz + cw[k] + h * GW);
#pragma unroll
                for (int k = 0; k < PP_K; ++k)
                    if (k < nk && cw[k] >= 0) {
#pragma unroll
                        for (int h = 0; h < W; ++h) all = all && (uint32_t)(raw[k][h] >> 32) == ep;
                        zc[k] = L::join(raw[k]);
                    }
                return all;
            }) && good;
            if (!good) sFailA = 1;
        } else if (w.limit <= 0) {
            sFailA = 1;
        }
        __syncthreads();
        const Real rr = sA[0], rz = sA[1];
        if (sFailA | sFailB) { failed = true; break; }
        const Real beta = n > 0 ? div_by(rz, rz_old, inv_old) : Real(0);
#pragma unroll
        for (int k = 0; k < PP_K; ++k)
            if (k < nk && cw[k] >= 0) sP[tid + k * PP_T] = pdir(zc[k], sP[tid + k * PP_T], beta);
        if (wave == 0)
#pragma unroll
            for (int k = 0; k < PP_E; ++k)
                if (op[k] >= 0) { p[k] = pdir(z[k], p[k], beta); sP[op[k]] = p[k]; }
        __syncthreads();
        // ---- A p at the own rows: lane group (row, part) takes every gpr-th block of its row
        Real acc[2] = {Real(0), Real(0)};
        {
            Real xk[NBR + 1], xh[NBR + 1];
#pragma unroll
            for (int k = 0; k < NBR; ++k)
                if (k < nbr) {
                    xk[k] = sP[bx[k] + (tid & 15)];
                    if constexpr (DM > 16) xh[k] = sP[bx[k] + 16 + (tid & 15)];
                }
#pragma unroll
            for (int k = 0; k < NBR; ++k)
                if (k < nbr) {
                    pp_cols<0, DM>([&](int c) { return B[k][c]; }, xk[k], acc);
                    if constexpr (DM > 16) pp_cols<16, DM>([&](int c) { return B[k][c]; }, xh[k], acc);
                }
            for (int b = ls0 + part; b < ls1; b += gpr) {
                const Real* px = sP + sCidx[b];
                const Real* Bl = sS + b * dd + (j < d ? j : 0);
                auto col = [&](int c) { return Bl[min(c, d - 1) * d]; };   // past d, x is 0
                pp_cols<0, DM>(col, px[tid & 15], acc);
                if constexpr (DM > 16) pp_cols<16, DM>(col, px[16 + (tid & 15)], acc);
            }
        }
        sY[tid] = acc[0] + acc[1];
        rz_old = rz > Real(1e-32) ? rz : Real(1e-32);                   // the next update's beta divides by it
        inv_old = Real(1) / rz_old;
        // the end of update n - 1 (ba_solver.py:1222-1236); at n = 0 the norm of b
        const Real rnorm = sqrt(rr);
        bool stop = false;
        if (n == 0) {
            bnorm = rnorm > Real(1e-12) ? rnorm : Real(1e-12);          // torch.norm(b).clamp(min=1e-12)
        } else {
            if (rnorm < best) {
                best = rnorm;
                bestk = n;
#pragma unroll
                for (int k = 0; k < PP_E; ++k) xb_[k] = x[k];
            }
            const bool conv = rnorm <= Real(a.tol) * bnorm;
            if (conv) conv_at = n;
            stop = conv || !isfinite(rz) || n >= a.maxiter;
        }
        __syncthreads();
        if (stop) break;
        // ---- B: p.Ap = sum_e p_u(e) y_e + sum_u damp_u p_u^2, and the shared unknowns' sums
        if (wave == 1 && nwg > 1 && !xB.relay(w.limit, ep, lane)) sFailB = 1;
        if (wave == 0) {
            Real q[1 + NS], y[PP_E];
#pragma unroll
            for (int s = 0; s <= NS; ++s) q[s] = Real(0);
#pragma unroll
            for (int k = 0; k < PP_E; ++k) {
                y[k] = Real(0);
                if (u[k] >= 0) {
                    for (int c = 0; c < gpr; c += 8) {                  // 8 at a time in flight, no branches
                        Real t[8];
#pragma unroll
                        for (int h = 0; h < 8; ++h) t[h] = sY[oy[k] + min(c + h, gpr - 1) * GW];
#pragma unroll
                        for (int h = 0; h < 8; ++h) y[k] += c + h < gpr ? t[h] : Real(0);
                    }
                    q[0] += p[k] * y[k] + (counts[k] ? dmp[k] * p[k] * p[k] : Real(0));
#pragma unroll
                    for (int s = 0; s < NS; ++s) q[1 + s] += sh[k] == s ? y[k] : Real(0);
                }
            }
            wave_sums(q);
            if (nwg > 1) {
                xB.put(q, ep, lane);
                if (!xB.get(w.limit, ep, lane, q)) sFailB = 1;          // read after the next barrier
                wave_sums(q);
            }
            const Real alpha = rz / (q[0] > Real(1e-32) ? q[0] : Real(1e-32));
#pragma unroll
            for (int k = 0; k < PP_E; ++k)
                if (u[k] >= 0) {
                    Real ap = y[k];
#pragma unroll
                    for (int s = 0; s < NS; ++s) ap = sh[k] == s ? q[1 + s] : ap;
                    ap += dmp[k] * p[k];
                    x[k] += alpha * p[k];
                    r[k] -= alpha * ap;
                    z[k] = div_by(r[k], dA[k], iA[k]);
                }
            publish_a(ep + 1);
        }
        __syncthreads();         // nobody polls (and so crowds the memory path) before this workgroup has published
    }
    if (failed) {
        if (tid == 0) a.istate[6] = 1;
        return;
    }
#pragma unroll
    for (int k = 0; k < PP_E; ++k)
        if (u[k] >= 0 && counts[k]) av.x[u[k]] = conv_at ? x[k] : xb_[k];
    if (wg == 0 && tid == 0) {
        // the done flags as the launch sequence leaves them: both set after a stop before the cap
        const int last = (n + 1) & 1;
        a.istate[last] = 1;
        a.istate[1 - last] = n < a.maxiter;
        a.istate[IS_K] = n; a.istate[IS_CONV] = conv_at != 0; a.istate[IS_BESTK] = bestk;
        a.istate[IS_USEBEST] = conv_at == 0;
    }
}

// the flag "stopped before update n" (read once the launches before it have run) to memory the host reads
// (pinned host memory: a system-scope store)
__global__ void k_pcg_stopped(const int32_t* __restrict__ flag, int32_t* out) {
    if (threadIdx.x == 0) __hip_atomic_store(out, *flag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// result: x if converged else the best iterate
template <typename Real>
__global__ void __launch_bounds__(PCG_T) k_pcg_result(ba_pcg_args a) {
    const PcgV<Real> av(a);
    int64_t u = (int64_t)blockIdx.x * PCG_T + threadIdx.x;
    if (u < a.n_u && a.istate[IS_USEBEST]) av.x[u] = av.xbest[u];
}

}  // namespace ba

using namespace ba;

static inline unsigned nb_of(int64_t n) { return (unsigned)((n + PCG_T - 1) / PCG_T); }

// partial sums: PCG_NP per block of the update launch (one thread per unknown)
extern "C" int64_t ba_pcg_partials_size(int64_t n_u) {
    const int64_t m = n_u < 1 ? 1 : n_u;
    return PCG_NP * ((m + PCG_T - 1) / PCG_T);
}

namespace ba {
// The unknown-level rhs, damping and preconditioner diagonal (the first part of ba_pcg_solve), for
// the direct solve that shares them: rhs = P^T e_img, damp per leaf, diagA = clamp(P^T dg_img + damp).
int unknown_setup(const ba_pcg_args& a, hipStream_t st) {
    if (a.n_u == 0) return BA_OK;
    BA_REQUIRE(!a.real32, "the direct reduced solve runs in fp64 only (real32 = 0)");
    const unsigned nb = nb_of(a.n_u);
    const unsigned nbw = (unsigned)((a.n_u + PCG_T / 64 - 1) / (PCG_T / 64));
    hipLaunchKernelGGL(k_unk_setup<double>, dim3(nbw), dim3(PCG_T), 0, st, a);
    hipLaunchKernelGGL(k_leaf_max<double>, dim3(nb), dim3(PCG_T), 0, st, a);
    hipLaunchKernelGGL(k_leaf_damp<double>, dim3(nb), dim3(PCG_T), 0, st, a);
    BA_LAUNCHED();
    return BA_OK;
}
}  // namespace ba

// the launches of ba_pcg_solve_range (w null) and ba_pcg_solve_pairs_range in the working precision Real, GW
// lanes per block row
template <int GW, typename Real>
static void pcg_launch(const ba_pcg_args& a, const ba_pcg_pairs* w, int32_t it0, int32_t it1, int32_t finish,
                       int32_t* stopped_out, int64_t n_ent, hipStream_t st) {
    const unsigned nb = nb_of(a.n_u);
    const unsigned nbw = (unsigned)((a.n_u + PCG_T / 64 - 1) / (PCG_T / 64));        // wave per unknown (setup)
    if (it0 == 0) {                                  // the setup precedes iteration 0
        if (w != nullptr)
            hipLaunchKernelGGL(k_pcg_up_ptr, dim3(nb_of(a.n_imgs + 1)), dim3(PCG_T), 0, st, a.pair_i1, w->n_pairs,
                               a.n_imgs, w->up_ptr);
        else if (n_ent > 0)
            hipLaunchKernelGGL(k_rows_build<Real>, dim3((unsigned)((n_ent + PCG_T / 64 - 1) / (PCG_T / 64))),
                               dim3(PCG_T), 0, st, a, n_ent, GW);
        hipLaunchKernelGGL(k_unk_setup<Real>, dim3(nbw), dim3(PCG_T), 0, st, a);
        hipLaunchKernelGGL(k_leaf_max<Real>, dim3(nb), dim3(PCG_T), 0, st, a);
        hipLaunchKernelGGL(k_leaf_damp<Real>, dim3(nb), dim3(PCG_T), 0, st, a);
        hipLaunchKernelGGL(k_pcg_init<Real>, dim3(nb), dim3(PCG_T), 0, st, a);
        hipLaunchKernelGGL(k_pcg_init2<Real>, dim3(1), dim3(PCG_T), 0, st, a, (int)nb);
    }
    const dim3 rows((unsigned)a.n_imgs);
    auto decide = [&](int it) {                      // the decisions after update it - 1, then p_it or A p_it
        if (w != nullptr)
            hipLaunchKernelGGL(k_pcg_dir<Real>, dim3(nb_of((int64_t)a.n_imgs * PCG_GW)), dim3(PCG_T), 0, st, a, *w, it,
                               (int)nb);
        else
            hipLaunchKernelGGL((k_pcg_spmv<GW, Real>), rows, dim3(PCG_ST), 0, st, a, it, (int)nb);
    };
    for (int it = it0; it < it1; ++it) {
        decide(it);
        if (w != nullptr) {
            hipLaunchKernelGGL(k_pcg_pairs<Real>, rows, dim3(PCG_T), 0, st, a, *w, it);
            hipLaunchKernelGGL(k_pcg_cols<Real>, rows, dim3(PCG_T), 0, st, a, *w, it);
        }
        hipLaunchKernelGGL(k_pcg_update<Real>, dim3(nb), dim3(PCG_T), 0, st, a, it);
    }
    if (finish) {
        // the decisions after update it1 - 1 (after the last update, or a launch that returns at once once
        // the loop has stopped), then the result
        decide(it1);
        hipLaunchKernelGGL(k_pcg_result<Real>, dim3(nb), dim3(PCG_T), 0, st, a);
    } else if (stopped_out != nullptr) {
        hipLaunchKernelGGL(k_pcg_stopped, dim3(1), dim3(64), 0, st, a.istate + IS_DONE0 + (it1 & 1), stopped_out);
    }
}

static int pcg_range(const ba_pcg_args* args, const ba_pcg_pairs* w, int32_t it0, int32_t it1, int32_t finish,
                     int32_t* stopped_out, void* stream) {
    clear_error();
    BA_REQUIRE(args != nullptr, "null args");
    const ba_pcg_args& a = *args;
    hipStream_t st = (hipStream_t)stream;
    BA_REQUIRE(a.n_u >= 0 && a.d >= 1 && a.d <= 32 && a.maxiter >= 0, "bad sizes (1 <= d <= 32)");
    BA_REQUIRE(a.n_long >= 0 && a.n_long <= a.n_u && a.long_ptr != nullptr && a.long_idx != nullptr &&
                   (a.n_long == 0 || a.long_u != nullptr) && a.img_part != nullptr,
               "bad long-list unknowns or image partials");
    BA_REQUIRE(0 <= it0 && it0 <= it1 && it1 <= a.maxiter, "iteration range outside [0, maxiter]");
    if (a.n_u == 0) return BA_OK;
    {
        const void* need[] = {a.umap, a.inv_ptr, a.inv_src, a.leaf, a.row_ptr, a.row_ent, a.pair_i1, a.pair_i2,
                              a.S_pairs, a.e_img, a.dg_img, a.rhs, a.diagA, a.damp, a.x, a.xbest, a.r, a.z, a.p,
                              a.y_img, a.partials, a.state, a.istate};
        for (const void* q : need) BA_REQUIRE(q != nullptr, "null pointer in ba_pcg_args");
    }
    int64_t n_ent = 0;
    if (w != nullptr) {
        BA_REQUIRE(w->t != nullptr && w->p_img != nullptr && w->up_ptr != nullptr, "null pointer in ba_pcg_pairs");
        BA_REQUIRE(a.d <= PCG_GW, "the product by pair blocks takes d <= 16");
        BA_REQUIRE(w->n_pairs >= 0 && w->n_pairs < ((int64_t)1 << 30) && a.n_imgs >= 1, "bad pair or image count");
    } else {
        BA_REQUIRE(a.row_cap >= 0 && a.row_cap % (PCG_ST / 16) == 0, "row_cap must be a multiple of 8");
        n_ent = a.row_cap > 0 ? (int64_t)a.n_imgs * a.row_cap : a.n_row_ent;
        BA_REQUIRE(n_ent >= 0 && a.S_rows != nullptr && a.row_u != nullptr, "image-row block workspace missing");
    }
    if (a.d <= 16) {
        if (a.real32) pcg_launch<16, float>(a, w, it0, it1, finish, stopped_out, n_ent, st);
        else          pcg_launch<16, double>(a, w, it0, it1, finish, stopped_out, n_ent, st);
    } else {
        if (a.real32) pcg_launch<32, float>(a, w, it0, it1, finish, stopped_out, n_ent, st);
        else          pcg_launch<32, double>(a, w, it0, it1, finish, stopped_out, n_ent, st);
    }
    BA_LAUNCHED();
    return BA_OK;
}

extern "C" int ba_pcg_solve_range(const ba_pcg_args* args, int32_t it0, int32_t it1, int32_t finish,
                                  int32_t* stopped_out, void* stream) {
    return pcg_range(args, nullptr, it0, it1, finish, stopped_out, stream);
}

extern "C" int ba_pcg_solve_pairs_range(const ba_pcg_args* args, const ba_pcg_pairs* pairs, int32_t it0, int32_t it1,
                                        int32_t finish, int32_t* stopped_out, void* stream) {
    if (pairs == nullptr) {
        clear_error();
        BA_REQUIRE(false, "null pairs");
    }
    return pcg_range(args, pairs, it0, it1, finish, stopped_out, stream);
}

// Images per workgroup of the resident solve (0: it does not apply): of those whose rows fit, the one with the
// least estimated time of an iteration.  In cycles, measured at 8 to 1024 images: the two exchanges take about
// 5200 + 50 per workgroup up to 2 PP_G of them, and with relays 9500 + 45 per workgroup; a round of blocks takes 300
// from registers and 1000 from LDS (the register rounds of the other lane groups hide under it, so the longest row
// counts); entries beyond the first 64 another 500.
extern "C" int32_t ba_pcg_resident_plan(const int32_t* row_ptr, int32_t n_imgs, int32_t d, int32_t real32,
                                        int32_t n_shared, int32_t n_cu, int32_t* max_blk, int32_t* max_col) {
    if (row_ptr == nullptr || max_blk == nullptr || max_col == nullptr || n_imgs < 1 || n_imgs > 65535 || d < 1 ||
        d > 32 || n_shared < 0 || n_shared > PP_NS || n_cu < 1)
        return 0;
    const int gw = d <= 16 ? 16 : 32, nbr = pp_regs_of(pp_width(d), real32 != 0);
    const size_t R = real32 ? 4 : 8;
    int longest = 0, best = 0, best_cost = 0;
    for (int i = 0; i < n_imgs; ++i) longest = std::max(longest, row_ptr[i + 1] - row_ptr[i]);
    for (int m = std::min({n_imgs, PP_T / gw, 64 * PP_E / d}); m >= 1; --m) {
        const int nwg = (n_imgs + m - 1) / m, gpr = PP_T / gw / m;
        if (nwg > n_cu || nwg > PP_WG) break;
        int blk = 1, all = 1;
        for (int i = 0; i < n_imgs; i += m) {
            int more = 0;
            const int e = std::min(i + m, n_imgs);
            for (int q = i; q < e; ++q) more += std::max(0, row_ptr[q + 1] - row_ptr[q] - nbr * gpr);
            blk = std::max(blk, more);
            all = std::max(all, row_ptr[e] - row_ptr[i]);
        }
        const int col = std::min(all + m, n_imgs);
        if (col * gw > PP_K * PP_T) continue;
        if (pp_lds(d, gw, R, n_imgs, blk, col).total > PP_LDS) continue;
        const int rounds = (longest + gpr - 1) / gpr;
        const int cost = (nwg == 1 ? 0 : nwg <= 2 * PP_G ? 5200 + 50 * nwg : 9500 + 45 * nwg) +
                         300 * std::min(rounds, nbr) + 1000 * std::max(0, rounds - nbr) + (m * d > 64 ? 500 : 0);
        if (best == 0 || cost < best_cost) {
            best = m;
            best_cost = cost;
            *max_blk = blk;
            *max_col = col;
        }
    }
    return best;
}

extern "C" int64_t ba_pcg_resident_words(int32_t n_imgs, int32_t d, int32_t real32, int32_t m) {
    if (n_imgs < 1 || d < 1 || d > 32 || m < 1) return -1;
    const int64_t gw = d <= 16 ? 16 : 32, nwg = (n_imgs + m - 1) / m;
    if (nwg > PP_WG) return -1;
    if (real32) return n_imgs * gw + PpSums<2, float>::words_of((int)nwg) + PpSums<1 + PP_NS, float>::words_of((int)nwg);
    return 2 * n_imgs * gw + PpSums<2, double>::words_of((int)nwg) + PpSums<1 + PP_NS, double>::words_of((int)nwg);
}

template <int GW, int DM, int NS, typename Real>
static int resident_launch(ba_pcg_args a, ba_pcg_resident w, hipStream_t st) {
    const unsigned nb = nb_of(a.n_u);
    const unsigned nbw = (unsigned)((a.n_u + PCG_T / 64 - 1) / (PCG_T / 64));
    const int64_t nw = ba_pcg_resident_words(a.n_imgs, a.d, a.real32, w.m);
    const void* k = (const void*)k_pcg_resident<GW, DM, NS, Real>;
    const size_t lds = pp_lds(a.d, GW, sizeof(Real), a.n_imgs, w.max_blk, w.max_col).total;
    BA_REQUIRE(lds <= PP_LDS, "the image rows do not fit the LDS");
    BA_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_pp_clear, dim3(nb_of(nw)), dim3(PCG_T), 0, st, w.words, nw, a.istate);
    hipLaunchKernelGGL(k_unk_setup<Real>, dim3(nbw), dim3(PCG_T), 0, st, a);
    hipLaunchKernelGGL(k_leaf_max<Real>, dim3(nb), dim3(PCG_T), 0, st, a);
    hipLaunchKernelGGL(k_leaf_damp<Real>, dim3(nb), dim3(PCG_T), 0, st, a);
    BA_LAUNCHED();
    void* args[] = {&a, &w};
    const hipError_t e = hipLaunchCooperativeKernel(k, dim3((unsigned)((a.n_imgs + w.m - 1) / w.m)), dim3(PP_T), args,
                                                    (unsigned)lds, st);
    if (e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported) {
        // fewer CUs than the device reports (a process with a CU mask), or no cooperative launches: as after a
        // wait that gave up
        (void)hipGetLastError();
        hipLaunchKernelGGL(k_pp_refused, dim3(1), dim3(1), 0, st, a.istate);
        BA_LAUNCHED();
        return BA_OK;
    }
    BA_HIP(e);
    return BA_OK;
}

template <int NS, typename Real>
static int resident_width(const ba_pcg_args& a, const ba_pcg_resident& w, hipStream_t st) {
    switch (pp_width(a.d)) {
        case 9: return resident_launch<16, 9, NS, Real>(a, w, st);
        case 13: return resident_launch<16, 13, NS, Real>(a, w, st);
        case 16: return resident_launch<16, 16, NS, Real>(a, w, st);
        case 20: return resident_launch<32, 20, NS, Real>(a, w, st);
        case 25: return resident_launch<32, 25, NS, Real>(a, w, st);
        default: return resident_launch<32, 32, NS, Real>(a, w, st);
    }
}

extern "C" int ba_pcg_solve_resident(const ba_pcg_args* args, const ba_pcg_resident* res, void* stream) {
    clear_error();
    BA_REQUIRE(args != nullptr && res != nullptr, "null args");
    const ba_pcg_args& a = *args;
    const ba_pcg_resident& w = *res;
    BA_REQUIRE(a.n_u >= 1 && a.n_imgs >= 1 && a.n_imgs <= 65535 && a.d >= 1 && a.d <= 32 && a.maxiter >= 1 &&
                   a.maxiter < (1 << 30),
               "bad sizes (1 <= d <= 32, at most 65535 images, 1 <= maxiter < 2^30)");
    const void* need[] = {a.umap, a.inv_ptr, a.inv_src, a.leaf, a.row_ptr, a.row_ent, a.pair_i1, a.pair_i2, a.S_pairs,
                          a.e_img, a.dg_img, a.rhs, a.diagA, a.damp, a.x, a.state, a.istate, w.words};
    for (const void* q : need) BA_REQUIRE(q != nullptr, "null pointer in ba_pcg_args or ba_pcg_resident");
    const int gw = a.d <= 16 ? 16 : 32;
    BA_REQUIRE(w.n_shared >= 0 && w.n_shared <= PP_NS && (w.n_shared == 0 || w.shared_u != nullptr), "bad shared unknowns");
    BA_REQUIRE(w.m >= 1 && w.m <= PP_T / gw && w.m * a.d <= 64 * PP_E && (a.n_imgs + w.m - 1) / w.m <= PP_WG &&
                   w.max_blk >= 1 && w.max_col >= 1 && w.max_col * gw <= PP_K * PP_T,
               "bad resident plan");
    hipStream_t st = (hipStream_t)stream;
    if (w.n_shared == 0) return a.real32 ? resident_width<0, float>(a, w, st) : resident_width<0, double>(a, w, st);
    return a.real32 ? resident_width<PP_NS, float>(a, w, st) : resident_width<PP_NS, double>(a, w, st);
}

extern "C" int ba_pcg_solve(const ba_pcg_args* args, void* stream) {
    return ba_pcg_solve_range(args, 0, args != nullptr ? args->maxiter : 0, 1, nullptr, stream);
}

// The device address of host memory that the device can reach (pinned, mapped), or NULL: the target that
// ba_pcg_solve_range's stopped_out needs, checked before any kernel is handed it.
extern "C" void* ba_host_mapped_ptr(const void* host_ptr) {
    if (host_ptr == nullptr) return nullptr;
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, host_ptr) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (at.type != hipMemoryTypeHost || at.devicePointer == nullptr) return nullptr;
    return at.devicePointer;
}
