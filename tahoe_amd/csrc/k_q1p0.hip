// Q1P0 mean-dilatation hexahedron kernels: element forces and the
// forward-difference stiffness blocks, written to the buffers that k_rows.hip
// gathers by nodes and matrix rows (SimoQ1P0,
// tahoe/src/elements/continuum/solid/SimoQ1P0.cpp).
//
// Element force of a state (x current coordinates, u displacements),
// ComputeInternalForce (SimoQ1P0.cpp:390-439) with E = 0 and no phase field:
//   f = sum_q w det_q (J_bar/J_q) B_bar_q^T sigma(F_bar_q)
//   SetMeanGradient (:661-686): H = sum w det0, v = sum w det,
//     mean = sum (w det/v) dN/dx
//   F_bar = (v/(H J))^(1/3) F, F from reference derivatives (:286-296)
//   B_bar from SolidElementT::Set_B_bar (SolidElementT.cpp:1011-1041)
// With s = det_q J_bar/J_q, p = tr sigma / 3 and B_bar's mean dilatation
// written out, node a gets
//   f_a = sum_q s (sigma - p 1) dN_a/dx + mean_a sum_q s p,
// so the mean gradient enters once, after the sum, and the pressure's parts
// that cancel between B and B_bar are never formed.
#include "tg_internal.h"
#include "tg_kinematics.h"
#include "tg_element.h"

namespace tg {

__device__ __forceinline__ double allreduce8(double v)
{
    v += __shfl_xor(v, 1);
    v += __shfl_xor(v, 2);
    v += __shfl_xor(v, 4);
    return v;
}

// Stress of one integration point at F (det J > 0), with the element's mean
// dilatation (v/H)^(1/3): dev = sigma(F_bar) - p 1, p, and s / det =
// J_bar / J.  Returns false when the material refuses F_bar.
template <int MAT>
__device__ __forceinline__ bool q1p0_stress(double F[9], double J, double vH, double mu, double kappa, double dev[6],
                                            double& p, double& ratio)
{
    const double sc = cbrt(vH / J);
#pragma unroll
    for (int k = 0; k < 9; k++) F[k] *= sc;
    // the material sees F_bar (SimoQ1P0 passes it on as the mechanical F)
    const double Jbar = det3(F);
    double Jk, kin[6];
    const bool ok = material_stress<MAT>(mu, kappa, F, Jbar, Jk, kin, dev);
    p = (dev[0] + dev[1] + dev[2]) / 3.0;
    dev[0] -= p;
    dev[1] -= p;
    dev[2] -= p;
    ratio = Jbar / J;
    return ok;
}

// Residual: -f into the force buffer (FormKd(-1), SimoQ1P0.cpp:528-582).  8
// lanes per element, lane q its integration point; each node's sums over the
// points are scattered to the lane that owns the node (two reduce-scatters of
// 24 values, where the mean gradient used to be reduced to every lane).
template <int MAT>
__global__ void __launch_bounds__(256) k_q1p0_forces(int nel, const int* __restrict__ conn,
                                                     const unsigned* __restrict__ perm, const int* __restrict__ emat,
                                                     const double2* __restrict__ props,
                                                     const double* __restrict__ X, const double* __restrict__ U,
                                                     double* __restrict__ fe, int* __restrict__ status,
                                                     const int* __restrict__ slice_seg, int* __restrict__ segstat)
{
    __shared__ double sX[32][8][3], su[32][8][3];
    const int t = threadIdx.x, le = t >> 3, q = t & 7;
    const int e = blockIdx.x * 32 + le;
    const bool valid = e < nel;
    int node = 0;
    if (valid) {
        node = conn[8L * e + q];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            sX[le][q][c] = X[3L * node + c];
            su[le][q][c] = U[3L * node + c];
        }
    } else {
        // inert unit element so the shuffled element reductions stay finite
#pragma unroll
        for (int c = 0; c < 3; c++) {
            sX[le][q][c] = c == 0 ? (RA[q] + 1.0) * 0.5 : (c == 1 ? (SA[q] + 1.0) * 0.5 : (TA[q] + 1.0) * 0.5);
            su[le][q][c] = 0.0;
        }
    }
    __syncthreads();
    double2 mk = make_double2(1.0, 1.0);
    if (valid) mk = props[emat[e]];
    double d[3][8], F[9], J, det0;
    bool ok;
    parent_derivs(q, d);
    {
        double j0[9], ji[9], g0[3][8];
        jacobian([&](int a, int c) { return sX[le][a][c]; }, d, j0);
        det0 = det3(j0);
        ok = det0 > 0.0;
        inv3(j0, det0, ji);
        spatial_derivs(ji, d, g0);
        deformation_gradient([&](int a, int c) { return su[le][a][c]; }, g0, F);
        J = det3(F);
        ok &= J > 0.0;
    }
    double jc[9], jci[9], n[3][8];
    jacobian([&](int a, int c) { return sX[le][a][c] + su[le][a][c]; }, d, jc);
    const double det = det3(jc);
    ok &= det > 0.0;
    inv3(jc, det, jci);
    spatial_derivs(jci, d, n);
    const double H = allreduce8(det0);  // weights 1
    const double v = allreduce8(det);
    double r[24], mean[3], f[3];
#pragma unroll
    for (int a = 0; a < 8; a++)
#pragma unroll
        for (int i = 0; i < 3; i++) r[3 * a + i] = ok ? det * n[i][a] : 0.0;
    reduce_scatter8(r, q, mean);
    double dev[6], p, ratio;
    ok &= q1p0_stress<MAT>(F, J, v / H, mk.x, mk.y, dev, p, ratio);
    const double s = det * ratio;
#pragma unroll
    for (int a = 0; a < 8; a++) {
        const double nx = n[0][a], ny = n[1][a], nz = n[2][a];
        r[3 * a + 0] = ok ? s * (dev[0] * nx + dev[5] * ny + dev[4] * nz) : 0.0;
        r[3 * a + 1] = ok ? s * (dev[5] * nx + dev[1] * ny + dev[3] * nz) : 0.0;
        r[3 * a + 2] = ok ? s * (dev[4] * nx + dev[3] * ny + dev[2] * nz) : 0.0;
    }
    reduce_scatter8(r, q, f);
    const double P = allreduce8(ok ? s * p : 0.0) / v;
    if (valid) {
        double* out = fe + 3 * (8L * e + rank_of(perm[e], q));
#pragma unroll
        for (int i = 0; i < 3; i++) out[i] = -(f[i] + mean[i] * P);
    }
    if (valid && !ok) {
        // the context's flag, and the flag of the element's problem in a batch
        atomicOr(status, 7);
        atomicOr(&segstat[slice_seg[node >> 6]], 7);
    }
}

// Stiffness: the reference's forward difference (FormStiffness,
// SimoQ1P0.cpp:446-525): for each element dof col, u_col += eps and x_col +=
// eps, K(:,col) = (f(u+eps) - f(u))/eps, eps = 1e-7; its upper entries (row <=
// col) go to the block buffer.
//
// One lane per perturbed state: 25 lanes (24 columns and the unperturbed
// one) per element, QE elements per workgroup, each lane looping over the
// integration points.  A perturbed coordinate changes one row of the Jacobian
// and of F by a multiple of one node's derivatives, so the lanes share the
// element's unperturbed Jacobians, F and reference derivatives in LDS, and no
// value crosses lanes until f(u) is subtracted.  (One integration point per
// lane and 25 evaluations in sequence kept 8 lanes per element busy, 7
// workgroups for a colour of a 12^3 cube, and spent 93 shuffles an
// evaluation.)  Bound by FP64 issue: 141 k elements 0.70 ms, 1,728 elements 22
// us; the colour passes took 4.3 and 1.19 ms.
constexpr int QE = 10;
constexpr int QIP = 43;  // per integration point: Jacobian 9, F 9, dN/dX 24, det0

template <int MAT>
__global__ void __launch_bounds__(256) k_q1p0_blocks(int nel, const int* __restrict__ conn,
                                                     const unsigned* __restrict__ perm, const int* __restrict__ emat,
                                                     const double2* __restrict__ props,
                                                     const double* __restrict__ X, const double* __restrict__ U,
                                                     double* __restrict__ eb, int* __restrict__ status)
{
    __shared__ double sX[QE][8][3], su[QE][8][3], sd[8][24], sf[QE][24];
    __shared__ double sip[QE * 8 * QIP > QE * 324 ? QE * 8 * QIP : QE * 324];
    const int t = threadIdx.x;
    const int e0 = blockIdx.x * QE;
    bool ok = true;
    if (t < 8 * QE) {
        const int le = t >> 3, q = t & 7;
        if (e0 + le < nel) {
            const int node = conn[8L * (e0 + le) + q];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                sX[le][q][c] = X[3L * node + c];
                su[le][q][c] = U[3L * node + c];
            }
        }
    }
    __syncthreads();
    if (t < 8 * QE) {
        const int le = t >> 3, q = t & 7;
        double d[3][8];
        parent_derivs(q, d);
        if (le == 0)
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int a = 0; a < 8; a++) sd[q][8 * k + a] = d[k][a];
        if (e0 + le < nel) {
            double j[9], ji[9], g[3][8], F[9];
            double* ip = sip + (le * 8 + q) * QIP;
            jacobian([&](int a, int c) { return sX[le][a][c]; }, d, j);
            const double det0 = det3(j);
            ok &= det0 > 0.0;
            inv3(j, det0, ji);
            spatial_derivs(ji, d, g);
            deformation_gradient([&](int a, int c) { return su[le][a][c]; }, g, F);
            jacobian([&](int a, int c) { return sX[le][a][c] + su[le][a][c]; }, d, j);
#pragma unroll
            for (int k = 0; k < 9; k++) {
                ip[k] = j[k];
                ip[9 + k] = F[k];
            }
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int a = 0; a < 8; a++) ip[18 + 8 * k + a] = g[k][a];
            ip[42] = det0;
        }
    }
    __syncthreads();
    const int le = t / 25, col = t - 25 * le;
    const bool on = t < 25 * QE && e0 + le < nel;
    const int pa = col < 24 ? col / 3 : 0, pi = col < 24 ? col % 3 : 0;
    const double eps = 1.0e-7;
    double f[24], mean[24];
    double v = 0.0;
    if (on) {
        const double2 mk = props[emat[e0 + le]];
        const double* ip0 = sip + le * 8 * QIP;
        // what the perturbation changes x and u by, as rounded
        const double x = sX[le][pa][pi] + su[le][pa][pi], u = su[le][pa][pi];
        const double ex = col < 24 ? (x + eps) - x : 0.0, eu = col < 24 ? (u + eps) - u : 0.0;
        const double ex0 = pi == 0 ? ex : 0.0, ex1 = pi == 1 ? ex : 0.0, ex2 = pi == 2 ? ex : 0.0;
        const double eu0 = pi == 0 ? eu : 0.0, eu1 = pi == 1 ? eu : 0.0, eu2 = pi == 2 ? eu : 0.0;
        auto current = [&](int q, double (&j)[9]) {
            const double* ip = ip0 + q * QIP;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double dk = sd[q][8 * k + pa];
                j[3 * k] = ip[3 * k] + ex0 * dk;
                j[3 * k + 1] = ip[3 * k + 1] + ex1 * dk;
                j[3 * k + 2] = ip[3 * k + 2] + ex2 * dk;
            }
        };
        double H = 0.0;
#pragma unroll 1
        for (int q = 0; q < 8; q++) {
            double j[9];
            current(q, j);
            const double det = det3(j);
            ok &= det > 0.0;
            v += det;
            H += ip0[q * QIP + 42];
        }
        const double vH = v / H;
#pragma unroll
        for (int k = 0; k < 24; k++) f[k] = mean[k] = 0.0;
        double P = 0.0;
#pragma unroll 1
        for (int q = 0; q < 8; q++) {
            const double* ip = ip0 + q * QIP;
            double j[9], c[9], F[9], dev[6], p, ratio;
            current(q, j);
            const double det = det3(j);
            inv3(j, 1.0, c);  // det times the inverse
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double gk = ip[18 + 8 * k + pa];
                F[3 * k] = ip[9 + 3 * k] + eu0 * gk;
                F[3 * k + 1] = ip[9 + 3 * k + 1] + eu1 * gk;
                F[3 * k + 2] = ip[9 + 3 * k + 2] + eu2 * gk;
            }
            const double J = det3(F);
            ok &= J > 0.0;
            ok &= q1p0_stress<MAT>(F, J, vH, mk.x, mk.y, dev, p, ratio);
            P += det * ratio * p;
#pragma unroll
            for (int k = 0; k < 6; k++) dev[k] *= ratio;
#pragma unroll
            for (int a = 0; a < 8; a++) {
                const double d0 = sd[q][a], d1 = sd[q][8 + a], d2 = sd[q][16 + a];
                // det dN_a/dx
                const double nx = c[0] * d0 + c[1] * d1 + c[2] * d2;
                const double ny = c[3] * d0 + c[4] * d1 + c[5] * d2;
                const double nz = c[6] * d0 + c[7] * d1 + c[8] * d2;
                mean[3 * a] += nx;
                mean[3 * a + 1] += ny;
                mean[3 * a + 2] += nz;
                f[3 * a] += dev[0] * nx + dev[5] * ny + dev[4] * nz;
                f[3 * a + 1] += dev[5] * nx + dev[1] * ny + dev[3] * nz;
                f[3 * a + 2] += dev[4] * nx + dev[3] * ny + dev[2] * nz;
            }
        }
        P /= v;
#pragma unroll
        for (int k = 0; k < 24; k++) f[k] = ok ? f[k] + mean[k] * P : 0.0;
        if (col == 24)
#pragma unroll
            for (int k = 0; k < 24; k++) sf[le][k] = f[k];
    }
    __syncthreads();  // past the last read of sip, and f(u) is there
    if (on && col < 24) {
        const unsigned pm = perm[e0 + le];
        const int rb = rank_of(pm, pa);
        double* out = sip + 324 * le;
#pragma unroll
        for (int a = 0; a < 8; a++) {
            if (a > pa) continue;
            const int ra = rank_of(pm, a);
            double* b = out + 9 * pair_index(min(ra, rb), max(ra, rb));
#pragma unroll
            for (int i = 0; i < 3; i++)
                if (a < pa || i <= pi) b[ra <= rb ? 3 * i + pi : 3 * pi + i] = (f[3 * a + i] - sf[le][3 * a + i]) / eps;
        }
    }
    __syncthreads();
    const int n = 324 * min(QE, nel - e0);
    for (int x = t; x < n; x += 256) eb[324L * e0 + x] = sip[x];
    if (!ok) atomicOr(status, 7);
}

void launch_q1p0_forces(tg_ctx* c, const double* u)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((c->nel + 31) / 32), dim3(256), 0, c->stream, c->nel, c->dconn.p, c->r_perm.p,
                           c->dmat.p, c->dmatprops.p, c->dX.p, u, c->r_force.p, c->dstatus.p, c->seg.d_slice_seg.p,
                           c->seg.d_segstat.p);
    };
    if (c->material_model == TG_MAT_STVENANT)
        go(k_q1p0_forces<MAT_STVENANT>);
    else
        go(k_q1p0_forces<MAT_SIMO>);
    TG_HIP(hipGetLastError());
}

void launch_q1p0_blocks(tg_ctx* c, const double* u)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((c->nel + QE - 1) / QE), dim3(256), 0, c->stream, c->nel, c->dconn.p,
                           c->r_perm.p, c->dmat.p, c->dmatprops.p, c->dX.p, u, c->r_blocks.p, c->dstatus.p);
    };
    if (c->material_model == TG_MAT_STVENANT)
        go(k_q1p0_blocks<MAT_STVENANT>);
    else
        go(k_q1p0_blocks<MAT_SIMO>);
    TG_HIP(hipGetLastError());
}

}  // namespace tg
