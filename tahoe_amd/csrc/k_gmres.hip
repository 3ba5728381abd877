// Restarted GMRES(m) with left preconditioning on the device: the linear
// solve of the Newton-Krylov solver (newton_krylov_solver, NLSolver_NK::
// Iterate/GMRES, NLSolver_NK.cpp:76-238).
//
// Same iteration as the reference: each restart cycle starts from
// r = M^-1 (b - A x), beta = |r|, and stops when the Givens-rotated residual
// |g_{j+1}| < rtol * beta of that cycle; Givens rotations [c s; -s c]; back
// substitution skipping |H_ii| <= 1e-14; at most maxit Arnoldi steps (3 n_eq
// when maxit <= 0).  The Arnoldi orthogonalisation is classical Gram-Schmidt
// applied twice (all j+1 projections of a pass in one multi-dot kernel and
// one update kernel) instead of the reference's modified Gram-Schmidt, which
// needs one reduction per basis vector; two CGS passes are as stable as MGS.
// M is the context's preconditioner (Jacobi as in the reference, or block
// Jacobi / multigrid).  The small Hessenberg work runs on the host.  Vectors
// live in node space [nnd][3] (prescribed dofs zero throughout).
#include <cmath>
#include <cstring>

#include "tg_internal.h"

namespace tg {

namespace {

constexpr int GB = 256;   // threads per block
constexpr int GNB = 512;  // blocks of the partial-sum kernels

inline unsigned nblocks(long n) { return (unsigned)((n + GB - 1) / GB); }

// y = A x on the block operator (storage MT, FP64 sums), or y = M A x with m,
// the point Jacobi preconditioner 1/diag.  A slice a workgroup, its NW waves
// share the row's slots and wave 0 adds their sums in order: nine waves to 640
// slices, three beyond (as the PCG's products, k_pcg.hip).  With a lane per row,
// a chain of 27 blocks, problems of 64 to 576 elements took 13.9 us here and 3.0
// more for 1/diag, and take 5.1 (their steps are bound by the launches); a
// correction of 30^3 elements 2.66 -> 2.43 ms, 50^3 mixed 5.42 -> 5.10 ms.
template <class MT, int NW>
__global__ void __launch_bounds__(64 * NW) k_gm_spmv(int nnd, const int* __restrict__ sbase,
                                                     const int* __restrict__ swidth, const int* __restrict__ col,
                                                     const MT* __restrict__ val, const double* __restrict__ m,
                                                     const double* __restrict__ x, double* __restrict__ y)
{
    __shared__ double red[NW][3][64];
    const int s = blockIdx.x, l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int a = 64 * s + l;
    const bool own = a < nnd;
    const long b0 = sbase[s];
    const int w = swidth[s], per = (w + NW - 1) / NW;
    const int q1 = min(w, (wv + 1) * per);
    double yi[3] = {0.0, 0.0, 0.0};
    // padding slots hold zeros and multiply the row's own entries
#pragma unroll 3
    for (int q = wv * per; q < q1; q++) {
        const long blk = b0 + q;
        const int cr = col[blk * 64 + l];
        const int c = cr >= 0 ? cr : own ? a : 0;
        const double x0 = x[3L * c], x1 = x[3L * c + 1], x2 = x[3L * c + 2];
        const MT* v = val + blk * 576 + l;
#pragma unroll
        for (int i = 0; i < 3; i++)
            yi[i] += (double)v[192 * i] * x0 + (double)v[192 * i + 64] * x1 + (double)v[192 * i + 128] * x2;
    }
#pragma unroll
    for (int i = 0; i < 3; i++) red[wv][i][l] = yi[i];
    __syncthreads();
    if (wv > 0 || !own) return;
    for (int j = 1; j < NW; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) yi[i] += red[j][i][l];
#pragma unroll
    for (int i = 0; i < 3; i++) y[3L * a + i] = m ? m[3L * a + i] * yi[i] : yi[i];
}

// z = M^-1 y for the point and block Jacobi preconditioners
__global__ void __launch_bounds__(GB) k_gm_jacobi(long n3, const double* __restrict__ dinv, const double* __restrict__ y,
                                                  double* __restrict__ z)
{
    const long k = (long)blockIdx.x * GB + threadIdx.x;
    if (k < n3) z[k] = dinv[k] * y[k];
}

__global__ void __launch_bounds__(GB) k_gm_block(int nnd, const double* __restrict__ binv, const double* __restrict__ y,
                                                 double* __restrict__ z)
{
    const int a = blockIdx.x * GB + threadIdx.x;
    if (a >= nnd) return;
    const double* b = binv + 9L * a;
    const double r0 = y[3L * a], r1 = y[3L * a + 1], r2 = y[3L * a + 2];
#pragma unroll
    for (int i = 0; i < 3; i++) z[3L * a + i] = b[3 * i] * r0 + b[3 * i + 1] * r1 + b[3 * i + 2] * r2;
}

// w = b - w
__global__ void __launch_bounds__(GB) k_gm_bminus(long n3, const double* __restrict__ b, double* __restrict__ w)
{
    const long k = (long)blockIdx.x * GB + threadIdx.x;
    if (k < n3) w[k] = b[k] - w[k];
}

// part[i][blk] = partial of V_i . w for vector i = blockIdx.y (V_i = V + i * n3).
// A workgroup per run and vector: one that goes through the vectors in turn,
// two barriers each, took 29 us at the end of a cycle of 100 steps on small
// problems (64 to 576 elements, mean of all steps 7.7 us) and takes 2.4 so.
__global__ void __launch_bounds__(GB) k_gm_mdot(long n3, const double* __restrict__ V, const double* __restrict__ w,
                                                double* __restrict__ part)
{
    __shared__ double red[GB / 64];
    const double* v = V + (long)blockIdx.y * n3;
    double s = 0.0;
    for (long k = (long)blockIdx.x * GB + threadIdx.x; k < n3; k += (long)gridDim.x * GB) s += v[k] * w[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int q = 0; q < GB / 64; q++) t += red[q];
        part[(long)blockIdx.y * gridDim.x + blockIdx.x] = t;
    }
}

// out[i] = host[i] = sum of part[i][0..np) (one block per i, fixed order); host
// is pinned memory
__global__ void __launch_bounds__(GB) k_gm_fin(const double* __restrict__ part, int np, double* __restrict__ out,
                                               double* __restrict__ host)
{
    __shared__ double red[GB / 64];
    const int i = blockIdx.x;
    double s = 0.0;
    for (int k = threadIdx.x; k < np; k += GB) s += part[(long)i * np + k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int q = 0; q < GB / 64; q++) t += red[q];
        out[i] = t;
        host[i] = t;
    }
}

// w -= sum_i h[i] V_i  (sign = -1), or x += sum_i h[i] V_i (sign = +1)
__global__ void __launch_bounds__(GB) k_gm_combine(long n3, const double* __restrict__ V, int j1,
                                                   const double* __restrict__ h, double sign, double* __restrict__ w)
{
    const long k = (long)blockIdx.x * GB + threadIdx.x;
    if (k >= n3) return;
    double s = 0.0;
#pragma unroll 8
    for (int i = 0; i < j1; i++) s += h[i] * V[(long)i * n3 + k];
    w[k] += sign * s;
}

// v = w * s
__global__ void __launch_bounds__(GB) k_gm_scale(long n3, const double* __restrict__ w, double s, double* __restrict__ v)
{
    const long k = (long)blockIdx.x * GB + threadIdx.x;
    if (k < n3) v[k] = s * w[k];
}

}  // namespace

template <class MT>
static void gmres_t(tg_ctx* c, const MT* val, const double* b, double* x, double rtol, int maxit, tg_lin_stats* st)
{
    const int nnd = c->nnd;
    const long n3 = 3L * nnd;
    const int m = c->gmres_restart;
    Gmres& G = c->gm;
    if (G.m != m || G.n3 != n3) {
        G.V.alloc((size_t)(m + 1) * n3);
        G.w.alloc(n3);
        G.q.alloc(n3);
        G.part.alloc((size_t)(m + 1) * GNB);
        G.h.alloc(2 * (m + 1) + 1);
        G.m = m;
        G.n3 = n3;
    }
    if (maxit <= 0) maxit = 3 * c->n_eq;
    const unsigned vb = nblocks(n3), nb = (unsigned)((nnd + GB - 1) / GB);
    const unsigned pb = (unsigned)std::min<long>(GNB, std::max<long>(1, (n3 + GB - 1) / GB));
    auto spmv = [&](const double* in, const double* dinv, double* out) {
        TimedRegion tr(c, T_SPMV);
        const unsigned ns = (unsigned)((nnd + 63) / 64);
        auto go = [&](auto kernel, int nw) {
            hipLaunchKernelGGL(kernel, dim3(ns), dim3(64 * nw), 0, c->stream, nnd, c->op.d_slice_base.p,
                               c->op.d_slice_width.p, c->op.d_col.p, val, dinv, in, out);
        };
        if (nnd <= 64 * 640)
            go(k_gm_spmv<MT, 9>, 9);
        else
            go(k_gm_spmv<MT, 3>, 3);
    };
    auto precondition = [&](const double* in, double* out) {
        TimedRegion tr(c, c->precond == TG_PC_AMG ? T_PRECOND : T_VECTOR);
        if (c->precond == TG_PC_AMG)
            amg_vcycle(c, in, out, nullptr);
        else if (c->precond == TG_PC_BLOCK_JACOBI)
            hipLaunchKernelGGL(k_gm_block, dim3(nb), dim3(GB), 0, c->stream, nnd, c->vbinv.p, in, out);
        else
            hipLaunchKernelGGL(k_gm_jacobi, dim3(vb), dim3(GB), 0, c->stream, n3, c->vdinv.p, in, out);
    };
    // An Arnoldi step leaves its projections and its norm in G.h and in pinned
    // memory: two passes of m + 1 and one value (m is at most 1,000).  The host
    // needs them only at the end of the step, so a step has one wait (three and
    // three copies before; with k_gm_mdot, a Newton solve of 64, 225 and 576
    // elements: 11.0 -> 5.7, 17.8 -> 8.2 and 22.0 -> 9.6 ms).
    const int nh = 2 * (m + 1) + 1;
    if ((size_t)nh > HOST_STAGE) fail(TG_OUT_OF_RANGE, "GMRES restart exceeds the staging buffer");
    const double* hh = c->hstage;
    // V_0..V_{j1-1} . w -> G.h[at ..]
    auto project = [&](int j1, const double* V, const double* w, int at) {
        TimedRegion tr(c, T_VECTOR);
        hipLaunchKernelGGL(k_gm_mdot, dim3(pb, (unsigned)j1), dim3(GB), 0, c->stream, n3, V, w, G.part.p);
        hipLaunchKernelGGL(k_gm_fin, dim3(j1), dim3(GB), 0, c->stream, G.part.p, (int)pb, G.h.p + at,
                           c->hstage + at);
    };
    auto orthogonalise = [&](int j1, int at) {
        project(j1, G.V.p, G.w.p, at);
        TimedRegion tr(c, T_VECTOR);
        hipLaunchKernelGGL(k_gm_combine, dim3(vb), dim3(GB), 0, c->stream, n3, G.V.p, j1, G.h.p + at, -1.0, G.w.p);
    };
    std::vector<double> H((size_t)(m + 1) * m), g((size_t)m + 1), cs((size_t)m), sn((size_t)m), y((size_t)m);
    auto HH = [&](int i, int j) -> double& { return H[(size_t)i * m + j]; };
    TG_HIP(hipMemsetAsync(x, 0, sizeof(double) * n3, c->stream));
    int total = 0, steps = 0;
    bool done = false;
    double beta0 = -1.0, last = 0.0;
    while (!done && total < maxit) {
        // r = M^-1 (b - A x)
        spmv(x, nullptr, G.q.p);
        {
            TimedRegion tr(c, T_VECTOR);
            hipLaunchKernelGGL(k_gm_bminus, dim3(vb), dim3(GB), 0, c->stream, n3, b, G.q.p);
        }
        precondition(G.q.p, G.w.p);
        project(1, G.w.p, G.w.p, nh - 1);
        TG_HIP(hipStreamSynchronize(c->stream));
        const double beta = std::sqrt(hh[nh - 1]);
        if (beta0 < 0.0) beta0 = beta;
        last = beta;
        if (beta == 0.0) {
            done = true;
            break;
        }
        const double tol_abs = rtol * beta;
        if (tol_abs == 0.0) {
            done = true;
            break;
        }
        hipLaunchKernelGGL(k_gm_scale, dim3(vb), dim3(GB), 0, c->stream, n3, G.w.p, 1.0 / beta, G.V.p);
        std::fill(g.begin(), g.end(), 0.0);
        g[0] = beta;
        int j_end = 0;
        for (int j = 0; j < m && total < maxit; j++, total++) {
            j_end = j;
            steps++;
            const bool point = c->precond != TG_PC_AMG && c->precond != TG_PC_BLOCK_JACOBI;
            spmv(G.V.p + (long)j * n3, point ? c->vdinv.p : nullptr, point ? G.w.p : G.q.p);
            if (!point) precondition(G.q.p, G.w.p);
            // two classical Gram-Schmidt passes
            orthogonalise(j + 1, 0);
            orthogonalise(j + 1, m + 1);
            project(1, G.w.p, G.w.p, nh - 1);
            TG_HIP(hipStreamSynchronize(c->stream));
            for (int i = 0; i <= j; i++) HH(i, j) = hh[i] + hh[m + 1 + i];
            const double hn = std::sqrt(hh[nh - 1]);
            HH(j + 1, j) = hn;
            if (hn > 0.0)
                hipLaunchKernelGGL(k_gm_scale, dim3(vb), dim3(GB), 0, c->stream, n3, G.w.p, 1.0 / hn,
                                   G.V.p + (long)(j + 1) * n3);
            for (int i = 0; i < j; i++) {
                const double t = cs[i] * HH(i, j) + sn[i] * HH(i + 1, j);
                HH(i + 1, j) = -sn[i] * HH(i, j) + cs[i] * HH(i + 1, j);
                HH(i, j) = t;
            }
            const double den = std::sqrt(HH(j, j) * HH(j, j) + HH(j + 1, j) * HH(j + 1, j));
            cs[j] = den > 0.0 ? HH(j, j) / den : 1.0;
            sn[j] = den > 0.0 ? HH(j + 1, j) / den : 0.0;
            double t = cs[j] * HH(j, j) + sn[j] * HH(j + 1, j);
            HH(j + 1, j) = -sn[j] * HH(j, j) + cs[j] * HH(j + 1, j);
            HH(j, j) = t;
            t = cs[j] * g[j] + sn[j] * g[j + 1];
            g[j + 1] = -sn[j] * g[j] + cs[j] * g[j + 1];
            g[j] = t;
            last = std::fabs(g[j + 1]);
            if (last < tol_abs) {
                j_end = j;
                done = true;
                break;
            }
        }
        for (int i = j_end; i >= 0; i--) {
            double sum = g[i];
            for (int l = i + 1; l <= j_end; l++) sum -= HH(i, l) * y[l];
            y[i] = std::fabs(HH(i, i)) > 1.0e-14 ? sum / HH(i, i) : 0.0;
        }
        TG_HIP(hipMemcpyAsync(G.h.p, y.data(), sizeof(double) * (j_end + 1), hipMemcpyHostToDevice, c->stream));
        {
            TimedRegion tr(c, T_VECTOR);
            hipLaunchKernelGGL(k_gm_combine, dim3(vb), dim3(GB), 0, c->stream, n3, G.V.p, j_end + 1, G.h.p, 1.0, x);
        }
        TG_HIP(hipStreamSynchronize(c->stream));  // y outlives its copy
    }
    TG_HIP(hipGetLastError());
    if (st) {
        st->iterations = steps;
        st->converged = done ? 1 : 0;
        st->rel_residual = beta0 > 0.0 ? last / beta0 : 0.0;
    }
}

void gmres_solve(tg_ctx* c, const double* b, double* x, double rtol, int maxit, tg_lin_stats* st)
{
    if (c->seg.nseg != 1) fail(TG_BAD_INPUT, "GMRES needs a single problem (no segments)");
    if (mixed_operator(c))
        gmres_t<float>(c, c->op.d_val32.p, b, x, rtol, maxit, st);
    else
        gmres_t<double>(c, c->op.d_val.p, b, x, rtol, maxit, st);
}

}  // namespace tg
