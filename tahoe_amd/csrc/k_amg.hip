// Aggregation multigrid preconditioner: coarse operators, smoothers and the
// V-cycle on the device (the structure is built by tg_amg.cpp).
//
// Smoother: Chebyshev polynomial in D^-1 A (Adams, Brezina, Hu and
// Tuminaro, J. Comput. Phys. 188 (2003) 593-610; the three-term recurrence
// of Saad, Iterative Methods for Sparse Linear Systems, Alg. 12.1) on
// [lmax / 14, lmax], with lmax a power-iteration estimate of the largest
// eigenvalue of D^-1 A raised by 10 %.  Pre- and post-smoothing use the same
// polynomial and the coarse correction is a Galerkin product, so the V-cycle
// is a symmetric positive definite preconditioner for CG.  Matrices below
// the fine level are FP32 (a preconditioner needs no more); all vectors and
// sums are FP64.
#include <cmath>
#include <cstring>

#include "tg_internal.h"

namespace tg {

namespace {

constexpr int AB = 256;          // threads per block of the vector/level kernels
// Smoothing interval [lmax / CHEB_RATIO, lmax]: the coarse levels take what
// lies below.  PCG iterations of one Newton step (128^3 mixed / 64^3 FP64 / 24^3
// to 1e-10): ratio 30 94 / 82 / 141, 16 87 / 78 / 132, 12 87 / 78 / 131, 8 91 /
// 80 / 133, 4 101 / 87 / 148.
constexpr double CHEB_RATIO = 14.0;
// With one step (level_degree) the interval is [lmax / 4, lmax], a damped
// Jacobi step with 1.6 / lmax: 128^3 mixed, fine and first coarse level so,
// PCG iterations of a Newton step: ratio 4 109, 10 114; 96^3: 3 112, 4 112.
constexpr double JACOBI_RATIO = 4.0;
constexpr double CHEB_BOOST = 1.1;
constexpr int POWER_ITS = 12;

inline unsigned blocks_for(long n) { return (unsigned)((n + AB - 1) / AB); }

__device__ __forceinline__ bool skip(const double* done) { return done && *done != 0.0; }

// Level 0: the solver's sliced-ELL operator (3x3 blocks), one lane per node.
// add: y += the products of slots k0 .. k1 - 1 of the row of node t (lane l of
// the slice at b0).  Padding slots (column -1) hold zeros and multiply the
// row's own entries, so no branch stands between the loads.  NT: non-temporal
// loads, for an operator that the last-level cache cannot hold (op_streams).
template <class MT, bool NT>
struct Op0 {
    static constexpr int NC = 3;
    int n;
    const int* sbase;
    const int* swidth;
    const int* col;
    const MT* val;
    __device__ __forceinline__ void add(long b0, int k0, int k1, int l, int t, const double* __restrict__ x, double (&y)[3]) const
    {
#pragma unroll 3
        for (int q = k0; q < k1; q++) {
            const long blk = b0 + q;
            const int* pc = col + blk * 64 + l;
            const int cr = NT ? __builtin_nontemporal_load(pc) : *pc;
            const int c = cr < 0 ? t : cr;
            const MT* pv = val + blk * 576 + l;
            double u[9], xc[3];
#pragma unroll
            for (int m = 0; m < 9; m++) u[m] = (double)(NT ? __builtin_nontemporal_load(pv + 64 * m) : pv[64 * m]);
#pragma unroll
            for (int j = 0; j < 3; j++) xc[j] = x[3L * c + j];
#pragma unroll
            for (int r = 0; r < 3; r++)
#pragma unroll
                for (int j = 0; j < 3; j++) y[r] += u[3 * r + j] * xc[j];
        }
    }
};

// Levels >= 1: sliced 6x6 FP32 blocks, one lane per node and 6 outputs.  The
// values of a slot are kept as nine groups of four, a group's 64 lanes side by
// side (amg_at), so a lane takes a block by nine 16-byte loads; padding slots
// are zero.  SYM: a lower block (column below the row) is read as its upper
// partner's transpose, slot part[slot], of the same bits: half the level's
// values come from HBM and half from the caches.  16-byte loads make that pay:
// a partner's lanes start anywhere in a cache line, so a 256-byte load of 64
// floats takes three lines for two, one of 1 KB nine for eight.  65^3 nodes
// (1.07 GB): 236 us with 4-byte loads, 216 with 16-byte ones, 175 so; with
// 4-byte loads the symmetric read took 266.
template <bool SYM>
struct OpC {
    static constexpr int NC = 6;
    int n;
    const int* sbase;
    const int* swidth;
    const int* col;
    const int* part;
    const float* val;
    __device__ __forceinline__ void add(long b0, int k0, int k1, int l, int t, const double* __restrict__ x, double (&y)[6]) const
    {
#pragma unroll(SYM ? 3 : 1)
        for (int q = k0; q < k1; q++) {
            int e = (int)(b0 + q) * 64 + l;
            const int cr = col[e];
            const int c = cr < 0 ? t : cr;
            const bool tr = SYM && c < t;
            if (tr) e = part[e];
            float u[36];
            double xc[6];
#pragma unroll
            for (int m = 0; m < 9; m++) {
                const float4 g = *(const float4*)(val + amg_at(e, 4 * m));
                u[4 * m] = g.x;
                u[4 * m + 1] = g.y;
                u[4 * m + 2] = g.z;
                u[4 * m + 3] = g.w;
            }
#pragma unroll
            for (int j = 0; j < 6; j++) xc[j] = x[6L * c + j];
#pragma unroll
            for (int r = 0; r < 6; r++)
#pragma unroll
                for (int j = 0; j < 6; j++) y[r] += (double)(tr ? u[6 * j + r] : u[6 * r + j]) * xc[j];
        }
    }
};

// what follows a product q at dof j
struct EStore {  // y = A x
    double* y;
    __device__ __forceinline__ void operator()(long j, double q) const { y[j] = q; }
};
// Chebyshev step: r -= A d_prev; d_next = c1 d_prev + c2 D^-1 r; x += d_next
// (+ d_prev when the pass started from a nonzero x)
struct EStep {
    const double *dinv, *dprev, *coef;
    double *dnext, *r, *x;
    int ci, add_prev;
    __device__ __forceinline__ void operator()(long j, double q) const
    {
        const double ri = r[j] - q, dp = dprev[j];
        r[j] = ri;
        const double dn = coef[ci] * dp + coef[ci + 1] * dinv[j] * ri;
        dnext[j] = dn;
        x[j] += (add_prev ? dp : 0.0) + dn;
    }
};
// the first step of a pass from zero, d0 = D^-1 f / theta (k_amg_pre): r = f -
// A d0, then as above with x = d0 + d1
struct EFirst {
    const double *dinv, *f, *coef, *d0;
    double *dnext, *r, *x;
    __device__ __forceinline__ void operator()(long j, double q) const
    {
        const double ri = f[j] - q, dp = d0[j];
        r[j] = ri;
        const double dn = coef[1] * dp + coef[2] * dinv[j] * ri;
        dnext[j] = dn;
        x[j] = dp + dn;
    }
};
struct EResid {  // r -= A d
    double* r;
    __device__ __forceinline__ void operator()(long j, double q) const { r[j] -= q; }
};
struct EDefect {  // r = f - A x
    const double* f;
    double* r;
    __device__ __forceinline__ void operator()(long j, double q) const { r[j] = f[j] - q; }
};
struct EJacobi {  // x = x0 + D^-1 (f - A x0) / theta
    const double *dinv, *f, *coef, *x0;
    double* x;
    __device__ __forceinline__ void operator()(long j, double q) const { x[j] = x0[j] + coef[0] * dinv[j] * (f[j] - q); }
};
struct EPost {  // start of post-smoothing: r = f - A x; d0 = D^-1 r / theta
    const double *dinv, *f, *coef;
    double *r, *d0;
    __device__ __forceinline__ void operator()(long j, double q) const
    {
        const double ri = f[j] - q;
        r[j] = ri;
        d0[j] = coef[0] * dinv[j] * ri;
    }
};

// A product with a level's operator and what follows it: a slice a workgroup,
// its NW waves share the row's slots and wave 0 adds their sums in order.  A
// lane per row instead walks its 27 blocks alone: at 128^3 the coarse levels of
// 72, 12 and 2 slices took 30-40 us a product so and take 6-8 shared, 544 slices
// 38 and 27.  ranges: each XCD takes a contiguous range of slices.  The large levels are
// bound by what passes the L2s: 2.15 M nodes FP32, 2.3 GB, 452 us with a lane per
// row, 432 so when lower blocks came from their partners, 419 with three waves
// and non-temporal loads; 275 k nodes 76 with the partners, 48 without; 270 k
// nodes of 6 dofs (1.07 GB) 236 and, as OpC reads them now, 165 us.
template <class Op, int NW, class E>
__global__ void __launch_bounds__(64 * NW) k_amg_rows(Op op, const double* __restrict__ x, E e, int ranges,
                                                         const double* done)
{
    if (skip(done)) return;
    const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = ranges ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    if (s >= (op.n + 63) >> 6) return;
    const int t = 64 * s + l;
    const bool own = t < op.n;
    const long b0 = op.sbase[s];
    const int w = op.swidth[s], per = (w + NW - 1) / NW;
    double q[Op::NC];
#pragma unroll
    for (int i = 0; i < Op::NC; i++) q[i] = 0.0;
    op.add(b0, wv * per, min(w, (wv + 1) * per), l, own ? t : 0, x, q);
    __shared__ double red[NW][Op::NC][64];
#pragma unroll
    for (int i = 0; i < Op::NC; i++) red[wv][i][l] = q[i];
    __syncthreads();
    if (wv > 0) return;
    for (int j = 1; j < NW; j++)
#pragma unroll
        for (int i = 0; i < Op::NC; i++) q[i] += red[j][i][l];
    if (own)
#pragma unroll
        for (int i = 0; i < Op::NC; i++) e((long)Op::NC * t + i, q[i]);
}

// first direction of a smoothing pass from zero
__global__ void __launch_bounds__(AB) k_amg_pre(long nd, const double* __restrict__ dinv, const double* __restrict__ f,
                                                const double* __restrict__ coef, double* __restrict__ d0,
                                                const double* done)
{
    if (skip(done)) return;
    const long j = (long)blockIdx.x * AB + threadIdx.x;
    if (j < nd) d0[j] = coef[0] * dinv[j] * f[j];
}

// fc[A][c] = sum over members i of A of P_i^T r_i, four members' loads at a
// time
template <int BS>
__global__ void __launch_bounds__(AB) k_amg_restrict(int nc, const int* __restrict__ mptr,
                                                     const int* __restrict__ mem, const float* __restrict__ P,
                                                     const double* __restrict__ r, double* __restrict__ fc,
                                                     const double* done)
{
    if (skip(done)) return;
    const long t = (long)blockIdx.x * AB + threadIdx.x;
    if (t >= 6L * nc) return;
    const int a = (int)(t / 6), c = (int)(t - 6L * a);
    const int m1 = mptr[a + 1];
    double s = 0.0;
    for (int m = mptr[a]; m < m1; m += 4) {
        float p[4][BS];
        double v[4][BS];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = mem[min(m + u, m1 - 1)];
#pragma unroll
            for (int q = 0; q < BS; q++) {
                p[u][q] = P[(long)i * BS * 6 + 6 * q + c];
                v[u][q] = r[(long)i * BS + q];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (m + u < m1)
#pragma unroll
                for (int q = 0; q < BS; q++) s += (double)p[u][q] * v[u][q];
    }
    fc[t] = s;
}

// x_i += w P_i xc[agg(i)]
template <int BS>
__global__ void __launch_bounds__(AB) k_amg_prolong(int n, const int* __restrict__ agg,
                                                    const float* __restrict__ P, const double* __restrict__ xc,
                                                    double w, double* __restrict__ x, const double* done)
{
    if (skip(done)) return;
    const long t = (long)blockIdx.x * AB + threadIdx.x;
    if (t >= (long)n * BS) return;
    const int i = (int)(t / BS);
    const int a = agg[i];
    const float* p = P + 6 * t;
    const double xt = x[t];
    if (a < 0) return;
    const double* e = xc + 6L * a;
    x[t] = xt + w * ((double)p[0] * e[0] + (double)p[1] * e[1] + (double)p[2] * e[2] + (double)p[3] * e[3] +
                     (double)p[4] * e[4] + (double)p[5] * e[5]);
}

// coarsest level: x = C^-1 f (C^-1 dense, symmetric, column-major); a row's
// columns in four parts, added in order
__global__ void __launch_bounds__(4 * AB) k_amg_dense(int n, const double* __restrict__ cinv,
                                                      const double* __restrict__ f, double* __restrict__ x,
                                                      const double* done)
{
    if (skip(done)) return;
    __shared__ double red[3][AB];
    const int t = threadIdx.x & (AB - 1), part = threadIdx.x / AB;
    const int r = blockIdx.x * AB + t;
    const int per = (n + 3) / 4, c1 = min(n, (part + 1) * per);
    double s = 0.0;
    if (r < n)
#pragma unroll 8
        for (int c = part * per; c < c1; c++) s += cinv[(long)c * n + r] * f[c];
    if (part > 0) red[part - 1][t] = s;
    __syncthreads();
    if (part == 0 && r < n) x[r] = ((s + red[0][t]) + red[1][t]) + red[2][t];
}

// Galerkin product, fine level = the sliced-ELL operator: one wave per
// upper coarse block, lane (r, c) < 36 sums P_i^T A_ij P_j over the block's
// gather list in order; the block and its transpose partner are written.
template <class MT>
__global__ void __launch_bounds__(AB) k_amg_rap0(long nup, const int* __restrict__ up, const long* __restrict__ gptr,
                                                 const int* __restrict__ gl, const int* __restrict__ fcol,
                                                 const MT* __restrict__ fval, const float* __restrict__ P,
                                                 float* __restrict__ cval)
{
    const long u = (long)blockIdx.x * (AB / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (u >= nup || lane >= 36) return;
    const int r = lane / 6, c = lane - 6 * (lane / 6);
    double s = 0.0;
#pragma unroll 4
    for (long e = gptr[u]; e < gptr[u + 1]; e++) {
        const int fb = gl[2 * e], i = gl[2 * e + 1];
        const int j = fcol[fb];
        const MT* v = fval + (long)(fb >> 6) * 576 + (fb & 63);
        const float* pi = P + (long)i * 18 + r;
        const float* pj = P + (long)j * 18 + c;
        double t = 0.0;
#pragma unroll
        for (int p = 0; p < 3; p++) {
            const double ap = (double)v[(3 * p) * 64] * pj[0] + (double)v[(3 * p + 1) * 64] * pj[6] +
                              (double)v[(3 * p + 2) * 64] * pj[12];
            t += (double)pi[6 * p] * ap;
        }
        s += t;
    }
    const int ab = up[2 * u], ba = up[2 * u + 1];
    cval[amg_at(ab, 6 * r + c)] = (float)s;
    if (ba >= 0) cval[amg_at(ba, 6 * c + r)] = (float)s;
}

// Galerkin product, fine level = a sliced 6x6 level
__global__ void __launch_bounds__(AB) k_amg_rapc(long nup, const int* __restrict__ up, const long* __restrict__ gptr,
                                                 const int* __restrict__ gl, const int* __restrict__ fcol,
                                                 const float* __restrict__ fval, const float* __restrict__ P,
                                                 float* __restrict__ cval)
{
    const long u = (long)blockIdx.x * (AB / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (u >= nup || lane >= 36) return;
    const int r = lane / 6, c = lane - 6 * (lane / 6);
    double s = 0.0;
    for (long e = gptr[u]; e < gptr[u + 1]; e++) {
        const int fb = gl[2 * e], i = gl[2 * e + 1];
        const int j = fcol[fb];
        const float* pi = P + (long)i * 36 + r;
        const float* pj = P + (long)j * 36 + c;
        double t = 0.0;
#pragma unroll
        for (int p = 0; p < 6; p++) {
            double ap = 0.0;
#pragma unroll
            for (int q = 0; q < 6; q++) ap += (double)fval[amg_at(fb, 6 * p + q)] * pj[6 * q];
            t += (double)pi[6 * p] * ap;
        }
        s += t;
    }
    const int ab = up[2 * u], ba = up[2 * u + 1];
    cval[amg_at(ab, 6 * r + c)] = (float)s;
    if (ba >= 0) cval[amg_at(ba, 6 * c + r)] = (float)s;
}

// inverse diagonal of a sliced 6x6 level (0 for inactive dofs)
__global__ void __launch_bounds__(AB) k_amg_dinv(int n, const int* __restrict__ diagblk, const float* __restrict__ val,
                                                 double* __restrict__ dinv)
{
    const long t = (long)blockIdx.x * AB + threadIdx.x;
    if (t >= 6L * n) return;
    const int a = (int)(t / 6), r = (int)(t - 6L * a);
    const int e = diagblk[a];
    const double d = (double)val[amg_at(e, 7 * r)];
    dinv[t] = d > 0.0 ? 1.0 / d : 0.0;
}

// ---- power iteration for the largest eigenvalue of D^-1 A -----------------

__global__ void __launch_bounds__(AB) k_amg_rand(long nd, const double* __restrict__ dinv, double* __restrict__ v)
{
    const long j = (long)blockIdx.x * AB + threadIdx.x;
    if (j >= nd) return;
    // SplitMix64 of the index: a fixed start vector with no structure
    unsigned long long z = (unsigned long long)j + 0x9e3779b97f4a7c15ULL;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    z ^= z >> 31;
    const double u = (double)(z >> 11) * (1.0 / 9007199254740992.0);
    v[j] = dinv[j] != 0.0 ? 2.0 * u - 1.0 : 0.0;
}

// part[b] = partial sums of a.b (KIND 0) or a.a / dinv over dinv != 0 (KIND 1)
template <int KIND>
__global__ void __launch_bounds__(AB) k_amg_part(long nd, const double* __restrict__ a, const double* __restrict__ b,
                                                 double* __restrict__ part)
{
    __shared__ double red[AB / 64];
    double s = 0.0;
    for (long j = (long)blockIdx.x * AB + threadIdx.x; j < nd; j += (long)gridDim.x * AB) {
        if (KIND == 0)
            s += a[j] * b[j];
        else if (b[j] != 0.0)
            s += a[j] * a[j] / b[j];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < AB / 64; w++) t += red[w];
        part[blockIdx.x] = t;
    }
}

__global__ void __launch_bounds__(AB) k_amg_fin(const double* __restrict__ part, int np, double* __restrict__ out)
{
    __shared__ double red[AB / 64];
    double s = 0.0;
    for (int j = threadIdx.x; j < np; j += AB) s += part[j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < AB / 64; w++) t += red[w];
        *out = t;
    }
}

// v = D^-1 w / sqrt(nrm2) with nrm2 = |D^-1 w|^2 computed beforehand into *nrm2
__global__ void __launch_bounds__(AB) k_amg_scale(long nd, const double* __restrict__ w,
                                                  const double* __restrict__ nrm2, double* __restrict__ v)
{
    const long j = (long)blockIdx.x * AB + threadIdx.x;
    if (j >= nd) return;
    const double s = *nrm2 > 0.0 ? 1.0 / sqrt(*nrm2) : 0.0;
    v[j] = w[j] * s;
}

// w = D^-1 w
__global__ void __launch_bounds__(AB) k_amg_jac(long nd, const double* __restrict__ dinv, double* __restrict__ w)
{
    const long j = (long)blockIdx.x * AB + threadIdx.x;
    if (j >= nd) return;
    w[j] *= dinv[j];
}

constexpr int NPART = 1024;

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

template <bool SYM>
static OpC<SYM> opc(const AmgLevel& L)
{
    return {L.n, L.d_sbase.p, L.d_swidth.p, L.d_col.p, L.d_part.p, L.d_val.p};
}

template <class Op, class E>
static void launch_rows(tg_ctx* c, const Op& op, const double* x, const E& e, const double* done, int nw)
{
    const unsigned nb = (unsigned)((op.n + 63) / 64 + 7) / 8 * 8;
    const int ranges = op.n < 1 << 19;  // as the PCG's product (k_pcg.hip: k_share_spmv)
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(nb), dim3(64 * nw), 0, c->stream, op, x, e, ranges, done); };
    if (nw == 9)
        go(k_amg_rows<Op, 9, E>);
    else
        go(k_amg_rows<Op, 3, E>);
}

// y = A_l x and what follows.  Nine waves share a row up to 640 slices and where
// lower blocks come from their partners, three otherwise.
template <class E>
static void level_rows(tg_ctx* c, int l, const double* x, const E& e, const double* done)
{
    const Bsell& B = c->op;
    if (l > 0) {
        const AmgLevel& A = *c->amg.lv[l];
        if (A.n >= AMG_SYM_NODES)
            launch_rows(c, opc<true>(A), x, e, done, 9);
        else
            launch_rows(c, opc<false>(A), x, e, done, A.n <= 64 * 640 ? 9 : 3);
    } else {
        auto go = [&](const auto& op) { launch_rows(c, op, x, e, done, c->nnd <= 64 * 640 ? 9 : 3); };
        if (op_streams(c, sizeof(float)))
            go(Op0<float, true>{c->nnd, B.d_slice_base.p, B.d_slice_width.p, B.d_col.p, B.d_val32.p});
        else
            go(Op0<float, false>{c->nnd, B.d_slice_base.p, B.d_slice_width.p, B.d_col.p, B.d_val32.p});
    }
}

// Chebyshev degree of a level's smoothing passes.  Untuned, the levels that
// memory bounds take one step, two products a cycle instead of four: the PCG
// iterations grow by a fifth and each costs two fifths less.  Mixed precision,
// ms a Newton step and PCG iterations, degree 2 everywhere / 1 at the fine level
// / 1 at the first coarse level too: 128^3 440 (86) / 379 (99) / 341 (109), 96^3
// 214 / 180 / 170, 80^3 127 / 110 / 108, 56^3 50.8 / 46.7 / 47.8, 48^3 27.4 /
// 26.8 / 27.5, 32^3 16.8 / 17.2 / 17.9.  So from 3 * 2^17 dofs of a level: 2^17
// nodes of the fine one, 2^16 of a coarse one.  The rule holds in FP64 (64^3 63
// and 71 ms with degree 2 everywhere, 128^3 380 and 451) and for nearly
// incompressible problems, one solve to 1e-3: Q1P0 nu 0.499 52^3 FP64 35 and 50
// ms, 64^3 mixed 331 and 383, nu 0.49 82^3 25 and 40; total-Lagrangian nu 0.49
// 96^3 40 and 148.
static int level_degree(const tg_ctx* c, int l)
{
    const AmgLevel& A = *c->amg.lv[l];
    return amg_degree(c, (long)A.n * A.bs);
}

static double* level_dinv(tg_ctx* c, int l) { return l == 0 ? c->vdinv.p : c->amg.lv[l]->dinv; }

static void reduce(tg_ctx* c, int kind, long nd, const double* a, const double* b, double* out)
{
    Amg& G = c->amg;
    const unsigned nb = std::min<long>(NPART, std::max<long>(1, blocks_for(nd)));
    if (kind == 0)
        hipLaunchKernelGGL(k_amg_part<0>, dim3(nb), dim3(AB), 0, c->stream, nd, a, b, G.d_part.p);
    else
        hipLaunchKernelGGL(k_amg_part<1>, dim3(nb), dim3(AB), 0, c->stream, nd, a, b, G.d_part.p);
    hipLaunchKernelGGL(k_amg_fin, dim3(1), dim3(AB), 0, c->stream, G.d_part.p, (int)nb, out);
}

// Largest eigenvalue of D^-1 A on level l by power iteration: the Rayleigh
// quotient (v.Av)/(v.Dv) is left in red[0] / red[1].
static void power_iteration(tg_ctx* c, int l, long nd, const double* dinv, double* v, double* w, double* red)
{
    const unsigned vb = blocks_for(nd);
    hipLaunchKernelGGL(k_amg_rand, dim3(vb), dim3(AB), 0, c->stream, nd, dinv, v);
    for (int it = 0; it < POWER_ITS; it++) {
        level_rows(c, l, v, EStore{w}, nullptr);
        hipLaunchKernelGGL(k_amg_jac, dim3(vb), dim3(AB), 0, c->stream, nd, dinv, w);
        reduce(c, 0, nd, w, w, red + 2);
        hipLaunchKernelGGL(k_amg_scale, dim3(vb), dim3(AB), 0, c->stream, nd, w, red + 2, v);
    }
    level_rows(c, l, v, EStore{w}, nullptr);
    reduce(c, 0, nd, v, w, red);
    reduce(c, 1, nd, v, dinv, red + 1);
}

// Dense inverse of the coarsest level by LDL^T: inactive dofs (zero
// diagonal) and non-positive pivots get zero rows and columns.
static void coarse_inverse(const AmgLevel& L, const std::vector<float>& val, std::vector<double>& inv)
{
    const int n = 6 * L.n;
    std::vector<double> A((size_t)n * n, 0.0);
    for (int a = 0; a < L.n; a++)
        for (int q = L.rowptr[a]; q < L.rowptr[a + 1]; q++) {
            const int b = L.col[q], e = L.slot[q];
            for (int r = 0; r < 6; r++)
                for (int s = 0; s < 6; s++) A[(size_t)(6 * a + r) * n + 6 * b + s] = val[amg_at(e, 6 * r + s)];
        }
    double dmax = 0.0;
    for (int i = 0; i < n; i++) dmax = std::max(dmax, A[(size_t)i * n + i]);
    // in-place LDL^T (lower triangle holds L, diagonal holds D)
    std::vector<char> live((size_t)n, 1);
    for (int j = 0; j < n; j++) {
        double d = A[(size_t)j * n + j];
        for (int k = 0; k < j; k++)
            if (live[k]) d -= A[(size_t)j * n + k] * A[(size_t)j * n + k] * A[(size_t)k * n + k];
        if (!(d > 1e-12 * dmax)) {
            live[j] = 0;
            A[(size_t)j * n + j] = 0.0;
            for (int i = j + 1; i < n; i++) A[(size_t)i * n + j] = 0.0;
            continue;
        }
        A[(size_t)j * n + j] = d;
        for (int i = j + 1; i < n; i++) {
            double s = A[(size_t)i * n + j];
            for (int k = 0; k < j; k++)
                if (live[k]) s -= A[(size_t)i * n + k] * A[(size_t)j * n + k] * A[(size_t)k * n + k];
            A[(size_t)i * n + j] = s / d;
        }
    }
    inv.assign((size_t)n * n, 0.0);
    std::vector<double> y((size_t)n);
    for (int e = 0; e < n; e++) {
        if (!live[e]) continue;
        std::fill(y.begin(), y.end(), 0.0);
        y[e] = 1.0;
        for (int i = 0; i < n; i++) {  // L y = e
            if (!live[i]) {
                y[i] = 0.0;
                continue;
            }
            double s = y[i];
            for (int k = 0; k < i; k++) s -= A[(size_t)i * n + k] * y[k];
            y[i] = s;
        }
        for (int i = 0; i < n; i++) y[i] = live[i] ? y[i] / A[(size_t)i * n + i] : 0.0;
        for (int i = n - 1; i >= 0; i--) {  // L^T x = y
            if (!live[i]) continue;
            double s = y[i];
            for (int k = i + 1; k < n; k++) s -= A[(size_t)k * n + i] * y[k];
            y[i] = s;
        }
        for (int i = 0; i < n; i++) inv[(size_t)e * n + i] = live[i] ? y[i] : 0.0;
    }
}

template <class MT>
static void amg_numeric_t(tg_ctx* c, const MT* val0)
{
    Amg& G = c->amg;
    const int L = (int)G.lv.size();
    TimedRegion tr(c, T_PRECOND);
    // coarse operators, finest first
    for (int l = 0; l + 1 < L; l++) {
        AmgLevel& F = *G.lv[l];
        AmgLevel& C = *G.lv[l + 1];
        const unsigned nb = (unsigned)((F.nup + AB / 64 - 1) / (AB / 64));
        if (nb > 0) {
            if (l == 0)
                hipLaunchKernelGGL(k_amg_rap0<MT>, dim3(nb), dim3(AB), 0, c->stream, F.nup, F.d_up.p, F.d_gptr.p,
                                   F.d_glist.p, c->op.d_col.p, val0, F.d_P.p, C.d_val.p);
            else
                hipLaunchKernelGGL(k_amg_rapc, dim3(nb), dim3(AB), 0, c->stream, F.nup, F.d_up.p, F.d_gptr.p,
                                   F.d_glist.p, F.d_col.p, F.d_val.p, F.d_P.p, C.d_val.p);
        }
        hipLaunchKernelGGL(k_amg_dinv, dim3(blocks_for(6L * C.n)), dim3(AB), 0, c->stream, C.n, C.d_diagblk.p,
                           C.d_val.p, C.dinv);
        TG_HIP(hipGetLastError());
    }
    // smoother intervals
    for (int l = 0; l + 1 < L; l++) {
        AmgLevel& A = *G.lv[l];
        const long nd = (long)A.n * A.bs;
        double* red = G.d_red.p + 16 * l;
        power_iteration(c, l, nd, level_dinv(c, l), A.d_d0.p, A.d_d1.p, red);
        TG_HIP(hipGetLastError());
    }
    std::vector<double> red(16 * (size_t)L);
    TG_HIP(hipMemcpyAsync(red.data(), G.d_red.p, sizeof(double) * red.size(), hipMemcpyDeviceToHost, c->stream));
    const AmgLevel& Cst = *G.lv[L - 1];
    std::vector<float> cval((size_t)Cst.nslots * 36);
    TG_HIP(hipMemcpyAsync(cval.data(), Cst.d_val.p, sizeof(float) * cval.size(), hipMemcpyDeviceToHost, c->stream));
    TG_HIP(hipStreamSynchronize(c->stream));
    std::vector<double> coef(8 * (size_t)L, 0.0);
    for (int l = 0; l + 1 < L; l++) {
        const double num = red[16 * l], den = red[16 * l + 1];
        double lmax = den > 0.0 ? num / den : 1.0;
        if (!(lmax > 0.0) || !std::isfinite(lmax)) lmax = 1.0;
        lmax *= CHEB_BOOST;
        G.lv[l]->lmax = lmax;
        const int degree = level_degree(c, l);
        const double lmin = lmax / (degree == 1 ? JACOBI_RATIO : CHEB_RATIO);
        const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin), sigma = theta / delta;
        double* cf = coef.data() + 8 * l;
        cf[0] = 1.0 / theta;
        double rho = 1.0 / sigma;
        for (int s = 1; s < degree; s++) {
            const double rn = 1.0 / (2.0 * sigma - rho);
            cf[2 * s - 1] = rn * rho;
            cf[2 * s] = 2.0 * rn / delta;
            rho = rn;
        }
    }
    std::vector<double> inv;
    coarse_inverse(Cst, cval, inv);
    TG_HIP(hipMemcpyAsync(G.d_coef.p, coef.data(), sizeof(double) * coef.size(), hipMemcpyHostToDevice, c->stream));
    TG_HIP(hipMemcpyAsync(G.d_cinv.p, inv.data(), sizeof(double) * inv.size(), hipMemcpyHostToDevice, c->stream));
    TG_HIP(hipStreamSynchronize(c->stream));  // host vectors outlive their copies
}

// The multigrid works on the FP32 copy of the fine operator in either
// precision (the solver's own operator when it is FP32; refreshed from the
// FP64 one by the caller otherwise): a preconditioner needs no more, and the
// smoother's fine-level products (two to four a cycle) move half the bytes.
// The coarse levels' numeric set-up (Galerkin products, smoother intervals,
// coarsest inverse) for the current fine operator.  With reuse = k > 0 one
// set-up serves the next k tangents of the same Newton solve too: the
// V-cycle then smooths with the current fine operator and corrects with the
// coarse operators of an earlier tangent of that solve (Galerkin products of
// an SPD matrix, so the V-cycle stays an SPD preconditioner; only the PCG
// count may change).  A new load, state or step (tg_apply_kbc,
// tg_set_displacement, tg_close_step, tg_reset_step) clears `since`: the
// tangents of a failed attempt never serve the next one.
void amg_numeric(tg_ctx* c)
{
    Amg& G = c->amg;
    if (G.lv.empty()) amg_setup(c);
    if (G.reuse > 0 && G.since >= 0 && G.since < G.reuse) {
        G.since++;
        return;
    }
    amg_numeric_t<float>(c, c->op.d_val32.p);
    G.since = 0;
}

// pre-smoothing from zero, then r = f - A x; with one step x stays in d0
static void smooth_down(tg_ctx* c, int l, const double* f, double* x, AmgLevel& A, const double* cf, const double* done)
{
    const double* dinv = level_dinv(c, l);
    const long nd = (long)A.n * A.bs;
    const int degree = level_degree(c, l);
    double *dp = A.d_d1.p, *dn = A.d_d0.p;
    hipLaunchKernelGGL(k_amg_pre, dim3(blocks_for(nd)), dim3(AB), 0, c->stream, nd, dinv, f, cf, dn, done);
    if (degree == 1) {
        level_rows(c, l, dn, EDefect{f, A.d_r.p}, done);
        return;
    }
    level_rows(c, l, dn, EFirst{dinv, f, cf, dn, dp, A.d_r.p, x}, done);
    for (int s = 2; s < degree; s++) {
        level_rows(c, l, dp, EStep{dinv, dp, cf, dn, A.d_r.p, x, 2 * s - 1, 0}, done);
        std::swap(dp, dn);
    }
    level_rows(c, l, dp, EResid{A.d_r.p}, done);
}

static void smooth_up(tg_ctx* c, int l, const double* f, double* x, AmgLevel& A, const double* cf, const double* done)
{
    const double* dinv = level_dinv(c, l);
    const int degree = level_degree(c, l);
    if (degree == 1) {
        level_rows(c, l, A.d_d0.p, EJacobi{dinv, f, cf, A.d_d0.p, x}, done);
        return;
    }
    level_rows(c, l, x, EPost{dinv, f, cf, A.d_r.p, A.d_d0.p}, done);
    double *dp = A.d_d0.p, *dn = A.d_d1.p;
    for (int s = 1; s < degree; s++) {
        level_rows(c, l, dp, EStep{dinv, dp, cf, dn, A.d_r.p, x, 2 * s - 1, s == 1 ? 1 : 0}, done);
        std::swap(dp, dn);
    }
}

// z = M^-1 f by one V-cycle; every kernel is a no-op once *done != 0 (the
// solve has converged), so a captured chunk of iterations stays valid.
void amg_vcycle(tg_ctx* c, const double* f0, double* z, const double* done)
{
    Amg& G = c->amg;
    const int L = (int)G.lv.size();
    for (int l = 0; l + 1 < L; l++) {
        AmgLevel& A = *G.lv[l];
        AmgLevel& C = *G.lv[l + 1];
        smooth_down(c, l, l == 0 ? f0 : A.d_f.p, l == 0 ? z : A.d_x.p, A, G.d_coef.p + 8 * l, done);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(blocks_for(6L * C.n)), dim3(AB), 0, c->stream, C.n, A.d_mptr.p, A.d_mem.p,
                               A.d_P.p, A.d_r.p, C.d_f.p, done);
        };
        if (l == 0)
            go(k_amg_restrict<3>);
        else
            go(k_amg_restrict<6>);
    }
    AmgLevel& Cst = *G.lv[L - 1];
    hipLaunchKernelGGL(k_amg_dense, dim3(blocks_for(G.ncd)), dim3(4 * AB), 0, c->stream, G.ncd, G.d_cinv.p, Cst.d_f.p,
                       Cst.d_x.p, done);
    for (int l = L - 2; l >= 0; l--) {
        AmgLevel& A = *G.lv[l];
        AmgLevel& C = *G.lv[l + 1];
        double* x = l == 0 ? z : A.d_x.p;
        double* xp = level_degree(c, l) == 1 ? A.d_d0.p : x;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(blocks_for((long)A.n * A.bs)), dim3(AB), 0, c->stream, A.n, A.d_agg.p,
                               A.d_P.p, C.d_x.p, 0.01 * G.weight, xp, done);
        };
        if (l == 0)
            go(k_amg_prolong<3>);
        else
            go(k_amg_prolong<6>);
        smooth_up(c, l, l == 0 ? f0 : A.d_f.p, x, A, G.d_coef.p + 8 * l, done);
    }
    TG_HIP(hipGetLastError());
}


}  // namespace tg
