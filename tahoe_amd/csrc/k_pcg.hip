// Segmented Jacobi-preconditioned conjugate gradients.
//
// A context holds one problem or a batch of independent problems packed as
// a disjoint union ("segments"), each starting at a multiple of 64 nodes.
// Every segment runs its own CG: its own dot products, alpha, beta and
// stopping test, all kept on the device.  Reductions are per slice of 64
// nodes (one wave, never shared by two segments) and then per segment in
// slice order, so a segment's arithmetic -- and its result -- is the same
// alone and inside any batch.  A single problem is the one-segment case.
//
// This file is compiled without FMA contraction (tahoe_amd/build.py): each
// expression rounds as written, so the iteration's variants below, which
// share their expressions, agree bit for bit.
//
// The reference has no linear CG; this is the textbook method (Saad,
// Iterative Methods for Sparse Linear Systems, Alg. 9.1) on the reference's
// building blocks: Multx (MSRMatrixT.cpp:385-420), Jacobi scaling
// (DiagonalMatrixT.cpp:267-324) and InnerProduct (SolverT.cpp:854-860).
#include <cstring>

#include <type_traits>

#include "tg_internal.h"

namespace tg {

constexpr int PB = 256;  // threads (= nodes) per block, 4 slices
constexpr int FB = 1024; // threads of the per-segment finalize blocks

// v of the lane that DPP control CTRL names, for a double
template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, true));
}

// Sum over the wave, the same bits in every lane: lanes 1 and 2 apart by
// quad permutes, 4 and 8 apart by mirroring 8 and 16 lanes (whose halves
// each hold one value by then), the rows of 16 and the halves by row swaps.
// All in the vector registers; a butterfly of __shfl_xor goes through LDS
// twelve times, about 0.4 us that every kernel of a short iteration pays.
// All 64 lanes must be active.
__device__ __forceinline__ double wsum(double v)
{
    v += dpp<0xB1>(v);    // quad_perm 1,0,3,2
    v += dpp<0x4E>(v);    // quad_perm 2,3,0,1
    v += dpp<0x141>(v);   // row_half_mirror
    v += dpp<0x140>(v);   // row_mirror
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    return v;
}

__device__ __forceinline__ double* sf(double* s, int field, int nseg, int seg) { return s + (long)field * nseg + seg; }

// z = M^-1 r at node a.  PC = 0: Jacobi, m = 1/diag [nnd][3]
// (DiagonalMatrixT); PC = 1: 3x3 nodal block Jacobi, m = inverse diagonal
// blocks [nnd][9] (row-major, prescribed rows and columns zero); PC = 2:
// multigrid, m = z itself, computed beforehand by a V-cycle.
template <int PC>
__device__ __forceinline__ void precondition(const double* __restrict__ m, long a, const double (&r)[3], double (&z)[3])
{
    if (PC == 2) {
#pragma unroll
        for (int i = 0; i < 3; i++) z[i] = m[3 * a + i];
    } else if (PC == 0) {
#pragma unroll
        for (int i = 0; i < 3; i++) z[i] = m[3 * a + i] * r[i];
    } else {
        const double* b = m + 9 * a;
#pragma unroll
        for (int i = 0; i < 3; i++) z[i] = b[3 * i] * r[0] + b[3 * i + 1] * r[1] + b[3 * i + 2] * r[2];
    }
}

// ---- partials -> per-segment totals -----------------------------------------
//
// A segment's slices are taken in groups of GS = 4; a group's sum is
// ((s0 + s1) + s2) + s3 (missing slices 0), lane l of a wave adds groups l,
// l + 64, ... in order, and the lanes are summed by wsum.  A kernel whose
// workgroups own a group each writes one partial per group, a kernel with a
// workgroup per slice one per slice (GROUPED = false: the reader adds four).
// The order depends only on the segment's own slice count, never on other
// segments.
constexpr int GS = 4;

// lane sums over n partials (groups, or slices) from part[k * stride]; this
// wave takes every wstep-th run of 64 groups, from run w0
template <int NV, bool GROUPED>
__device__ __forceinline__ void lane_sums(const double* part, long stride, int n, int w0, int wstep, double (&x)[NV])
{
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < NV; k++) x[k] = 0.0;
    const int per = GROUPED ? 1 : GS;
#pragma unroll 4
    for (int base = 64 * per * w0; base < n; base += 64 * per * wstep) {
        const int s = base + per * l;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const double* q = part + k * stride + s;
            if (GROUPED) {
                x[k] += s < n ? q[0] : 0.0;
            } else {
                const double a0 = s < n ? q[0] : 0.0, a1 = s + 1 < n ? q[1] : 0.0;
                const double a2 = s + 2 < n ? q[2] : 0.0, a3 = s + 3 < n ? q[3] : 0.0;
                x[k] += ((a0 + a1) + a2) + a3;
            }
        }
    }
}

// Sum of the partials of a segment of at most FOLD_SLICES slices by one
// wave, the same in every lane.  Any kernel that needs a total forms it by
// itself, so an iteration needs no kernel that does only that: at 16^3
// elements (77 slices) such a kernel took 4 us of a 28 us iteration, twice.
constexpr int FOLD_SLICES = PCG_FOLD_SLICES;
template <int NV, bool GROUPED>
__device__ __forceinline__ void wave_total(const double* part, long stride, int n, double (&tot)[NV])
{
    lane_sums<NV, GROUPED>(part, stride, n, 0, 1, tot);
#pragma unroll
    for (int k = 0; k < NV; k++) tot[k] = wsum(tot[k]);
}

// The same total by one block of FB threads: a segment of at most
// FOLD_SLICES slices exactly as wave_total sums it (by wave 0); a larger one
// with wave w taking every (FB / 64)-th run and the wave sums added in
// order.  The result is in thread 0.
template <int NV, bool GROUPED>
__device__ __forceinline__ void seg_total(const double* part, long stride, int n, int nsl, double (&tot)[NV])
{
    const int t = threadIdx.x;
    if (nsl <= FOLD_SLICES) {
        if (t < 64) wave_total<NV, GROUPED>(part, stride, n, tot);
        return;
    }
    __shared__ double red[NV][FB / 64];
    double x[NV];
    lane_sums<NV, GROUPED>(part, stride, n, t >> 6, FB / 64, x);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const double y = wsum(x[k]);
        if ((t & 63) == 0) red[k][t >> 6] = y;
    }
    __syncthreads();
    if (t == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) {
            double y = 0.0;
            for (int w = 0; w < FB / 64; w++) y += red[k][w];
            tot[k] = y;
        }
}

// Segment tables as the kernels take them.  grp[i] = (first slice, slices,
// segment, -) of group i; seg g owns slices [seg_slice[g], seg_slice[g + 1])
// and groups [seg_grp[g], seg_grp[g + 1]).
struct SegTab {
    const int* slice_seg;
    const int* seg_slice;
    const int* seg_grp;
    const int4* grp;
    int nseg;
    long nslices;
    __device__ __forceinline__ int slices(int g) const { return seg_slice[g + 1] - seg_slice[g]; }
    __device__ __forceinline__ int groups(int g) const { return seg_grp[g + 1] - seg_grp[g]; }
};

// The group's partials of this workgroup's up to GS waves (PB threads, wave
// w = slice w of the group), from per-lane values already summed by wsum:
// thread 0 writes part[k * stride + group].
template <int NV>
__device__ __forceinline__ void group_partials(const double (&v)[NV], double* part, long stride, const bool (&on)[NV])
{
    __shared__ double red[NV][GS];
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < NV; k++)
        if ((t & 63) == 0) red[k][t >> 6] = v[k];
    __syncthreads();
    if (t == 0)
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (on[k]) part[k * stride + blockIdx.x] = ((red[k][0] + red[k][1]) + red[k][2]) + red[k][3];
}

// slots of r.z and the iteration count before (o) and after the iteration
__device__ __forceinline__ double* slot_rz(double* sc, int o, int nseg, int g) { return sf(sc, o ? S_RZ1 : S_RZ, nseg, g); }
__device__ __forceinline__ double* slot_it(double* sc, int o, int nseg, int g) { return sf(sc, o ? S_IT1 : S_IT0, nseg, g); }

// End of an iteration of segment g with tot = (r.z, r.r): beta = rz'/rz,
// stop on ||r||^2 <= rtol^2 ||b||^2 or the iteration cap.  Several waves may
// form the same decision in one kernel, so the values of the iteration
// before (slot o) are kept and the new ones go to slot o ^ 1; the owner (one
// lane per segment) writes.  Returns whether the segment is done.
__device__ __forceinline__ bool seg_advance(const double (&tot)[2], double* sc, int nseg, int g, int o, bool owner,
                                            int* ndone, double& beta)
{
    const double it = *slot_it(sc, o, nseg, g) + 1.0;
    beta = tot[0] / *slot_rz(sc, o, nseg, g);
    const bool done = tot[1] <= *sf(sc, S_THRESH, nseg, g) || it >= *sf(sc, S_MAXIT, nseg, g);
    if (owner) {
        *slot_rz(sc, o ^ 1, nseg, g) = tot[0];
        *slot_it(sc, o ^ 1, nseg, g) = it;
        *sf(sc, S_ITER, nseg, g) = it;
        *sf(sc, S_BETA, nseg, g) = beta;
        *sf(sc, S_RR, nseg, g) = tot[1];
        if (done) {
            *sf(sc, S_DONE, nseg, g) = 1.0;
            atomicAdd(ndone, 1);
        }
    }
    return done;
}

// x = 0, r = b, z = p = M^-1 b; per segment rz = b.M^-1 b, bb = b.b.  b and z
// may be one array.
template <int PC>
__global__ void __launch_bounds__(PB) k_seg_init(SegTab T, int nnd, const double* b, const double* __restrict__ m,
                                                 double* __restrict__ x, double* __restrict__ r,
                                                 double* __restrict__ p, double* z, double* __restrict__ part)
{
    const int4 gr = T.grp[blockIdx.x];
    const int a = 64 * gr.x + threadIdx.x;
    double v[2] = {0.0, 0.0};
    if ((int)(threadIdx.x >> 6) < gr.y && a < nnd) {
        double bi[3], zi[3];
#pragma unroll
        for (int i = 0; i < 3; i++) bi[i] = b[3L * a + i];
        precondition<PC>(m, a, bi, zi);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const long k = 3L * a + i;
            x[k] = 0.0;
            r[k] = bi[i];
            p[k] = zi[i];
            if (PC != 2 && z) z[k] = zi[i];
            v[0] += bi[i] * zi[i];
            v[1] += bi[i] * bi[i];
        }
    }
    v[0] = wsum(v[0]);
    v[1] = wsum(v[1]);
    group_partials<2>(v, part, T.nslices, {true, true});
}

__global__ void __launch_bounds__(FB) k_seg_fin_init(SegTab T, const double* __restrict__ part,
                                                     const int* __restrict__ active, double* __restrict__ sc,
                                                     double rtol, int maxit, int* __restrict__ ndone)
{
    const int g = blockIdx.x, nseg = T.nseg;
    double tot[2];
    seg_total<2, true>(part + T.seg_grp[g], T.nslices, T.groups(g), T.slices(g), tot);
    if (threadIdx.x == 0) {
        *sf(sc, S_RZ, nseg, g) = tot[0];
        *sf(sc, S_BB, nseg, g) = tot[1];
        *sf(sc, S_RR, nseg, g) = tot[1];
        *sf(sc, S_ITER, nseg, g) = 0.0;
        *sf(sc, S_IT0, nseg, g) = 0.0;
        *sf(sc, S_BETA, nseg, g) = 0.0;  // the fused iteration forms p_0 = z_0 + 0 p
        *sf(sc, S_THRESH, nseg, g) = rtol * rtol * tot[1];
        *sf(sc, S_MAXIT, nseg, g) = (double)maxit;
        const bool done = !active[g] || tot[1] == 0.0 || maxit <= 0;
        *sf(sc, S_DONE, nseg, g) = done ? 1.0 : 0.0;
        if (done) atomicAdd(ndone, 1);
    }
}

// Workgroup -> rows.  Workgroups are dealt to the 8 XCDs round-robin, and
// each XCD has its own L2; with XCD = true workgroup w takes the row range
// (w % 8) * (G / 8) + w / 8 (G a multiple of 8), so each XCD sweeps one
// contiguous eighth of the rows and the x entries its rows gather (the
// neighbouring node layers) stay in its L2.
template <bool XCD>
__device__ __forceinline__ int row_block()
{
    if (!XCD) return blockIdx.x;
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

// The 9 values of block slot blk of lane l, row-major (v[3 r + q]).  With
// SYM a lower block (column node below the row node) is read as the
// transpose of its upper partner, whose first value index tpos holds: the
// operator is symmetric by construction (a lower block is a copy of its
// partner), so the values are the same, while the partner's row, just
// streamed by a nearby workgroup, serves them from L2 or the last-level
// cache instead of HBM.  Only the lanes of lower blocks read tpos.
template <class MT, bool SYM, bool NT = false>
__device__ __forceinline__ void block_values(const MT* __restrict__ bval, const int* __restrict__ tpos, long blk,
                                             int l, bool lower, double v[9])
{
    long base = blk * 9 * 64 + l;
    const bool tr = SYM && lower;
    if (tr) base = tpos[blk * 64 + l];
    double u[9];
#pragma unroll
    for (int m = 0; m < 9; m++) u[m] = (double)(NT ? __builtin_nontemporal_load(bval + base + m * 64) : bval[base + m * 64]);
    v[0] = u[0];
    v[4] = u[4];
    v[8] = u[8];
    v[1] = tr ? u[3] : u[1];
    v[3] = tr ? u[1] : u[3];
    v[2] = tr ? u[6] : u[2];
    v[6] = tr ? u[2] : u[6];
    v[5] = tr ? u[7] : u[5];
    v[7] = tr ? u[5] : u[7];
}

// A row's sum over its blocks k = 0 .. w-1 is formed in groups of RG
// consecutive slots: each group from zero in slot order, the groups added in
// order.  So one lane can sum a whole row, or the waves of a workgroup can
// take a group each, with the same rounding.  Nine groups of three are the
// 27 blocks of an interior node of a hexahedral mesh.
constexpr int RG = 3;
constexpr int SHARE_WAVES = 3; // waves of a workgroup of k_share_spmv

// y += A_blk x for one slot of a row
__device__ __forceinline__ void block_mac(const double (&v)[9], double x0, double x1, double x2, double (&y)[3])
{
    y[0] += v[0] * x0 + v[1] * x1 + v[2] * x2;
    y[1] += v[3] * x0 + v[4] * x1 + v[5] * x2;
    y[2] += v[6] * x0 + v[7] * x1 + v[8] * x2;
}

// One lane's row sum: x(c, x0, x1, x2) gives the vector at node c.  UNR:
// padding slots (column -1) hold zero values: they multiply the row's own x,
// which keeps the loop branch-free so its loads can be issued ahead; adding
// the zero products leaves the sums unchanged.
template <class MT, bool UNR, bool SYM, bool NT = false, class X>
__device__ __forceinline__ void row_sum(const int* __restrict__ bcol, const MT* __restrict__ bval,
                                        const int* __restrict__ tpos, long b0, int w, int l, int a, X x,
                                        double (&y)[3])
{
    y[0] = y[1] = y[2] = 0.0;
    int k = 0;
    for (; k + RG <= w; k += RG) {
        double g[3] = {0.0, 0.0, 0.0};
#pragma unroll(UNR ? RG : 1)
        for (int i = 0; i < RG; i++) {
            const long blk = b0 + k + i;
            const int cr = NT ? __builtin_nontemporal_load(bcol + blk * 64 + l) : bcol[blk * 64 + l];
            if (!UNR && cr < 0) continue;
            const int c = cr < 0 ? a : cr;
            double x0, x1, x2, v[9];
            x(c, x0, x1, x2);
            block_values<MT, SYM, NT>(bval, tpos, blk, l, c < a, v);
            block_mac(v, x0, x1, x2, g);
        }
#pragma unroll
        for (int i = 0; i < 3; i++) y[i] += g[i];
    }
    if (k < w) {
        double g[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
        for (; k < w; k++) {
            const long blk = b0 + k;
            const int cr = NT ? __builtin_nontemporal_load(bcol + blk * 64 + l) : bcol[blk * 64 + l];
            if (!UNR && cr < 0) continue;
            const int c = cr < 0 ? a : cr;
            double x0, x1, x2, v[9];
            x(c, x0, x1, x2);
            block_values<MT, SYM, NT>(bval, tpos, blk, l, c < a, v);
            block_mac(v, x0, x1, x2, g);
        }
#pragma unroll
        for (int i = 0; i < 3; i++) y[i] += g[i];
    }
}

// q = A p on the block operator, with per-slice partials of p.q.  MT is the
// storage type of the operator values (double, or float in mixed
// precision); products and sums are FP64.  NT: an operator that the last-level
// cache cannot hold (op_streams) is read past it by non-temporal loads, which
// leaves the caches to the vectors: 384 RVEs of edge 4-24 (1.2 GB) 88.4 ms a
// solve without, 84.6 with.
template <class MT, bool XCD, bool UNR, bool SYM, bool NT = false>
__global__ void __launch_bounds__(PB) k_seg_spmv(SegTab T, int nnd,
                                                 const int* __restrict__ sbase, const int* __restrict__ swidth,
                                                 const int* __restrict__ bcol, const MT* __restrict__ bval,
                                                 const int* __restrict__ tpos, const double* __restrict__ x,
                                                 double* __restrict__ y, double* __restrict__ ppq,
                                                 const double* __restrict__ sc)
{
    const int a = row_block<XCD>() * PB + threadIdx.x;
    const int s = __builtin_amdgcn_readfirstlane(a >> 6), l = a & 63;
    if (s >= T.nslices) return;
    const int g = T.slice_seg[s];
    if (*sf((double*)sc, S_DONE, T.nseg, g) != 0.0) return;
    double dv = 0.0;
    if (a < nnd) {
        double yi[3];
        row_sum<MT, UNR, SYM, NT>(bcol, bval, tpos, sbase[s], swidth[s], l, a, [&](int c, double& x0, double& x1, double& x2) {
            x0 = x[3L * c];
            x1 = x[3L * c + 1];
            x2 = x[3L * c + 2];
        }, yi);
        y[3L * a] = yi[0];
        y[3L * a + 1] = yi[1];
        y[3L * a + 2] = yi[2];
        dv = yi[0] * x[3L * a] + yi[1] * x[3L * a + 1] + yi[2] * x[3L * a + 2];
    }
    dv = wsum(dv);
    if (l == 0) ppq[s] = dv;
}

// The same product with a row shared by three waves, a workgroup a slice:
// from 2^17 nodes, where the operator's bytes bound it.  A wave takes nine
// consecutive slots, leaves each group's sum in LDS and wave 0 adds the groups
// in order: bitwise k_seg_spmv.  Three short chains a row keep more loads in
// flight than one of 27 blocks.  NT: an operator that the last-level cache
// cannot hold (op_streams) is read past it by non-temporal loads, which leaves
// the caches to the vectors.  XCD: below 2^19 nodes; beyond, slices in
// index order.  ms a Newton step, Jacobi, rtol 1e-3, symmetric read (7) /
// XCD / XCD NT / index order NT: mixed 140 k nodes 69.5 / 54.8 / 59.3 / 64.5,
// 275 k 127 / 112 / 109 / 110, 531 k 290 / 278 / 258 / 254, 912 k 617 / 608 /
// 570 / 559, 2.15 M 1344 / 1442 / 1372 / 1339 (FP32: 5.5 TB/s); FP64 140 k 99.9
// / 89.5 / 87.2 / 93.0, 275 k 188 / 187 / 162 / 168, 531 k 422 / 440 / 404 /
// 404, 912 k 891 / 961 / 906 / 896.
template <class MT, bool XCD, bool NT>
__global__ void __launch_bounds__(64 * SHARE_WAVES) k_share_spmv(SegTab T, int nnd, const int* __restrict__ sbase,
                                                                 const int* __restrict__ swidth,
                                                                 const int* __restrict__ bcol,
                                                                 const MT* __restrict__ bval,
                                                                 const double* __restrict__ x, double* __restrict__ y,
                                                                 double* __restrict__ ppq, const double* __restrict__ sc)
{
    constexpr int GW = 3, ROUND = SHARE_WAVES * GW * RG;  // groups a wave and slots a workgroup take at a time
    __shared__ double red[SHARE_WAVES * GW][3][64];
    const int s = row_block<XCD>(), l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (s >= T.nslices) return;
    const int g = T.slice_seg[s];
    if (*sf((double*)sc, S_DONE, T.nseg, g) != 0.0) return;
    const int a = 64 * s + l;
    const bool own = a < nnd;
    const long b0 = sbase[s];
    const int w = swidth[s];
    double yi[3] = {0.0, 0.0, 0.0};
    for (int r0 = 0; r0 < w; r0 += ROUND) {
#pragma unroll 1
        for (int j = 0; j < GW; j++) {
            const int k0 = r0 + RG * (GW * wv + j);
            if (k0 >= w) break;
            // past the row's last slot that slot again (not used): no branch
            // stands around a load
            double xc[RG][3];
            MT v[RG][9];
#pragma unroll
            for (int i = 0; i < RG; i++) {
                const long blk = b0 + min(k0 + i, w - 1);
                const int* pc = bcol + blk * 64 + l;
                const int cr = NT ? __builtin_nontemporal_load(pc) : *pc;
                const int c = cr >= 0 ? cr : own ? a : 0;
                const MT* pv = bval + blk * 576 + l;
#pragma unroll
                for (int m = 0; m < 9; m++) v[i][m] = NT ? __builtin_nontemporal_load(pv + 64 * m) : pv[64 * m];
#pragma unroll
                for (int m = 0; m < 3; m++) xc[i][m] = x[3L * c + m];
            }
            double gs[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < RG; i++) {
                double vd[9];
#pragma unroll
                for (int m = 0; m < 9; m++) vd[m] = (double)v[i][m];
                if (k0 + i < w) block_mac(vd, xc[i][0], xc[i][1], xc[i][2], gs);
            }
#pragma unroll
            for (int i = 0; i < 3; i++) red[GW * wv + j][i][l] = gs[i];
        }
        __syncthreads();
        if (wv == 0)
            for (int j = 0; j < SHARE_WAVES * GW && r0 + RG * j < w; j++)
#pragma unroll
                for (int i = 0; i < 3; i++) yi[i] += red[j][i][l];
        if (r0 + ROUND < w) __syncthreads();
    }
    if (wv > 0) return;
    double dv = 0.0;
    if (own) {
#pragma unroll
        for (int i = 0; i < 3; i++) y[3L * a + i] = yi[i];
        dv = yi[0] * x[3L * a] + yi[1] * x[3L * a + 1] + yi[2] * x[3L * a + 2];
    }
    dv = wsum(dv);
    if (l == 0) ppq[s] = dv;
}

__global__ void __launch_bounds__(FB) k_seg_fin_alpha(SegTab T, const double* __restrict__ ppq, int o,
                                                      double* __restrict__ sc)
{
    const int g = blockIdx.x;
    if (*sf(sc, S_DONE, T.nseg, g) != 0.0) return;
    double tot[1];
    seg_total<1, false>(ppq + T.seg_slice[g], 0, T.slices(g), T.slices(g), tot);
    if (threadIdx.x == 0) *sf(sc, S_ALPHA, T.nseg, g) = *slot_rz(sc, o, T.nseg, g) / tot[0];
}

// x += alpha p, r -= alpha q; partials of r.M^-1 r and r.r (with the
// multigrid, r.r only: r.z follows the V-cycle).  One workgroup per group.
// FOLD: alpha = r.z / p.q from the slice partials of p.q, else from its
// scalar slot.  With z given, M^-1 r is kept for the direction.
template <int PC, bool FOLD>
__global__ void __launch_bounds__(PB) k_seg_update(SegTab T, int nnd, const double* __restrict__ p,
                                                   const double* __restrict__ q, const double* __restrict__ m,
                                                   double* __restrict__ x, double* __restrict__ r,
                                                   double* __restrict__ z, const double* __restrict__ ppq,
                                                   double* __restrict__ part, int o, double* sc)
{
    const int4 gr = T.grp[blockIdx.x];
    const int g = gr.z, nseg = T.nseg;
    if (*sf(sc, S_DONE, nseg, g) != 0.0) return;
    // the vectors first: their loads are in flight while the total is formed
    const int a = 64 * gr.x + threadIdx.x;
    const bool own = (int)(threadIdx.x >> 6) < gr.y && a < nnd;
    double xi[3], ri[3], pi[3], qi[3], mi[PC == 1 ? 9 : 3];
    const long k0 = own ? 3L * a : 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        pi[i] = p[k0 + i];
        qi[i] = q[k0 + i];
        ri[i] = r[k0 + i];
        xi[i] = x[k0 + i];
    }
    if (PC != 2)
#pragma unroll
        for (int i = 0; i < (PC == 1 ? 9 : 3); i++) mi[i] = m[(PC == 1 ? 3 : 1) * k0 + i];
    double alpha;
    if (FOLD) {
        double tot[1];
        wave_total<1, false>(ppq + T.seg_slice[g], 0, T.slices(g), tot);
        alpha = *slot_rz(sc, o, nseg, g) / tot[0];
    } else {
        alpha = *sf(sc, S_ALPHA, nseg, g);
    }
    double v[2] = {0.0, 0.0};
    if (own) {
        double zi[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            x[k0 + i] = xi[i] + alpha * pi[i];
            ri[i] = ri[i] - alpha * qi[i];
            r[k0 + i] = ri[i];
        }
        if (PC != 2) precondition<PC>(mi, 0, ri, zi);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            if (PC != 2) v[0] += ri[i] * zi[i];
            v[1] += ri[i] * ri[i];
        }
        if (PC != 2 && z)
#pragma unroll
            for (int i = 0; i < 3; i++) z[k0 + i] = zi[i];
    }
    if (PC != 2) v[0] = wsum(v[0]);
    v[1] = wsum(v[1]);
    group_partials<2>(v, part, T.nslices, {PC != 2, true});
}

// the end of an iteration, one workgroup per segment
__global__ void __launch_bounds__(FB) k_seg_fin_beta(SegTab T, const double* __restrict__ part, int o,
                                                     double* __restrict__ sc, int* __restrict__ ndone)
{
    const int g = blockIdx.x;
    if (*sf(sc, S_DONE, T.nseg, g) != 0.0) return;
    double tot[2], beta;
    seg_total<2, true>(part + T.seg_grp[g], T.nslices, T.groups(g), T.slices(g), tot);
    if (threadIdx.x == 0) seg_advance(tot, sc, T.nseg, g, o, true, ndone, beta);
}

// p = M^-1 r + beta p.  FOLD: the end of the iteration (beta, the stopping
// test) from the partials, else beta from its scalar slot.  PC = 2: m holds
// M^-1 r itself.
template <int PC, bool FOLD>
__global__ void __launch_bounds__(PB) k_seg_direction(SegTab T, int nnd, const double* __restrict__ r,
                                                      const double* __restrict__ m, double* __restrict__ p,
                                                      const double* __restrict__ part, int o, double* sc, int* ndone)
{
    const int4 gr = T.grp[blockIdx.x];
    const int g = gr.z, nseg = T.nseg;
    if (*sf(sc, S_DONE, nseg, g) != 0.0) return;
    const int a = 64 * gr.x + threadIdx.x;
    const bool own = (int)(threadIdx.x >> 6) < gr.y && a < nnd;
    const long k0 = own ? 3L * a : 0;
    double ri[3], pi[3], zi[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        ri[i] = PC == 2 ? 0.0 : r[k0 + i];
        pi[i] = p[k0 + i];
    }
    precondition<PC>(m, k0 / 3, ri, zi);
    double beta;
    if (FOLD) {
        double tot[2];
        wave_total<2, true>(part + T.seg_grp[g], T.nslices, T.groups(g), tot);
        if (seg_advance(tot, sc, nseg, g, o, gr.x == T.seg_slice[g] && threadIdx.x == 0, ndone, beta)) return;
    } else {
        beta = *sf(sc, S_BETA, nseg, g);
    }
    if (!own) return;
#pragma unroll
    for (int i = 0; i < 3; i++) p[k0 + i] = zi[i] + beta * pi[i];
}

// ---- persistent iteration: one workgroup per small segment ----------------
//
// A segment of at most PERSIST_MAX slices (PW = 1024 nodes) keeps its
// whole CG loop inside one workgroup of PW threads, thread t owning node
// 64 sb + t: its x and r stay in registers, the direction p in LDS
// (the SpMV gathers neighbours from there), the per-slice partials and the
// segment scalars in registers; only the operator is read from memory (L2)
// each iteration, and no kernel is launched per iteration.  The arithmetic
// is the kernel-per-step iteration's, in the same order: the row sums of
// row_sum, the updates of k_seg_update and k_seg_direction, and each
// per-segment total summed as wave_total sums it, by every wave for itself
// from the partials in LDS (one barrier per total).  So the iterates are
// bitwise those of the kernel-per-step iteration.  The loop ends on the
// segment's own stopping test or iteration cap, as seg_advance decides; the
// final x, r, p and scalars are written back as that iteration leaves them.
constexpr int PW = FB;
constexpr int PERSIST_MAX = PW / 64;
static_assert(PERSIST_MAX == PCG_PERSIST_MAX, "the host's threshold cap is the kernel's slice capacity");

// per-segment totals of the NV x nsl partials lp, in every lane, in
// wave_total's order (nsl <= 16: lanes 0..3 hold four each)
template <int NV>
__device__ __forceinline__ void wave_total_lds(const double (&lp)[2][PERSIST_MAX], int nsl, double (&tot)[NV])
{
    const int s = 4 * (threadIdx.x & 63);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const double a0 = s < nsl ? lp[k][s] : 0.0, a1 = s + 1 < nsl ? lp[k][s + 1] : 0.0;
        const double a2 = s + 2 < nsl ? lp[k][s + 2] : 0.0, a3 = s + 3 < nsl ? lp[k][s + 3] : 0.0;
        tot[k] = wsum(0.0 + (((a0 + a1) + a2) + a3));
    }
}

template <class MT, int PC>
__global__ void __launch_bounds__(PW) k_pcg_persistent(const int* __restrict__ segs, int nnd,
                                                       const int* __restrict__ seg_slice,
                                                       const int* __restrict__ sbase, const int* __restrict__ swidth,
                                                       const int* __restrict__ bcol, const MT* __restrict__ bval,
                                                       const double* __restrict__ m, double* __restrict__ x,
                                                       double* __restrict__ r, double* __restrict__ p, int nseg,
                                                       double* __restrict__ sc, int* __restrict__ ndone)
{
    __shared__ double sp[PW][3];
    __shared__ double lpq[2][PERSIST_MAX], lrz[2][PERSIST_MAX];
    const int g = segs[blockIdx.x];
    const int sb = seg_slice[g], nsl = seg_slice[g + 1] - sb;
    const int t = threadIdx.x, l = t & 63;
    const int s = sb + (t >> 6);          // this thread's slice
    const int base = 64 * sb;             // first node of the segment
    const int a = base + t;               // this thread's node
    const bool own = (t >> 6) < nsl && a < nnd;
    if (*sf(sc, S_DONE, nseg, g) != 0.0) return;
    double rz = *sf(sc, S_RZ, nseg, g), rr = 0.0, iter = 0.0;
    const double thresh = *sf(sc, S_THRESH, nseg, g), maxit = *sf(sc, S_MAXIT, nseg, g);
    double xi[3] = {0, 0, 0}, ri[3] = {0, 0, 0}, zi[3] = {0, 0, 0}, pi[3] = {0, 0, 0};
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (own) {
            xi[i] = x[3L * a + i];
            ri[i] = r[3L * a + i];
            pi[i] = p[3L * a + i];
        }
        sp[t][i] = pi[i];
    }
    __syncthreads();
    for (;;) {
        // q = A p and the slice partial of p.q
        double qi[3] = {0, 0, 0};
        {
            double dv = 0.0;
            if (own) {
                row_sum<MT, true, false>(bcol, bval, nullptr, sbase[s], swidth[s], l, a,
                                         [&](int c, double& x0, double& x1, double& x2) {
                                             x0 = sp[c - base][0];
                                             x1 = sp[c - base][1];
                                             x2 = sp[c - base][2];
                                         }, qi);
                dv = qi[0] * pi[0] + qi[1] * pi[1] + qi[2] * pi[2];
            }
            dv = wsum(dv);
            if (l == 0 && (t >> 6) < nsl) lpq[0][t >> 6] = dv;
        }
        __syncthreads();
        double pq[1];
        wave_total_lds<1>(lpq, nsl, pq);
        const double al = rz / pq[0];
        // x += alpha p, r -= alpha q, z = M^-1 r; slice partials of r.z, r.r (k_seg_update)
        {
            double v0 = 0.0, v1 = 0.0;
            if (own) {
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    xi[i] += al * pi[i];
                    ri[i] = ri[i] - al * qi[i];
                }
                precondition<PC>(m, a, ri, zi);
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    v0 += ri[i] * zi[i];
                    v1 += ri[i] * ri[i];
                }
            }
            v0 = wsum(v0);
            v1 = wsum(v1);
            if (l == 0 && (t >> 6) < nsl) {
                lrz[0][t >> 6] = v0;
                lrz[1][t >> 6] = v1;
            }
        }
        __syncthreads();
        // the end of the iteration (seg_advance), the same in every lane
        double tot[2];
        wave_total_lds<2>(lrz, nsl, tot);
        iter = iter + 1.0;
        const double be = tot[0] / rz;
        rz = tot[0];
        rr = tot[1];
        if (tot[1] <= thresh || iter >= maxit) break;
        // p = M^-1 r + beta p (every wave is past this iteration's reads of
        // sp: they came before the first barrier)
        if (own)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                pi[i] = zi[i] + be * pi[i];
                sp[t][i] = pi[i];
            }
        __syncthreads();
    }
    if (own)
#pragma unroll
        for (int i = 0; i < 3; i++) {
            x[3L * a + i] = xi[i];
            r[3L * a + i] = ri[i];
            p[3L * a + i] = pi[i];
        }
    if (t == 0) {
        *sf(sc, S_ITER, nseg, g) = iter;
        *sf(sc, S_RZ, nseg, g) = rz;
        *sf(sc, S_RR, nseg, g) = rr;
        *sf(sc, S_DONE, nseg, g) = 1.0;
        atomicAdd(ndone, 1);
    }
}

// ---- fused iteration: the direction formed inside the SpMV ------------------
//
// The direction update p = z + beta p_old is formed inside the SpMV -- for
// the SpMV's own rows, which it stores, and for every neighbour it gathers --
// so the separate direction pass (and its reads of r, z and p) disappears;
// p is double-buffered (the SpMV reads p_old of its neighbours while it
// writes p of its own rows).  With the totals folded into the kernels that
// need them, an iteration is two kernels: this one, which first closes the
// iteration before (beta, the stopping test: seg_advance) from the update's
// partials, and the update, which forms alpha from this one's.  A device-
// scope fence per wave instead (one kernel per iteration) would write back
// and invalidate the XCD's L2 each time.

// z at dof k: Jacobi (m = 1/diag) or kept by the update / the multigrid (m = z)
template <int PC>
__device__ __forceinline__ double zval(const double* __restrict__ m, const double* __restrict__ r, long k)
{
    return PC == 2 ? m[k] : m[k] * r[k];
}

// beta of segment g for the SpMV of slice s, closing the iteration before
// when `close`; returns whether the segment is done
__device__ __forceinline__ bool direction_beta(const SegTab& T, const double* part, int g, int s, bool owner_lane,
                                               bool close, int o, double* sc, int* ndone, double& beta)
{
    if (!close) {
        beta = *sf(sc, S_BETA, T.nseg, g);
        return false;
    }
    double tot[2];
    wave_total<2, true>(part + T.seg_grp[g], T.nslices, T.groups(g), tot);
    return seg_advance(tot, sc, T.nseg, g, o, s == T.seg_slice[g] && owner_lane, ndone, beta);
}

template <class MT, int PC, bool XCD, bool UNR, bool SYM>
__global__ void __launch_bounds__(PB) k_fused_spmv(SegTab T, int nnd,
                                                   const int* __restrict__ sbase, const int* __restrict__ swidth,
                                                   const int* __restrict__ bcol, const MT* __restrict__ bval,
                                                   const int* __restrict__ tpos,
                                                   const double* __restrict__ m, const double* __restrict__ r,
                                                   const double* __restrict__ pold, double* __restrict__ pnew,
                                                   double* __restrict__ y, const double* __restrict__ part,
                                                   double* __restrict__ ppq, int close, int o, double* sc, int* ndone)
{
    const int a = row_block<XCD>() * PB + threadIdx.x;
    const int s = __builtin_amdgcn_readfirstlane(a >> 6), l = a & 63;
    if (s >= T.nslices) return;
    const int g = T.slice_seg[s];
    if (*sf(sc, S_DONE, T.nseg, g) != 0.0) return;
    double beta;
    if (direction_beta(T, part, g, s, l == 0, close, o, sc, ndone, beta)) return;
    double dv = 0.0;
    if (a < nnd) {
        double yi[3], p3[3];
        row_sum<MT, UNR, SYM>(bcol, bval, tpos, sbase[s], swidth[s], l, a, [&](int c, double& x0, double& x1, double& x2) {
            x0 = zval<PC>(m, r, 3L * c) + beta * pold[3L * c];
            x1 = zval<PC>(m, r, 3L * c + 1) + beta * pold[3L * c + 1];
            x2 = zval<PC>(m, r, 3L * c + 2) + beta * pold[3L * c + 2];
        }, yi);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            p3[i] = zval<PC>(m, r, 3L * a + i) + beta * pold[3L * a + i];
            pnew[3L * a + i] = p3[i];
            y[3L * a + i] = yi[i];
        }
        dv = yi[0] * p3[0] + yi[1] * p3[1] + yi[2] * p3[2];
    }
    dv = wsum(dv);
    if (l == 0) ppq[s] = dv;
}

// The fused SpMV with a row's groups of slots dealt to the NW waves of a
// workgroup, one workgroup per slice: at a few hundred slices a lane that
// walks 27 blocks by itself is a chain of dependent loads on a nearly idle
// chip (FP64, 77 slices: 17.2 us a launch with a lane per row, 6.3 with nine
// waves; 363 slices: 23.1 and 12.5 with five, where the 48 MB operator comes
// from the last-level cache at 3.8 TB/s).  z holds M^-1 r.  Wave 0 closes the iteration before while the other
// waves' first loads are in flight; the group sums meet in LDS and wave 0
// adds them in order, so the product is bitwise k_fused_spmv's.  Each XCD
// takes a contiguous range of slices (row_block), so the gathered vectors
// stay in its L2 (1,077 slices, FP32: 27.7 us per iteration in launch order,
// 25.4 so).
// PRE: the gathers, too, are issued before beta is known (more registers).
template <class MT, int NW, bool PRE>
__global__ void __launch_bounds__(64 * NW) k_split_spmv(SegTab T, int nnd,
                                                        const int* __restrict__ sbase, const int* __restrict__ swidth,
                                                        const int* __restrict__ bcol, const MT* __restrict__ bval,
                                                        const double* __restrict__ z, const double* __restrict__ pold,
                                                        double* __restrict__ pnew, double* __restrict__ y,
                                                        const double* __restrict__ part, double* __restrict__ ppq,
                                                        int close, int o, double* sc, int* ndone)
{
    __shared__ double red[NW][3][64];
    __shared__ double sbeta;
    __shared__ int sdone;
    const int s = row_block<true>(), l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (s >= T.nslices) return;
    const int a = 64 * s + l;
    const int g = T.slice_seg[s];
    const long b0 = sbase[s];
    const int w = swidth[s];
    // the owner may set the flag while this kernel runs: a wave that sees it
    // skips its loads, and wave 0 comes to the same decision for them all
    const bool was_done = *sf(sc, S_DONE, T.nseg, g) != 0.0;
    const bool own = a < nnd;
    int c[RG];
    MT v[RG][9];
    double zc[PRE ? RG : 1][3], pc[PRE ? RG : 1][3];
    // slots k0 .. k0 + RG - 1, k0 < w; past the row's last slot that slot
    // again (not used), so no branch stands around a load
    auto load_group = [&](int k0) {
#pragma unroll
        for (int i = 0; i < RG; i++) {
            const long blk = b0 + min(k0 + i, w - 1);
            const int cr = bcol[blk * 64 + l];
            c[i] = own && cr >= 0 ? cr : (own ? a : 0);
#pragma unroll
            for (int m = 0; m < 9; m++) v[i][m] = bval[(blk * 9 + m) * 64 + l];
        }
        if (PRE)
#pragma unroll
            for (int i = 0; i < RG; i++)
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    zc[PRE ? i : 0][m] = z[3L * c[i] + m];
                    pc[PRE ? i : 0][m] = pold[3L * c[i] + m];
                }
    };
    if (!was_done && RG * wv < w) load_group(RG * wv);
    if (wv == 0) {
        double b = 0.0;
        const bool d = was_done || direction_beta(T, part, g, s, l == 0, close, o, sc, ndone, b);
        if (l == 0) {
            sbeta = b;
            sdone = d;
        }
    }
    __syncthreads();
    if (sdone) return;
    const double beta = sbeta;
    double yi[3] = {0.0, 0.0, 0.0};
    for (int r0 = 0; r0 < w; r0 += RG * NW) {
        const int k0 = r0 + RG * wv;
        if (k0 < w) {
            if (r0 > 0) load_group(k0);
            double gs[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < RG; i++) {
                double xv[3], vd[9];
#pragma unroll
                for (int m = 0; m < 3; m++)
                    xv[m] = PRE ? zc[PRE ? i : 0][m] + beta * pc[PRE ? i : 0][m] : z[3L * c[i] + m] + beta * pold[3L * c[i] + m];
#pragma unroll
                for (int m = 0; m < 9; m++) vd[m] = (double)v[i][m];
                if (k0 + i < w) block_mac(vd, xv[0], xv[1], xv[2], gs);
            }
#pragma unroll
            for (int i = 0; i < 3; i++) red[wv][i][l] = gs[i];
        }
        __syncthreads();
        if (wv == 0)
            for (int j = 0; j < NW && r0 + RG * j < w; j++)
#pragma unroll
                for (int i = 0; i < 3; i++) yi[i] += red[j][i][l];
        if (r0 + RG * NW < w) __syncthreads();
    }
    if (wv > 0) return;
    double dv = 0.0;
    if (own) {
        double p3[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            p3[i] = z[3L * a + i] + beta * pold[3L * a + i];
            pnew[3L * a + i] = p3[i];
            y[3L * a + i] = yi[i];
        }
        dv = yi[0] * p3[0] + yi[1] * p3[1] + yi[2] * p3[2];
    }
    dv = wsum(dv);
    if (l == 0) ppq[s] = dv;
}

// per-segment dot product a.b into out[seg]: partials per group, then totals
__global__ void __launch_bounds__(PB) k_seg_dot(SegTab T, int nnd, const double* __restrict__ x,
                                                const double* __restrict__ y, double* __restrict__ part)
{
    const int4 gr = T.grp[blockIdx.x];
    const int a = 64 * gr.x + threadIdx.x;
    double v[1] = {0.0};
    if ((int)(threadIdx.x >> 6) < gr.y && a < nnd)
#pragma unroll
        for (int i = 0; i < 3; i++) v[0] += x[3L * a + i] * y[3L * a + i];
    v[0] = wsum(v[0]);
    group_partials<1>(v, part, 0, {true});
}

__global__ void __launch_bounds__(FB) k_seg_fin_dot(SegTab T, const double* __restrict__ part, double* __restrict__ out)
{
    const int g = blockIdx.x;
    double tot[1];
    seg_total<1, true>(part + T.seg_grp[g], 0, T.groups(g), T.slices(g), tot);
    if (threadIdx.x == 0) out[g] = tot[0];
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

static unsigned node_blocks(const tg_ctx* c) { return (unsigned)((c->nnd + PB - 1) / PB); }

static SegTab seg_tab(const tg_ctx* c)
{
    const Segments& S = c->seg;
    return SegTab{S.d_slice_seg.p, S.d_seg_slice.p, S.d_seg_grp.p, S.d_grp.p, S.nseg, S.nslices};
}

// f(std::integral_constant<int, v>) for the SpMV variant v = 0..7 (bit 0
// XCD row ranges, bit 1 unrolled loop, bit 2 symmetric read), so every
// variant is its own kernel instance.
template <class F>
static void spmv_dispatch(int v, F f)
{
    switch (v & 7) {
    case 0: f(std::integral_constant<int, 0>{}); break;
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    default: f(std::integral_constant<int, 7>{}); break;
    }
}

void segment_dots(tg_ctx* c, const double* a, const double* b, double* host_out)
{
    {
        TimedRegion tr(c, T_VECTOR);
        const SegTab T = seg_tab(c);
        hipLaunchKernelGGL(k_seg_dot, dim3((unsigned)c->seg.ngroups), dim3(PB), 0, c->stream, T, c->nnd, a, b,
                           c->seg.d_part.p);
        hipLaunchKernelGGL(k_seg_fin_dot, dim3(c->seg.nseg), dim3(FB), 0, c->stream, T, c->seg.d_part.p, c->seg.d_out.p);
        TG_HIP(hipGetLastError());
    }
    TG_HIP(hipMemcpyAsync(host_out, c->seg.d_out.p, sizeof(double) * c->seg.nseg, hipMemcpyDeviceToHost, c->stream));
    TG_HIP(hipStreamSynchronize(c->stream));
}

template <class MT, int PC>
static void pcg_loop(tg_ctx* c, const MT* val, const double* m, const double* b, double* x, double* r, double* p,
                     double* q, double rtol, int maxit, const int* d_active, const PcgWork& W, tg_lin_stats* st);

template <class MT>
void pcg_run(tg_ctx* c, const MT* val, const double* dinv, const double* b, double* x, double* r, double* p,
             double* q, double rtol, int maxit, const int* d_active, int nactive, tg_lin_stats* st,
             const PcgWork* work)
{
    (void)nactive;
    PcgWork W;
    if (work) {
        W = *work;
    } else {
        // the context's own reductions, scalars and done count; the second
        // direction buffer of the fused iteration is allocated on first use
        if (pcg_fused(c) && c->vp2.n != 3 * (size_t)c->nnd) c->vp2.alloc(3 * (size_t)c->nnd);
        W = PcgWork{c->seg.d_part.p, c->seg.d_part.p + 2 * c->seg.nslices, c->seg.d_scal.p, c->seg.d_ndone.p, c->vp2.p,
                    c->vz.p, true};
    }
    if (c->precond == TG_PC_BLOCK_JACOBI)
        pcg_loop<MT, 1>(c, val, c->vbinv.p, b, x, r, p, q, rtol, maxit, d_active, W, st);
    else if (c->precond == TG_PC_AMG)
        pcg_loop<MT, 2>(c, val, c->amg.lv[0]->d_x.p, b, x, r, p, q, rtol, maxit, d_active, W, st);
    else
        pcg_loop<MT, 0>(c, val, dinv, b, x, r, p, q, rtol, maxit, d_active, W, st);
}

template <class MT, int PC>
static void pcg_loop(tg_ctx* c, const MT* val, const double* dinv, const double* b, double* x, double* r, double* p,
                     double* q, double rtol, int maxit, const int* d_active, const PcgWork& W, tg_lin_stats* st)
{
    Segments& S = c->seg;
    const long ns = S.nslices;
    const int nseg = S.nseg;
    const unsigned nb = node_blocks(c), ng = (unsigned)S.ngroups;
    const SegTab T = seg_tab(c);
    TG_HIP(hipMemsetAsync(W.ndone, 0, sizeof(int), c->stream));
    // multigrid: dinv is the z vector; *done of the single segment gates the V-cycle
    const double* done = W.scal + S_DONE * nseg;
    if (PC == 2) {
        TimedRegion tr(c, T_PRECOND);
        amg_vcycle(c, b, (double*)dinv, nullptr);
    }
    // The totals are formed inside the kernels that need them (FOLD) when no
    // segment has more than FOLD_SLICES slices and the work space has room
    // for the partials of p.q beside those of r.z and r.r; the multigrid
    // needs r.r before its cycle and r.z after it, and keeps its finalize
    // kernels.
    const bool fold = PC != 2 && W.ppq && S.max_slices <= FOLD_SLICES;
    const bool fused = pcg_fused(c) && (PC != 1 || fold);
    // M^-1 r kept by the update: for the folded fused iteration, whose SpMV
    // gathers it, and for block Jacobi, whose direction would form it again
    // from the 3x3 blocks
    const bool keep_z = PC != 2 && W.z && (fold ? fused || PC == 1 : false);
    double* z = keep_z ? W.z : nullptr;
    {
        TimedRegion tr(c, T_VECTOR);
        hipLaunchKernelGGL(k_seg_init<PC>, dim3(ng), dim3(PB), 0, c->stream, T, c->nnd, b, dinv, x, r, p, z, W.part);
        hipLaunchKernelGGL(k_seg_fin_init, dim3(nseg), dim3(FB), 0, c->stream, T, W.part, d_active, W.scal, rtol, maxit,
                           W.ndone);
    }
    // small segments: the whole iteration in one persistent workgroup each
    // (the list is built at set-up and when the threshold changes)
    const int npers = PC == 2 || S.persist_built != pcg_persist(c) ? 0 : (int)S.h_persist.size();
    if (npers > 0) {
        TimedRegion tr(c, T_SPMV);
        hipLaunchKernelGGL((k_pcg_persistent<MT, PC>), dim3(npers), dim3(PW), 0, c->stream, S.d_persist.p, c->nnd,
                           S.d_seg_slice.p, c->op.d_slice_base.p, c->op.d_slice_width.p, c->op.d_col.p, val, dinv, x,
                           r, p, nseg, W.scal, W.ndone);
        TG_HIP(hipGetLastError());
    }
    if (npers < nseg) {
    // even: direction buffers and scalar slots alternate.  An iteration with the
    // multigrid is some 60 kernels: chunks of two keep the launches queued past
    // the last iteration few (chunks of eight cost 1.6 ms a solve at 128^3)
    const int CHUNK = PC == 2 ? 2 : 16;
    double* pbuf[2] = {p, nullptr};
    if (fused) {
        if (!W.p2) fail(TG_GENERAL_FAIL, "fused PCG iteration without its second direction buffer");
        pbuf[1] = W.p2;
    }
    const int variant = spmv_variant(c);
    double* ppq = fold ? W.ppq : W.part;
    // rows split over the waves of a workgroup
    const int split = fold && fused ? pcg_split(c) : 0;
    // the unfused iteration's product: 1..4 by three waves a row (+ 1 streaming,
    // + 2 contiguous ranges of slices for the XCDs), 5 the batch's variant
    // streaming, 0 the variant as it is
    const bool streams = op_streams(c, sizeof(MT));
    const int share = fused || c->spmv_xcd >= 0 ? 0
                      : pcg_share(c, sizeof(MT)) ? 1 + (streams ? 1 : 0) + (c->nnd < 1 << 19 ? 2 : 0)
                                                 : (variant == 2 && streams ? 5 : 0);
    auto update = [&](const double* pk, int o) {
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(ng), dim3(PB), 0, c->stream, T, c->nnd, pk, q, dinv, x, r, z, ppq, W.part, o,
                               W.scal);
        };
        if (fold)
            go(k_seg_update<PC, true>);
        else
            go(k_seg_update<PC, false>);
    };
    auto fin_alpha = [&](int o) {
        hipLaunchKernelGGL(k_seg_fin_alpha, dim3(nseg), dim3(FB), 0, c->stream, T, ppq, o, W.scal);
    };
    auto fin_beta = [&](int o) {
        hipLaunchKernelGGL(k_seg_fin_beta, dim3(nseg), dim3(FB), 0, c->stream, T, W.part, o, W.scal, W.ndone);
    };
    auto precond_pass = [&]() {
        TimedRegion tr(c, T_PRECOND);
        amg_vcycle(c, r, (double*)dinv, done);
        hipLaunchKernelGGL(k_seg_dot, dim3(ng), dim3(PB), 0, c->stream, T, c->nnd, r, dinv, W.part);
    };
    // the fused SpMV of iteration k; folded, it closes iteration k - 1 itself
    // (slot o = (k - 1) & 1), except in the first iteration of a chunk, which
    // finds beta in its scalar slot
    auto spmv_fused = [&](int k) {
        TimedRegion tr(c, T_SPMV);
        const double* pold = pbuf[k & 1];
        double* pnew = pbuf[(k + 1) & 1];
        const int close = fold && k > 0, o = (k + 1) & 1;
        auto go_split = [&](auto kernel, int nw) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)(ns + 7) / 8 * 8), dim3(64 * nw), 0, c->stream, T, c->nnd, c->op.d_slice_base.p,
                               c->op.d_slice_width.p, c->op.d_col.p, val, z, pold, pnew, q, W.part, ppq, close, o,
                               W.scal, W.ndone);
        };
        if (split == 9) {
            go_split(k_split_spmv<MT, 9, true>, 9);
            return;
        }
        if (split == 5) {
            go_split(k_split_spmv<MT, 5, false>, 5);
            return;
        }
        if (split == 3) {
            go_split(k_split_spmv<MT, 3, false>, 3);
            return;
        }
        spmv_dispatch(variant, [&](auto V) {
            constexpr int v = decltype(V)::value;
            auto go = [&](auto kernel, const double* m) {
                hipLaunchKernelGGL(kernel, dim3((v & 1) ? (nb + 7) / 8 * 8 : nb), dim3(PB), 0, c->stream, T, c->nnd,
                                   c->op.d_slice_base.p, c->op.d_slice_width.p, c->op.d_col.p, val, c->op.d_tpos.p, m,
                                   r, pold, pnew, q, W.part, ppq, close, o, W.scal, W.ndone);
            };
            if (PC == 2 || z)
                go(k_fused_spmv<MT, 2, (v & 1) != 0, (v & 2) != 0, (v & 4) != 0>, z ? z : dinv);
            else if constexpr (PC == 0)
                go(k_fused_spmv<MT, 0, (v & 1) != 0, (v & 2) != 0, (v & 4) != 0>, dinv);
        });
    };
    auto issue_fused = [&]() {
        for (int k = 0; k < CHUNK; k++) {
            spmv_fused(k);
            {
                TimedRegion tr(c, T_VECTOR);
                if (!fold) fin_alpha(k & 1);
                update(pbuf[(k + 1) & 1], k & 1);
            }
            if (PC == 2) precond_pass();
            if (!fold || k == CHUNK - 1) {
                TimedRegion tr(c, T_VECTOR);
                fin_beta(k & 1);
            }
        }
    };
    auto issue_chunk = [&]() {
        if (fused) {
            issue_fused();
            return;
        }
        for (int k = 0; k < CHUNK; k++) {
            {
                TimedRegion tr(c, T_SPMV);
                auto go_share = [&](auto kernel) {
                    hipLaunchKernelGGL(kernel, dim3((unsigned)(ns + 7) / 8 * 8), dim3(64 * SHARE_WAVES), 0, c->stream, T,
                                       c->nnd, c->op.d_slice_base.p, c->op.d_slice_width.p, c->op.d_col.p, val, p, q, ppq,
                                       W.scal);
                };
                if (share == 4)
                    go_share(k_share_spmv<MT, true, true>);
                else if (share == 3)
                    go_share(k_share_spmv<MT, true, false>);
                else if (share == 2)
                    go_share(k_share_spmv<MT, false, true>);
                else if (share == 1)
                    go_share(k_share_spmv<MT, false, false>);
                auto go = [&](auto kernel, unsigned blocks) {
                    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(PB), 0, c->stream, T, c->nnd, c->op.d_slice_base.p,
                                       c->op.d_slice_width.p, c->op.d_col.p, val, c->op.d_tpos.p, p, q, ppq, W.scal);
                };
                if (share == 5)
                    go(k_seg_spmv<MT, false, true, false, true>, nb);
                else if (share == 0)
                    spmv_dispatch(variant, [&](auto V) {
                        constexpr int v = decltype(V)::value;
                        go(k_seg_spmv<MT, (v & 1) != 0, (v & 2) != 0, (v & 4) != 0>, (v & 1) ? (nb + 7) / 8 * 8 : nb);
                    });
            }
            {
                TimedRegion tr(c, T_VECTOR);
                if (!fold) fin_alpha(k & 1);
                update(p, k & 1);
            }
            if (PC == 2) precond_pass();
            {
                TimedRegion tr(c, T_VECTOR);
                if (!fold) fin_beta(k & 1);
                auto go = [&](auto kernel, const double* m) {
                    hipLaunchKernelGGL(kernel, dim3(ng), dim3(PB), 0, c->stream, T, c->nnd, r, m, p, W.part, k & 1,
                                       W.scal, W.ndone);
                };
                if (!fold)
                    go(k_seg_direction<PC, false>, dinv);
                else if (z)
                    go(k_seg_direction<2, true>, z);
                else
                    go(k_seg_direction<PC, true>, dinv);
            }
        }
    };
    // The chunk's kernels only ever see the same pointers, so one capture
    // serves every later solve of this context with the same vectors; the
    // iteration state lives in device memory (done flags make finished
    // segments' work a no-op).  The graph holds kernel nodes only.
    const bool graph = W.graph && c->pcg_graph && !c->timing.enabled;
    if (graph) {
        // every address and size the chunk's launches take (tg_initialize
        // also drops the graph, as buffers may come back at old addresses)
        const void* key[24] = {val, dinv, x, r, p, q, W.part, W.scal, W.ndone,
                               (const void*)(long)(PC + 4L * (variant + 8L * ((int)fused + 2L * (split + 16L * (share + 8L * c->amg.gen))))),
                               (const void*)(long)sizeof(MT), (const void*)(long)c->nnd, (const void*)(long)nseg,
                               (const void*)ns, S.d_grp.p, S.d_slice_seg.p, c->op.d_slice_base.p,
                               c->op.d_slice_width.p, c->op.d_col.p, pbuf[1], z,
                               c->amg.lv.empty() ? nullptr : (const void*)c->amg.lv[0], c->op.d_tpos.p};
        if (!c->pg.exec || std::memcmp(key, c->pg.key, sizeof key) != 0) {
            drop_pcg_graph(c);
            TG_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
            issue_chunk();
            TG_HIP(hipStreamEndCapture(c->stream, &c->pg.graph));
            TG_HIP(hipGraphInstantiate(&c->pg.exec, c->pg.graph, nullptr, nullptr, 0));
            std::memcpy(c->pg.key, key, sizeof key);
        }
    }
    // (tg_create made the two poll events)
    // Chunk k+1 is queued before chunk k's done count is read, so the GPU
    // never waits for the host; a chunk queued after every segment finished
    // does nothing.
    int issued = 0, chunks = 0;
    for (;;) {
        if (graph)
            TG_HIP(hipGraphLaunch(c->pg.exec, c->stream));
        else
            issue_chunk();
        TG_HIP(hipGetLastError());
        issued += CHUNK;
        const int slot = chunks & 1;
        TG_HIP(hipMemcpyAsync(c->hstatus + 2 + slot, W.ndone, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        TG_HIP(hipEventRecord(c->poll_ev[slot], c->stream));
        chunks++;
        if (issued >= maxit) break;
        if (chunks >= 2) {
            const int prev = (chunks - 2) & 1;
            TG_HIP(hipEventSynchronize(c->poll_ev[prev]));
            if (c->hstatus[2 + prev] >= nseg) break;
        }
    }
    }  // npers < nseg
    TG_HIP(hipStreamSynchronize(c->stream));
    // per-segment results
    if (S.h_scal.size() != (size_t)S_NSCAL * nseg) S.h_scal.resize((size_t)S_NSCAL * nseg);
    TG_HIP(hipMemcpyAsync(S.h_scal.data(), W.scal, sizeof(double) * S_NSCAL * nseg, hipMemcpyDeviceToHost,
                          c->stream));
    TG_HIP(hipStreamSynchronize(c->stream));
    if (st) {
        // aggregate: max iterations, worst relative residual, all converged
        st->iterations = 0;
        st->rel_residual = 0.0;
        st->converged = 1;
        for (int g = 0; g < nseg; g++) {
            const double it = S.h_scal[(size_t)S_ITER * nseg + g];
            const double bb = S.h_scal[(size_t)S_BB * nseg + g];
            const double rr = S.h_scal[(size_t)S_RR * nseg + g];
            const double th = S.h_scal[(size_t)S_THRESH * nseg + g];
            st->iterations = std::max(st->iterations, (int)it);
            if (bb > 0.0) st->rel_residual = std::max(st->rel_residual, sqrt(rr / bb));
            if (rr > th) st->converged = 0;
        }
    }
}

template void pcg_run<double>(tg_ctx*, const double*, const double*, const double*, double*, double*, double*,
                              double*, double, int, const int*, int, tg_lin_stats*, const PcgWork*);
template void pcg_run<float>(tg_ctx*, const float*, const double*, const double*, double*, double*, double*,
                             double*, double, int, const int*, int, tg_lin_stats*, const PcgWork*);

}  // namespace tg
