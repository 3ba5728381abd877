// Assembly by rows: the element kernels write their forces and stiffness
// blocks to buffers, all elements in one launch, and a gather sums each
// node's, in ascending element order, and writes every result once.  No
// colours, no read-modify-write of the matrix, no clearing pass: the sums
// depend only on a node's own elements, so a problem's result is the same
// alone and in any batch, run to run.
//
// Buffers.  The nodes of an element are ranked by their numbers.  Force
// buffer: [element][rank][3].  Block buffer: [element][36][9], the 3x3 blocks
// of rank pairs (r, s), r <= s, row by row: the node of rank r needs the
// 8 - r consecutive blocks of its row, so a gather reads contiguous runs.
// Only the upper entries of a diagonal block are written.
#include "tg_internal.h"
#include "tg_element.h"

namespace tg {

namespace {

// ---- structure --------------------------------------------------------------

// ranks of element e's nodes: 4 bits per local node
__global__ void k_ranks(int nel, const int* __restrict__ conn, unsigned* __restrict__ perm)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nel) return;
    int n[8];
#pragma unroll
    for (int a = 0; a < 8; a++) n[a] = conn[8L * e + a];
    unsigned p = 0;
#pragma unroll
    for (int a = 0; a < 8; a++) {
        int r = 0;
#pragma unroll
        for (int b = 0; b < 8; b++) r += n[b] < n[a];
        p |= (unsigned)r << (4 * a);
    }
    perm[e] = p;
}

// each node's list of (8 element + rank) codes ascending (the lists come
// from atomic appends; insertion sort, at most 8 entries on a hexahedral grid)
__global__ void k_sort_lists(int nnd, const int* __restrict__ ptr, int* __restrict__ list)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nnd) return;
    const int p0 = ptr[a], n = ptr[a + 1] - p0;
    for (int i = 1; i < n; i++) {
        const int x = list[p0 + i];
        int j = i;
        while (j > 0 && list[p0 + j - 1] > x) {
            list[p0 + j] = list[p0 + j - 1];
            j--;
        }
        list[p0 + j] = x;
    }
}

// slot index of each row's diagonal block (the number of its lower blocks),
// the row's upper slots, and their largest number over all rows
__global__ void k_row_upper(int nnd, const int* __restrict__ sbase, const int* __restrict__ swidth,
                            const int* __restrict__ bcol, int2* __restrict__ upper, int* __restrict__ most)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nnd) return;
    const int s = a >> 6, l = a & 63;
    int lo = 0, n = 0;
    for (int k = 0; k < swidth[s]; k++) {
        const int c = bcol[((long)sbase[s] + k) * 64 + l];
        if (c < 0) break;
        n++;
        lo += c < a;
    }
    upper[a] = make_int2(lo, n - lo);
    atomicMax(most, n - lo);
}

// rslot[e][r][j] = upper slot (0: the diagonal) of the row of rank r that
// block (r, r + j) of element e goes to; one thread per (element, rank)
__global__ void k_row_slots(int nel, const int* __restrict__ conn, const unsigned* __restrict__ perm,
                            const int* __restrict__ sbase, const int* __restrict__ bcol,
                            const int2* __restrict__ upper, unsigned char* __restrict__ rslot)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 8L * nel) return;
    const int e = (int)(t >> 3), r = (int)(t & 7);
    const unsigned p = perm[e];
    int node[8];  // by rank
#pragma unroll
    for (int a = 0; a < 8; a++) {
        const int x = conn[8L * e + a];
        const int ra = (p >> (4 * a)) & 7;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (ra == q) node[q] = x;
    }
    int A = node[0];
#pragma unroll
    for (int q = 1; q < 8; q++)
        if (r == q) A = node[q];
    const int2 up = upper[A];
    const long base = ((long)sbase[A >> 6] + up.x) * 64 + (A & 63);
    unsigned long long out = 0;
    int k = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        if (q < r) continue;
        while (k < up.y - 1 && bcol[base + 64L * k] < node[q]) k++;  // columns ascend as the ranks do
        out |= (unsigned long long)(unsigned char)k << (8 * (q - r));
    }
    reinterpret_cast<unsigned long long*>(rslot)[t] = out;
}

// the partner of an upper off-diagonal block, coded -index - 2, beside the
// lower blocks' partners (which stay >= 0)
__global__ void k_upper_partners(long n, const int* __restrict__ tpos_in, int* __restrict__ tpos)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int t = tpos_in[i];
    if (t < 0) return;
    // value index t = (blk * 9) * 64 + l of the upper block
    const long blk = (t >> 6) / 9, l = t & 63;
    tpos[blk * 64 + l] = -(int)(((i >> 6) * 9) * 64 + (i & 63)) - 2;
}

// ---- residual ---------------------------------------------------------------

// R = the sum of each node's element forces, plus the applied forces, zero at
// prescribed dofs; one thread per dof (88 k elements: 11 us after an element
// pass of 39 us; eight colour passes took 110 us).  Block partials of R.R for the norm,
// and with req given the active entries in equation order.
__global__ void __launch_bounds__(256) k_node_residual(long n3, const int* __restrict__ ptr,
                                                       const int* __restrict__ list, const double* __restrict__ fe,
                                                       const int* __restrict__ eqn, const double* __restrict__ fext,
                                                       double* __restrict__ R, double* __restrict__ req,
                                                       double* __restrict__ part)
{
    __shared__ double red[4];
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    double s = 0.0;
    if (t < n3) {
        const int a = (int)(t / 3), i = (int)(t - 3L * a);
        const int p0 = ptr[a], p1 = ptr[a + 1], eq = eqn[t];
        for (int p = p0; p < p1; p += 8) {
            double v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = p + k < p1 ? fe[3L * list[p + k] + i] : 0.0;
#pragma unroll
            for (int k = 0; k < 8; k++) s += v[k];
        }
        if (fext) s += fext[t];
        if (eq < 0) s = 0.0;
        R[t] = s;
        if (req && eq >= 0) req[eq] = s;
    }
    double v = s * s;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// ||R||^2 from the block partials and the status flag, into host memory
__global__ void __launch_bounds__(1024) k_fin_residual(const double* __restrict__ part, int n,
                                                       const int* __restrict__ status, double* __restrict__ out)
{
    __shared__ double red[16];
    double v = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) v += part[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < 16; w++) s += red[w];
        out[0] = s;
        out[1] = (double)*status;
    }
}

// ---- stiffness ----------------------------------------------------------------

constexpr int GR = 32;  // rows of a workgroup (half a slice), 8 lanes each

// Rows of half a slice: 8 lanes per row add the row's blocks of its elements,
// in list order, into LDS (a row's lanes are in one wave, so its sums need
// no barrier); then 32 consecutive lanes write one component of their rows'
// blocks: the operator block and its transpose in the partner's row, the MSR
// values, and 1/diag.  Prescribed dofs (src < 0) give zeros.
// BT: block buffer and sums, MT: MSR values, OT: operator.
// Bound by memory: the block buffer read once, every operator and MSR value
// written once.  67 k nodes FP64: 144 us for 0.43 GB (3.0 TB/s); with the
// element pass 168 us.  The colour passes with their clearing, expansion and
// 1/diag took 265 + 18 + 105 us there; 1.15 M nodes FP32: 1.94 + 1.56 ms
// against 2.30 + 1.05 ms, and the set-up's slot maps (4.7 ms) are gone.
template <class BT, class MT, class OT>
__global__ void __launch_bounds__(256) k_gather_rows(int nnd, int n_eq, int up_most, const int* __restrict__ sbase,
                                                     const int* __restrict__ swidth, const int* __restrict__ tpos,
                                                     const int* __restrict__ src, const int2* __restrict__ upper,
                                                     const int* __restrict__ ptr, const int* __restrict__ list,
                                                     const unsigned char* __restrict__ rslot,
                                                     const BT* __restrict__ eb, MT* __restrict__ val,
                                                     OT* __restrict__ out, double* __restrict__ dinv)
{
    extern __shared__ unsigned char lds_raw[];
    BT* acc = reinterpret_cast<BT*>(lds_raw);
    const int stride = 9 * up_most + 1;  // odd: consecutive rows fall into different banks
    const int s = blockIdx.x >> 1, h = blockIdx.x & 1;
    const int row0 = 64 * s + GR * h;
    if (blockIdx.x == 0 && threadIdx.x == 0) val[n_eq] = MT(0);  // the entry between diagonal and rows is no value
    {
        const int row = threadIdx.x >> 3, t = threadIdx.x & 7;
        const int a = row0 + row;
        if (a < nnd) {
            BT* my = acc + row * stride;
            const int nup9 = 9 * upper[a].y;
            for (int x = t; x < nup9; x += 8) my[x] = BT(0);
            // value x = t + 8 m of a run is component c of block j of it
            const int p1 = ptr[a + 1];
            for (int p = ptr[a]; p < p1; p += 2) {
                // two elements' loads in flight before their sums
                BT v[2][9];
                unsigned long long sl[2];
                int len[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const bool in = p + q < p1;
                    const int code = in ? list[p + q] : 0;
                    const int e = code >> 3, r = code & 7;
                    len[q] = in ? 9 * (8 - r) : 0;
                    sl[q] = reinterpret_cast<const unsigned long long*>(rslot)[code];
                    const BT* run = eb + 324L * e + 9 * pair_index(r, r);
#pragma unroll
                    for (int m = 0; m < 9; m++) v[q][m] = t + 8 * m < len[q] ? run[t + 8 * m] : BT(0);
                }
#pragma unroll
                for (int q = 0; q < 2; q++)
#pragma unroll
                    for (int m = 0; m < 9; m++)
                        if (t + 8 * m < len[q]) {
                            const int j = t >= m ? m : m - 1, c = t >= m ? t - m : t - m + 9;
                            my[9 * (int)((sl[q] >> (8 * j)) & 255) + c] += v[q][m];
                        }
                // (lanes of a row read sums other lanes wrote: the wave's LDS
                // operations stay in this order)
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    __syncthreads();
    const int row = threadIdx.x & 31, a = row0 + row, l = GR * h + row;
    const long b0 = sbase[s];
    const int w = swidth[s];
    const int2 up = a < nnd ? upper[a] : make_int2(0, 0);
    const BT* my = acc + row * stride;
    for (int k = threadIdx.x >> 5; k < w; k += 8) {
        const int kk = k - up.x;
        if (a < nnd && kk < 0) continue;  // a lower block: written by its partner's row
        const long o = (b0 + k) * 576 + l;
        if (a >= nnd || kk >= up.y) {
#pragma unroll
            for (int c = 0; c < 9; c++) out[o + 64 * c] = OT(0);
            continue;
        }
        const int lp = -tpos[(b0 + k) * 64 + l] - 2;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const int c = 3 * i + j;
                // a diagonal block holds its upper entries
                const BT x = my[9 * kk + (kk == 0 && j < i ? 3 * j + i : c)];
                const int sv = src[o + 64 * c];
                const BT v = sv >= 0 ? x : BT(0);
                out[o + 64 * c] = (OT)v;
                if (sv >= 0 && (kk > 0 || j >= i)) val[sv] = (MT)v;
                if (kk > 0) out[lp + 64 * (3 * j + i)] = (OT)v;
                if (kk == 0 && i == j) dinv[3L * a + i] = v != BT(0) ? 1.0 / (double)v : 0.0;
            }
    }
    // rows of nodes that no element uses
    if (a < nnd && up.y == 0 && threadIdx.x < GR)
#pragma unroll
        for (int i = 0; i < 3; i++) dinv[3L * a + i] = 0.0;
}

unsigned grid(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

// largest number of upper blocks of a row whose half slice fits in LDS with
// FP64 sums (64 KB): a row of a hexahedral grid has 14
constexpr int ROWS_UP_MOST = 27;

void rows_structure(tg_ctx* c)
{
    const int nnd = c->nnd, nel = c->nel;
    const Bsell& B = c->op;
    hipLaunchKernelGGL(k_sort_lists, dim3(grid(nnd, 256)), dim3(256), 0, c->stream, nnd, c->g_neptr.p, c->g_nelist.p);
    c->r_perm.alloc((size_t)nel);
    hipLaunchKernelGGL(k_ranks, dim3(grid(nel, 256)), dim3(256), 0, c->stream, nel, c->dconn.p, c->r_perm.p);
    c->r_upper.alloc((size_t)nnd);
    TG_HIP(hipMemsetAsync(c->g_flag.p, 0, sizeof(int), c->stream));
    hipLaunchKernelGGL(k_row_upper, dim3(grid(nnd, 256)), dim3(256), 0, c->stream, nnd, B.d_slice_base.p,
                       B.d_slice_width.p, B.d_col.p, c->r_upper.p, c->g_flag.p);
    TG_HIP(hipGetLastError());
    TG_HIP(hipMemcpyAsync(&c->r_up_most, c->g_flag.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    TG_HIP(hipStreamSynchronize(c->stream));
    c->r_slot.alloc(64 * (size_t)nel);
    hipLaunchKernelGGL(k_row_slots, dim3(grid(8L * nel, 256)), dim3(256), 0, c->stream, nel, c->dconn.p, c->r_perm.p,
                       B.d_slice_base.p, B.d_col.p, c->r_upper.p, c->r_slot.p);
    hipLaunchKernelGGL(k_upper_partners, dim3(grid(B.nblocks_padded, 256)), dim3(256), 0, c->stream, B.nblocks_padded,
                       B.d_tpos.p, B.d_tpos.p);
    TG_HIP(hipGetLastError());
    c->r_force.alloc(24 * (size_t)nel);
    c->dpart_r.alloc(grid(3L * nnd, 256));
}

void rows_buffers(tg_ctx* c)
{
    const size_t n = 324 * (size_t)c->nel;
    if (mixed_stiffness(c)) {
        if (c->r_blocks32.n != n) c->r_blocks32.alloc(n);
    } else if (c->r_blocks.n != n) {
        c->r_blocks.alloc(n);
    }
}

bool rows_assembly(const tg_ctx* c) { return !c->stiff_explicit && c->r_up_most <= ROWS_UP_MOST; }

void launch_node_residual(tg_ctx* c, double* R_node, double* R_eq)
{
    const long n3 = 3L * c->nnd;
    const unsigned nb = grid(n3, 256);
    hipLaunchKernelGGL(k_node_residual, dim3(nb), dim3(256), 0, c->stream, n3, c->g_neptr.p, c->g_nelist.p,
                       c->r_force.p, c->deqn.p, c->dfext.p, R_node, R_eq, c->dpart_r.p);
    TG_HIP(hipGetLastError());
}

void launch_residual_result(tg_ctx* c)
{
    hipLaunchKernelGGL(k_fin_residual, dim3(1), dim3(1024), 0, c->stream, c->dpart_r.p, (int)grid(3L * c->nnd, 256),
                       c->dstatus.p, c->hscal);
    TG_HIP(hipGetLastError());
}

void launch_gather_rows(tg_ctx* c)
{
    const Bsell& B = c->op;
    const unsigned g = 2u * (unsigned)B.nslices;
    const size_t row = (size_t)(9 * std::max(c->r_up_most, 1) + 1) * GR;
    const int most = std::max(c->r_up_most, 1);
    auto go = [&](auto kernel, size_t vb, const auto* eb, auto* val, auto* out) {
        hipLaunchKernelGGL(kernel, dim3(g), dim3(256), row * vb, c->stream, c->nnd, c->n_eq, most, B.d_slice_base.p,
                           B.d_slice_width.p, B.d_tpos.p, B.d_src.p, c->r_upper.p, c->g_neptr.p, c->g_nelist.p,
                           c->r_slot.p, eb, val, out, c->vdinv.p);
    };
    if (mixed_stiffness(c))
        go(k_gather_rows<float, float, float>, sizeof(float), c->r_blocks32.p, c->dval32.p, B.d_val32.p);
    else if (mixed_operator(c))
        go(k_gather_rows<double, double, float>, sizeof(double), c->r_blocks.p, c->dval.p, B.d_val32.p);
    else
        go(k_gather_rows<double, double, double>, sizeof(double), c->r_blocks.p, c->dval.p, B.d_val.p);
    TG_HIP(hipGetLastError());
}

}  // namespace tg
