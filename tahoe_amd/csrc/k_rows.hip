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
// the row's upper slots, and their largest number over all rows; for each
// upper slot 8 x (active dofs of the row's neighbours between it and the
// diagonal) + mask of its node's active dofs: with the row's pointer, where
// the block's MSR values are (a slice's rows one after the other)
__global__ void k_row_upper(int nnd, const int* __restrict__ sbase, const int* __restrict__ swidth,
                            const int* __restrict__ bcol, const unsigned char* __restrict__ act,
                            int2* __restrict__ upper, unsigned short* __restrict__ runs, int* __restrict__ most)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    int lo = 0, n = 0;
    if (a < nnd) {
        const int s = a >> 6, l = a & 63;
        int run = 0;
        for (int k = 0; k < swidth[s]; k++) {
            const long at = ((long)sbase[s] + k) * 64 + l;
            const int c = bcol[at];
            if (c < 0) break;
            n++;
            lo += c < a;
            if (c < a) continue;
            const int mask = act[c];
            runs[64L * sbase[s] + (long)l * swidth[s] + k] = (unsigned short)(8 * run + mask);
            if (c > a) run += __popc(mask);
        }
        upper[a] = make_int2(lo, n - lo);
    }
    int m = n - lo;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) atomicMax(most, m);
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

__global__ void k_most_to_host(const int* __restrict__ most, double* __restrict__ out) { *out = (double)*most; }

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
constexpr int GQ = 2;   // elements whose loads are in flight

// What a wave's lanes have written to LDS is there for its other lanes, and
// nothing they read later is read before: an ordering for the compiler (one
// wave's LDS operations stay in order), no instruction of its own.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Rows of half a slice: 8 lanes per row add the row's blocks of its elements,
// in list order, into LDS, a block a lane (a row's lanes are in one wave, so
// its sums need no barrier), and write the row's MSR values and 1/diag; then
// 32 consecutive lanes write one component of their rows' blocks, the operator
// block and its transpose in the partner's row.  Prescribed dofs give zeros.
// BT: block buffer and sums, MT: MSR values, OT: operator.
// Bound by memory: the block buffer read once, every operator and MSR value
// written once.  67 k nodes FP64: 105 us for 0.37 GB (3.5 TB/s); with the
// element pass 224 us.  The colour passes with their clearing, expansion and
// 1/diag took 265 + 18 + 105 us there; 2.15 M nodes FP32: 2.13 + 2.35 ms.
// (With single values a lane and the expansion's map of 36 B a block read
// beside it the gather took 144 us and 3.25 ms.)
template <class BT, class MT, class OT>
__global__ void __launch_bounds__(256) k_gather_rows(int nnd, int n_eq, int up_most, const int* __restrict__ sbase,
                                                     const int* __restrict__ swidth, const int* __restrict__ tpos,
                                                     const int2* __restrict__ upper,
                                                     const unsigned short* __restrict__ runs,
                                                     const int* __restrict__ eqn, const int* __restrict__ bindx,
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
    const long b0 = sbase[s];
    const int w = swidth[s];
    if (blockIdx.x == 0 && threadIdx.x == 0) val[n_eq] = MT(0);  // the entry between diagonal and rows is no value
    {
        const int row = threadIdx.x >> 3, t = threadIdx.x & 7;
        const int a = row0 + row;
        if (a < nnd) {
            BT* my = acc + row * stride;
            const int2 up = upper[a];
            for (int x = t; x < 9 * up.y; x += 8) my[x] = BT(0);
            wave_lds_fence();
            // lane t takes block t of a run
            const int p1 = ptr[a + 1];
            for (int p = ptr[a]; p < p1; p += GQ) {
                // GQ elements' loads in flight before their sums
                BT v[GQ][9];
                int slot[GQ];
#pragma unroll
                for (int q = 0; q < GQ; q++) {
                    const int code = list[min(p + q, p1 - 1)];
                    const int e = code >> 3, r = code & 7;
                    const int j = min(t, 7 - r);
                    slot[q] = p + q < p1 && t == j ? rslot[8L * code + j] : -1;
                    const BT* blk = eb + 324L * e + 9 * (pair_index(r, r) + j);
#pragma unroll
                    for (int c = 0; c < 9; c++) v[q][c] = blk[c];
                }
#pragma unroll
                for (int q = 0; q < GQ; q++) {
                    if (slot[q] >= 0)
#pragma unroll
                        for (int c = 0; c < 9; c++) my[9 * slot[q] + c] += v[q][c];
                    wave_lds_fence();  // lanes of a row read sums that other lanes wrote
                }
            }
            // MSR values: row r[i] lists the node's own later dofs, then the
            // neighbours'.  What is no entry becomes zero for the operator.
            int r[3], first[3], own = 0;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                r[i] = eqn[3L * a + i];
                own |= (r[i] >= 0) << i;
            }
#pragma unroll
            for (int i = 0; i < 3; i++) first[i] = r[i] >= 0 ? bindx[r[i]] + __popc(own >> (i + 1)) : 0;
            const unsigned short* run = runs + 64 * b0 + (long)(GR * h + row) * w + up.x;
            for (int kk = t; kk < up.y; kk += 8) {
                const int rm = run[kk], mask = rm & 7;
                BT* x = my + 9 * kk;
                if (kk == 0) {
                    // a diagonal block holds its upper entries
#pragma unroll
                    for (int i = 0; i < 3; i++)
#pragma unroll
                        for (int j = i; j < 3; j++) {
                            const bool act = r[i] >= 0 && r[j] >= 0;
                            const BT y = act ? x[3 * i + j] : BT(0);
                            x[3 * i + j] = x[3 * j + i] = y;
                            if (act)
                                val[i == j ? r[i] : first[i] - __popc(own >> j)] = (MT)y;
                            if (i == j) dinv[3L * a + i] = y != BT(0) ? 1.0 / (double)y : 0.0;
                        }
                } else {
                    const int at = rm >> 3;
#pragma unroll
                    for (int i = 0; i < 3; i++)
#pragma unroll
                        for (int j = 0; j < 3; j++) {
                            if (r[i] >= 0 && ((mask >> j) & 1))
                                val[first[i] + at + __popc(mask & ((1 << j) - 1))] = (MT)x[3 * i + j];
                            else
                                x[3 * i + j] = BT(0);
                        }
                }
            }
            // rows of nodes that no element uses: an empty diagonal (nothing
            // clears the MSR values before this pass)
            if (up.y == 0 && t < 3) {
                const int e = eqn[3L * a + t];
                if (e >= 0) val[e] = MT(0);
                dinv[3L * a + t] = 0.0;
            }
        }
    }
    __syncthreads();
    const int row = threadIdx.x & 31, a = row0 + row, l = GR * h + row;
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
                const OT v = (OT)my[9 * kk + 3 * i + j];
                out[o + 64 * (3 * i + j)] = v;
                if (kk > 0) out[lp + 64 * (3 * j + i)] = v;
            }
    }
}

unsigned grid(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

// largest number of upper blocks of a row whose half slice fits in LDS with
// FP64 sums (64 KB): a row of a hexahedral grid has 14
constexpr int ROWS_UP_MOST = 27;

// (the caller waits for the stream before it reads the widest row, hscal[0])
void rows_structure(tg_ctx* c)
{
    const int nnd = c->nnd, nel = c->nel;
    const Bsell& B = c->op;
    hipLaunchKernelGGL(k_sort_lists, dim3(grid(nnd, 256)), dim3(256), 0, c->stream, nnd, c->g_neptr.p, c->g_nelist.p);
    c->r_perm.alloc((size_t)nel);
    hipLaunchKernelGGL(k_ranks, dim3(grid(nel, 256)), dim3(256), 0, c->stream, nel, c->dconn.p, c->r_perm.p);
    c->r_upper.alloc((size_t)nnd);
    c->r_run.alloc((size_t)B.nblocks_padded);
    TG_HIP(hipMemsetAsync(c->g_flag.p, 0, sizeof(int), c->stream));
    hipLaunchKernelGGL(k_row_upper, dim3(grid(nnd, 256)), dim3(256), 0, c->stream, nnd, B.d_slice_base.p,
                       B.d_slice_width.p, B.d_col.p, c->g_mask.p, c->r_upper.p, c->r_run.p, c->g_flag.p);
    c->r_slot.alloc(64 * (size_t)nel);
    hipLaunchKernelGGL(k_row_slots, dim3(grid(8L * nel, 256)), dim3(256), 0, c->stream, nel, c->dconn.p, c->r_perm.p,
                       B.d_slice_base.p, B.d_col.p, c->r_upper.p, c->r_slot.p);
    TG_HIP(hipGetLastError());
    // the widest row decides whether the rows are used: read with the rest
    hipLaunchKernelGGL(k_most_to_host, dim3(1), dim3(1), 0, c->stream, c->g_flag.p, c->hscal);
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
                           B.d_slice_width.p, B.d_tpos.p, c->r_upper.p, c->r_run.p, c->deqn.p, c->dbindx.p,
                           c->g_neptr.p, c->g_nelist.p,
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
