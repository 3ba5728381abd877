// Structure of the equation system built on the device: the node graph
// (element lists per node, then each node's sorted unique neighbours), the
// solver operator's sliced layout and block columns, and the row pointers
// of the upper MSR pattern.  The reference builds the same structure on the
// host in FEManagerT::SetEquationSystem (tahoe/src/main/FEManagerT.cpp:
// 2248-2313) through GraphT::MakeGraph (toolbox/src/graph/GraphT.cpp:376-456)
// and MSRBuilderT::GenerateMSR (toolbox/src/graph/MSRBuilderT.cpp:134-181).
// Every output is a function of the mesh and the equation numbers alone
// (sorted lists, counts, prefix sums), so the atomics used to gather the
// element lists leave no trace in the results.
#include <hipcub/hipcub.hpp>

#include "tg_internal.h"

namespace tg {

namespace {

// ---- equation numbers ---------------------------------------------------------
// NodeManagerT::SetEquationNumbers (tahoe/src/nodes/NodeManagerT.cpp:712-760)
// -> FieldT::InitEquations/SetEquations (tahoe/src/nodes/FieldT.cpp:635-690):
// dofs with a kinematic card get none, the others 0.. in node-major, dof-minor
// order (the interface counts from 1).

__global__ void k_all_active(long n, int* __restrict__ eqn)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) eqn[k] = 1;
}

__global__ void k_prescribed(long n, const int* __restrict__ idx, int* __restrict__ eqn)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) eqn[idx[k]] = 0;
}

// eqn: 1 where active, sum: their inclusive sum; mask[a] = node a's active dofs
__global__ void k_numbers(int nnd, const int* __restrict__ sum, int* __restrict__ eqn, unsigned char* __restrict__ mask)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nnd) return;
    int m = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const bool act = eqn[3L * a + i] != 0;
        eqn[3L * a + i] = act ? sum[3L * a + i] - 1 : -1;
        m |= act << i;
    }
    mask[a] = (unsigned char)m;
}

// a few integers for the host, written straight into its memory
__global__ void k_to_host(const int* __restrict__ a, const int* __restrict__ b, const long long* __restrict__ l,
                          double* __restrict__ out)
{
    if (a) out[0] = (double)*a;
    if (b) out[1] = (double)*b;
    if (l) out[2] = (double)*l;
}

// ---- node graph ---------------------------------------------------------------

// incidence k of the connectivity (element k / 8, node conn[k]): count per
// node into cnt[node + 1]
__global__ void k_ne_count(long n8, const int* __restrict__ conn, int* __restrict__ cnt)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n8) atomicAdd(&cnt[conn[k] + 1], 1);
}

// incidence k into its node's list, as 8 element + the node's rank among the
// element's nodes (order within a list is arbitrary here: only sets are read
// from it until rows_structure sorts it)
__global__ void k_ne_fill(long n8, const int* __restrict__ conn, int* __restrict__ fill, int* __restrict__ list)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n8) return;
    const int a = conn[k];
    const int* c = conn + (k & ~7L);
    int r = 0;
#pragma unroll
    for (int b = 0; b < 8; b++) r += c[b] < a;
    list[atomicAdd(&fill[a], 1)] = (int)(k & ~7L) + r;
}

// candidate t of a node whose element list starts at p0: node t % 8 of the
// (t / 8)-th element
__device__ __forceinline__ int candidate(const int* conn, const int* list, int p0, int t)
{
    return conn[(long)(list[p0 + (t >> 3)] & ~7) + (t & 7)];
}

// The distinct values among one wave's n <= 64 K candidates (lane l of pass k
// holds candidate 64 k + l, lanes past the last one a value above every node):
// their number, and per held candidate whether it is its value's first
// occurrence (bit k of first) and how many distinct values lie below it.
template <int K>
__device__ __forceinline__ int distinct(int n, const int (&v)[K], int& first, int (&below)[K])
{
    const int lane = threadIdx.x & 63;
    unsigned long long rest[K];  // candidates whose value has not been taken
    int m = 0;
    first = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
        below[k] = 0;
        rest[k] = __ballot(64 * k + lane < n);
    }
#pragma unroll
    for (int k = 0; k < K; k++)
        while (rest[k]) {
            const int l = __ffsll(rest[k]) - 1;
            const int x = __builtin_amdgcn_readlane(v[k], l);
            m++;
            first |= (lane == l) << k;
#pragma unroll
            for (int q = 0; q < K; q++) {
                rest[q] &= ~(unsigned long long)__ballot(v[q] == x);
                below[q] += x < v[q];
            }
        }
    return m;
}

// FILL = false: deg[a] = the number of distinct candidates of node a (its
// neighbours, itself included).  FILL = true: those neighbours ascending
// into nlist[nptr[a] ..), each at the number of distinct candidates below it.
// One wave per node, its candidates in the lanes' registers.  More than 64
// elements on a node raise the flag.  Bound by the chain of a node's distinct
// values (27 inside a grid): 2,200 nodes 8 + 9 us, 1.09 M nodes 325 + 414 us.
// With a lane per node and its candidates in LDS they took 52 + 122 us (34
// waves, each with 64 x 64 dependent reads) and 427 + 1,142 us.
template <bool FILL>
__global__ void __launch_bounds__(256) k_neighbours(int nnd, const int* __restrict__ ne_ptr,
                                                   const int* __restrict__ list, const int* __restrict__ conn,
                                                   long long* __restrict__ deg, const long long* __restrict__ nptr,
                                                   int* __restrict__ nlist, int* __restrict__ flag)
{
    const int lane = threadIdx.x & 63;
    const int a = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (a >= nnd) return;
    const int p0 = ne_ptr[a], ne = ne_ptr[a + 1] - p0;
    if (ne > 64) {
        if (!FILL && lane == 0) {
            atomicOr(flag, 1);
            deg[a] = 0;
        }
        return;
    }
    auto node = [&](auto pass) {
        constexpr int K = decltype(pass)::value;
        const int n = 8 * ne;
        int v[K], below[K], first;
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = 64 * k + lane < n ? candidate(conn, list, p0, 64 * k + lane) : 0x7fffffff;
        const int m = distinct<K>(n, v, first, below);
        if (FILL) {
#pragma unroll
            for (int k = 0; k < K; k++)
                if ((first >> k) & 1) nlist[nptr[a] + below[k]] = v[k];
        } else if (lane == 0) {
            deg[a] = m;
        }
    };
    if (ne <= 8)
        node(std::integral_constant<int, 1>{});
    else
        node(std::integral_constant<int, 8>{});
}

// widest row of each slice of 64 nodes; one wave per slice
__global__ void __launch_bounds__(256) k_slice_width(int nnd, int nslices, const long long* __restrict__ deg,
                                                     int* __restrict__ swidth)
{
    const int s = blockIdx.x * 4 + (threadIdx.x >> 6), a = 64 * s + (threadIdx.x & 63);
    if (s >= nslices) return;
    int w = a < nnd ? (int)deg[a] : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) w = max(w, __shfl_xor(w, o));
    if ((threadIdx.x & 63) == 0) swidth[s] = w;
}

// block columns: row node a (slice s, lane l) lists its neighbours in its
// first deg[a] slots, -1 after them and in rows past the last node
__global__ void k_block_columns(int nnd, int nslices, const int* __restrict__ sbase, const int* __restrict__ swidth,
                                const long long* __restrict__ nptr, const int* __restrict__ nlist,
                                int* __restrict__ col)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = a >> 6, l = a & 63;
    if (s >= nslices) return;
    const long long o = a < nnd ? nptr[a] : 0;
    const int d = a < nnd ? (int)(nptr[a + 1] - o) : 0;
    for (int k = 0; k < swidth[s]; k++)
        col[((long)sbase[s] + k) * 64 + l] = k < d ? nlist[o + k] : -1;
}

// MSR row lengths (equation numbers grow with (node, dof)): row (a, i)
// holds the active dofs of a after i and every active dof of each
// neighbour b > a; a node that no element uses has no neighbours, itself
// included, and empty rows.  rl[0] = n_eq + 1 and rl[r + 1] = the length of row r,
// so that the inclusive sum of rl is bindx[0 .. n_eq].
__global__ void k_msr_rowlen(int nnd, int n_eq, const long long* __restrict__ nptr, const int* __restrict__ nlist,
                             const int* __restrict__ eqn, const unsigned char* __restrict__ mask,
                             long long* __restrict__ rl)
{
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a == 0) rl[0] = n_eq + 1;
    if (a >= nnd) return;
    if (nptr[a + 1] == nptr[a]) return;  // a node of no element couples nothing: empty rows
    int later = 0;
    for (long long k = nptr[a]; k < nptr[a + 1]; k++) {
        const int b = nlist[k];
        if (b > a) later += __popc(mask[b]);
    }
    for (int i = 0; i < 3; i++) {
        const int r = eqn[3L * a + i];
        if (r < 0) continue;
        int own = 0;
        for (int j = i + 1; j < 3; j++) own += eqn[3L * a + j] >= 0;
        rl[r + 1] = later + own;
    }
}

__global__ void k_narrow(long n, const long long* __restrict__ in, int* __restrict__ out)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = (int)in[k];
}

// MSR value ranges of the rows of each half slice (32 nodes): off-diagonal
// [bindx[r0], bindx[r1]) and diagonal [r0, r1) for the active rows r0 .. r1 - 1
// of its nodes (node-major equations: consecutive), (0, 0, 0, 0) without
// any; most[h] = the values the expansion stages for it.
__global__ void k_half_slice_ranges(int nnd, int nhalf, const int* __restrict__ eqn, const int* __restrict__ bindx,
                                    int4* __restrict__ rng, long long* __restrict__ most)
{
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= nhalf) return;
    int r0 = -1, r1 = -1;
    for (int a = 32 * h; a < 32 * h + 32 && a < nnd; a++)
        for (int i = 0; i < 3; i++) {
            const int e = eqn[3L * a + i];
            if (e < 0) continue;
            if (r0 < 0) r0 = e;
            r1 = e + 1;
        }
    if (r0 < 0) {
        rng[h] = make_int4(0, 0, 0, 0);
        most[h] = 0;
        return;
    }
    rng[h] = make_int4(bindx[r0], bindx[r1], r0, r1);
    most[h] = (long long)(bindx[r1] - bindx[r0]) + (r1 - r0);
}

unsigned grid(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// out[k] = in[0] + .. + in[k], k < n (temporary storage in c->g_scan)
template <class T>
void inclusive_sum(tg_ctx* c, const T* in, T* out, long n)
{
    size_t bytes = 0;
    TG_HIP(hipcub::DeviceScan::InclusiveSum(nullptr, bytes, in, out, (int)n, c->stream));
    if (c->g_scan.n < bytes) c->g_scan.alloc(bytes);
    TG_HIP(hipcub::DeviceScan::InclusiveSum(c->g_scan.p, bytes, in, out, (int)n, c->stream));
}

}  // namespace

// Equation numbers (deqn) and the nodes' masks of active dofs (g_mask) from
// the prescribed dofs' indices (dkbc_idx).
void launch_equation_numbers(tg_ctx* c, long nkbc)
{
    const long n3 = 3L * c->nnd;
    int* sum = reinterpret_cast<int*>(c->vwork.p);  // scratch until the first solve
    c->g_mask.alloc((size_t)c->nnd);
    hipLaunchKernelGGL(k_all_active, dim3(grid(n3, 256)), dim3(256), 0, c->stream, n3, c->deqn.p);
    if (nkbc > 0)
        hipLaunchKernelGGL(k_prescribed, dim3(grid(nkbc, 256)), dim3(256), 0, c->stream, nkbc, c->dkbc_idx.p,
                           c->deqn.p);
    inclusive_sum(c, c->deqn.p, sum, n3);
    hipLaunchKernelGGL(k_numbers, dim3(grid(c->nnd, 256)), dim3(256), 0, c->stream, c->nnd, sum, c->deqn.p,
                       c->g_mask.p);
    TG_HIP(hipGetLastError());
}

// the interface's equation numbers (from 1, prescribed -1), copied when they
// are first asked for
const std::vector<int>& host_eqnos(tg_ctx* c)
{
    if (!c->eqnos_ready) {
        c->eqnos.resize(3 * (size_t)c->nnd);
        TG_HIP(hipMemcpyAsync(c->eqnos.data(), c->deqn.p, sizeof(int) * c->eqnos.size(), hipMemcpyDeviceToHost,
                              c->stream));
        TG_HIP(hipStreamSynchronize(c->stream));
        for (int& e : c->eqnos) e = e >= 0 ? e + 1 : -1;
        c->eqnos_ready = true;
    }
    return c->eqnos;
}

// Node graph on the device: g_neptr/g_nelist (elements per node), g_deg and
// g_nptr/g_nlist (sorted unique neighbours per node); n_eq with the graph's
// size, in one read.
void device_node_graph(tg_ctx* c)
{
    const int nnd = c->nnd;
    const long n8 = 8L * c->nel;
    if (n8 > 0x7fffffffL) fail(TG_OUT_OF_RANGE, "connectivity exceeds 32-bit indexing");
    c->g_neptr.alloc((size_t)nnd + 1);
    c->g_nelist.alloc((size_t)n8);
    c->g_deg.alloc((size_t)nnd);
    c->g_nptr.alloc((size_t)nnd + 1);
    c->g_flag.alloc(1);
    c->g_fill.alloc((size_t)nnd + 1);
    TG_HIP(hipMemsetAsync(c->g_fill.p, 0, sizeof(int) * ((size_t)nnd + 1), c->stream));
    TG_HIP(hipMemsetAsync(c->g_flag.p, 0, sizeof(int), c->stream));
    // counts into fill[a + 1], their sums into neptr, then fill = the list starts
    hipLaunchKernelGGL(k_ne_count, dim3(grid(n8, 256)), dim3(256), 0, c->stream, n8, c->dconn.p, c->g_fill.p);
    inclusive_sum(c, c->g_fill.p, c->g_neptr.p, (long)nnd + 1);
    TG_HIP(hipMemcpyAsync(c->g_fill.p, c->g_neptr.p, sizeof(int) * nnd, hipMemcpyDeviceToDevice, c->stream));
    hipLaunchKernelGGL(k_ne_fill, dim3(grid(n8, 256)), dim3(256), 0, c->stream, n8, c->dconn.p, c->g_fill.p,
                       c->g_nelist.p);
    hipLaunchKernelGGL(k_neighbours<false>, dim3(grid(nnd, 4)), dim3(256), 0, c->stream, nnd, c->g_neptr.p,
                       c->g_nelist.p, c->dconn.p, c->g_deg.p, nullptr, nullptr, c->g_flag.p);
    // nptr[0] = 0, nptr[a + 1] = deg[0] + .. + deg[a]
    TG_HIP(hipMemsetAsync(c->g_nptr.p, 0, sizeof(long long), c->stream));
    inclusive_sum(c, c->g_deg.p, c->g_nptr.p + 1, (long)nnd);
    const int* last_sum = reinterpret_cast<const int*>(c->vwork.p) + (3L * nnd - 1);
    hipLaunchKernelGGL(k_to_host, dim3(1), dim3(1), 0, c->stream, last_sum, c->g_flag.p, c->g_nptr.p + nnd, c->hscal);
    TG_HIP(hipGetLastError());
    TG_HIP(hipStreamSynchronize(c->stream));
    c->n_eq = (int)c->hscal[0];
    if (c->hscal[1] != 0.0) fail(TG_OUT_OF_RANGE, "a node is shared by more than 64 elements");
    if (c->hscal[2] > 2147483647.0) fail(TG_OUT_OF_RANGE, "node graph exceeds 32-bit indexing");
    c->g_nlist.alloc((size_t)c->hscal[2]);
    hipLaunchKernelGGL(k_neighbours<true>, dim3(grid(nnd, 4)), dim3(256), 0, c->stream, nnd, c->g_neptr.p,
                       c->g_nelist.p, c->dconn.p, c->g_deg.p, c->g_nptr.p, c->g_nlist.p, c->g_flag.p);
    TG_HIP(hipGetLastError());
}

// The solver operator's layout (slice widths and bases, block columns, the
// blocks' partners) and the MSR row pointers from the device node graph.  The
// MSR columns follow when they are asked for (tg_get_msr_bindx), the
// expansion's maps when it first runs.  Allocates the MSR value arrays (their
// length is known only here).
void device_structure(tg_ctx* c)
{
    Bsell& B = c->op;
    const int nnd = c->nnd, n_eq = c->n_eq;
    B.nslices = (nnd + 63) / 64;
    B.d_slice_width.alloc(B.nslices);
    B.d_slice_base.alloc((size_t)B.nslices + 1);
    hipLaunchKernelGGL(k_slice_width, dim3(grid(B.nslices, 4)), dim3(256), 0, c->stream, nnd, B.nslices, c->g_deg.p,
                       B.d_slice_width.p);
    // (the widths' sum is at most the graph's size, which fits an int)
    TG_HIP(hipMemsetAsync(B.d_slice_base.p, 0, sizeof(int), c->stream));
    inclusive_sum(c, B.d_slice_width.p, B.d_slice_base.p + 1, (long)B.nslices);
    // MSR row pointers, summed in 64 bits
    c->g_rowlen.alloc((size_t)n_eq + 1);
    c->g_rows.alloc((size_t)n_eq + 1);
    TG_HIP(hipMemsetAsync(c->g_rowlen.p, 0, sizeof(long long) * ((size_t)n_eq + 1), c->stream));
    hipLaunchKernelGGL(k_msr_rowlen, dim3(grid(nnd, 256)), dim3(256), 0, c->stream, nnd, n_eq, c->g_nptr.p,
                       c->g_nlist.p, c->deqn.p, c->g_mask.p, c->g_rowlen.p);
    inclusive_sum(c, c->g_rowlen.p, c->g_rows.p, (long)n_eq + 1);
    hipLaunchKernelGGL(k_to_host, dim3(1), dim3(1), 0, c->stream, B.d_slice_base.p + B.nslices, nullptr,
                       c->g_rows.p + n_eq, c->hscal);
    TG_HIP(hipGetLastError());
    TG_HIP(hipStreamSynchronize(c->stream));
    B.nblocks_padded = (long)c->hscal[0] * 64;
    if (B.nblocks_padded * 9 > 0x7fffffffL) fail(TG_OUT_OF_RANGE, "block operator exceeds 32-bit indexing");
    if (c->hscal[2] > 2147483647.0) fail(TG_OUT_OF_RANGE, "MSR pattern exceeds 32-bit indexing");
    c->msr_len = (long)c->hscal[2];
    B.d_col.alloc((size_t)B.nblocks_padded);
    B.d_tpos.alloc((size_t)B.nblocks_padded);
    B.d_val.alloc((size_t)B.nblocks_padded * 9);
    c->dbindx.alloc((size_t)c->msr_len);
    c->dval.alloc((size_t)c->msr_len);
    c->dval32.alloc(mixed_stiffness(c) ? (size_t)c->msr_len : 0);
    hipLaunchKernelGGL(k_block_columns, dim3(grid(64L * B.nslices, 256)), dim3(256), 0, c->stream, nnd, B.nslices,
                       B.d_slice_base.p, B.d_slice_width.p, c->g_nptr.p, c->g_nlist.p, B.d_col.p);
    hipLaunchKernelGGL(k_narrow, dim3(grid((long)n_eq + 1, 256)), dim3(256), 0, c->stream, (long)n_eq + 1,
                       c->g_rows.p, c->dbindx.p);
    TG_HIP(hipGetLastError());
    launch_build_tpos(c);
    c->cols_ready = false;
    c->src_ready = false;
}

// What the expansion of the MSR values into the operator needs: the value map
// and the half slices' value ranges; built when it first runs on a mesh (the
// assembly by rows writes the operator itself).
void expansion_structure(tg_ctx* c)
{
    if (c->src_ready) return;
    Bsell& B = c->op;
    B.d_src.alloc((size_t)B.nblocks_padded * 9);
    launch_build_src(c);
    const int nhalf = 2 * B.nslices;
    B.d_srange.alloc((size_t)nhalf);
    c->g_most.alloc((size_t)nhalf);
    hipLaunchKernelGGL(k_half_slice_ranges, dim3(grid(nhalf, 256)), dim3(256), 0, c->stream, c->nnd, nhalf, c->deqn.p,
                       c->dbindx.p, B.d_srange.p, c->g_most.p);
    TG_HIP(hipGetLastError());
    std::vector<long long> most((size_t)nhalf);
    TG_HIP(hipMemcpyAsync(most.data(), c->g_most.p, sizeof(long long) * nhalf, hipMemcpyDeviceToHost, c->stream));
    TG_HIP(hipStreamSynchronize(c->stream));
    B.lds_values = most.empty() ? 0 : (long)*std::max_element(most.begin(), most.end());
    c->src_ready = true;
}

}  // namespace tg
