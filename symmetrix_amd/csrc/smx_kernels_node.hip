// Node-level kernels for gfx950: symmetric contraction, MFMA channel mixing,
// readout tail, integer list preparation and caller-side force reduction.
#include "smx_device.hpp"
#include "smx_kernels.hpp"
#include "smx_host_model.hpp"

#include <algorithm>

namespace smx {

// ===========================================================================
// Integer list preparation
namespace {

constexpr int SCAN_BLOCK = 1024;

// exclusive scan of one 1024-element tile held by a 1024-thread block
__device__ int block_scan_exclusive(int v, int* total)
{
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(incl, off, 64);
        if (lane >= off) incl += t;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    if (w == 0) {
        int s = lane < 16 ? wsum[lane] : 0;
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const int t = __shfl_up(s, off, 64);
            if (lane >= off) s += t;
        }
        if (lane < 16) wsum[lane] = s;
    }
    __syncthreads();
    const int base = w ? wsum[w - 1] : 0;
    *total = wsum[15];
    __syncthreads();
    return base + incl - v;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_tiles(const int* in, int* out, int n, int* block_sums)
{
    const int i = blockIdx.x * SCAN_BLOCK + threadIdx.x;
    const int v = i < n ? in[i] : 0;
    int total;
    const int ex = block_scan_exclusive(v, &total);
    if (i < n) out[i] = ex;
    if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}
// scan of the per-tile sums (up to 1024 tiles per pass, looped) and write of out[n]
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_sums(int* block_sums, int nb, int* out, int n)
{
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += SCAN_BLOCK) {
        const int i = b0 + threadIdx.x;
        const int v = i < nb ? block_sums[i] : 0;
        int total;
        const int ex = block_scan_exclusive(v, &total);
        if (i < nb) block_sums[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) out[n] = carry;
}
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_add(int* out, int n, const int* block_sums)
{
    const int i = blockIdx.x * SCAN_BLOCK + threadIdx.x;
    if (i < n) out[i] += block_sums[blockIdx.x];
}

// Histogram of the keys, and the place that every entry took inside its bucket (whatever order the atomics leave: readers
// order the bucket by entry).  Keys outside [0, rows) are left out and raise bit 1 of *flag (if not null).
__global__ void k_count_ranked(const int* key, long n, int rows, int* count, int* rank, int* flag)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const int j = key[i];
        if (j >= 0 && j < rows) rank[i] = atomicAdd(&count[j], 1);
        else if (flag) atomicOr(flag, 1);
    }
}
// Placement of entries that know their place inside the bucket: no atomics.  The counters are dead by now: they are cleared
// here, so that the next list build finds them at zero without a launch of its own.
// With a guard (arrays that no host code has looked at): when the checks of this evaluation raised its status word, the CSR
// offsets, the sender lists and the species groups are set to "no edges, no nodes", so that no later kernel of the
// evaluation uses an unchecked integer as an address; the status goes into the sticky word the host reads at its next
// synchronising call and, raised or not, into the word the later kernels read.
__global__ void k_place_ranked(const int* key, const int* rank, long n, int rows, int* start, int* list, int* count,
                               InputGuard g)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < rows) count[i] = 0;
    if (g.status) {
        const int st = *g.status;
        if (i == 0) {
            *g.live = st;
            if (st) *g.sticky |= st;   // one thread of one launch on the stream: no other writer
        }
        if (st) {
            if (i < g.n_first) g.first_neigh[i] = 0;
            if (i < g.n_tstart) g.tstart[i] = 0;
            if (i <= rows) start[i] = 0;
            return;
        }
    }
    if (i < n) {
        const int j = key[i];
        if (j >= 0 && j < rows) list[start[j] + rank[i]] = (int)i;
    }
}
// Ascending order inside every bucket, in memory: for readers that take a window of the edges (the others order a bucket in
// LDS as they read it).  One wavefront per bucket.
constexpr int SORT_LDS = 1024;
__global__ __launch_bounds__(64) void k_sort_buckets(const int* start, int rows, int* list, int* spare)
{
    __shared__ __align__(16) int buf[SORT_LDS];
    const int j = blockIdx.x;
    const int s0 = start[j], n = start[j + 1] - s0;
    if (n <= 1) return;
    const int* sorted = wave_sorted_bucket<SORT_LDS>(list, s0, n, buf, threadIdx.x, spare);
    if (sorted == buf)
        for (int t = threadIdx.x; t < n; t += 64) list[s0 + t] = sorted[t];
}
// One block scans an array, or picks a species out of it, 16 consecutive elements per thread at a time: bound by the latency of a
// load and of the block's scan per round, so that a round takes as many as there are registers for.
// Up to 1 024 elements one per thread: 24 to 501 atoms, the launch of the node lists 9.0, 11.2 and 8.1 us against 10.4, 12.5 and 10.6.
constexpr int SCAN_ITEMS = 16;
template <int ITEMS>
__device__ __forceinline__ void load_items(const int* in, int n, int i0, int beyond, int (&v)[ITEMS])
{
    if (i0 + ITEMS <= n) {
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) v[q] = in[i0 + q];
    } else {
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) {
            const int x = in[min(i0 + q, n - 1)];      // (no branches: all loads go out together)
            v[q] = i0 + q < n ? x : beyond;
        }
    }
}
// species group t of a block of its own: where it begins (the number of atoms of smaller species), and its atoms in ascending
// order.  (One block with counters in the LDS for all species took a serial chain of same-address atomics, two per atom.)
// N > 0: without an element there is no round that fills v.
template <int ITEMS>
__device__ void type_group_items(const int* node_types, int N, int T, int t, int* tstart, int* perm)
{
    int before = 0, v[ITEMS];
    for (int b0 = 0; b0 < N; b0 += SCAN_BLOCK * ITEMS) {
        load_items(node_types, N, b0 + (int)threadIdx.x * ITEMS, -1, v);
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) before += v[q] >= 0 && v[q] < t;
    }
    int place;
    if (N <= SCAN_BLOCK * ITEMS) {
        // one round holds all atoms, and one scan both sums, 16 bits each
        int mine = 0, total;
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) mine += v[q] == t;
        int to = block_scan_exclusive(before << 16 | mine, &total) & 0xffff;
        place = total >> 16;
        to += place;
#pragma unroll
        for (int q = 0; q < ITEMS; ++q)
            if (v[q] == t) perm[to++] = (int)threadIdx.x * ITEMS + q;
        if (threadIdx.x == 0) {
            tstart[t] = place;
            if (t == T - 1) tstart[T] = place + (total & 0xffff);
        }
        return;
    }
    block_scan_exclusive(before, &place);
    if (threadIdx.x == 0) tstart[t] = place;
    for (int b0 = 0; b0 < N; b0 += SCAN_BLOCK * ITEMS) {
        const int i0 = b0 + (int)threadIdx.x * ITEMS;
        load_items(node_types, N, i0, -1, v);
        int mine = 0, total;
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) mine += v[q] == t;
        int to = place + block_scan_exclusive(mine, &total);
#pragma unroll
        for (int q = 0; q < ITEMS; ++q)
            if (v[q] == t) perm[to++] = i0 + q;
        place += total;
    }
    if (t == T - 1 && threadIdx.x == 0) tstart[T] = place;
}
__device__ __forceinline__ void type_group_body(const int* node_types, int N, int T, int t, int* tstart, int* perm)
{
    if (N <= SCAN_BLOCK) type_group_items<1>(node_types, N, T, t, tstart, perm);
    else type_group_items<SCAN_ITEMS>(node_types, N, T, t, tstart, perm);
}
__global__ __launch_bounds__(SCAN_BLOCK) void k_type_groups(const int* node_types, int N, int T, int* tstart, int* perm)
{
    type_group_body(node_types, N, T, blockIdx.x, tstart, perm);
}
__global__ void k_check_range(const int* v, long n, int limit, int* flags)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && (v[i] < 0 || v[i] >= limit)) atomicOr(flags, 1);
}
__global__ void k_check_r(const double* r, long n, double r_cut, int* flags)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !(r[i] > 0.0 && r[i] < r_cut)) atomicOr(flags, 2);
}
template <typename T>
__global__ void k_fill(T* p, long n, T v)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
template <typename TS, typename TD>
__global__ void k_convert(const TS* s, TD* d, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = (TD)s[i];
}
inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// whole scan in one block (tiles visited in order with a running carry): one launch
// instead of three while the array is short
template <int ITEMS>
__device__ void scan_single_items(const int* in, int* out, int n)
{
    int carry = 0, v[ITEMS];
    for (int b0 = 0; b0 < n; b0 += SCAN_BLOCK * ITEMS) {
        const int i0 = b0 + (int)threadIdx.x * ITEMS;
        load_items(in, n, i0, 0, v);
        int sum = 0, total;
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) { const int x = v[q]; v[q] = sum; sum += x; }
        const int ex = carry + block_scan_exclusive(sum, &total);
        if (i0 + ITEMS <= n) {
#pragma unroll
            for (int q = 0; q < ITEMS; ++q) out[i0 + q] = ex + v[q];
        } else {
#pragma unroll
            for (int q = 0; q < ITEMS; ++q)
                if (i0 + q < n) out[i0 + q] = ex + v[q];
        }
        carry += total;
    }
    if (threadIdx.x == 0) out[n] = carry;
}
__device__ __forceinline__ void scan_single_body(const int* in, int* out, int n)
{
    if (n <= SCAN_BLOCK) scan_single_items<1>(in, out, n); else scan_single_items<SCAN_ITEMS>(in, out, n);
}
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_single(const int* in, int* out, int n)
{
    scan_single_body(in, out, n);
}
__device__ void node_lists_part(const int* num_neigh, int N, int* first_neigh, const int* node_types, int T,
                                int* tstart, int* perm, const int* key, long n, int rows, int* count, int* rank,
                                const InputChecks& chk)
{
    // the node lists do not depend on each other: a block for the scan, and one for every species
    if (blockIdx.x == 0) {
        scan_single_body(num_neigh, first_neigh, N);
        __syncthreads();   // first_neigh, written by this block, is read back below
        if (chk.status && threadIdx.x == 0 && ((first_neigh[N] != (int)chk.num_edges) | (first_neigh[chk.num_local_nodes] != (int)n)))
            atomicOr(chk.status, 1);
        return;
    }
    if ((int)blockIdx.x <= T) { type_group_body(node_types, N, T, (int)blockIdx.x - 1, tstart, perm); return; }
    const long first = (long)(blockIdx.x - 1 - T) * SCAN_BLOCK + threadIdx.x, step = (long)(gridDim.x - 1 - T) * SCAN_BLOCK;
    for (long i = first; i < n; i += step) {
        const int j = key[i];
        if (j >= 0 && j < rows) rank[i] = atomicAdd(&count[j], 1);   // the entry's place inside its bucket
        else if (chk.status) atomicOr(chk.status, 1);
    }
    if (chk.status) {
        int bad = 0;
        for (long i = first; i < N; i += step) bad |= (num_neigh[i] < 0) | (node_types[i] < 0) | (node_types[i] >= T);
        // species and length of every edge (layer 0 covers the edges of ghost receivers as well)
        for (long i = first; i < chk.num_edges; i += step) {
            const int t = chk.neigh_types[i];
            const double rr = chk.r[i];
            bad |= (t < 0 || t >= T) ? 1 : 0;
            bad |= (rr > 0.0 && rr < chk.r_cut) ? 0 : 2;
        }
        if (bad) atomicOr(chk.status, bad);
    }
}
// The node-level lists of one evaluation and its sender histogram in one launch: blocks 0 to T form the node lists
// (first_neigh = exclusive scan of num_neigh, the species groups), the other blocks count the
// senders (counters at zero on entry), which does not depend on the node lists.  With a ticket, the block that finishes last
// turns the histogram into the sender offsets: a launch of its own costs 6 to 8 us of a small evaluation, but the fences of
// the ticket cost more than that over many blocks (83 blocks, 3 000 atoms: 21 us with the ticket, 19 without; 80 us over 2 048),
// so the launcher hands out tickets to small grids only.  Larger ones are bound by the atomics (50 000 atoms, 3.9 million
// edges: 92 us while one block each formed the node lists an element per thread at a time, now 60, the scan behind it 43 and
// 14; 20 011 atoms 41 and 19, now 26 and 7).
// With `chk.status` set the launch also checks everything the later kernels use as an address or a table argument
// (species, sender rows, edge lengths, counts that add up to the edge totals) and raises bits in the status word.
__global__ __launch_bounds__(SCAN_BLOCK) void k_node_lists_count(const int* num_neigh, int N, int* first_neigh,
                                                                const int* node_types, int T, int* tstart, int* perm,
                                                                const int* key, long n, int rows, int* count, int* rank,
                                                                int* sstart, int* ticket, InputChecks chk)
{
    node_lists_part(num_neigh, N, first_neigh, node_types, T, tstart, perm, key, n, rows, count, rank, chk);
    if (!ticket) return;
    // every block's counts are out before it takes its ticket
    __shared__ int last;
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        last = atomicAdd(ticket, 1) == (int)gridDim.x - 1;
        __threadfence();
    }
    __syncthreads();
    if (!last) return;
    scan_single_body(count, sstart, rows);
    if (threadIdx.x == 0) *ticket = 0;
}
// the same checks as separate work for lists too long for the single-block scan
__global__ void k_check_counts(const int* num_neigh, int N, const int* first_neigh, int num_local_nodes, long num_edges,
                               long num_local_edges, int* status)
{
    int bad = 0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) bad |= num_neigh[i] < 0;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        bad |= (first_neigh[N] != (int)num_edges) | (first_neigh[num_local_nodes] != (int)num_local_edges);
    if (bad) atomicOr(status, 1);
}
}  // namespace

hipError_t launch_node_lists_count(const int* num_neigh, int N, int* first_neigh, const int* node_types, int T,
                                   int* tstart, int* perm, const int* key, long n, int rows, int* count, int* rank,
                                   int* sstart, int* ticket, const InputChecks& chk, hipStream_t s)
{
    if (N <= 0 || N > 64 * SCAN_BLOCK || T <= 0) return hipErrorInvalidValue;
    const long work = chk.status ? std::max(n, chk.num_edges) : n;
    const unsigned counting = (unsigned)std::max<long>(1, std::min<long>((work + SCAN_BLOCK - 1) / SCAN_BLOCK, 2048));
    const bool with_scan = counting <= 48;
    hipLaunchKernelGGL(k_node_lists_count, dim3(1 + T + counting), dim3(SCAN_BLOCK), 0, s, num_neigh, N, first_neigh,
                       node_types, T, tstart, perm, key, n, rows, count, rank, sstart, with_scan ? ticket : nullptr, chk);
    if (!with_scan) hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(SCAN_BLOCK), 0, s, count, sstart, rows);
    return hipGetLastError();
}
hipError_t launch_check_counts(const int* num_neigh, int N, const int* first_neigh, int num_local_nodes, long num_edges,
                               long num_local_edges, int* status, hipStream_t s)
{
    if (N > 0)
        hipLaunchKernelGGL(k_check_counts, dim3(std::min<unsigned>(nblk(N, 256), 1024u)), dim3(256), 0, s, num_neigh, N,
                           first_neigh, num_local_nodes, num_edges, num_local_edges, status);
    return hipGetLastError();
}

hipError_t launch_scan_exclusive(const int* in, int* out, int n, int* block_sums, hipStream_t s)
{
    if (n <= 64 * SCAN_BLOCK) {
        hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(SCAN_BLOCK), 0, s, in, out, n);
        return hipGetLastError();
    }
    const int nb = (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
    hipLaunchKernelGGL(k_scan_tiles, dim3(nb), dim3(SCAN_BLOCK), 0, s, in, out, n, block_sums);
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_BLOCK), 0, s, block_sums, nb, out, n);
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(SCAN_BLOCK), 0, s, out, n, block_sums);
    return hipGetLastError();
}

hipError_t launch_sender_lists(const int* gather, long E, int rows, int* count, int* rank, int* sstart, int* slist,
                               int* block_sums, bool counted, int* range_flag, hipStream_t s, const InputGuard& guard)
{
    if (rows <= 0) return hipSuccess;
    if (!counted) {
        if (E > 0) hipLaunchKernelGGL(k_count_ranked, dim3(nblk(E, 256)), dim3(256), 0, s, gather, E, rows, count, rank, range_flag);
        hipError_t err = launch_scan_exclusive(count, sstart, rows, block_sums, s);
        if (err != hipSuccess) return err;
    }
    // (the counters and the guard's bookkeeping ride on this launch, so it also runs for an empty edge list)
    const long threads = std::max<long>({E, (long)rows + 1, (long)guard.n_first, (long)guard.n_tstart});
    hipLaunchKernelGGL(k_place_ranked, dim3(nblk(threads, 256)), dim3(256), 0, s, gather, rank, E, rows, sstart, slist, count, guard);
    return hipGetLastError();
}
hipError_t launch_sort_buckets(const int* start, int rows, int* list, int* spare, hipStream_t s)
{
    if (rows > 0) hipLaunchKernelGGL(k_sort_buckets, dim3(rows), dim3(64), 0, s, start, rows, list, spare);
    return hipGetLastError();
}

hipError_t launch_type_groups(const int* node_types, int N, int T, int* tcount, int* tstart, int* cursor,
                              int* perm, int* block_sums, hipStream_t s)
{
    (void)tcount; (void)cursor; (void)block_sums;
    if (T <= 0) return hipSuccess;
    if (N <= 0) return launch_fill<int>(tstart, (long)T + 1, 0, s);   // empty groups: the kernel needs an element to load
    hipLaunchKernelGGL(k_type_groups, dim3(T), dim3(SCAN_BLOCK), 0, s, node_types, N, T, tstart, perm);
    return hipGetLastError();
}

hipError_t launch_check_range(const int* v, long n, int limit, int* flags, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_check_range, dim3(nblk(n, 256)), dim3(256), 0, s, v, n, limit, flags);
    return hipGetLastError();
}
hipError_t launch_check_r(const double* r, long n, double r_cut, int* flags, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_check_r, dim3(nblk(n, 256)), dim3(256), 0, s, r, n, r_cut, flags);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_fill(T* p, long n, T v, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_fill<T>, dim3(nblk(n, 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}
template hipError_t launch_fill<double>(double*, long, double, hipStream_t);
template hipError_t launch_fill<float>(float*, long, float, hipStream_t);
template hipError_t launch_fill<int>(int*, long, int, hipStream_t);
template <typename TS, typename TD>
hipError_t launch_convert(const TS* src, TD* dst, long n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL((k_convert<TS, TD>), dim3(nblk(n, 256)), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}
template hipError_t launch_convert<double, float>(const double*, float*, long, hipStream_t);
template hipError_t launch_convert<float, double>(const float*, double*, long, hipStream_t);
template hipError_t launch_convert<double, double>(const double*, double*, long, hipStream_t);
template hipError_t launch_convert<float, float>(const float*, float*, long, hipStream_t);

// ===========================================================================
// Symmetric contraction.  Atoms are grouped by species (list preparation); a
// thread owns one channel of two atoms of the same species, so every coefficient
// it loads (coalesced over channels, [species][monomial][K]) serves two
// evaluations.  The monomial indices come from the model file: the same for
// every lane, but not compile-time, so the 16 variables of each atom live in an
// LDS column ([17][block], slot 16 = the constant 1) that is only ever read in
// the loops.  The polynomial is walked once per variable v: the entries of list
// v give dP/dx_v = sum w x_fa x_fb in a register, written straight to M_grad;
// the monomials that start with v come first in the list, and
// P = sum_v x_v * (their partial sum).
namespace {
constexpr int POLY_BLOCK = 128;
// Atoms per thread: as many as fill one 16-byte LDS word, so that one ds_read_b128 brings a variable of
// all of them and every loaded coefficient serves them all.  (Twice as many was measured slower: fewer
// blocks than the chip holds at once.)
template <typename F> constexpr int poly_nb() { return 16 / (int)sizeof(F); }
typedef int __attribute__((address_space(4))) ConstInt;
template <typename F, int N>
struct alignas(16) PolyVec {
    F v[N];
};

// POLY_VG groups of POLY_BLOCK threads share the variables of a block in LDS; group g walks the lists of
// the variables v = g, g + POLY_VG, ...  A block is latency bound (every list entry needs a coefficient
// from L2), so spreading the 16 lists of an atom group over four times as many wavefronts shortens the
// kernel by nearly that factor.
constexpr int POLY_VG = POLY_GROUPS;
static_assert(16 % POLY_VG == 0 && POLY_BLOCK % 64 == 0 && POLY_SPARE_CHUNKS >= 2, "list layout and the kernel's walk must agree");

// Threads of a block: POLY_VG variable groups of PB threads each; thread `tid` of a group owns channel tid % CB of
// atom group tid / CB (AG atom groups of poly_nb atoms per block, PB = AG * CB rounded up to whole wavefronts).
// With K = 96 two atom groups fill three wavefronts exactly, where one group alone would leave a third of two
// wavefronts without a channel.
struct PolyShape {
    int CB, AG, PB;   // channels per block, atom groups per block, threads per variable group
};
static PolyShape poly_shape(int K, long atom_groups)
{
    PolyShape sh;
    sh.CB = K <= POLY_BLOCK ? K : POLY_BLOCK;
    sh.AG = 1;
    double best = 1e30;   // idle lanes per used lane; ties keep the smaller block
    for (int a = 1; a <= 4; a *= 2) {
        const int used = a * sh.CB, pb = (used + 63) / 64 * 64;
        if (a > 1 && pb > 192) break;
        if (a > 1 && atom_groups / a < 2 * 256) break;   // fewer than two blocks per CU: the lanes gained do not pay
        const double waste = (double)(pb - used) / used;
        if (waste < best - 1e-12) { best = waste; sh.AG = a; }
    }
    sh.PB = (sh.AG * sh.CB + 63) / 64 * 64;
    return sh;
}

template <typename F, int PB>
__global__ __launch_bounds__(PB * POLY_VG) void k_poly(const PolyParams<F> a, const PolyShape sh)
{
    constexpr int NB = poly_nb<F>();
    extern __shared__ __align__(16) unsigned char poly_smem[];
    PolyVec<F, NB>* Xs = reinterpret_cast<PolyVec<F, NB>*>(poly_smem);          // [17][PB]
    PolyVec<F, NB>* fsum = Xs + 17 * PB;                                         // [POLY_VG][PB]
    auto X = [&](int q) { return Xs + q * PB; };
    // the group index is the same for a whole wavefront: as a scalar it keeps the walk through the lists
    // (indices, chunk counts, coefficient rows) in scalar registers and scalar loads
    const int tid = threadIdx.x % PB, vg = __builtin_amdgcn_readfirstlane(threadIdx.x / PB);
    const int ag = tid / sh.CB, kloc = tid - ag * sh.CB;
    const bool tlive = ag < sh.AG;
    constexpr int VPG = 16 / POLY_VG;   // variables per group
    // species segment and atom groups of this block row
    const int kblocks = (a.K + sh.CB - 1) / sh.CB;
    int type = -1, sg = blockIdx.x / kblocks, seg0 = 0, seg_n = 0;
    for (int t = 0; t < a.T; ++t) {
        const int n_t = a.tstart[t + 1] - a.tstart[t];
        const int sgroups = ((n_t + NB - 1) / NB + sh.AG - 1) / sh.AG;
        if (sg < sgroups) { type = t; seg0 = a.tstart[t]; seg_n = n_t; break; }
        sg -= sgroups;
    }
    if (type < 0) return;
    const int grp = sg * sh.AG + (tlive ? ag : 0);
    const int k = (blockIdx.x % kblocks) * sh.CB + kloc;
    const bool klive = tlive && k < a.K;
    const unsigned kk = klive ? k : a.K - 1;
    int node[NB];
    bool nlive[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int j = grp * NB + b;
        nlive[b] = tlive && j < seg_n;
        node[b] = a.perm[seg0 + (j < seg_n ? j : seg_n - 1)];
    }
    for (int q = vg; q < 17; q += POLY_VG) {
        PolyVec<F, NB> x;
#pragma unroll
        for (int b = 0; b < NB; ++b) x.v[b] = q < 16 ? a.A[((size_t)node[b] * 16 + q) * a.K + kk] : F(1);
        X(q)[tid] = x;
    }
    __syncthreads();
    for (int pl = 0; pl < a.NP; ++pl) {
        // the lists are read-only model data, the same for every lane: through the constant address space
        // they are fetched by scalar loads
        const ConstInt* pki = (const ConstInt*)a.packed[pl];
        auto pk = [&](int ch) { return make_int4(pki[4 * ch], pki[4 * ch + 1], pki[4 * ch + 2], pki[4 * ch + 3]); };
        const ConstInt* nch = (const ConstInt*)a.chunks[pl];
        // scalar base in the global address space; the lane adds kk
        typedef const F __attribute__((address_space(1))) GlobalF;
        GlobalF* coef = (GlobalF*)a.coef[pl] + (size_t)type * (a.num_entries[pl] + 1) * a.K;
        F f[NB], g[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) f[b] = g[b] = F(0);
        // this group's chunks are contiguous and start at c
        int c = 0;
        for (int q = 0; q < 2 * VPG * vg; ++q) c += nch[q];
        auto weights = [&](const int4& e, F (&w)[4]) {
            const int e4[4] = {e.x, e.y, e.z, e.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) w[q] = (coef + (size_t)(e4[q] & 0xffff) * a.K)[kk];
        };
        // indices two chunks ahead and coefficients one chunk ahead of the arithmetic, across the variables
        // of the group; the list ends with spare chunks of padding entries, so nothing here depends on where
        // the group's range stops
        int4 cur = pk(c), nxt = pk(c + 1);
        F w[4];
        weights(cur, w);
        // The gradients of the group's variables stay in registers until all lists are walked: a store between
        // the lists would sit in front of the next coefficient loads, whose wait would then wait for it too.
        F gs[VPG][NB];
#pragma unroll
        for (int t = 0; t < VPG; ++t) {
            const int v = vg + POLY_VG * t;
            const int n0 = nch[2 * (VPG * vg + t)], n1 = nch[2 * (VPG * vg + t) + 1];
#pragma unroll
            for (int b = 0; b < NB; ++b) g[b] = F(0);
            for (int i = 0; i < n0 + n1; ++i, ++c) {
                F wn[4];
                weights(nxt, wn);
                const int4 nn = pk(c + 2);
                const int e4[4] = {cur.x, cur.y, cur.z, cur.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int ia = (e4[q] >> 16) & 0xff, ib = (e4[q] >> 24) & 0xff;
                    const PolyVec<F, NB> xa = X(ia)[tid], xb = X(ib)[tid];
#pragma unroll
                    for (int b = 0; b < NB; ++b) g[b] += w[q] * (xa.v[b] * xb.v[b]);
                }
                cur = nxt; nxt = nn;
#pragma unroll
                for (int q = 0; q < 4; ++q) w[q] = wn[q];
                if (i + 1 == n0) {
                    // the monomials that start with v are done: their sum times x_v is v's share of P
                    const PolyVec<F, NB> xv = X(v)[tid];
#pragma unroll
                    for (int b = 0; b < NB; ++b) f[b] += xv.v[b] * g[b];
                }
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) gs[t][b] = g[b];
        }
#pragma unroll
        for (int t = 0; t < VPG; ++t)
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (klive && nlive[b])
                    a.M_grad[(((size_t)node[b] * a.NP + pl) * 16 + vg + POLY_VG * t) * a.K + k] = gs[t][b];
        // P = sum of the groups' shares, added in group order
        {
            PolyVec<F, NB> fv;
#pragma unroll
            for (int b = 0; b < NB; ++b) fv.v[b] = f[b];
            fsum[vg * PB + tid] = fv;
        }
        __syncthreads();
        if (vg == 0) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                F t = F(0);
#pragma unroll
                for (int g2 = 0; g2 < POLY_VG; ++g2) t += fsum[g2 * PB + tid].v[b];
                if (klive && nlive[b]) a.M[((size_t)node[b] * a.NP + pl) * a.K + k] = t;
            }
        }
        __syncthreads();
    }
}


template <typename F, int V>
struct alignas(sizeof(F) * V > 16 ? 16 : sizeof(F) * V) RevVec {
    F v[V];
};
// four consecutive channels per thread when K allows 16/32-byte accesses (V = 4), else one
template <typename F, int V>
__global__ void k_poly_reverse(long total_v, int NP, int K, const F* M_grad, const F* M_adj, F* A_adj)
{
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;  // over [N][16][K / V]
    if (idx >= total_v) return;
    const int KV = K / V;
    const int kq = (int)(idx % KV) * V;
    const long t = idx / KV;
    const int lm = (int)(t % 16);
    const long i = t / 16;
    RevVec<F, V> s;
#pragma unroll
    for (int j = 0; j < V; ++j) s.v[j] = F(0);
    for (int p = 0; p < NP; ++p) {
        const RevVec<F, V> g = *reinterpret_cast<const RevVec<F, V>*>(M_grad + ((i * NP + p) * 16 + lm) * K + kq);
        const RevVec<F, V> m = *reinterpret_cast<const RevVec<F, V>*>(M_adj + (i * NP + p) * K + kq);
#pragma unroll
        for (int j = 0; j < V; ++j) s.v[j] += g.v[j] * m.v[j];
    }
    *reinterpret_cast<RevVec<F, V>*>(A_adj + (i * 16 + lm) * K + kq) = s;
}
}  // namespace

template <typename F>
hipError_t launch_poly(const PolyParams<F>& p, hipStream_t s)
{
    if (p.num_nodes <= 0) return hipSuccess;
    if (p.table_slabs) return launch_poly_spec<F>(p, s);   // standard product basis (smx_kernels_poly.hip)
    if (p.mode != 0) return hipErrorInvalidValue;   // the general kernel has the one mode
    const PolyShape sh = poly_shape(p.K, (p.num_nodes + poly_nb<F>() - 1) / poly_nb<F>());
    const int kblocks = (p.K + sh.CB - 1) / sh.CB;
    const int per_block = poly_nb<F>() * sh.AG;
    const unsigned sgroups = (unsigned)((p.num_nodes + per_block - 1) / per_block + p.T);
    const size_t lds = (size_t)(17 + POLY_VG) * sh.PB * 16;
    auto go = [&](auto pbc) -> hipError_t {
        constexpr int PB = decltype(pbc)::value;
        static bool attr_done = false;   // per instantiation
        if (!attr_done) {
            hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(k_poly<F, PB>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
            if (err != hipSuccess) return err;
            attr_done = true;
        }
        hipLaunchKernelGGL((k_poly<F, PB>), dim3(sgroups * kblocks), dim3(PB * POLY_VG), lds, s, p, sh);
        return hipGetLastError();
    };
    switch (sh.PB) {
    case 64: return go(std::integral_constant<int, 64>{});
    case 128: return go(std::integral_constant<int, 128>{});
    case 192: return go(std::integral_constant<int, 192>{});
    default: return hipErrorInvalidValue;
    }
}
template hipError_t launch_poly<double>(const PolyParams<double>&, hipStream_t);
template hipError_t launch_poly<float>(const PolyParams<float>&, hipStream_t);

template <typename F>
hipError_t launch_poly_reverse(int N, int NP, int K, const F* M_grad, const F* M_adj, F* A_adj, hipStream_t s)
{
    if (N <= 0) return hipSuccess;
    if (K % 4 == 0) {
        const long total = (long)N * 16 * (K / 4);
        hipLaunchKernelGGL((k_poly_reverse<F, 4>), dim3(nblk(total, 256)), dim3(256), 0, s, total, NP, K, M_grad, M_adj, A_adj);
    } else {
        const long total = (long)N * 16 * K;
        hipLaunchKernelGGL((k_poly_reverse<F, 1>), dim3(nblk(total, 256)), dim3(256), 0, s, total, NP, K, M_grad, M_adj, A_adj);
    }
    return hipGetLastError();
}
template hipError_t launch_poly_reverse<double>(int, int, int, const double*, const double*, double*, hipStream_t);
template hipError_t launch_poly_reverse<float>(int, int, int, const float*, const float*, float*, hipStream_t);

// ===========================================================================
// Readout tail
// The whole readout tail in one launch (mace.cpp:876-903, multilayer_perceptron.cpp:76-150): the K -> 16 -> 1
// network on H2 with its gradient (H2_adj), the linear readout of H1's scalar block, the atomic energy, and the
// seed of H1_adj (readout weights in the scalar block of the first N rows, zero elsewhere).  A block serves 16
// nodes; thread (node, hidden unit) forms one hidden activation with the K products taken in ascending order.
namespace {
template <typename F>
__global__ __launch_bounds__(256) void k_readout_fused(int N, int rows, int K, int num_LM, const int* node_types,
                                                       const double* E0, const double* w1, const double* W1,
                                                       const double* w2, double scale, const F* H1, const double* H2,
                                                       double* H2_adj, F* H1_adj, double* node_energies,
                                                       int zero_energies, double* energies_copy, const int* guard,
                                                       int* guard_clear, double* guard_forces, double* guard_copy, long guard_forces_n)
{
    extern __shared__ double rsm[];
    // every reader of the check word has run (the sender lists come before the readout): clean for the next evaluation
    if (guard_clear && blockIdx.x == 0 && threadIdx.x == 0) *guard_clear = 0;
    if (guard && *guard) {
        // unchecked species indices: no table lookup, the energies say so; so do the edge forces, which the
        // adjoint kernels of this evaluation will not touch (they see no edges)
        const int i = blockIdx.x * 16 + (threadIdx.x >> 4);
        if ((threadIdx.x & 15) == 0 && i < N) {
            node_energies[i] = __builtin_nan("");
            if (energies_copy) energies_copy[i] = __builtin_nan("");
        }
        for (long t = (long)blockIdx.x * 256 + threadIdx.x; t < guard_forces_n; t += (long)gridDim.x * 256) {
            guard_forces[t] = __builtin_nan("");
            if (guard_copy) guard_copy[t] = __builtin_nan("");
        }
        return;
    }
    const int ldw = K + 1;                 // rows of W1 start two banks apart
    double* W = rsm;                       // [16][K + 1]
    double* hg = W + 16 * ldw;             // [16 nodes][16]
    double* X = hg + 256;                  // [16 nodes][K]: the block's rows of H2
    for (int t = threadIdx.x; t < 16 * K; t += 256) {
        W[(t / K) * ldw + t % K] = W1[t];
        const size_t src = (size_t)blockIdx.x * 16 * K + t;
        X[t] = src < (size_t)N * K ? H2[src] : 0.0;
    }
    __syncthreads();
    const int n = threadIdx.x >> 4, h = threadIdx.x & 15;
    const int i = blockIdx.x * 16 + n;
    double e = 0.0, g = 0.0;
    if (i < N) {
        const double* h2 = X + n * K;
        double s = 0.0;
#pragma unroll 8
        for (int k = 0; k < K; ++k) s += W[h * ldw + k] * h2[k];
        // multilayer_perceptron.cpp:107-113: scaled SiLU and its derivative
        const double sig = 1.0 / (1.0 + exp(-s));
        e = w2[h] * (scale * s * sig);
        g = w2[h] * (scale * sig + scale * s * sig * (1 - sig));
        const F* Hs = H1 + (size_t)i * num_LM * K;
        for (int k = h; k < K; k += 16) e += w1[k] * (double)Hs[k];
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) e += __shfl_xor(e, off, 64);
    hg[threadIdx.x] = g;
    if (h == 0 && i < N) {
        const double en = (zero_energies ? 0.0 : node_energies[i]) + E0[node_types[i]] + e;
        node_energies[i] = en;
        if (energies_copy) energies_copy[i] = en;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 16 * K; t += 256) {
        const int n2 = t / K, k = t - n2 * K;
        const int i2 = blockIdx.x * 16 + n2;
        if (i2 < N) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < 16; ++q) s += hg[n2 * 16 + q] * W[q * ldw + k];
            H2_adj[(size_t)i2 * K + k] = s;
        }
    }
    const int width = num_LM * K;
    for (int t = threadIdx.x; t < 16 * width; t += 256) {
        const int n2 = t / width, c = t - n2 * width;
        const int row = blockIdx.x * 16 + n2;
        if (row < rows) H1_adj[(size_t)row * width + c] = (c < K && row < N) ? (F)w1[c] : F(0);
    }
}
}  // namespace

template <typename F>
hipError_t launch_readout_fused(int N, int rows, int K, int num_LM, const int* node_types, const double* atomic_energies,
                                const double* w1, const double* W1, const double* w2, double scale, const F* H1,
                                const double* H2, double* H2_adj, F* H1_adj, double* node_energies, int zero_energies,
                                double* energies_copy, const int* guard, int* guard_clear, double* guard_forces,
                                double* guard_copy, long guard_forces_n, hipStream_t s)
{
    if (rows < N) return hipErrorInvalidValue;
    if (rows <= 0) return hipSuccess;
    const size_t lds = ((size_t)16 * (K + 1) + 256 + (size_t)16 * K) * sizeof(double);
    if (lds > 160 * 1024) return hipErrorInvalidValue;    // K beyond about 630 channels
    if (lds > 64 * 1024) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(k_readout_fused<F>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL(k_readout_fused<F>, dim3((rows + 15) / 16), dim3(256), lds, s, N, rows, K, num_LM, node_types,
                       atomic_energies, w1, W1, w2, scale, H1, H2, H2_adj, H1_adj, node_energies, zero_energies,
                       energies_copy, guard, guard_clear, guard_forces, guard_copy, guard_forces_n);
    return hipGetLastError();
}
template hipError_t launch_readout_fused<double>(int, int, int, int, const int*, const double*, const double*, const double*, const double*, double, const double*, const double*, double*, double*, double*, int, double*, const int*, int*, double*, double*, long, hipStream_t);
template hipError_t launch_readout_fused<float>(int, int, int, int, const int*, const double*, const double*, const double*, const double*, double, const float*, const double*, double*, float*, double*, int, double*, const int*, int*, double*, double*, long, hipStream_t);


// ===========================================================================
// Caller-side reductions: per-edge forces -> per-atom forces, virial.
// One wavefront per atom and step: the edges on which the atom is the sender are ordered in LDS, its lanes add them up (and
// the edges of its receivers, which are contiguous) in a fixed assignment and a fixed tree, so the sums are
// bit-reproducible.  A wavefront's share of the virial stays in its registers; every block leaves one partial sum.
// Bound by latency at small sizes (one thread per atom, as this was before: 52 us at 107 atoms, 31 us at 501), by the
// gather of 24-byte forces at large ones.
namespace {
constexpr int GATHER_CAP = 512;
__device__ __forceinline__ bool no_result(const int* flag, const int* skipped) { return (flag && *flag) || (skipped && *skipped); }
__device__ __forceinline__ void add_virial(double (&v)[6], const double* d, const double* f)
{
    const double x = d[0], y = d[1], z = d[2];
    v[0] += x * f[0]; v[1] += y * f[1]; v[2] += z * f[2];
    v[3] += 0.5 * (x * f[1] + y * f[0]); v[4] += 0.5 * (x * f[2] + z * f[0]); v[5] += 0.5 * (y * f[2] + z * f[1]);
}
// The block that finishes last adds up the partial sums of the virial, in a fixed order.  (A launch of its own for that: 4 to 5 us of a
// small evaluation.)  The sums and the count of finished blocks go past the L2 of a die, by themselves: a fence would write back and
// drop everything in it.
template <bool BEHIND>
__global__ __launch_bounds__(256) void k_force_gather(const ForceGather a, double* virial)
{
    __shared__ __align__(16) int bucket[4][GATHER_CAP];
    __shared__ double red[4][6];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double v[6] = {0, 0, 0, 0, 0, 0};
    const bool nothing = no_result(a.flag, a.skipped);     // (asked for here, needed at the end)
    for (int at = blockIdx.x * 4 + wave; at < a.num_atoms; at += gridDim.x * 4) {
        double fx = 0, fy = 0, fz = 0;
        if (a.send_start) {
            const int s0 = a.send_start[at], n = a.send_start[at + 1] - s0;
            const int* sorted = wave_sorted_bucket<GATHER_CAP>(a.send_list, s0, n, bucket[wave], lane, a.send_spare);
            for (int t = lane; t < n; t += 64) {
                const int e = sorted[t];
                if (a.senders && a.senders[e] != at) *a.differ = 1;
                const double* f = a.forces + 3 * (size_t)e;
                fx += f[0]; fy += f[1]; fz += f[2];
            }
        }
        // nodes whose receivers belong to this atom: a list of them, or node at itself
        const int n0 = a.node_start ? a.node_start[at] : at;
        const int n1 = a.node_start ? a.node_start[at + 1] : (at < a.num_nodes ? at + 1 : at);
        for (int q = n0; q < n1; ++q) {
            const int node = a.node_list ? a.node_list[q] : q;
            for (int e = a.first_neigh[node] + lane; e < a.first_neigh[node + 1]; e += 64) {
                const double* f = a.forces + 3 * (size_t)e;
                fx -= f[0]; fy -= f[1]; fz -= f[2];
                if (a.partial) add_virial(v, a.xyz + 3 * (size_t)e, f);
            }
        }
        if (a.atom_forces) {
            fx = wave_sum(fx); fy = wave_sum(fy); fz = wave_sum(fz);
            if (nothing) fx = fy = fz = __builtin_nan("");
            if (lane < 3) a.atom_forces[3 * (size_t)at + lane] = lane == 0 ? fx : (lane == 1 ? fy : fz);
        }
        wave_lds_sync();   // the next atom's bucket overwrites this one's
    }
    if (!a.partial) return;
    // Edges behind those of the nodes (the last counts covered the leading nodes of a longer edge list): every edge is in the
    // virial.
    if constexpr (BEHIND)
        for (long e = a.node_edges + (long)blockIdx.x * 256 + threadIdx.x; e < a.num_edges; e += (long)gridDim.x * 256)
            add_virial(v, a.xyz + 3 * (size_t)e, a.forces + 3 * (size_t)e);
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const double t = wave_sum(v[q]);
        if (lane == 0) red[wave][q] = t;
    }
    __shared__ int last;
    __syncthreads();
    if (wave == 0) {
        if (lane < 6)
            __hip_atomic_store(a.partial + (size_t)blockIdx.x * 6 + lane, (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the sums have arrived before the block counts as finished
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane == 0) last = __hip_atomic_fetch_add(a.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    for (int q = wave; q < 6; q += 4) {
        double t = 0.0;
        const int n = (int)gridDim.x;
        for (int b0 = lane; b0 < n; b0 += 8 * 64) {
            double x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                x[j] = __hip_atomic_load(a.partial + (size_t)min(b0 + 64 * j, n - 1) * 6 + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int j = 0; j < 8; ++j) t += b0 + 64 * j < n ? x[j] : 0.0;
        }
        t = wave_sum(t);
        if (lane == 0) virial[q] = nothing ? __builtin_nan("") : t;
    }
    if (threadIdx.x == 0) *a.ticket = 0;
}
}  // namespace

int force_gather_blocks(int num_atoms) { return std::min(std::max((num_atoms + 3) / 4, 1), 2048); }
hipError_t launch_force_gather(const ForceGather& g, double* virial, hipStream_t s)
{
    const int nb = force_gather_blocks(g.num_atoms);
    if ((g.partial != nullptr) != (virial != nullptr) || (virial && !g.ticket)) return hipErrorInvalidValue;
    if (g.num_edges > g.node_edges) hipLaunchKernelGGL(k_force_gather<true>, dim3(nb), dim3(256), 0, s, g, virial);
    else hipLaunchKernelGGL(k_force_gather<false>, dim3(nb), dim3(256), 0, s, g, virial);
    return hipGetLastError();
}

}  // namespace smx
