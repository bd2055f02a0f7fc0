// Full neighbour list on the device in the canonical order of this library:
// receivers ascending; within a receiver senders ascending; several periodic
// images of one sender ordered by the index of their image shift (the caller
// lists the shifts in lexicographic order of their integer triples).
//
// The arithmetic that decides membership and fills xyz and r is spelled out
// with round-to-nearest intrinsics (no fused multiply-add), in the order
//     image = x_j + shift;  d = image - x_i;  r2 = (d0*d0 + d1*d1) + d2*d2
// so that the list is bit-identical to the host builder
// (symmetrix_amd/neighbors.py), whatever the compiler would contract.
#include "smx_device.hpp"
#include "smx_kernels.hpp"

namespace smx {

namespace {

struct Cand {
    double d0, d1, d2, r2;
};
__device__ __forceinline__ Cand displacement(const double* pos, int i, int j, const double* sv)
{
    Cand c;
    c.d0 = __dsub_rn(__dadd_rn(pos[3 * (size_t)j], sv[0]), pos[3 * (size_t)i]);
    c.d1 = __dsub_rn(__dadd_rn(pos[3 * (size_t)j + 1], sv[1]), pos[3 * (size_t)i + 1]);
    c.d2 = __dsub_rn(__dadd_rn(pos[3 * (size_t)j + 2], sv[2]), pos[3 * (size_t)i + 2]);
    c.r2 = __dadd_rn(__dadd_rn(__dmul_rn(c.d0, c.d0), __dmul_rn(c.d1, c.d1)), __dmul_rn(c.d2, c.d2));
    return c;
}

__device__ __forceinline__ int bin_of(double x, double lo, double inv_bs, int nb)
{
    return min(max((int)floor((x - lo) * inv_bs), 0), nb - 1);
}

// per-block minima and maxima of the coordinates: part[block][6]
__global__ __launch_bounds__(256) void k_nl_bbox(const double* pos, int N, double* part)
{
    __shared__ double red[6][256];
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int i = blockIdx.x * 256 + threadIdx.x; i < N; i += gridDim.x * 256)
        for (int k = 0; k < 3; ++k) {
            const double v = pos[3 * (size_t)i + k];
            lo[k] = fmin(lo[k], v); hi[k] = fmax(hi[k], v);
        }
    for (int k = 0; k < 3; ++k) { red[k][threadIdx.x] = lo[k]; red[3 + k][threadIdx.x] = hi[k]; }
    __syncthreads();
    for (int off = 128; off >= 1; off >>= 1) {
        if ((int)threadIdx.x < off)
            for (int k = 0; k < 3; ++k) {
                red[k][threadIdx.x] = fmin(red[k][threadIdx.x], red[k][threadIdx.x + off]);
                red[3 + k][threadIdx.x] = fmax(red[3 + k][threadIdx.x], red[3 + k][threadIdx.x + off]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void k_nl_bin_count(const double* pos, int N, NlGrid g, int* atom_bin, int* bin_count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int b0 = bin_of(pos[3 * (size_t)i], g.lo[0], g.inv_bs[0], g.nb[0]);
    const int b1 = bin_of(pos[3 * (size_t)i + 1], g.lo[1], g.inv_bs[1], g.nb[1]);
    const int b2 = bin_of(pos[3 * (size_t)i + 2], g.lo[2], g.inv_bs[2], g.nb[2]);
    const int b = (b0 * g.nb[1] + b1) * g.nb[2] + b2;
    atom_bin[i] = b;
    atomicAdd(&bin_count[b], 1);
}
__global__ void k_nl_bin_fill(int N, const int* atom_bin, const int* bin_start, int* bin_cursor, int* bin_atoms)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int b = atom_bin[i];
    bin_atoms[bin_start[b] + atomicAdd(&bin_cursor[b], 1)] = i;
}

// Where a receiver's entries begin, without launches for counting and for the prefix sum: every block publishes the number
// of its entries, before it waits for anything, and adds up those of the blocks before it.  No block depends on another one
// running: after a bounded number of looks (blocks before it that have not started, whatever else is on the chip) a block
// counts the entries of all receivers before its own itself, `count_of` by the wavefront that calls.  A published number
// carries the tag of the launch, so nothing is cleared between launches.  The last block hands the total to the host while the
// entries are still being written.  (Counting, prefix sum and writing were three launches and the total a copy: 28 us of a
// 24-atom list, 15 us of an update at 501 atoms.)
template <typename CountOf>
__device__ __forceinline__ long chained_offset(const NlChain& ch, int c, int wave, int lane, CountOf&& count_of)
{
    __shared__ int counts[4];
    __shared__ long long parts[4];
    if (lane == 0) counts[wave] = c;
    __syncthreads();
    const unsigned sum = (unsigned)counts[0] + (unsigned)counts[1] + (unsigned)counts[2] + (unsigned)counts[3];
    if (threadIdx.x == 0)
        __hip_atomic_store(&ch.sums[blockIdx.x], ch.tag | sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    long long before = 0;
    bool all = true;
    for (unsigned b0 = 0; all && b0 < blockIdx.x; b0 += 4 * 256) {
        unsigned long long v[4];
        all = false;
        for (int look = 0; !all && look < ch.rounds; ++look) {
            all = true;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const unsigned b = b0 + q * 256 + threadIdx.x;
                v[q] = b < blockIdx.x ? __hip_atomic_load(&ch.sums[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ch.tag;
                all = all && (v[q] >> 32) == (ch.tag >> 32);
            }
        }
        if (all) {
#pragma unroll
            for (int q = 0; q < 4; ++q) before += (long long)(v[q] & 0xffffffffull);
        }
    }
    all = !__any(!all);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) before += __shfl_xor(before, off);
    if (lane == 0) parts[wave] = all ? before : -1;
    __syncthreads();
    if (parts[0] < 0 || parts[1] < 0 || parts[2] < 0 || parts[3] < 0) {
        before = 0;
        for (int k = wave; k < 4 * (int)blockIdx.x; k += 4) before += count_of(k);
        __syncthreads();      // everybody has seen who gave up
        if (lane == 0) parts[wave] = before;
        __syncthreads();
    }
    before = parts[0] + parts[1] + parts[2] + parts[3];
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        const unsigned long long total = (unsigned long long)before + sum;
        __hip_atomic_store(ch.host_total, ch.tag | (total > 0x7fffffffull ? 0xffffffffull : total), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
    for (int w = 0; w < wave; ++w) before += counts[w];
    return (long)before;
}

// One wavefront per receiver.  Its lanes first test 64 image shifts at a time against the bounding box of the atoms; for
// every shift that can hold neighbours the senders are walked 64 at a time: ALL false, the runs of atoms in the bins that
// the cutoff sphere of the shifted receiver touches (bins along the last axis are adjacent in memory, so a run is a row of
// bins); ALL true, every atom, without bins (short lists: binning is three launches, and a small cell is one bin anyway).
// COUNT counts.  FILL and CHAIN collect the keys sender * num_shifts + shift index in LDS and write them in ascending
// order, which is the canonical edge order, FILL at offsets it is given, CHAIN at offsets it finds itself; EMIT writes the
// edge arrays as well (a list without a skin: every candidate is an edge, at the positions of the search).
// Bound by latency: a receiver takes about nine dependent steps (one thread per receiver, as this was before, took as many
// as there are candidate pairs: 570 us against 8 us at 107 atoms in a cell smaller than twice the cutoff).
constexpr int SORT_KEYS = 256;   // keys per wavefront that are ordered in LDS (2 KB each, four wavefronts per block)
enum NlMode { COUNT, FILL, CHAIN };
enum { KEYS_NONE, KEYS_LDS, KEYS_GLOBAL };
using NlEdges = NlEdgeArrays;
__device__ __forceinline__ void emit_edge(const NlEdges& o, size_t e, int j, int s, const Cand& cd)
{
    o.neigh_indices[e] = j;
    o.neigh_types[e] = o.types ? o.types[j] : 0;
    o.neigh_shift[3 * e] = o.shift_int[3 * s]; o.neigh_shift[3 * e + 1] = o.shift_int[3 * s + 1];
    o.neigh_shift[3 * e + 2] = o.shift_int[3 * s + 2];
    o.xyz[3 * e] = cd.d0; o.xyz[3 * e + 1] = cd.d1; o.xyz[3 * e + 2] = cd.d2;
    o.r[e] = __dsqrt_rn(cd.r2);
}
template <NlMode MODE, bool ALL, bool EMIT>
__global__ __launch_bounds__(256) void k_nl_search(const double* pos, int N, NlGrid g, const int* bin_start,
                                                   const int* bin_atoms, int num_shifts, const double* shift_vec,
                                                   int zero_shift, double r_cut, double r2cut, int* count,
                                                   int* first, long capacity, long long* keys, long long* sorted,
                                                   NlEdges out, NlChain chain)
{
    __shared__ long long buf[MODE != COUNT ? 4 : 1][MODE != COUNT ? SORT_KEYS : 1];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + wave;
    const bool real = i < N;
    if (MODE != CHAIN && !real) return;
    const double reach = r_cut * (1.0 + 1e-9) + 1e-12;
    // the keys of receiver i in the order of the walk, to where HOW says; how many there are
    auto search = [&](auto how, int i, long e0) {
        constexpr int HOW = decltype(how)::value;
        const double xi[3] = {pos[3 * (size_t)i], pos[3 * (size_t)i + 1], pos[3 * (size_t)i + 2]};
        int c = 0;
        for (int s0 = 0; s0 < num_shifts; s0 += 64) {
            bool here = s0 + lane < num_shifts;
            if (here) {
                const double* sv = shift_vec + 3 * (s0 + lane);
                for (int k = 0; k < 3; ++k) {
                    const double q = xi[k] - sv[k];   // senders within reach of q see the receiver through shift s
                    here = here && !(q + reach < g.lo[k] || q - reach > g.hi[k]);
                }
            }
            for (unsigned long long todo = __ballot(here); todo; todo &= todo - 1) {
                const int s = s0 + __ffsll((long long)todo) - 1;
                const double sv[3] = {shift_vec[3 * s], shift_vec[3 * s + 1], shift_vec[3 * s + 2]};
                auto walk = [&](int t0, int t1) {
                    for (int tb = t0; tb < t1; tb += 64) {
                        const int t = tb + lane;
                        bool hit = false;
                        int j = 0;
                        if (t < t1) {
                            j = ALL ? t : bin_atoms[t];
                            hit = !(j == i && s == zero_shift) && displacement(pos, i, j, sv).r2 < r2cut;
                        }
                        const unsigned long long mask = __ballot(hit);
                        if (HOW != KEYS_NONE && hit) {
                            const int at = c + __popcll(mask & ((1ull << lane) - 1ull));
                            const long long key = (long long)j * num_shifts + s;
                            if (HOW == KEYS_GLOBAL) keys[(size_t)e0 + at] = key;
                            else if (at < SORT_KEYS) buf[wave][at] = key;
                        }
                        c += __popcll(mask);
                    }
                };
                if constexpr (ALL) {
                    walk(0, N);
                } else {
                    int blo[3], bhi[3];
                    for (int k = 0; k < 3; ++k) {
                        const double q = xi[k] - sv[k];
                        blo[k] = bin_of(q - reach, g.lo[k], g.inv_bs[k], g.nb[k]);
                        bhi[k] = bin_of(q + reach, g.lo[k], g.inv_bs[k], g.nb[k]);
                    }
                    for (int b0 = blo[0]; b0 <= bhi[0]; ++b0)
                        for (int b1 = blo[1]; b1 <= bhi[1]; ++b1) {
                            const int row = (b0 * g.nb[1] + b1) * g.nb[2];
                            walk(bin_start[row + blo[2]], bin_start[row + bhi[2] + 1]);
                        }
                }
            }
        }
        return c;
    };
    constexpr std::integral_constant<int, KEYS_NONE> none{};
    constexpr std::integral_constant<int, KEYS_LDS> to_lds{};
    constexpr std::integral_constant<int, KEYS_GLOBAL> to_memory{};
    if constexpr (MODE == COUNT) {
        const int c = search(none, i, 0);
        if (lane == 0) count[i] = c;
    } else {
        long e0;
        int n;
        if constexpr (MODE == CHAIN) {
            n = real ? search(to_lds, i, 0) : 0;
            e0 = chained_offset(chain, n, wave, lane, [&](int k) { return search(none, k, 0); });
            if (!real) return;
            if (lane == 0) {
                first[i] = (int)e0;
                if (i == N - 1) first[N] = (int)(e0 + n);
            }
        } else {
            e0 = first[i]; n = first[i + 1] - (int)e0;
        }
        if (EMIT && lane == 0) {
            out.first[i] = (int)e0; out.num_neigh[i] = n;
            if (i == N - 1) out.first[N] = (int)(e0 + n);
        }
        // room for the whole list was taken before its length was known: what does not fit is not written (the host looks
        // at the total and takes more room)
        if (e0 + n > capacity) return;
        const bool in_lds = n <= SORT_KEYS;
        if (!in_lds) search(to_memory, i, e0);
        else if (MODE == FILL) search(to_lds, i, e0);
        // rank of every key among the receiver's keys (they are distinct)
        if (in_lds) wave_lds_sync();
        else __threadfence();
        for (int a = lane; a < n; a += 64) {
            const long long key = in_lds ? buf[wave][a] : keys[(size_t)e0 + a];
            int rank = 0;
            if (in_lds) {
                for (int b = 0; b < n; ++b) rank += buf[wave][b] < key ? 1 : 0;
            } else {
                for (int b = 0; b < n; ++b) rank += keys[(size_t)e0 + b] < key ? 1 : 0;
            }
            sorted[(size_t)e0 + rank] = key;
            if constexpr (EMIT) {
                const int j = (int)(key / num_shifts), s = (int)(key % num_shifts);
                emit_edge(out, (size_t)e0 + rank, j, s, displacement(pos, i, j, shift_vec + 3 * s));
            }
        }
    }
}

// One wavefront per receiver walks its sorted candidates with the current positions and keeps those inside
// the cutoff, in order.  COUNT counts; FILL writes the edge arrays at first[i] + (number kept before), CHAIN counts, finds
// first[i] and writes.
// (room for `capacity` edges was taken before their number was known: none is written past it)
template <NlMode MODE>
__global__ __launch_bounds__(256) void k_nl_filter(const double* pos, int N, const int* cfirst, const long long* sorted,
                                                   long room, int num_shifts, const double* shift_vec, double r2cut,
                                                   int* count, int* first, long capacity, NlEdges out, NlChain chain)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + wave;
    const bool real = i < N;
    if (MODE != CHAIN && !real) return;
    // candidates that did not fit were not written to `sorted`
    const bool there = cfirst[N] <= room;
    // kept candidates of receiver i
    auto walk = [&](auto emit, int i, size_t e0) {
        const int c0 = cfirst[i], n = there ? cfirst[i + 1] - c0 : 0;
        int kept = 0;
        for (int a0 = 0; a0 < n; a0 += 64) {
            const int a = a0 + lane;
            bool pass = false;
            int j = 0, s = 0;
            Cand cd{};
            if (a < n) {
                const long long key = sorted[(size_t)c0 + a];
                j = (int)(key / num_shifts); s = (int)(key % num_shifts);
                cd = displacement(pos, i, j, shift_vec + 3 * s);
                pass = cd.r2 < r2cut;
            }
            const unsigned long long mask = __ballot(pass);
            if (decltype(emit)::value && pass) emit_edge(out, e0 + kept + __popcll(mask & ((1ull << lane) - 1ull)), j, s, cd);
            kept += __popcll(mask);
        }
        return kept;
    };
    if constexpr (MODE == FILL) {
        if (!there || first[N] > capacity) return;
        walk(std::true_type{}, i, (size_t)first[i]);
    } else {
        const int kept = real ? walk(std::false_type{}, i, 0) : 0;
        if (real && lane == 0) count[i] = kept;
        if constexpr (MODE == CHAIN) {
            const long e0 = chained_offset(chain, kept, wave, lane, [&](int k) { return walk(std::false_type{}, k, 0); });
            if (!real) return;
            if (lane == 0) {
                first[i] = (int)e0;
                if (i == N - 1) first[N] = (int)(e0 + kept);
            }
            if (e0 + kept <= capacity) walk(std::true_type{}, i, (size_t)e0);
        }
    }
}

__global__ __launch_bounds__(256) void k_bring(uint4* to, const uint4* from, unsigned n)
{
    const unsigned t = blockIdx.x * 256 + threadIdx.x;
    if (t < n) to[t] = from[t];
}

}  // namespace

hipError_t launch_bring(void* to, const void* from_host, size_t n, hipStream_t s)
{
    if (n % 16 || n / 16 > 0x7fffffffu) return hipErrorInvalidValue;
    if (n) hipLaunchKernelGGL(k_bring, dim3((unsigned)((n / 16 + 255) / 256)), dim3(256), 0, s, static_cast<uint4*>(to),
                              static_cast<const uint4*>(from_host), (unsigned)(n / 16));
    return hipGetLastError();
}
hipError_t launch_nl_bbox(const double* pos, int N, double* part, int nblocks, hipStream_t s)
{
    hipLaunchKernelGGL(k_nl_bbox, dim3(nblocks), dim3(256), 0, s, pos, N, part);
    return hipGetLastError();
}
hipError_t launch_nl_bins(const double* pos, int N, const NlGrid& g, int* atom_bin, int* bin_count, hipStream_t s)
{
    if (N > 0) hipLaunchKernelGGL(k_nl_bin_count, dim3((N + 255) / 256), dim3(256), 0, s, pos, N, g, atom_bin, bin_count);
    return hipGetLastError();
}
hipError_t launch_nl_bin_fill(int N, const int* atom_bin, const int* bin_start, int* bin_cursor, int* bin_atoms,
                              hipStream_t s)
{
    if (N > 0) hipLaunchKernelGGL(k_nl_bin_fill, dim3((N + 255) / 256), dim3(256), 0, s, N, atom_bin, bin_start, bin_cursor, bin_atoms);
    return hipGetLastError();
}
hipError_t launch_nl_search(bool fill, const double* pos, int N, const NlGrid& g, const int* bin_start,
                            const int* bin_atoms, int num_shifts, const double* shift_vec, int zero_shift,
                            double r_cut, int* count, int* first, long capacity, long long* keys, long long* sorted,
                            const NlEdgeArrays* edges, const NlChain* chain, hipStream_t s)
{
    if (N <= 0) return hipSuccess;
    const NlEdges o = edges ? *edges : NlEdges{};
    const NlChain ch = chain ? *chain : NlChain{};
    const bool all = bin_start == nullptr;
    if (all && !(fill && chain)) return hipErrorInvalidValue;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nl_blocks(N)), dim3(256), 0, s, pos, N, g, bin_start, bin_atoms, num_shifts, shift_vec,
                           zero_shift, r_cut, r_cut * r_cut, count, first, capacity, keys, sorted, o, ch);
    };
    if (!fill) go(k_nl_search<COUNT, false, false>);
    else if (!chain) { if (edges) go(k_nl_search<FILL, false, true>); else go(k_nl_search<FILL, false, false>); }
    else if (all) { if (edges) go(k_nl_search<CHAIN, true, true>); else go(k_nl_search<CHAIN, true, false>); }
    else { if (edges) go(k_nl_search<CHAIN, false, true>); else go(k_nl_search<CHAIN, false, false>); }
    return hipGetLastError();
}
hipError_t launch_nl_filter(bool fill, const double* pos, int N, const int* cfirst, const long long* sorted, long room, int num_shifts,
                            const double* shift_vec, double r_cut, int* count, int* first, long capacity,
                            const NlEdgeArrays* edges, const NlChain* chain, hipStream_t s)
{
    if (N <= 0) return hipSuccess;
    const NlEdges o = edges ? *edges : NlEdges{};
    const NlChain ch = chain ? *chain : NlChain{};
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nl_blocks(N)), dim3(256), 0, s, pos, N, cfirst, sorted, room, num_shifts, shift_vec,
                           r_cut * r_cut, count, first, capacity, o, ch);
    };
    if (!fill) go(k_nl_filter<COUNT>);
    else if (!chain) go(k_nl_filter<FILL>);
    else go(k_nl_filter<CHAIN>);
    return hipGetLastError();
}

}  // namespace smx
