// H2, the readout tail and reverse_H2 in one launch (mace.cpp:820-903).  All three work on one atom's
// rows only.  A block takes tiles of 16 atoms of one species (species groups of the list preparation) through:
//   H2 = H1[l=0] . W_H1[type] + M1 . W_M1 on the matrix cores (wavefront w owns columns 16 w to 16 w + 15),
//   the K -> 16 -> 1 network with its gradient hg [16 atoms][16 hidden units], energies,
//   H2_adj = hg . W1, H1_adj[l=0] = w1 + hg . (W1 W_H1[type]^T), M1_adj = hg . (W1 W_M1^T).
// The gradient of H2 has rank 16, so its products with the K x K matrices are taken once, at load, and what is left of them
// here is an eighth of the products for H2 (K = 128).  Sums over k run in one fixed order per output element, independent of the
// atom's tile mates; inside groups of 8, k is permuted on both operands so that a lane reads 16 bytes of a row at once.
//
// Bound by the matrix instructions for H2 (64 cycles each, K / 2 per wavefront and tile) once the chip is full, by the latency of
// the phases below for one tile per block.  The weights of H2 stay in registers over the tiles of a block (they are 256 KB at
// K = 128, twice what the matrix instructions of a tile leave time to read), the rows of the next tile are on their way during
// the second half of this one.  Against one tile per block with all four K x K products: 50 000 atoms, 128 channels 356 -> 112 us,
// 24 999 atoms 198 -> 78 us, 20 011 atoms, 96 channels 98 -> 53 us, 3 000 atoms 23.4 -> 18.3 us.
//
// Compiled without the hoisting of machine instructions out of loops: it kept the constants of exp in 22 registers over the
// tiles, and spilled as many weights (K = 96).  At three wavefronts per SIMD 96 channels still spill 12 registers (single 2).
#include "smx_device.hpp"
#include "smx_kernels.hpp"

#include <algorithm>

namespace smx {

namespace {
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
constexpr int kTailLd = 18;      // doubles of a row in the 16-column tiles: 16-byte reads of eight rows meet all banks
constexpr int tail_blocks_per_cu(int KT) { return KT == 6 ? 2 : 8 / KT; }      // by registers
template <typename F, int KT>
__global__ __launch_bounds__(64 * KT, KT == 6 ? 3 : 2) void k_tail_fused(const TailParams<F> p, int per)
{
    extern __shared__ __align__(16) double tsm[];
    constexpr int K = 16 * KT, T = 64 * KT, ld = K + 4;   // (rows 8 banks apart, as above)
    typedef F F4 __attribute__((ext_vector_type(4)));
    double* XA = tsm;                        // [16][ld] H1[l=0] rows
    double* XB = XA + 16 * ld;               // [16][ld] M1 rows
    double* part = XB + 16 * ld;             // [KT][16][kTailLd] columns of H2 by wavefront, then its part of the hidden units
    double* hg = part + KT * 16 * kTailLd;   // [16 atoms][kTailLd]
    double* W1s = hg + 16 * kTailLd;         // [16 hidden][ld]
    // [8][T] operands of two adjoint products, by thread: the product for H2 needs the registers
    double* const back = W1s + 16 * ld + threadIdx.x;
    __shared__ double w1_s[K], w2_s[16];
    __shared__ int node_s[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int width = p.num_LM * K;
    // every reader of the check word has run (the sender lists come before the readout): clean for the next evaluation
    if (p.guard_clear && blockIdx.x == 0 && tid == 0) *p.guard_clear = 0;
    if (p.guard && *p.guard) {
        // the inputs of this evaluation failed their checks and the species groups are empty: the energies say so
        for (long i = (long)blockIdx.x * T + tid; i < p.N; i += (long)gridDim.x * T) {
            p.node_energies[i] = __builtin_nan("");
            if (p.energies_copy) p.energies_copy[i] = __builtin_nan("");
        }
        // ... and so do the edge forces, which the adjoint kernels will not touch (they see no edges)
        for (long t = (long)blockIdx.x * T + tid; t < p.guard_forces_n; t += (long)gridDim.x * T) {
            p.guard_forces[t] = __builtin_nan("");
            if (p.guard_copy) p.guard_copy[t] = __builtin_nan("");
        }
        return;
    }
    // rows beyond the atoms (ghost rows of H1_adj) are cleared by all blocks together
    {
        const long ghost = (long)(p.rows - p.N) * width;
        for (long t = (long)blockIdx.x * T + tid; t < ghost; t += (long)gridDim.x * T)
            p.H1_adj[(size_t)p.N * width + t] = F(0);
    }
    // tiles first to first + per - 1, those that there are
    int index = blockIdx.x * per;
    const int last = min(index + per, p.N / 16 + p.T) - 1;
    RowTile at = row_tile(p.tstart, p.T, index, lane);
    auto advance = [&]() {
        if ((at.tile + 1) * 16 < at.seg_n && index < last) { ++at.tile; ++index; return; }
        for (at.type = -1; at.type < 0 && index < last;) at = row_tile(p.tstart, p.T, ++index, lane);
    };
    if (at.type < 0) advance();
    if (at.type < 0) return;
    auto node_of = [&](int row) { return at.tile * 16 + row < at.seg_n ? p.perm[at.seg0 + at.tile * 16 + row] : -1; };
    int r = lane & 15, g = lane >> 4, col = wave * 16 + r;
    // one 4-element piece of a row per thread
    int row = tid / (K / 4), k4 = tid % (K / 4) * 4;
    int node = node_of(row);      // of this thread's row
    F4 h1 = {}, m1 = {};
    auto fetch = [&]() {
        const size_t nd = max(node, 0);      // (rows of no atom repeat atom 0 and are not stored)
        h1 = *reinterpret_cast<const F4*>(p.H1 + nd * width + k4);
        m1 = *reinterpret_cast<const F4*>(p.M1 + nd * K + k4);
    };
    fetch();
    // element of a [K][K] matrix in operand order: row 8 (q / 2) + 2 g + q % 2, column col, as scalar base and 32 bits per lane
    const unsigned lane_bytes = (unsigned)(2 * g * K + col) * 8;
    auto operand = [&](const double* w, int q) {
        return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(w + (8 * (q / 2) + q % 2) * K) + lane_bytes);
    };
    double b1[K / 4], b2[K / 4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        W1s[row * ld + k4 + u] = p.W1[row * K + k4 + u];
        back[u * T] = operand(p.V_M1, u);
    }
#pragma unroll
    for (int q = 0; q < K / 4; ++q) b2[q] = operand(p.W_M1, q);
    if (tid < K) w1_s[tid] = p.w1[tid];
    if (tid < 16) w2_s[tid] = p.w2[tid];
    int type = -1;
    for (int i = 0; at.type >= 0; ++i) {
        if (at.type != type) {
            type = at.type;
            const double* WH = p.W_H1 + (size_t)type * K * K;
#pragma unroll
            for (int q = 0; q < K / 4; ++q) b1[q] = operand(WH, q);
#pragma unroll
            for (int u = 0; u < 4; ++u) back[(4 + u) * T] = operand(p.V_H1 + (size_t)type * 16 * K, u);
        }
        // (the compiler would keep every address that depends on these over the loop, and spill weights for them)
        asm volatile("" : "+v"(r), "+v"(g), "+v"(col), "+v"(row), "+v"(k4));
        int* const nodes = node_s[i & 1];
        if (k4 == 0) nodes[row] = node;
        {
            double* a = XA + row * ld + k4;
            double* b = XB + row * ld + k4;
#pragma unroll
            for (int t = 0; t < 4; ++t) { a[t] = (double)h1[t]; b[t] = (double)m1[t]; }
        }
        // the blocks of H1_adj other than l = 0 start at zero
        if (node >= 0)
            for (int LM = 1; LM < p.num_LM; ++LM) *reinterpret_cast<F4*>(p.H1_adj + (size_t)node * width + LM * K + k4) = F4{};
        __syncthreads();
        // ---- H2 tile
        advance();
        if (at.type >= 0) node = node_of(row);
        double* const mine = part + wave * 16 * kTailLd;
        {
            f64x4 acc1 = {0, 0, 0, 0}, acc2 = {0, 0, 0, 0};
            const double* a = XA + r * ld + 2 * g;
            const double* b = XB + r * ld + 2 * g;
            // (reads one group ahead, and no further: the compiler would take all of them first and spill)
            f64x2 va[2], vb[2];
            auto read = [&](int q) {
                va[q & 1] = *reinterpret_cast<const f64x2*>(a + 8 * q);
                vb[q & 1] = *reinterpret_cast<const f64x2*>(b + 8 * q);
            };
            read(0);
#pragma unroll
            for (int q = 0; q < K / 8; ++q) {
                if (q + 1 < K / 8) read(q + 1);
                asm volatile("" ::: "memory");
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(va[q & 1][t], b1[2 * q + t], acc1, 0, 0, 0);
                    acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(vb[q & 1][t], b2[2 * q + t], acc2, 0, 0, 0);
                }
            }
            int nd[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) nd[q] = nodes[4 * q + g];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double v = acc1[q] + acc2[q];
                mine[(4 * q + g) * kTailLd + r] = v;
                if (nd[q] >= 0) p.H2[(size_t)nd[q] * K + col] = v;
            }
        }
        wave_lds_sync();
        // this wavefront's columns in the sums of the hidden units
        {
            f64x4 acc = {0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f64x2 v = *reinterpret_cast<const f64x2*>(mine + r * kTailLd + 8 * j + 2 * g);
                const f64x2 w = *reinterpret_cast<const f64x2*>(W1s + r * ld + wave * 16 + 8 * j + 2 * g);
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v[0], w[0], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v[1], w[1], acc, 0, 0, 0);
            }
            wave_lds_sync();
#pragma unroll
            for (int q = 0; q < 4; ++q) mine[(4 * q + g) * kTailLd + r] = acc[q];
        }
        __syncthreads();
        // ---- readout network, energies (16 lanes an atom, one per hidden unit)
        for (int u = wave * 64 + 16 * g + r; u < 256; u += T) {
            const int n = u >> 4, h = u & 15, nd = nodes[n];
            double s = 0.0, e = 0.0;
#pragma unroll
            for (int w = 0; w < KT; ++w) s += part[(w * 16 + n) * kTailLd + h];
#pragma unroll
            for (int w = 0; w < KT; ++w) e += w1_s[16 * w + h] * XA[n * ld + 16 * w + h];
            // multilayer_perceptron.cpp:107-113: scaled SiLU and its derivative
            const double sig = 1.0 / (1.0 + exp(-s));
            e += w2_s[h] * (p.scale * s * sig);
            hg[n * kTailLd + h] = w2_s[h] * (p.scale * sig + p.scale * s * sig * (1 - sig));
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) e += __shfl_xor(e, off, 64);
            if (h == 0 && nd >= 0) {
                const double en = (p.zero_energies ? 0.0 : p.node_energies[nd]) + p.E0[type] + e;
                p.node_energies[nd] = en;
                if (p.energies_copy) p.energies_copy[nd] = en;
            }
        }
        __syncthreads();
        // ---- adjoints
        if (at.type >= 0) fetch();
        {
            int nd[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) nd[q] = nodes[4 * q + g];
            const f64x2 v[2] = {*reinterpret_cast<const f64x2*>(hg + r * kTailLd + 2 * g),
                                *reinterpret_cast<const f64x2*>(hg + r * kTailLd + 8 + 2 * g)};
            // (one after another, for the registers of one)
            auto product = [&](const double* w, int step0, int step, auto store) {
                asm volatile("" ::: "memory");
                f64x4 acc = {0, 0, 0, 0};
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v[u / 2][u % 2], w[(u / 2) * step0 + (u % 2) * step], acc, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (nd[q] >= 0) store((size_t)nd[q], acc[q]);
            };
            product(W1s + 2 * g * ld + col, 8 * ld, ld, [&](size_t n, double x) { p.H2_adj[n * K + col] = x; });
            const double seed = (double)(F)w1_s[col];
            product(back + 4 * T, 2 * T, T, [&](size_t n, double x) { p.H1_adj[n * width + col] = (F)(seed + x); });
            product(back, 2 * T, T, [&](size_t n, double x) { p.M1_adj[n * K + col] = (F)x; });
        }
    }
}
}  // namespace

template <typename F>
size_t tail_fused_lds(int K) { return ((size_t)3 * 16 * (K + 4) + (size_t)(K + 16) * kTailLd + 8 * 4 * (size_t)K) * sizeof(double); }
bool tail_fused_ok(int K) { return K == 32 || K == 48 || K == 64 || K == 96 || K == 128; }

template <typename F, int KT>
static hipError_t launch_tail_fused_t(const TailParams<F>& p, hipStream_t s)
{
    const size_t lds = tail_fused_lds<F>(p.K);
    if (lds > 64 * 1024) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(k_tail_fused<F, KT>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    // a block per tile while the chip holds them all at once, then as many tiles to each of the blocks that it holds
    const int tiles = (p.N + 15) / 16 + p.T, at_once = std::max(p.num_cus, 1) * tail_blocks_per_cu(KT), per = (tiles + at_once - 1) / at_once;
    hipLaunchKernelGGL((k_tail_fused<F, KT>), dim3((unsigned)((tiles + per - 1) / per)), dim3(64 * KT), lds, s, p, per);
    return hipGetLastError();
}
template <typename F>
hipError_t launch_tail_fused(const TailParams<F>& p, hipStream_t s)
{
    if (p.rows < p.N || !tail_fused_ok(p.K) || p.T <= 0) return hipErrorInvalidValue;
    if (p.rows <= 0) return hipSuccess;
    switch (p.K / 16) {
    case 2: return launch_tail_fused_t<F, 2>(p, s);
    case 3: return launch_tail_fused_t<F, 3>(p, s);
    case 4: return launch_tail_fused_t<F, 4>(p, s);
    case 6: return launch_tail_fused_t<F, 6>(p, s);
    default: return launch_tail_fused_t<F, 8>(p, s);
    }
}
template hipError_t launch_tail_fused<double>(const TailParams<double>&, hipStream_t);
template hipError_t launch_tail_fused<float>(const TailParams<float>&, hipStream_t);

}  // namespace smx
