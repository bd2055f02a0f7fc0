// The node-local stages between two aggregations in one launch each, for systems that do not fill the chip with row tiles.
//
//   k_chain0   A0 = Phi0 . W, M0 = polynomials of A0, H1 = M0 . W                    (mace.cpp:158-178, 349-370, 397-418)
//   k_chain1   A1 = Phi1 . W, M1, H2, readouts, their adjoints back to M1_adj and the seed of H1_adj, dPhi1
//              (mace.cpp:607-640, 759-903)
//   k_chain2   H1_adj += messages, M0_adj = H1_adj . W^T, A0_adj, dPhi0              (mace.cpp:372-436, 579-604, 180-236)
//
// All of them touch the rows of one atom only, so a thread block takes one atom through all of its stages, with everything
// between them in LDS.  As launches of their own the stages of a small system were a row of dependent launches of 6 to 20 us,
// each of which waited for its first loads and filled a few CUs: 24 atoms, 96 channels, double precision 96 us in eight launches,
// in chains 10 + 18 + 11; 107 atoms, 128 channels, l <= 1: 170 us in ten, in chains 17 + 43 + 33.
// The aggregation before a chain and its adjoint behind it touch the rows of one receiver and its edges, and go into the same launch
// for scalar features where that pays (smx_chain_edges.hpp; the rule is the caller's): 24 atoms 8 + 10, 7 + 18 + 13 and 11 + 12 us in
// seven launches, now 17 + 33 + 19 in three, and a device-resident evaluation 87 -> 78; 256 atoms 102 -> 86, single precision 501
// atoms 97 -> 87.
// Bound by what one CU reads, at 64 bytes per cycle: 295 KB of weights (96 channels, double, one A-basis product), 470 KB of spline
// coefficients (38 edges); between them by the latency of dependent loads.
//
// Products.  A wavefront owns 16 columns and 8 of the 16 (l, m): either l = 0 and 3 or l = 1 and 2, which is the same work.  Its
// four 16-lane rows share the inner index (every row a quarter of each piece of 64 bytes) and are added up at the end.  Weights
// come from memory in the operand order of k_linear (1 KB per instruction, a few pieces ahead).  Operands are read from LDS with
// the lanes of a row holding different (l, m), and v_fmac with a DPP row broadcast brings them to all columns.  Rows lie 64 bytes
// further than a multiple of 128 apart in LDS: four rows and the four quarters of a piece meet all banks.
// (Four atoms per block, which share every weight, came out behind the row tiles of k_linear where those fill the chip: 3 000
// atoms, 96 channels, double: 53 + 106 + 84 us against 60 + 112 + 61.)
#include "smx_chain_edges.hpp"
#include "smx_paths.hpp"
#include "smx_poly_body.hpp"

#include <algorithm>

namespace smx {

namespace {

constexpr int kPad = 64;       // bytes behind a row in LDS
__device__ __forceinline__ int lm_of_slot(int set, int slot) { return set == 0 ? (slot == 0 ? 0 : 8 + slot) : 1 + slot; }
__device__ __forceinline__ int slot_of_quad(int quad, int g) { return 4 * quad + ((g & 1) << 1 | g >> 1); }

// Sums over the four 16-lane rows of four values: row 0 ends with the first, row 2 with the second, row 1 with the third, row 3
// with the fourth (slot_of_quad).
template <typename F>
__device__ __forceinline__ F sum_rows4(F q0, F q1, F q2, F q3)
{
    swap_halves(q0, q1);
    swap_halves(q2, q3);
    F a = q0 + q1, b = q2 + q3;
    swap_rows(a, b);
    return a + b;
}

// One product of an atom's rows with 16 columns, for the (l, m) of a set: see above.  SAME: both l of a set have as many pieces.
template <typename F, bool SAME>
struct Product {
    static constexpr int V = 16 / (int)sizeof(F);
    // pieces of weights requested ahead; a row of 32 channels has this many pieces, so every number of them is a multiple
    static constexpr int AHEAD = sizeof(F) == 8 ? 4 : 2;
    typedef F VV __attribute__((ext_vector_type(V)));
    VV w[AHEAD][2];
    const F* wp[2];           // the lane's place in the weights of the two l of the set
    int steps[2];             // pieces of their inner index
    __device__ __forceinline__ void request(int c, int at)
    {
#pragma unroll
        for (int j = 0; j < 2; ++j) w[at][j] = *reinterpret_cast<const VV*>(wp[j] + (size_t)max(min(c, steps[j] - 1), 0) * (64 * V));
    }
    __device__ __forceinline__ void begin()
    {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) request(d, d);
    }
    // row: the operand row of slot lane % 8, at the lane's quarter of the first piece; out: slots slot_of_quad(0 and 1, lane / 16)
    template <int SET>
    __device__ __forceinline__ void run_set(const unsigned char* row, F (&out)[2])
    {
        constexpr int NA = SET == 0 ? 1 : 3;      // slots of the first l
        F acc[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[q] = F(0);
        const int n = SAME ? steps[0] : max(steps[0], steps[1]);
        VV a[2];                // operands of this piece and the next
        auto fetch = [&](int c, VV& to) { to = *reinterpret_cast<const VV*>(row + min(c, n - 1) * 64); };
        fetch(0, a[0]);
        for (int c0 = 0; c0 < n; c0 += AHEAD)
            static_for<0, AHEAD>([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                const int c = c0 + d;
                fetch(c + 1, a[(d + 1) & 1]);
                // (two wait states between a move of an operand, which the compiler may place here, and its broadcast)
                asm volatile("s_nop 1" : "+v"(a[d & 1]));
                auto part = [&](auto bc, auto ec, auto lc) {
                    constexpr int l = decltype(lc)::value;
                    if (!SAME && c >= steps[l]) return;
                    static_for<0, V>([&](auto vc) {
                        constexpr int v = decltype(vc)::value;
                        static_for<decltype(bc)::value, decltype(ec)::value>([&](auto qc) {
                            fmac_lane<decltype(qc)::value>(acc[decltype(qc)::value], a[d & 1][v], w[d][l][v]);
                        });
                    });
                };
                part(std::integral_constant<int, 0>{}, std::integral_constant<int, NA>{}, std::integral_constant<int, 0>{});
                part(std::integral_constant<int, NA>{}, std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
                // the piece is done with: its registers take the next weights (otherwise the compiler collects the requests
                // behind the arithmetic of all pieces)
#pragma unroll
                for (int q = 0; q < 8; ++q) pin(acc[q]);
                request(c + AHEAD, d);
                __builtin_amdgcn_sched_barrier(0);
            });
#pragma unroll
        for (int j = 0; j < 2; ++j) out[j] = sum_rows4<F>(acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]);
    }
    __device__ __forceinline__ void run(int set, const unsigned char* row, F (&out)[2])
    {
        if (set == 0) run_set<0>(row, out);
        else run_set<1>(row, out);
    }
};

// Block -> atom, in the order of the species groups: blocks that run together read the same weights.
struct BlockAtom {
    int type, node;       // species (-1: nothing to do)
};
__device__ __forceinline__ BlockAtom block_atom(const int* perm, const int* tstart, int T, int lane)
{
    const int at = blockIdx.x;
    if (at >= tstart[T]) return {-1, 0};      // (the lists of a skipped evaluation are empty)
    int type = 0;
    for (int t0 = 1; t0 < T; t0 += 64) type += __popcll(__ballot(t0 + lane < T && tstart[min(t0 + lane, T)] <= at));
    return {type, __builtin_amdgcn_readfirstlane(perm[at])};
}

constexpr int chain_threads(int K) { return 8 * K; }      // two sets of (l, m) for every 16 columns
// Wavefronts per SIMD the kernels are compiled for: one block of 128 channels on a CU, two of 64, four of 32, and two of 96 channels
// in single precision.  There k_chain1 spills 12 registers with the edges (l = 0) and 2 without, k_chain0 of l <= 2 with the edges 7,
// which pays where CUs have a second block: evaluations, us, with six / with four and nothing spilled: l = 0, 24 atoms 57 / 57, 107
// 65 / 64, 256 76 / 74, 300 93 / 107, 501 98 / 114, 1 000 171 / 203; l <= 1, 107 120 / 118, 256 144 / 142, 500 216 / 225; l <= 2, 24
// 156 / 151, 256 221 / 218, 400 337 / 351.  In double precision k_chain1 of l = 0 with the edges spills 2 registers from 64 channels on,
// k_chain0 of l <= 2 with the edges 4 at 32 channels.
template <typename F> constexpr int chain_waves(int K) { return sizeof(F) == 4 && K == 96 ? 6 : 4; }

// The products of a few rows per atom (polynomials, scalar features) with K x K weights: a thread takes 16 bytes of columns and a
// slice of the inner index, one slice in SLICES (all threads take part unless that were too many partial sums).
template <int NV> constexpr int mix_slices() { return NV > 4 ? 4 : 16; }
// acc[v] += sum over the slice, COUNT long, of x[k'][v] W(v)[k'][columns]: NV values of x per k', NW matrices of which value v
// takes which(v)
template <typename F, int NV, int NW, int COUNT, int K>
struct Mix {
    static constexpr int V = 16 / (int)sizeof(F), AHEAD = COUNT * NW <= 8 ? COUNT : 8 / NW;
    typedef F VV __attribute__((ext_vector_type(V)));
    VV w[AHEAD][NW];
    const F* wp;
    unsigned matrix;
    __device__ __forceinline__ Mix(const F* W, unsigned matrix_stride, int column, int first) : wp(W + (size_t)first * K + column), matrix(matrix_stride) {}
    __device__ __forceinline__ void request(int i)
    {
#pragma unroll
        for (int j = 0; j < NW; ++j) w[i % AHEAD][j] = *reinterpret_cast<const VV*>(wp + (size_t)j * matrix + (size_t)i * K);
    }
    __device__ __forceinline__ void begin()
    {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) request(d);
    }
    template <typename Which>
    __device__ __forceinline__ void run(const F* x, VV (&acc)[NV], Which which)
    {
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = VV(F(0));
        static_for<0, COUNT>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            static_for<0, NV>([&](auto vc) {
                constexpr int v = decltype(vc)::value;
                acc[v] += x[i * NV + v] * w[i % AHEAD][which(vc)];
            });
            if constexpr (i + AHEAD < COUNT) request(i + AHEAD);
        });
    }
};

// x . W of an atom's NV rows, x[K][NV] in LDS: the sums of the slices in red[slice][v][k], to be added up by mixed().  Value v is a
// row of degree l(v) and takes matrix l.  The barrier before the product is in here (between the requests and the first use).
template <typename F, int NV, int NW, int K>
__device__ __forceinline__ void mix_rows(const F* x, const F* W, F* red, int tid)
{
    constexpr int S = mix_slices<NV>(), count = K / S, V = 16 / (int)sizeof(F);
    using M = Mix<F, NV, NW, count, K>;
    const int sl = tid / (K / V), col = (tid - sl * (K / V)) * V;
    M mix(W, K * K, col, min(sl, S - 1) * count);
    if (sl < S) mix.begin();
    __syncthreads();
    if (sl < S) {
        typename M::VV acc[NV];
        mix.run(x + sl * count * NV, acc, [](auto vc) { return lm_l(decltype(vc)::value); });
#pragma unroll
        for (int v = 0; v < NV; ++v) *reinterpret_cast<typename M::VV*>(red + (sl * NV + v) * K + col) = acc[v];
    }
    __syncthreads();
}
template <typename F, int NV, int K>
__device__ __forceinline__ F mixed(const F* red, int t)
{
    F s = red[t];
#pragma unroll
    for (int j = 1; j < mix_slices<NV>(); ++j) s += red[j * NV * K + t];
    return s;
}

// coefficients of a channel's polynomials: every 256 bytes 16 of them
template <typename F, int K>
__device__ __forceinline__ const unsigned char* coefficients(const F* coef, int groups16, int type, int k)
{
    return reinterpret_cast<const unsigned char*>(coef) + (((size_t)type * (K / 16) + k / 16) * groups16 * 16 + k % 16) * 16;
}

// groups of coefficients requested ahead: as many as the registers hold
template <typename F> constexpr int kCoefAhead = sizeof(F) == 8 ? 3 : 4;
template <typename F, int LM, int AHEAD = kCoefAhead<F>> using Coef = PolyCoef<F, LM, AHEAD>;

// The polynomial of output slot 0 of all channels, value and gradient, in kSlices parts by groups of wavefronts:
// part[slice][17][K] gets the sums over the slice, gradient before value; polynomial_value() adds them up.  Evaluations with one, two and
// four slices, us: 96 channels, double 24 atoms 78.8 / 77.6 / 80.2, 107 81.8 / 80.7 / 83.6, 600 215 / 213 / 223; 64 channels 200 62.7 /
// 61.1 / 63.5; single, 96 channels 501 89.6 / 88.6 / 89.5.
constexpr int kSlices = 2;
template <typename F, int K> constexpr size_t slice_bytes() { return (size_t)kSlices * 17 * K * sizeof(F); }
template <typename F, int K, unsigned RS>
struct SlicedPolynomial {
    static constexpr int per = (K + 63) / 64 * 64;
    static_assert(chain_threads(K) / per >= kSlices, "a group of wavefronts for every slice");
    Coef<F, 0> coef;
    int slot, k;
    bool own;
    __device__ __forceinline__ SlicedPolynomial(const F* from, int groups16, int type, int tid)
        : coef(coefficients<F, K>(from, groups16, type, min(tid % per, K - 1)), 256), slot(__builtin_amdgcn_readfirstlane(tid / per)),
          k(tid % per), own(tid % per < K) {}
    __device__ __forceinline__ void begin()
    {
        static_for<0, kSlices>([&](auto sc) {
            if (slot == decltype(sc)::value) coef.template begin<poly_slice<F, 0>(decltype(sc)::value, kSlices)>();
        });
    }
    // rows: the variables, rows RS bytes apart
    __device__ __forceinline__ void run(const unsigned char* rows, F* part)
    {
        if (slot >= kSlices) return;
        F x[16], g[16], f = F(0);
#pragma unroll
        for (int q = 0; q < 16; ++q) { x[q] = *reinterpret_cast<const F*>(rows + q * RS + min(k, K - 1) * sizeof(F)); g[q] = F(0); }
        static_for<0, kSlices>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if (slot == s) poly_spec_run<F, 0, 0, false, kCoefAhead<F>, poly_slice<F, 0>(s, kSlices), poly_slice<F, 0>(s + 1, kSlices)>(coef, x, g, f, F(1));
        });
        if (!own) return;
#pragma unroll
        for (int q = 0; q < 16; ++q) part[(slot * 17 + q) * K + k] = g[q];
        part[(slot * 17 + 16) * K + k] = f;
    }
};
template <typename F, int K>
__device__ __forceinline__ F polynomial_value(const F* part, int t)      // entry t of [17][K]
{
    F s = part[t];
#pragma unroll
    for (int j = 1; j < kSlices; ++j) s += part[j * 17 * K + t];
    return s;
}

// An atom's operand rows into LDS, 16 bytes at a time, all of a thread's words requested before the first is stored;
// row_of(lme): the LDS row of a memory row
template <typename F, int ROWS, int K, typename RowOf>
__device__ __forceinline__ void stage_rows(const F* from, unsigned char* dst, RowOf row_of)
{
    constexpr unsigned KW = K * sizeof(F) / 16, WORDS = ROWS * KW, T = chain_threads(K), N = (WORDS + T - 1) / T;
    uint4 v[N];
    static_for<0, (int)N>([&](auto jc) {      // (a thread without a word of its own takes the last one)
        v[decltype(jc)::value] = reinterpret_cast<const uint4*>(from)[min(decltype(jc)::value * T + threadIdx.x, WORDS - 1)];
    });
    static_for<0, (int)N>([&](auto jc) {
        const unsigned w = decltype(jc)::value * T + threadIdx.x;
        if (WORDS % T == 0 || w < WORDS) *reinterpret_cast<uint4*>(dst + w * 16 + row_of(w / KW) * kPad) = v[decltype(jc)::value];
    });
}

// ---------------------------------------------------------------------------
// EDGES (here and below): the aggregation before the node-local stages, or its adjoint behind them, in the same launch.
template <typename F, int LH, int K, bool EDGES>
__global__ __launch_bounds__(chain_threads(K), chain_waves<F>(K)) void k_chain0(const ChainParams<F> p, const AggParams<F> agg)
{
    constexpr int NP = (LH + 1) * (LH + 1), V = 16 / (int)sizeof(F), KC = 4 * V, T = chain_threads(K);
    constexpr unsigned RS = K * sizeof(F) + kPad;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const BlockAtom b = block_atom(p.perm, p.tstart, p.T, lane);
    if (b.type < 0) return;
    const size_t node = b.node;
    const int type = b.type;
    F* xm = reinterpret_cast<F*>(smem + p.lds_front);       // [K][NP]: M0
    const int ct = wave >> 1, set = wave & 1, column = ct * 16 + r16;
    if constexpr (EDGES) {
        F sum[2];
        ChainEdges<F, K>(wave, lane).forward(agg, (int)node, type, smem + p.lds_part, tid, lane, sum);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = tid + j * T, row = t / K;
            *reinterpret_cast<F*>(smem + row * RS + (t - row * K) * sizeof(F)) = sum[j];
            if constexpr (LH == 0) agg.out[node * 16 * K + t] = sum[j];     // (A0 may be asked for, and is formed from them)
        }
    }
    Product<F, true> prod;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int l = set == 0 ? 3 * j : 1 + j;
        prod.wp[j] = p.W + ((size_t)l * p.T + type) * K * K + ((size_t)ct * (K / KC) * 64 + lane) * V;
        prod.steps[j] = K / KC;
    }
    prod.begin();
    if constexpr (!EDGES) stage_rows<F, 16, K>(p.Phi + node * 16 * K, smem, [](unsigned row) { return row; });
    __syncthreads();
    F out[2];
    prod.run(set, smem + lm_of_slot(set, r16 & 7) * RS + g * 16, out);
    auto leave = [&]() {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int lm = lm_of_slot(set, slot_of_quad(j, g));
            *reinterpret_cast<F*>(smem + lm * RS + column * sizeof(F)) = out[j];
            if constexpr (LH > 0) p.A[(node * 16 + lm) * K + column] = out[j];
        }
    };
    if constexpr (LH == 0) {
        SlicedPolynomial<F, K, RS> poly(p.coef, poly_spec_offset(NP) / V, type, tid);
        poly.begin();
        __syncthreads();
        leave();
        __syncthreads();
        F* part = reinterpret_cast<F*>(smem + p.lds_part);
        poly.run(smem, part);
        __syncthreads();
        for (int t = tid; t < 17 * K; t += T) {
            const F s = polynomial_value<F, K>(part, t);
            if (t < 16 * K) p.M_grad[node * 16 * K + t] = s;
            else {
                xm[t - 16 * K] = s;
                p.M[node * K + t - 16 * K] = s;
            }
        }
    } else {
        // polynomials: K threads each, in whole wavefronts
        constexpr int per = (K + 63) / 64 * 64, slots = T / per;
        const int slot = __builtin_amdgcn_readfirstlane(tid / per), k = min(tid - slot * per, K - 1);
        const bool own = tid - slot * per < K;
        const unsigned char* coef = coefficients<F, K>(p.coef, poly_spec_offset(NP) / V, type, k);
        Coef<F, 0> first(coef, 256);
        if (slot == 0) first.begin();
        __syncthreads();
        leave();
        __syncthreads();
        static_for<0, NP>([&](auto pc) {
            constexpr int lm = decltype(pc)::value;
            if (lm % slots != slot) return;
            F x[16], gr[16], f = F(0);
#pragma unroll
            for (int q = 0; q < 16; ++q) { x[q] = *reinterpret_cast<const F*>(smem + q * RS + k * sizeof(F)); gr[q] = F(0); }
            if constexpr (lm == 0) poly_spec_run<F, 0, 1, false>(first, x, gr, f, F(1));
            else {
                Coef<F, lm> next(coef, 256);
                next.begin();
                poly_spec_run<F, lm, 1, false>(next, x, gr, f, F(1));
            }
            if (!own) return;
            xm[k * NP + lm] = f;
            p.M[(node * NP + lm) * K + k] = f;
        });
    }
    F* red = reinterpret_cast<F*>(smem);
    mix_rows<F, NP, LH + 1, K>(xm, p.WH1, red, tid);
    for (int t = tid; t < NP * K; t += T) p.H1[node * NP * K + t] = mixed<F, NP, K>(red, t);
}

// ---------------------------------------------------------------------------
// (EDGES: scalar hidden features with a diagonal coupling)
template <typename F, int LH, int K, bool EDGES>
__global__ __launch_bounds__(chain_threads(K), chain_waves<F>(K)) void k_chain1(const ChainParams<F> p, const TailParams<F> q, const AggParams<F> agg)
{
    static_assert(!EDGES || LH == 0, "scalar hidden features");
    using PT = Paths<LH>;
    constexpr int NLM = (LH + 1) * (LH + 1), NE = PT::NE, V = 16 / (int)sizeof(F), KC = 4 * V, S = mix_slices<1>();
    constexpr int T = chain_threads(K), width = NLM * K;
    constexpr unsigned RS = K * sizeof(F) + kPad;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    // the readout's part for skipped evaluations and ghost rows: see k_tail_fused
    if (q.guard_clear && blockIdx.x == 0 && tid == 0) *q.guard_clear = 0;
    if (q.guard && *q.guard) {
        for (long i = (long)blockIdx.x * T + tid; i < q.N; i += (long)gridDim.x * T) {
            q.node_energies[i] = __builtin_nan("");
            if (q.energies_copy) q.energies_copy[i] = __builtin_nan("");
        }
        for (long t = (long)blockIdx.x * T + tid; t < q.guard_forces_n; t += (long)gridDim.x * T) {
            q.guard_forces[t] = __builtin_nan("");
            if (q.guard_copy) q.guard_copy[t] = __builtin_nan("");
        }
        return;
    }
    {
        const long ghost = (long)(q.rows - q.N) * width;
        for (long t = (long)blockIdx.x * T + tid; t < ghost; t += (long)gridDim.x * T) q.H1_adj[(size_t)q.N * width + t] = F(0);
    }
    const BlockAtom b = block_atom(p.perm, p.tstart, p.T, lane);
    if (b.type < 0) return;
    const size_t node = b.node;
    const int type = b.type;
    // LDS: operand rows, then the 16 rows of the A-basis in their place, then what the tail needs (in double), then the
    // adjoint rows; H1[l = 0] and M1 behind them
    double* red = reinterpret_cast<double*>(smem);                // [S][K]
    double* h2 = red + S * K;                                     // [K]
    double* dots = h2 + K;                                        // [17]
    double* hg = dots + 17;                                       // [16]
    double* xh = reinterpret_cast<double*>(smem + p.lds_front);   // [2][K]: H1[l = 0] and M1
    const int ct = wave >> 1, set = wave & 1, column = ct * 16 + r16;
    constexpr int nel[4] = {PT::num_e(0), PT::num_e(1), PT::num_e(2), PT::num_e(3)};
    constexpr int lme0[4] = {PT::lme_off(0), PT::lme_off(1), PT::lme_off(2), PT::lme_off(3)};
    auto nel_of = [&](int l) { return l == 0 ? nel[0] : (l == 1 ? nel[1] : (l == 2 ? nel[2] : nel[3])); };
    auto lme_of = [&](int l) { return l == 0 ? lme0[0] : (l == 1 ? lme0[1] : (l == 2 ? lme0[2] : lme0[3])); };
    auto blocks_before = [&](int l) { return (l > 0 ? nel[0] : 0) + (l > 1 ? nel[1] : 0) + (l > 2 ? nel[2] : 0); };   // matrices
    Product<F, (LH < 2)> prod;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int l = set == 0 ? 3 * j : 1 + j;
        prod.steps[j] = nel_of(l) * (K / KC);
        prod.wp[j] = p.W + (size_t)blocks_before(l) * K * K + ((size_t)ct * prod.steps[j] * 64 + lane) * V;
    }
    if constexpr (EDGES) {
        F sum[2];
        ChainEdges<F, K>(wave, lane).forward(agg, (int)node, type, smem + p.lds_part, tid, lane, sum);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = tid + j * T, row = t / K;
            *reinterpret_cast<F*>(smem + row * RS + (t - row * K) * sizeof(F)) = sum[j];
            agg.out[node * 16 * K + t] = sum[j];
        }
        prod.begin();
    } else {
        prod.begin();
        stage_rows<F, NE, K>(p.Phi + node * NE * K, smem, [&](unsigned lme) {
            const int l = lme < (unsigned)lme0[1] ? 0 : (lme < (unsigned)lme0[2] ? 1 : (lme < (unsigned)lme0[3] ? 2 : 3));
            const unsigned in = lme - lme_of(l);
            return (unsigned)(l * l) + (l == 0 ? 0u : (l == 1 ? in / nel[1] : (l == 2 ? in / nel[2] : in / nel[3])));
        });
    }
    const bool own = tid < K;                  // this thread's channel
    const int k = own ? tid : 0;
    if (own) xh[k] = (double)q.H1[node * width + k];
    __syncthreads();
    F out[2];
    {
        const int lm = lm_of_slot(set, r16 & 7), l = lm_l(lm);
        prod.run(set, smem + (unsigned)(lme_of(l) + (lm - l * l) * nel_of(l)) * (K * sizeof(F)) + lm * kPad + g * 16, out);
    }
    SlicedPolynomial<F, K, RS> poly(p.coef, poly_spec_offset(1) / V, type, tid);
    poly.begin();
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<F*>(smem + lm_of_slot(set, slot_of_quad(j, g)) * RS + column * sizeof(F)) = out[j];
    __syncthreads();
    // M1; its gradient stays with the threads that formed it
    F gr[2];
    {
        F* part = reinterpret_cast<F*>(smem + p.lds_part);
        poly.run(smem, part);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            gr[j] = polynomial_value<F, K>(part, tid + j * T);
            p.M_grad[node * 16 * K + tid + j * T] = gr[j];
        }
        if (own) {
            const F f = polynomial_value<F, K>(part, 16 * K + k);
            xh[K + k] = (double)f;
            p.M[node * K + k] = f;
        }
    }
    // two products with K x K weights at once: the lower half of the slices takes the first matrix, the upper the second
    constexpr int count = 2 * K / S;
    using TM = Mix<double, 1, 1, count, K>;
    const int sl = tid / (K / 2), pair = (tid - sl * (K / 2)) * 2, from = (sl % (S / 2)) * count;
    const size_t typed = (size_t)type * K * K;
    // H2 = H1[l = 0] . W_H1[type] + M1 . W_M1
    {
        TM mix(sl < S / 2 ? q.W_H1 + typed : q.W_M1, 0, pair, from);
        mix.begin();
        __syncthreads();
        typename TM::VV acc[1];
        mix.run((sl < S / 2 ? xh : xh + K) + from, acc, [](auto) { return 0; });
        *reinterpret_cast<typename TM::VV*>(red + sl * K + pair) = acc[0];
        __syncthreads();
    }
    // what the gradient of the hidden units is multiplied with below: a channel of H2_adj, H1_adj[l = 0] or M1_adj
    const int back = tid / K, kb = tid - back * K;
    double v[16];
    if (back < 3) {
        const double* from_hg = back == 0 ? q.W1 : (back == 1 ? q.V_H1 + (size_t)type * 16 * K : q.V_M1);
#pragma unroll
        for (int h = 0; h < 16; ++h) v[h] = from_hg[h * K + kb];
    }
    if (own) {
        const double s = mixed<double, 1, K>(red, k);
        h2[k] = s;
        q.H2[node * K + k] = s;
    }
    __syncthreads();
    // 16 hidden units and the linear readout: eight lanes a sum
    if (tid < 192) {
        const int u = min(tid >> 3, 16), part = tid & 7;
        const double* w = u < 16 ? q.W1 + u * K : q.w1;
        const double* x = u < 16 ? h2 : xh;
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < K / 8; ++j) s += w[part + 8 * j] * x[part + 8 * j];
#pragma unroll
        for (int off = 4; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
        if (part == 0 && tid < 17 * 8) dots[u] = s;
    }
    __syncthreads();
    if (tid < 16) {
        // multilayer_perceptron.cpp:107-113: scaled SiLU and its derivative
        const double s = dots[tid], sig = 1.0 / (1.0 + exp(-s));
        double e = q.w2[tid] * (q.scale * s * sig);
        hg[tid] = q.w2[tid] * (q.scale * sig + q.scale * s * sig * (1 - sig));
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) e += __shfl_xor(e, off, 64);
        if (tid == 0) {
            const double en = (q.zero_energies ? 0.0 : q.node_energies[node]) + q.E0[type] + (e + dots[16]);
            q.node_energies[node] = en;
            if (q.energies_copy) q.energies_copy[node] = en;
        }
    }
    __syncthreads();
    // the weights of the adjoint product, for what follows the next two barriers
    auto aim_back = [&](int e) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int l = set == 0 ? 3 * j : 1 + j;
            prod.steps[j] = e < nel_of(l) ? K / KC : 0;
            prod.wp[j] = p.Wt + (size_t)(blocks_before(l) + min(e, nel_of(l) - 1)) * K * K + ((size_t)ct * (K / KC) * 64 + lane) * V;
        }
        prod.begin();
    };
    aim_back(0);
    // H2_adj = hg . W1, H1_adj[l = 0] = w1 + H2_adj . W_H1^T, M1_adj = H2_adj . W_M1^T
    if (back < 3) {
        double s = back == 1 ? (double)(F)q.w1[kb] : 0.0;
#pragma unroll
        for (int h = 0; h < 16; ++h) s += hg[h] * v[h];
        if (back == 0) q.H2_adj[node * K + kb] = s;
        else if (back == 1) q.H1_adj[node * width + kb] = (F)s;
        else {
            q.M1_adj[node * K + kb] = (F)s;
            xh[K + kb] = s;
        }
    }
    for (int t = K + tid; t < width; t += T) q.H1_adj[node * width + t] = F(0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int t = tid + j * T, row = t / K, c = t - row * K;
        *reinterpret_cast<F*>(smem + row * RS + c * sizeof(F)) = gr[j] * (F)xh[K + c];
    }
    __syncthreads();
    // dPhi1 = A1_adj . W^T, output block by output block
    constexpr int most = std::max(std::max(nel[0], nel[1]), std::max(nel[2], nel[3]));
    for (int e = 0; e < most; ++e) {
        if (e) aim_back(e);
        if (prod.steps[0] == 0 && prod.steps[1] == 0) continue;
        F o[2];
        prod.run(set, smem + lm_of_slot(set, r16 & 7) * RS + g * 16, o);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int lm = lm_of_slot(set, slot_of_quad(j, g)), l = lm_l(lm), n = nel_of(l);
            if (e < n) p.out[(node * NE + lme_of(l) + (lm - l * l) * n + e) * K + column] = o[j];
        }
        if constexpr (EDGES) {
            if (!agg.msg) return;          // (the messages do not fit their array: launches of their own)
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j) *reinterpret_cast<F*>(smem + lm_of_slot(set, slot_of_quad(j, g)) * RS + column * sizeof(F)) = o[j];
            __syncthreads();
            ChainEdges<F, K>(wave, lane).template adjoint<true>(agg, (int)node, type, smem, RS, smem + p.lds_part, tid, lane);
        }
    }
}

// ---------------------------------------------------------------------------
constexpr int kBucket = 256;       // edges of a sender that are put in order in LDS
constexpr int kPolySlots = 4;      // groups of wavefronts that share the polynomials of layer 0
template <int NP> constexpr int kMsgWords = NP == 1 ? 4 : 8;     // 16-byte words of messages that a thread brings at once
// In double precision l <= 1 spills 38 to 48 registers of the polynomials' adjoints (44 at 128 channels with the edges, 38 without, where
// the wavefronts of a block leave 128 registers each in any case), l <= 2 up to 8.  With the registers of one block per CU (K / 32
// wavefronts per SIMD) l <= 1 spills none up to 96 channels; evaluations, us, as it is / so: 32 channels 200 atoms 109 / 109, 1 000
// 246 / 245; 64 channels 48 121 / 120, 200 141 / 139, 768 390 / 404 (no second block on a CU); 96 channels, where there is one block
// either way, 107 159 / 158, 250 233 / 231, 500 427 / 425.
template <typename F, int LH, int K, bool EDGES>
__global__ __launch_bounds__(chain_threads(K), LH == 0 ? chain_waves<F>(K) : 4) void k_chain2(const ChainParams<F> p, const AggParams<F> agg)
{
    constexpr int NP = (LH + 1) * (LH + 1), V = 16 / (int)sizeof(F), KC = 4 * V, T = chain_threads(K), width = NP * K;
    constexpr unsigned RS = K * sizeof(F) + kPad;
    typedef F VV __attribute__((ext_vector_type(V)));
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) int bucket[kBucket], sorted[kBucket];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const BlockAtom b = block_atom(p.perm, p.tstart, p.T, lane);
    if (b.type < 0) return;
    const size_t node = b.node;
    const int type = b.type;
    F* xm = reinterpret_cast<F*>(smem + p.lds_front);       // [K][NP]: H1_adj
    F* ym = xm + width;                                     // [K][NP]: M0_adj
    F* red = reinterpret_cast<F*>(smem);                    // messages, then partial sums, before the operand rows
    const int ct = wave >> 1, set = wave & 1, column = ct * 16 + r16;
    Product<F, true> prod;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int l = set == 0 ? 3 * j : 1 + j;
        prod.wp[j] = p.Wt + ((size_t)l * p.T + type) * K * K + ((size_t)ct * (K / KC) * 64 + lane) * V;
        prod.steps[j] = K / KC;
    }
    // The messages to this atom, added to what is there in ascending edge order (the order of a sum by launches of their own,
    // chunk by chunk: same bits).  All threads bring messages into LDS, as many as fit, the next ones while a thread per column
    // adds up these.
    F sum[2];                    // this thread's columns: tid, tid + T (width is at most nine times K)
#pragma unroll
    for (int j = 0; j < 2; ++j) sum[j] = tid + j * T < width ? p.H1_adj[node * width + tid + j * T] : F(0);
    if (p.msg) {
        const int s0 = p.sstart[node], n = p.sstart[node + 1] - s0;
        const int* const list = p.slist + s0;
        if (n > kBucket) {
            if (wave == 0) wave_sort_in_memory(p.slist, s0, n, bucket, lane, p.spare);
        } else {
            // the rank of an edge is the number of smaller ones, counted by eight lanes
            for (int t = tid; t < n; t += T) bucket[t] = list[t];
            __syncthreads();
            for (int e0 = 0; e0 < n; e0 += T / 8) {
                const int e = e0 + (tid >> 3), v = bucket[min(e, n - 1)];
                int rank = 0;
                for (int t = tid & 7; t < n; t += 8) rank += bucket[t] < v;
                rank += __shfl_xor(rank, 1, 64); rank += __shfl_xor(rank, 2, 64); rank += __shfl_xor(rank, 4, 64);
                if (e < n && (tid & 7) == 0) sorted[rank] = v;
            }
        }
        __syncthreads();
        constexpr int UL = kMsgWords<NP>;
        constexpr unsigned mw = width / V, at_once = (unsigned)(UL * T) / mw;
        VV hold[UL];
        // (a word behind the last message repeats that one's; nothing is asked for where all threads are behind it)
        auto bring = [&](int first) {
            int e[UL];
#pragma unroll
            for (int q = 0; q < UL; ++q) {
                const int m = first + min((int)((q * T + tid) / mw), (int)at_once - 1);
                e[q] = n > kBucket ? list[min(m, n - 1)] : sorted[min(m, n - 1)];
            }
#pragma unroll
            for (int q = 0; q < UL; ++q)
                if (first + (int)(q * T / mw) < n)
                    hold[q] = __builtin_nontemporal_load(reinterpret_cast<const VV*>(p.msg + (size_t)e[q] * width) + (q * T + tid) % mw);
        };
        VV* stage = reinterpret_cast<VV*>(smem);
        if (n > 0) bring(0);
        for (int first = 0; first < n; first += at_once) {
            const int here = min((int)at_once, n - first);
#pragma unroll
            for (int q = 0; q < UL; ++q) stage[q * T + tid] = hold[q];
            __syncthreads();
            bring(first + at_once);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (tid + j * T < width) {
                    const F* col = reinterpret_cast<const F*>(smem) + tid + j * T;
#pragma unroll 8
                    for (int m = 0; m < here; ++m) sum[j] += col[(size_t)m * width];
                }
            __syncthreads();
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c = tid + j * T;
        if (c < width) {
            if (p.msg) p.H1_adj[node * width + c] = sum[j];
            xm[(c % K) * NP + c / K] = sum[j];
        }
    }
    // M0_adj = H1_adj . W^T
    mix_rows<F, NP, LH + 1, K>(xm, p.WH1, red, tid);
    for (int t = tid; t < width; t += T) {
        const F s = mixed<F, NP, K>(red, t);
        ym[(t % K) * NP + t / K] = s;
        p.M[node * width + t] = s;
    }
    if constexpr (LH == 0) prod.begin();
    __syncthreads();
    // A0_adj into the operand rows
    if constexpr (LH == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = tid + j * T, row = t / K, k = t - row * K;
            *reinterpret_cast<F*>(smem + row * RS + k * sizeof(F)) = p.M_grad[(node * 16 + row) * K + k] * ym[k];
        }
    } else {
        // the gradients again from the variables, every group of wavefronts some of the polynomials
        constexpr int per = (K + 63) / 64 * 64, slots = T / per < kPolySlots ? T / per : kPolySlots;
        const int slot = __builtin_amdgcn_readfirstlane(tid / per), k = tid - slot * per;
        F* part = reinterpret_cast<F*>(smem + p.lds_part);       // [slots][16][K]
        if (slot < slots && k < K) {
            F x[16], gr[16], f = F(0);
#pragma unroll
            for (int i = 0; i < 16; ++i) { x[i] = p.A[(node * 16 + i) * K + k]; gr[i] = F(0); }
            static_for<0, NP>([&](auto pc) {
                constexpr int lm = decltype(pc)::value;
                if (lm % slots != slot) return;
                asm volatile("" ::: "memory");      // (the coefficients of the other polynomials stay where they are)
                Coef<F, lm, 2> coef(coefficients<F, K>(p.coef, poly_spec_offset(NP) / V, type, k), 256);
                coef.begin();
                poly_spec_run<F, lm, 2, false>(coef, x, gr, f, ym[k * NP + lm]);
            });
#pragma unroll
            for (int i = 0; i < 16; ++i) part[(slot * 16 + i) * K + k] = gr[i];
        }
        prod.begin();
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = tid + j * T, row = t / K, kk = t - row * K;
            F s = part[t];
#pragma unroll
            for (int q = 1; q < slots; ++q) s += part[q * 16 * K + t];
            *reinterpret_cast<F*>(smem + row * RS + kk * sizeof(F)) = s;
        }
    }
    __syncthreads();
    F o[2];
    prod.run(set, smem + lm_of_slot(set, r16 & 7) * RS + g * 16, o);
#pragma unroll
    for (int j = 0; j < 2; ++j) p.out[(node * 16 + lm_of_slot(set, slot_of_quad(j, g))) * K + column] = o[j];
    if constexpr (EDGES) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<F*>(smem + lm_of_slot(set, slot_of_quad(j, g)) * RS + column * sizeof(F)) = o[j];
        __syncthreads();
        ChainEdges<F, K>(wave, lane).template adjoint<false>(agg, (int)node, type, smem, RS, smem + p.lds_edges, tid, lane);
    }
}

template <typename Kernel, typename... Args>
hipError_t launch_chain_t(Kernel kern, unsigned blocks, int threads, size_t lds, hipStream_t s, const Args&... args)
{
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    if (lds > 64 * 1024) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(threads), lds, s, args...);
    return hipGetLastError();
}
inline size_t round16(size_t n) { return (n + 15) / 16 * 16; }

template <typename Fn>
hipError_t with_degree(int L_max, Fn&& f)
{
    if (L_max == 0) return f(std::integral_constant<int, 0>{});
    if (L_max == 1) return f(std::integral_constant<int, 1>{});
    if (L_max == 2) return f(std::integral_constant<int, 2>{});
    return hipErrorInvalidValue;
}

}  // namespace

// Compiled in 24 parts, side by side: SMX_CHAIN_PART = 8 * chain + 2 * (K / 32 - 1) + (0: double, 1: float).
#ifndef SMX_CHAIN_PART
#error "define SMX_CHAIN_PART"
#endif
#if SMX_CHAIN_PART % 2 == 0
typedef double chain_t;
#else
typedef float chain_t;
#endif
constexpr int kK = 32 * (SMX_CHAIN_PART / 2 % 4 + 1);

#if SMX_CHAIN_PART / 8 == 0
template <typename F, int K>
hipError_t launch_chain0(ChainParams<F> p, const AggParams<F>* agg, int L_max, hipStream_t s)
{
    if (p.N <= 0) return hipSuccess;
    if (p.T <= 0) return hipErrorInvalidValue;
    return with_degree(L_max, [&](auto lc) {
        constexpr int LH = decltype(lc)::value, NP = (LH + 1) * (LH + 1);
        constexpr size_t rows = (size_t)16 * (K * sizeof(F) + kPad), sums = (size_t)mix_slices<NP>() * NP * K * sizeof(F);
        p.lds_front = (unsigned)round16(std::max(rows, sums));
        size_t lds = p.lds_front + (size_t)NP * K * sizeof(F);
        p.lds_part = (unsigned)round16(lds);
        if (LH == 0) lds = p.lds_part + slice_bytes<F, K>();
        if (!agg) return launch_chain_t(k_chain0<F, LH, K, false>, (unsigned)p.N, chain_threads(K), lds, s, p, AggParams<F>{});
        lds = std::max(lds, p.lds_part + ChainEdges<F, K>::fwd_bytes);
        return launch_chain_t(k_chain0<F, LH, K, true>, (unsigned)p.N, chain_threads(K), lds, s, p, *agg);
    });
}
template hipError_t launch_chain0<chain_t, kK>(ChainParams<chain_t>, const AggParams<chain_t>*, int, hipStream_t);
#elif SMX_CHAIN_PART / 8 == 1
template <typename F, int K>
hipError_t launch_chain1(ChainParams<F> p, const TailParams<F>& q, const AggParams<F>* agg, int L_max, hipStream_t s)
{
    if (q.rows <= 0) return hipSuccess;
    if (p.N <= 0 || p.T <= 0 || q.rows < q.N || q.N != p.N) return hipErrorInvalidValue;
    return with_degree(L_max, [&](auto lc) {
        constexpr int LH = decltype(lc)::value;
        constexpr size_t in = Paths<LH>::NE * K * sizeof(F) + 16 * kPad, rows = (size_t)16 * (K * sizeof(F) + kPad);
        constexpr size_t tail = ((size_t)(mix_slices<1>() + 1) * K + 33) * sizeof(double);
        p.lds_front = (unsigned)round16(std::max({in, rows, tail}));
        p.lds_part = (unsigned)round16(p.lds_front + (size_t)2 * K * sizeof(double));
        size_t lds = p.lds_part + slice_bytes<F, K>();
        if constexpr (LH == 0) {
            if (agg) {
                lds = std::max({lds, p.lds_part + ChainEdges<F, K>::fwd_bytes, p.lds_part + ChainEdges<F, K>::bwd_bytes});
                return launch_chain_t(k_chain1<F, LH, K, true>, (unsigned)p.N, chain_threads(K), lds, s, p, q, *agg);
            }
        }
        if (agg) return hipErrorInvalidValue;
        return launch_chain_t(k_chain1<F, LH, K, false>, (unsigned)p.N, chain_threads(K), lds, s, p, q, AggParams<F>{});
    });
}
template hipError_t launch_chain1<chain_t, kK>(ChainParams<chain_t>, const TailParams<chain_t>&, const AggParams<chain_t>*, int, hipStream_t);
#else
template <typename F, int K>
hipError_t launch_chain2(ChainParams<F> p, const AggParams<F>* agg, int L_max, hipStream_t s)
{
    if (p.N <= 0) return hipSuccess;
    if (p.T <= 0) return hipErrorInvalidValue;
    return with_degree(L_max, [&](auto lc) {
        constexpr int LH = decltype(lc)::value, NP = (LH + 1) * (LH + 1);
        constexpr size_t rows = (size_t)16 * (K * sizeof(F) + kPad), sums = (size_t)mix_slices<NP>() * NP * K * sizeof(F);
        constexpr size_t stage = (size_t)kMsgWords<NP> * 16 * chain_threads(K);
        p.lds_front = (unsigned)round16(std::max(rows, sums));
        size_t lds = p.lds_front + (size_t)2 * NP * K * sizeof(F);
        p.lds_part = (unsigned)round16(lds);
        p.lds_edges = (unsigned)round16(rows);
        if (LH > 0) lds = p.lds_part + (size_t)kPolySlots * 16 * K * sizeof(F);
        lds = std::max(lds, stage);
        if (!agg) return launch_chain_t(k_chain2<F, LH, K, false>, (unsigned)p.N, chain_threads(K), lds, s, p, AggParams<F>{});
        lds = std::max(lds, p.lds_edges + ChainEdges<F, K>::bwd_bytes);
        return launch_chain_t(k_chain2<F, LH, K, true>, (unsigned)p.N, chain_threads(K), lds, s, p, *agg);
    });
}
template hipError_t launch_chain2<chain_t, kK>(ChainParams<chain_t>, const AggParams<chain_t>*, int, hipStream_t);
#endif

}  // namespace smx
