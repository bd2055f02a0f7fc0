// The channel-mixing linears of the A-basis, their adjoints, and the symmetric contractions behind them, on the gfx950 matrix
// cores (MACE::compute_A0 / compute_A1, the linears of reverse_A0 / reverse_A1, compute_M0 / compute_M1).
//
// A row tile is 16 atoms with the same (l, m), so the 16 (l, m) of an atom are 16 tiles, and the accumulators of one
// wavefront (16 columns, 16 tiles) hold all 16 variables of an (atom, channel) in the registers of one lane: the polynomial of
// the contraction is evaluated where the product left its variables.  A separate contraction launch read and wrote them once
// more and was itself bound by that traffic and its ramp (3 000 atoms, 96 channels, fp64: 34 + 21 us for the two launches).
//
// A thread block takes 16 atoms (of one species where weights or polynomials depend on it) and WPB column tiles, one per
// wavefront.  Rows come through LDS in pieces of 64 bytes of each of the 256 rows, brought there by loads that bypass the
// registers, two pieces ahead of the matrix instructions; weights come from L2 in operand order (laid out at load), two pieces
// ahead in registers.  Every piece is the same number of loads (finished l repeat their last piece), so that the wait for a
// piece leaves the younger ones in flight.  Bound by the matrix instructions (16 x 16 x 4 in 32 cycles, 64 in double) from a few
// thousand atoms on, by the latency of the pieces below.
#include "smx_kernels.hpp"
#include "smx_poly_body.hpp"

#include <algorithm>

namespace smx {

namespace {

template <typename F> struct MatOp;
template <> struct MatOp<double> {
    typedef double acc_t __attribute__((ext_vector_type(4)));
    // register r of lane group g holds atom ...
    __device__ static int row(int g, int r) { return 4 * r + g; }
    __device__ static acc_t run(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
};
template <> struct MatOp<float> {
    typedef float acc_t __attribute__((ext_vector_type(4)));
    __device__ static int row(int g, int r) { return 4 * g + r; }
    __device__ static acc_t run(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

// The four 16-byte parts of a row's piece lie in LDS in an order that depends on the atom, so that the sixteen lanes that read
// the same part of sixteen atoms meet 256 different bytes, modulo 256.  That does not keep the banks apart: the counters show
// half of the LDS cycles of this read as conflicts, which fits eight lanes to 128 bytes at a time, where two lanes share every
// place.  (The LDS is busy for 6 % of the kernel's cycles at 3 000 atoms and for 15 % at 50 000, conflicts included.)
__device__ __forceinline__ int part_of(int slot, int atom) { return slot ^ ((atom >> 2) & 3); }
// 1 KB of a wavefront from global memory (16 bytes per lane) into LDS at `to` + 16 lane.  In assembly: next to the compiler's
// own form of this load it lets every read of the LDS, and every use of another load, wait for all loads in flight; here the
// loop below waits by count.  The LDS address goes through m0, which the load may read one wait state after the write (s_nop)
// and has read when it is issued; m0 belongs to the compiler and is given back as it was.
__device__ __forceinline__ void load_into_lds(const void* from, unsigned to)
{
    unsigned m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(m0) : "v"(from), "s"(to) : "memory");
}
// all but the N youngest loads have arrived, and every read of the LDS has
template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory"); }

// POLY: linear and contraction (one polynomial per channel, with gradients); else the linear alone.  (With several polynomials
// per channel, values only, a launch of their own came out ahead: the 4 to 9 polynomials of the four atoms of a lane in turn are a
// long chain for the few wavefronts here.)
template <typename F, int WPB, bool POLY, bool SCALED>
__global__ __launch_bounds__(64 * WPB, 2) void k_linear(const LinearParams<F> p)
{
    using Op = MatOp<F>;
    constexpr int V = 16 / (int)sizeof(F), KC = 4 * V;      // elements per 16 bytes, per piece
    constexpr int PIECE = 256 * 64, AHEAD = 2, BUFS = AHEAD + 1;
    constexpr int LOADS = (16 + WPB - 1) / WPB + 4 + (SCALED ? 1 : 0);     // of a wavefront per piece
    typedef F VV __attribute__((ext_vector_type(V)));
    extern __shared__ __align__(16) unsigned char lin_lds[];      // [BUFS][16 (l, m)][16 atoms][64]; later the coefficients
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;

    // Block -> (row tile, column block, output block e): the blocks that share rows are eight apart, on one die.
    const int cols = p.K / (16 * WPB), per = cols * p.num_e_max;
    const int rem = blockIdx.x % (8 * per), tile_index = blockIdx.x / (8 * per) * 8 + rem % 8;
    const int cb = rem / 8 % cols, e = rem / 8 / cols;
    int type = 0, tile = tile_index, seg0 = 0, seg_n = p.num_nodes;
    if (p.perm) {
        const RowTile at = row_tile(p.tstart, p.T, tile_index, lane);
        if (at.type < 0) return;
        type = at.type; tile = at.tile; seg0 = at.seg0; seg_n = at.seg_n;
    } else if (tile * 16 >= seg_n) {
        return;
    }
    // atom a of the tile; beyond the segment the last atom again, whose results are not stored
    auto node_of = [&](int a) {
        const int j = min(tile * 16 + a, seg_n - 1);
        return p.perm ? p.perm[seg0 + j] : j;
    };
    const int ct = cb * WPB + wave;           // column tile of this wavefront
    int steps[4];                             // pieces per l
#pragma unroll
    for (int l = 0; l < 4; ++l) steps[l] = e < p.num_e[l] ? p.inner[l] / KC : 0;
    const int nsteps = max(max(steps[0], steps[1]), max(steps[2], steps[3]));

    // rows into LDS: a load instruction brings 1 KB, the pieces of 16 atoms for one (l, m)
    const F* const from = p.A + (size_t)node_of(lane / 4) * p.a_node_stride + part_of(lane % 4, lane / 4) * V;
    const unsigned lds0 = (unsigned)(unsigned long long)(__attribute__((address_space(3))) unsigned char*)lin_lds;
    constexpr int ROUNDS = (16 + WPB - 1) / WPB;
    int row_lm[ROUNDS], row_off[ROUNDS], row_last[ROUNDS];      // (places left over repeat the last (l, m))
#pragma unroll
    for (int u = 0; u < ROUNDS; ++u) {
        const int lm = min(u * WPB + wave, 15);
        row_lm[u] = lm; row_off[u] = p.row_off[lm];
        row_last[u] = max((lm < 1 ? steps[0] : (lm < 4 ? steps[1] : (lm < 9 ? steps[2] : steps[3]))) - 1, 0);
    }
    auto stage = [&](int c, int slot) {
#pragma unroll
        for (int u = 0; u < ROUNDS; ++u)
            load_into_lds(from + row_off[u] + min(c, row_last[u]) * KC, lds0 + slot * PIECE + row_lm[u] * 1024);
    };
    VV b[BUFS][4], sc[BUFS];      // weights (and factors) of this piece and the AHEAD next ones
    const F* w_lane[4];
#pragma unroll
    for (int l = 0; l < 4; ++l)
        w_lane[l] = p.W + p.w_off[l] + (size_t)type * p.w_type_stride[l] +
                    ((size_t)(min(e, p.num_e[l] - 1) * (p.K / 16) + ct) * (p.inner[l] / KC) * 64 + lane) * V;
    const F* s_lane = SCALED ? p.scale + (size_t)node_of(r16) * p.K + g * V : nullptr;
    auto request = [&](int c, VV (&w)[4], VV& f) {
#pragma unroll
        for (int l = 0; l < 4; ++l) w[l] = *reinterpret_cast<const VV*>(w_lane[l] + (size_t)max(min(c, steps[l] - 1), 0) * 64 * V);
        if constexpr (SCALED) f = *reinterpret_cast<const VV*>(s_lane + c * KC);
    };

    typename Op::acc_t acc[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = {0, 0, 0, 0};
    static_for<0, AHEAD>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        request(min(c, nsteps - 1), b[c], sc[c]);
        stage(min(c, nsteps - 1), c);
    });
    auto step = [&](int c, auto slot_c) {
        constexpr int slot = decltype(slot_c)::value, ahead = (slot + AHEAD) % BUFS;
        // the piece requested AHEAD steps ago is in LDS for everybody after this, and everybody has read the piece of the step
        // before, whose slot the next request overwrites (no __syncthreads: its fence would wait for the younger pieces too)
        wait_loads<(AHEAD - 1) * LOADS>();
#pragma unroll
        for (int l = 0; l < 4; ++l) asm volatile("" : "+v"(b[slot][l]));      // (here, not after the requests below)
        if constexpr (SCALED) asm volatile("" : "+v"(sc[slot]));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        request(min(c + AHEAD, nsteps - 1), b[ahead], sc[ahead]);
        stage(min(c + AHEAD, nsteps - 1), ahead);
        const unsigned char* buf = lin_lds + slot * PIECE + r16 * 64 + part_of(g, r16) * 16;
        static_for<0, 4>([&](auto lc) {
            constexpr int l = decltype(lc)::value;
            if (c < steps[l]) {
                static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    VV a = *reinterpret_cast<const VV*>(buf + q * 1024);
                    if constexpr (SCALED) a *= sc[slot];
#pragma unroll
                    for (int t = 0; t < V; ++t) acc[q] = Op::run(a[t], b[slot][l][t], acc[q]);
                });
            }
        });
        asm volatile("" ::: "memory");
    };
    // BUFS steps a round, so that the registers of a piece are the same ones from its request to its use (steps past the last
    // one multiply nothing), and one way out of the loop, so that the waits need not allow for others
    for (int c = 0; c < nsteps; c += BUFS)
        static_for<0, BUFS>([&](auto sl) { step(c + decltype(sl)::value, sl); });
    wait_loads<0>();      // the pieces requested past the end land before the LDS changes hands

    const int col = ct * 16 + r16;
    int node[4];
    bool live[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int atom = Op::row(g, r);
        node[r] = node_of(atom);
        live[r] = tile * 16 + atom < seg_n;
    }
    if constexpr (!POLY) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (live[r]) {
                F* o = p.out + (size_t)node[r] * p.out_node_stride + (size_t)e * p.K + col;
                static_for<0, 16>([&](auto qc) {
                    constexpr int q = decltype(qc)::value, l = lm_l(q);
                    if (e < p.num_e[l]) o[p.out_off[q]] = acc[q][r];
                });
            }
    }
    if constexpr (POLY) {
        // coefficients of this block's channels: [column tile][16-byte group of monomials][16 channels]
        constexpr int G16 = poly_spec_padded(PolyTable<0>::N) / V;
        __syncthreads();
        {
            const uint4* src = reinterpret_cast<const uint4*>(p.coef) + ((size_t)type * (p.K / 16) + ct) * G16 * 16;
            uint4* dst = reinterpret_cast<uint4*>(lin_lds) + (size_t)wave * G16 * 16;
            for (int t = lane; t < G16 * 16; t += 64) dst[t] = src[t];
        }
        wave_lds_sync();      // a wavefront reads its own column tile only
        const unsigned char* slab = lin_lds + (size_t)wave * G16 * 256 + r16 * 16;
        for (int r = 0; r < 4; ++r) {
            F x[16], gr[16], f = F(0);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                x[q] = r == 0 ? acc[q][0] : (r == 1 ? acc[q][1] : (r == 2 ? acc[q][2] : acc[q][3]));
                gr[q] = F(0);
            }
            const int nd = r == 0 ? node[0] : (r == 1 ? node[1] : (r == 2 ? node[2] : node[3]));
            const bool lv = r == 0 ? live[0] : (r == 1 ? live[1] : (r == 2 ? live[2] : live[3]));
            poly_spec_body<F, 0, 0>(slab, 256, x, gr, f, F(1));
            if (lv) {
                p.M[(size_t)nd * p.K + col] = f;
#pragma unroll
                for (int q = 0; q < 16; ++q) p.M_grad[((size_t)nd * 16 + q) * p.K + col] = gr[q];
            }
        }
    }
}

template <typename F, int WPB, bool POLY, bool SCALED>
hipError_t launch_linear_t(const LinearParams<F>& p, hipStream_t s)
{
    size_t lds = 3 * (size_t)256 * 64;
    if (POLY) lds = std::max(lds, (size_t)WPB * poly_spec_padded(kPolyTableLen[0]) * 16 * sizeof(F));
    const long tiles = ((long)p.num_nodes + 15) / 16 + (p.perm ? p.T : 0);
    const long blocks = (tiles + 7) / 8 * 8 * (p.K / (16 * WPB)) * p.num_e_max;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_linear<F, WPB, POLY, SCALED>), dim3((unsigned)blocks), dim3(64 * WPB), lds, s, p);
    return hipGetLastError();
}

}  // namespace

// Column tiles of a block: all that divide evenly, up to four (48 KB of LDS a block: three blocks on a CU).
template <typename F>
hipError_t launch_linear(const LinearParams<F>& p, hipStream_t s)
{
    if (p.num_nodes <= 0) return hipSuccess;
    if (!linear_ok(p.K) || p.T <= 0 || (p.coef && (p.scale || p.num_e_max != 1))) return hipErrorInvalidValue;
    auto go = [&](auto pc, auto sc) -> hipError_t {
        constexpr bool POLY = decltype(pc)::value, SCALED = decltype(sc)::value;
        if (p.K % 64 == 0) return launch_linear_t<F, 4, POLY, SCALED>(p, s);
        if (p.K % 96 == 0) return launch_linear_t<F, 3, POLY, SCALED>(p, s);
        return launch_linear_t<F, 2, POLY, SCALED>(p, s);
    };
    if (p.coef) return go(std::true_type{}, std::false_type{});
    return p.scale ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

#ifndef SMX_LINEAR_PART
#error "define SMX_LINEAR_PART (0: double, 1: float)"
#endif
#if SMX_LINEAR_PART == 0
template hipError_t launch_linear<double>(const LinearParams<double>&, hipStream_t);
#else
template hipError_t launch_linear<float>(const LinearParams<float>&, hipStream_t);
#endif

}  // namespace smx
