// The channel-mixing linears of the A-basis, their adjoints, and the symmetric contractions behind them, on the gfx950 matrix
// cores (MACE::compute_A0 / compute_A1, the linears of reverse_A0 / reverse_A1, compute_M0 / compute_M1).
//
// A row tile is 16 atoms with the same (l, m), so the 16 (l, m) of an atom are 16 tiles, and the accumulators of one
// wavefront (16 columns, 16 or 8 of the tiles) hold the variables of an (atom, channel) in the registers of one lane: the polynomial
// of the contraction is evaluated where the product left its variables.  A separate contraction launch read and wrote them once
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

// The (l, m) that a wavefront takes: l = 0 and 3 (set 0) or l = 1 and 2 (set 1), eight each, or all 16 (set 2).
constexpr int slots_of(int set) { return set == 2 ? 16 : 8; }
constexpr int num_l(int set) { return set == 2 ? 4 : 2; }
constexpr int l_of(int set, int j) { return set == 2 ? j : (set == 0 ? 3 * j : 1 + j); }
constexpr int lm_of(int set, int slot) { return set == 2 ? slot : (set == 0 ? (slot == 0 ? 0 : 8 + slot) : 1 + slot); }

// The product of a wavefront: 16 atoms, 16 columns, a set of (l, m).
//   STAGED  (l, m) whose rows the block brings to LDS: those of the set, or all 16
template <typename F, int WPB, int SET, int STAGED, bool SCALED>
struct SetProduct {
    using Op = MatOp<F>;
    static constexpr int V = 16 / (int)sizeof(F), KC = 4 * V;      // elements per 16 bytes, per piece
    static constexpr int PIECE = STAGED * 1024, AHEAD = 2, BUFS = AHEAD + 1, ROUNDS = (STAGED + WPB - 1) / WPB;
    static constexpr int NL = num_l(SET), NS = slots_of(SET);
    static constexpr int LOADS = ROUNDS + NL + (SCALED ? 1 : 0);     // of a wavefront per piece
    typedef F VV __attribute__((ext_vector_type(V)));

    template <typename NodeOf>
    __device__ static __forceinline__ void run(const LinearParams<F>& p, unsigned char* lds, int wave, int lane, int ct, int e, int type,
                                               NodeOf node_of, typename Op::acc_t (&acc)[NS])
    {
        const int r16 = lane & 15, g = lane >> 4;
        int steps[4];                             // pieces per l
#pragma unroll
        for (int l = 0; l < 4; ++l) steps[l] = e < p.num_e[l] ? p.inner[l] / KC : 0;
        const int nsteps = STAGED == 16 ? max(max(steps[0], steps[1]), max(steps[2], steps[3])) : max(steps[l_of(SET, 0)], steps[l_of(SET, 1)]);

        // rows into LDS: a load instruction brings 1 KB, the pieces of 16 atoms for one (l, m)
        const F* const from = p.A + (size_t)node_of(lane / 4) * p.a_node_stride + part_of(lane % 4, lane / 4) * V;
        const unsigned lds0 = (unsigned)(unsigned long long)(__attribute__((address_space(3))) unsigned char*)lds;
        int row_at[ROUNDS], row_off[ROUNDS], row_last[ROUNDS];      // (places left over repeat the last (l, m))
#pragma unroll
        for (int u = 0; u < ROUNDS; ++u) {
            const int at = min(u * WPB + wave, STAGED - 1);
            const int lm = STAGED == 16 ? at : lm_of(SET, at);
            row_at[u] = at; row_off[u] = p.row_off[lm];
            row_last[u] = max((lm < 1 ? steps[0] : (lm < 4 ? steps[1] : (lm < 9 ? steps[2] : steps[3]))) - 1, 0);
        }
        auto stage = [&](int c, int slot) {
#pragma unroll
            for (int u = 0; u < ROUNDS; ++u)
                load_into_lds(from + row_off[u] + min(c, row_last[u]) * KC, lds0 + slot * PIECE + row_at[u] * 1024);
        };
        VV b[BUFS][NL], sc[BUFS];      // weights (and factors) of this piece and the AHEAD next ones
        const F* w_lane[NL];
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int l = l_of(SET, j);
            w_lane[j] = p.W + p.w_off[l] + (size_t)type * p.w_type_stride[l] +
                        ((size_t)(min(e, p.num_e[l] - 1) * (p.K / 16) + ct) * (p.inner[l] / KC) * 64 + lane) * V;
        }
        const F* s_lane = SCALED ? p.scale + (size_t)node_of(r16) * p.K + g * V : nullptr;
        auto request = [&](int c, VV (&w)[NL], VV& f) {
#pragma unroll
            for (int j = 0; j < NL; ++j)
                w[j] = *reinterpret_cast<const VV*>(w_lane[j] + (size_t)max(min(c, steps[l_of(SET, j)] - 1), 0) * 64 * V);
            if constexpr (SCALED) f = *reinterpret_cast<const VV*>(s_lane + c * KC);
        };
#pragma unroll
        for (int q = 0; q < NS; ++q) acc[q] = {0, 0, 0, 0};
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
            for (int j = 0; j < NL; ++j) asm volatile("" : "+v"(b[slot][j]));      // (here, not after the requests below)
            if constexpr (SCALED) asm volatile("" : "+v"(sc[slot]));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            request(min(c + AHEAD, nsteps - 1), b[ahead], sc[ahead]);
            stage(min(c + AHEAD, nsteps - 1), ahead);
            const unsigned char* buf = lds + slot * PIECE + r16 * 64 + part_of(g, r16) * 16;
            static_for<0, NL>([&](auto jc) {
                constexpr int j = decltype(jc)::value, l = l_of(SET, j);
                if (c < steps[l]) {
                    static_for<0, NS>([&](auto qc) {
                        constexpr int q = decltype(qc)::value, lm = lm_of(SET, q);
                        if constexpr (lm_l(lm) == l) {
                            VV a = *reinterpret_cast<const VV*>(buf + (STAGED == 16 ? lm : q) * 1024);
                            if constexpr (SCALED) a *= sc[slot];
#pragma unroll
                            for (int t = 0; t < V; ++t) acc[q] = Op::run(a[t], b[slot][j][t], acc[q]);
                        }
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
    }
};

// POLY: linear and contraction (one polynomial per channel, with gradients); else the linear alone.  (With several polynomials
// per channel, values only, a launch of their own came out ahead: the 4 to 9 polynomials of the four atoms of a lane in turn are a
// long chain for the few wavefronts here.)
//
// A wavefront takes half of the (l, m), eight tiles: with all 16, a few thousand atoms give the SIMDs one or two wavefronts each,
// and 3 000 atoms with 96 channels (1 128 wavefronts, 1 024 SIMDs) twice the time of an even share.  Half the registers also
// leaves room for more blocks, whose stores and first loads then go on under the products of others (those were 20 to 25 % of the
// time each).  All 16, and now, us: 3 000 atoms, 96 channels, double, with a contraction 51 / 42, without 42 / 32; 20 011 atoms,
// single 133 / 111 and 108 / 96; 24 999 atoms, 128 channels, double, without 302 / 268.  Without the contraction the halves are
// blocks of their own, which stage the rows of their half only.  With it both are in one block, and trade variables through LDS.
// Many atoms whose channels are multiples of 64 keep all 16 (l, m) (SPLIT false) with a contraction behind them, where a block of
// halves stages rows for half the columns, and in single precision without one and without factors: rules in launch_linear.
// Three wavefronts per SIMD with halves and a contraction: at 172 registers instead of 168 there were two, and an evaluation of
// 3 000 atoms, 96 channels, double took 462 us instead of 449 (four column tiles in double spill two registers for it).
template <typename F, int WPB, bool POLY, bool SCALED, bool SPLIT>
__global__ __launch_bounds__(64 * WPB, POLY && SPLIT ? 3 : 2) void k_linear(const LinearParams<F> p)
{
    using Op = MatOp<F>;
    constexpr int V = 16 / (int)sizeof(F);
    constexpr int CT = POLY && SPLIT ? WPB / 2 : WPB, SETS = POLY || !SPLIT ? 1 : 2;      // column tiles, blocks for the sets
    extern __shared__ __align__(16) unsigned char lin_lds[];      // [BUFS][8 or 16 (l, m)][16 atoms][64]; later the coefficients
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;

    // Block -> (row tile, column block, output block e, set): the blocks that share rows are eight apart, on one die.
    const int cols = p.K / (16 * CT), per = cols * p.num_e_max * SETS;
    const int rem = blockIdx.x % (8 * per), tile_index = blockIdx.x / (8 * per) * 8 + rem % 8;
    const int cb = rem / 8 % cols, e = rem / 8 / cols % p.num_e_max;
    const int set = !SPLIT ? 2 : (POLY ? wave & 1 : rem / 8 / cols / p.num_e_max);
    int type = 0, tile = tile_index, seg0 = 0, seg_n = p.num_nodes;
    if (p.perm) {
        const RowTile at = row_tile(p.tstart, p.T, tile_index, lane);
        if (at.type < 0) return;
        type = at.type; tile = at.tile; seg0 = at.seg0; seg_n = at.seg_n;
    } else if (tile * 16 >= seg_n) {
        return;
    }
    if (!POLY && SPLIT && (set == 0 ? e >= p.num_e[0] && e >= p.num_e[3] : e >= p.num_e[1] && e >= p.num_e[2])) return;
    // atom a of the tile; beyond the segment the last atom again, whose results are not stored
    auto node_of = [&](int a) {
        const int j = min(tile * 16 + a, seg_n - 1);
        return p.perm ? p.perm[seg0 + j] : j;
    };
    const int tile_in_block = POLY && SPLIT ? wave >> 1 : wave, ct = cb * CT + tile_in_block, col = ct * 16 + r16;      // column tile, column
    typename Op::acc_t acc[SPLIT ? 8 : 16];
    if constexpr (!SPLIT) SetProduct<F, WPB, 2, 16, SCALED>::run(p, lin_lds, wave, lane, ct, e, type, node_of, acc);
    else if (set == 0) SetProduct<F, WPB, 0, POLY ? 16 : 8, SCALED>::run(p, lin_lds, wave, lane, ct, e, type, node_of, acc);
    else SetProduct<F, WPB, 1, POLY ? 16 : 8, SCALED>::run(p, lin_lds, wave, lane, ct, e, type, node_of, acc);

    int node[4];
    bool live[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int atom = Op::row(g, r);
        node[r] = node_of(atom);
        live[r] = tile * 16 + atom < seg_n;
    }
    if constexpr (!POLY) {
        auto store = [&](auto set_c) {
            constexpr int SET = decltype(set_c)::value;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (live[r]) {
                    F* o = p.out + (size_t)node[r] * p.out_node_stride + (size_t)e * p.K + col;
                    static_for<0, slots_of(SET)>([&](auto qc) {
                        constexpr int q = decltype(qc)::value, lm = lm_of(SET, q), l = lm_l(lm);
                        if (e < p.num_e[l]) o[p.out_off[lm]] = acc[q][r];
                    });
                }
        };
        if constexpr (!SPLIT) store(std::integral_constant<int, 2>{});
        else if (set == 0) store(std::integral_constant<int, 0>{});
        else store(std::integral_constant<int, 1>{});
    }
    if constexpr (POLY) {
        // With halves, the two wavefronts of a column tile trade variables: the one ends with all 16 of a lane's atoms 0 and 1, the
        // other with those of atoms 2 and 3.
        constexpr int ATOMS = SPLIT ? 2 : 4;
        F x[ATOMS][16];
        if constexpr (SPLIT) {
            F* const mine = reinterpret_cast<F*>(lin_lds) + (size_t)wave * 16 * 64 + lane;
            const F* const other = reinterpret_cast<const F*>(lin_lds) + (size_t)(wave ^ 1) * 16 * 64 + lane;
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                mine[(2 * q) * 64] = set == 0 ? acc[q][2] : acc[q][0];
                mine[(2 * q + 1) * 64] = set == 0 ? acc[q][3] : acc[q][1];
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const F here = set == 0 ? acc[q][t] : acc[q][2 + t], there = other[(2 * q + t) * 64];
                    x[t][lm_of(0, q)] = set == 0 ? here : there;
                    x[t][lm_of(1, q)] = set == 0 ? there : here;
                }
        } else {
#pragma unroll
            for (int q = 0; q < 16; ++q)
#pragma unroll
                for (int t = 0; t < 4; ++t) x[t][q] = acc[q][t];
        }
        // coefficients of this block's channels: [column tile][16-byte group of monomials][16 channels]
        constexpr int G16 = poly_spec_padded(PolyTable<0>::N) / V;
        __syncthreads();
        {
            const uint4* src = reinterpret_cast<const uint4*>(p.coef) + ((size_t)type * (p.K / 16) + cb * CT) * G16 * 16;
            uint4* dst = reinterpret_cast<uint4*>(lin_lds);
            for (int t = tid; t < CT * G16 * 16; t += 64 * WPB) dst[t] = src[t];
        }
        __syncthreads();
        const unsigned char* slab = lin_lds + (size_t)tile_in_block * G16 * 256 + r16 * 16;
        const int first = SPLIT && set == 1 ? 2 : 0;
#pragma unroll 1
        for (int t = 0; t < ATOMS; ++t) {
            F v[16], gr[16], f = F(0);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                v[q] = t == 0 ? x[0][q] : (t == 1 ? x[1][q] : (t == 2 ? x[ATOMS - 2][q] : x[ATOMS - 1][q]));
                gr[q] = F(0);
            }
            const int r = first + t;
            const int nd = r == 0 ? node[0] : (r == 1 ? node[1] : (r == 2 ? node[2] : node[3]));
            const bool lv = r == 0 ? live[0] : (r == 1 ? live[1] : (r == 2 ? live[2] : live[3]));
            poly_spec_body<F, 0, 0>(slab, 256, v, gr, f, F(1));
            if (lv) {
                p.M[(size_t)nd * p.K + col] = f;
#pragma unroll
                for (int q = 0; q < 16; ++q) p.M_grad[((size_t)nd * 16 + q) * p.K + col] = gr[q];
            }
        }
    }
}

template <typename F, int WPB, bool POLY, bool SCALED, bool SPLIT = true>
hipError_t launch_linear_t(const LinearParams<F>& p, hipStream_t s)
{
    constexpr int CT = POLY && SPLIT ? WPB / 2 : WPB;
    size_t lds = 3 * (size_t)(POLY || !SPLIT ? 16 : 8) * 1024;
    if (POLY) lds = std::max({lds, (size_t)CT * poly_spec_padded(kPolyTableLen[0]) * 16 * sizeof(F), (size_t)WPB * 16 * 64 * sizeof(F)});
    const long tiles = ((long)p.num_nodes + 15) / 16 + (p.perm ? p.T : 0);
    const long blocks = (tiles + 7) / 8 * 8 * (p.K / (16 * CT)) * p.num_e_max * (POLY || !SPLIT ? 1 : 2);
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_linear<F, WPB, POLY, SCALED, SPLIT>), dim3((unsigned)blocks), dim3(64 * WPB), lds, s, p);
    return hipGetLastError();
}

}  // namespace

// Column tiles of a block: all that divide evenly, up to four (24 KB of LDS a block, 48 KB with all (l, m)); with a contraction
// two, each with both halves of the (l, m), or four without halves.
template <typename F>
hipError_t launch_linear(const LinearParams<F>& p, hipStream_t s)
{
    if (p.num_nodes <= 0) return hipSuccess;
    if (!linear_ok(p.K) || p.T <= 0 || (p.coef && (p.scale || p.num_e_max != 1))) return hipErrorInvalidValue;
    if constexpr (sizeof(F) == 4) {
        if (linear32_ok(p)) return launch_linear32(p, s);
    }
    const long whole = ((long)p.num_nodes + 15) / 16 * (p.K / 64);      // blocks of four column tiles, all (l, m)
    if (p.coef) {
        // Blocks with all (l, m) once there are enough to even out over 256 CUs, which hold two (double) or three at a time: A1 of
        // layers l <= 1 at 128 channels, halves / all: double 3 000 atoms 107 / 119 us, 9 000 276 / 305, 12 000 373 / 329,
        // 24 999 770 / 710; single 3 000 62 / 68, 4 500 95 / 100, 6 000 118 / 106, 50 000 830 / 735.
        if (p.K % 64 == 0 && whole > (sizeof(F) == 8 ? 1152 : 640)) return launch_linear_t<F, 4, true, false, false>(p, s);
        return launch_linear_t<F, 4, true, false>(p, s);
    }
    auto go = [&](auto sc) -> hipError_t {
        constexpr bool SCALED = decltype(sc)::value;
        if constexpr (sizeof(F) == 4 && !SCALED) {
            // Single precision without factors keeps all (l, m) over many atoms: the weights are read half as often.  Halves / all,
            // us: adjoint of A1 (output blocks), l <= 1, 128 channels 1 000 atoms 23 / 28, 2 000 42 / 38, 6 000 114 / 104, 50 000
            // 894 / 775, 64 channels 6 000 40 / 40, 8 000 51 / 48; A1 (longer sums) 128 channels 4 500 82 / 87, 6 000 98 / 91,
            // 50 000 779 / 705, 64 channels 8 000 40 / 40, 12 000 58 / 56; A0 and its adjoint 128 channels 8 000 57 / 68, 15 000
            // 103 / 101, 50 000 340 / 331, 64 channels 25 000 54 / 60, 35 000 80 / 81, 50 000 121 / 115.  With factors halves win
            // at every size (50 000 atoms 295 / 303), and in double (50 000 atoms, 96 channels 384 / 435; A0 24 999 atoms, 128
            // channels 277 / 317), and in columns of 96 (50 000 atoms 222 / 236).
            const int inner = std::max({p.inner[0], p.inner[1], p.inner[2], p.inner[3]});
            if (p.K % 64 == 0 && whole > (p.num_e_max > 1 ? 384 : (inner > p.K ? 640 : 2048))) return launch_linear_t<F, 4, false, false, false>(p, s);
        }
        if (p.K % 64 == 0) return launch_linear_t<F, 4, false, SCALED>(p, s);
        if (p.K % 96 == 0) return launch_linear_t<F, 3, false, SCALED>(p, s);
        return launch_linear_t<F, 2, false, SCALED>(p, s);
    };
    return p.scale ? go(std::true_type{}) : go(std::false_type{});
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
