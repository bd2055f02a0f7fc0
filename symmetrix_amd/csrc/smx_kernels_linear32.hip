// The channel-mixing linears of the A-basis, their adjoints and the contractions behind them in single precision at multiples of 96
// and 128 channels, on the bf16 matrix instructions (smx_kernels_linear.hip has the other ones, and says what a row tile and a set of
// (l, m) are).
//
// A number of 24 bits is the sum of three bf16 numbers of 8 bits each, rounded to nearest, exactly:  x = x0 + x1 + x2.  Of the nine
// products of two such numbers the six with indices up to 2 in sum are formed, exactly, and added in single precision; what is left
// out is x1 w2 + x2 w1 + x2 w2, with |x1| <= 2^-8 and |x2| <= 2^-17 of the leading bit of x: up to 1.002 2^-24 of the product.
// Both operands are multiplied by 2^24 first, so that the parts of every number down to the smallest one are normal numbers, and the sums by
// 2^-48.  Numbers above 2^103, infinities, NaN and sums above 2^80 end in an infinity or NaN for it: such sums are formed again, in
// single precision as they are (plain_sums).  Evaluations without and with that, us: 96 channels 20 011 atoms 1 331 / 1 333, 128 channels,
// l <= 2 3 000 1 433 / 1 435, 50 000 15 470 / 15 460.  v_mfma_f32_16x16x32_bf16 does 32 terms of a sum in 16 cycles, the single-precision
// instruction 4 in 32: six of them take 96 cycles for what took 256, and they round the sum six times instead of eight.  Error of
// the sums against 64 bits (2-norm, relative; the single-precision instruction / this): A0 96 channels 1.7e-7 / 1.2e-7, A1 128
// channels, l <= 1 3.3e-7 / 2.7e-7, l <= 2 4.4e-7 / 3.7e-7, adjoints of A1 2.0e-7 / 1.5e-7 and 2.1e-7 / 1.7e-7.
//
// A thread block takes 16 atoms (of one species where weights or polynomials depend on it), 16 or 32 columns per wavefront, and eight
// (l, m) per wavefront: l = 0 and 3 or l = 1 and 2.  Rows come from memory in pieces of 32 terms, into registers one piece ahead;
// every thread splits some of them and leaves the three parts in LDS in operand order (three pieces of 1 KB for an (l, m)), where
// all wavefronts read them: 3 KB for 12 matrix instructions, 64 of the 128 bytes per cycle of a CU.  Weights are split and laid out at
// load, and come from L2, one l ahead in registers.
//
// Bound by memory and by what does not overlap: of 230 us for A0 at 50 000 atoms, 128 channels (820 MB in and out; a copy of as much
// takes 160) 76 are matrix instructions, 25 the split, which the vector pipe does not do beside them, and loads and stores alone take
// 120 and 100.  Rows two pieces ahead (242 us), all of them at once (262), operands one (l, m) ahead (235), 16-byte stores by the
// transposed product (236) and two places in LDS (240) gave nothing where three blocks share a CU.
#include "smx_kernels.hpp"
#include "smx_poly_body.hpp"

#include <algorithm>

namespace smx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPiece = 32;       // terms of a sum per matrix instruction
constexpr float kBack = 1.0f / (kSplitScale * kSplitScale);

// the three parts of eight numbers
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&part)[3])
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f32x2 rest = {x[2 * j], x[2 * j + 1]};
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const bf16x2 h = __builtin_convertvector(rest, bf16x2);
            part[s][2 * j] = h[0]; part[s][2 * j + 1] = h[1];
            if (s < 2) rest -= __builtin_convertvector(h, f32x2);
        }
    }
}
// every LDS operation of the wavefront is done, and all wavefronts are here (__syncthreads would wait for the requested rows too)
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The eight (l, m) of a set: l = 0 and 3 (set 0) or l = 1 and 2 (set 1).
constexpr int l_of(int set, int j) { return set == 0 ? 3 * j : 1 + j; }
constexpr int lm_of(int set, int slot) { return set == 0 ? (slot == 0 ? 0 : 8 + slot) : 1 + slot; }
__device__ __forceinline__ int lm_of_slot(int set, int slot) { return set == 0 ? (slot == 0 ? 0 : 8 + slot) : 1 + slot; }
constexpr int slots_of_l(int set, int j) { return 2 * l_of(set, j) + 1; }

// The sums of a wavefront: 16 atoms, 32 columns, a set of (l, m).  STAGED: (l, m) that the block brings to LDS, those of the set or all
template <int WAVES, int COLS, int STAGED, int SET, bool SCALED>
struct SplitProduct {
    // With both sets in a block there is one block on a CU, which keeps two places for pieces and reads operands one (l, m) ahead (A1 and
    // its contraction, l <= 1, 50 000 atoms 577 us against 663); else other blocks work meanwhile.
    static constexpr bool DEEP = STAGED == 16;
    static constexpr int PLACES = DEEP ? 2 : 1;
    static constexpr int ROUNDS = (STAGED + WAVES - 1) / WAVES;
    template <typename NodeOf>
    __device__ static __forceinline__ void run(const LinearParams<float>& p, unsigned char* lds, int wave, int lane, int ct, int e, int type,
                                               NodeOf node_of, f32x4 (&acc)[8][COLS])
    {
        const int r16 = lane & 15, g = lane >> 4;
        int steps[4];                             // pieces per l
#pragma unroll
        for (int l = 0; l < 4; ++l) steps[l] = e < p.num_e[l] ? p.inner[l] / kPiece : 0;
        const int nsteps = STAGED == 16 ? max(max(steps[0], steps[1]), max(steps[2], steps[3])) : max(steps[l_of(SET, 0)], steps[l_of(SET, 1)]);

        // what this thread brings: eight terms of an atom's row for some (l, m)
        const int node = node_of(r16);
        const float* from[ROUNDS];
        int pieces[ROUNDS];
#pragma unroll
        for (int u = 0; u < ROUNDS; ++u) {
            const int at = u * WAVES + wave, lm = STAGED == 16 ? min(at, 15) : lm_of_slot(SET, min(at, 7));
            from[u] = p.A + (size_t)node * p.a_node_stride + p.row_off[lm] + 8 * g;
            pieces[u] = at >= STAGED ? 0 : (lm < 1 ? steps[0] : (lm < 4 ? steps[1] : (lm < 9 ? steps[2] : steps[3])));
        }
        const float* factor = SCALED ? p.scale + (size_t)node * p.K + 8 * g : nullptr;
        f32x4 x[ROUNDS][2], sc[2];
        // (pieces behind the last one: that one again, so that the number of loads in flight is the same everywhere)
        auto request = [&](int c) {
#pragma unroll
            for (int u = 0; u < ROUNDS; ++u) {
                const f32x4* row = reinterpret_cast<const f32x4*>(from[u] + max(min(c, pieces[u] - 1), 0) * kPiece);
                x[u][0] = row[0]; x[u][1] = row[1];
            }
            if constexpr (SCALED) {
                const f32x4* f = reinterpret_cast<const f32x4*>(factor + min(c, nsteps - 1) * kPiece);
                sc[0] = f[0]; sc[1] = f[1];
            }
        };
        auto leave = [&](int c) {
#pragma unroll
            for (int u = 0; u < ROUNDS; ++u)
                if (c < pieces[u]) {
                    float v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = x[u][j / 4][j % 4] * (SCALED ? sc[j / 4][j % 4] * kSplitScale : kSplitScale);
                    bf16x8 part[3];
                    split8(v, part);
                    unsigned char* to = lds + c % PLACES * (STAGED * 3072) + (u * WAVES + wave) * 3072 + lane * 16;
#pragma unroll
                    for (int s = 0; s < 3; ++s) *reinterpret_cast<bf16x8*>(to + s * 1024) = part[s];
                }
        };
        // weights of the two l of the set, 3 KB per column tile and piece
        const unsigned short* w_lane[2];
        unsigned w_tile[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int l = l_of(SET, j);
            w_tile[j] = (unsigned)(p.inner[l] / kPiece) * 1536;
            w_lane[j] = p.W_split + 3 * (p.w_off[l] + (size_t)type * p.w_type_stride[l]) +
                        (size_t)(min(e, p.num_e[l] - 1) * (p.K / 16) + COLS * ct) * w_tile[j] + lane * 8;
        }
        bf16x8 w[2][COLS][3];
        auto weights = [&](auto jc, int c) {
            constexpr int j = decltype(jc)::value;
            const int at = max(min(c, steps[l_of(SET, j)] - 1), 0);
#pragma unroll
            for (int t = 0; t < COLS; ++t)
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    w[j][t][s] = *reinterpret_cast<const bf16x8*>(w_lane[j] + t * w_tile[j] + (size_t)at * 1536 + s * 512);
        };
        auto product = [&](auto jc, int c) {
            constexpr int j = decltype(jc)::value, first = j == 0 ? 0 : slots_of_l(SET, 0), last = first + slots_of_l(SET, j) - 1;
            if (c >= steps[l_of(SET, j)]) return;
            const unsigned char* const buf = lds + c % PLACES * (STAGED * 3072);
            bf16x8 a[PLACES][3];      // the rows of this (l, m), and of the next
            auto fetch = [&](auto qc) {
                constexpr int q = decltype(qc)::value;
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    a[q % PLACES][s] = *reinterpret_cast<const bf16x8*>(buf + (STAGED == 16 ? lm_of(SET, q) : q) * 3072 + s * 1024 + lane * 16);
            };
            if constexpr (DEEP) fetch(std::integral_constant<int, first>{});
            static_for<first, last + 1>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if constexpr (!DEEP) fetch(qc);
                else if constexpr (q < last) fetch(std::integral_constant<int, q + 1>{});
                // the small products first
                static_for<0, 6>([&](auto oc) {
                    constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, iw[6] = {0, 2, 1, 0, 1, 0}, o = decltype(oc)::value;
#pragma unroll
                    for (int t = 0; t < COLS; ++t)
                        acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q % PLACES][ia[o]], w[j][t][iw[o]], acc[q][t], 0, 0, 0);
                });
                if constexpr (DEEP) {
                    if constexpr (q < last) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 6 * COLS, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        };
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int t = 0; t < COLS; ++t) acc[q][t] = f32x4{0, 0, 0, 0};
        using J0 = std::integral_constant<int, 0>;
        using J1 = std::integral_constant<int, 1>;
        request(0);
        asm volatile("" ::: "memory");      // (in this order, in which they are waited for)
        weights(J0{}, 0);
        asm volatile("" ::: "memory");
        // (weights, then rows, in the order in which they are waited for: a wait for the younger would be one for the older too)
        if constexpr (DEEP) {
            leave(0);
            request(1);
            for (int c = 0; c < nsteps; ++c) {
                lds_barrier();        // this piece is there, and everybody has read the one before
                weights(J1{}, c);
                asm volatile("" ::: "memory");
                product(J0{}, c);
                asm volatile("" ::: "memory");
                if (c + 1 < nsteps) leave(c + 1);
                weights(J0{}, c + 1);
                asm volatile("" ::: "memory");
                request(c + 2);
                asm volatile("" ::: "memory");
                product(J1{}, c);
            }
        } else {
            for (int c = 0; c < nsteps; ++c) {
                leave(c);
                weights(J1{}, c);
                asm volatile("" ::: "memory");
                request(c + 1);
                lds_barrier();
                product(J0{}, c);
                weights(J0{}, c + 1);
                product(J1{}, c);
                lds_barrier();        // everybody has read this piece
            }
        }
    }
};

// The sums of a wavefront as SplitProduct leaves them, scaled back; those that are not finite as products in single precision.
template <int COLS, int SET, bool SCALED, typename NodeOf>
__device__ __forceinline__ void plain_sums(const LinearParams<float>& p, int lane, int ct, int e, int type, NodeOf node_of, f32x4 (&acc)[8][COLS])
{
    float none[4] = {0.0f, 0.0f, 0.0f, 0.0f};      // NaN if a sum is not finite
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int t = 0; t < COLS; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                none[r] = fmaf(acc[q][t][r], 0.0f, none[r]);
                acc[q][t][r] *= kBack;
            }
    const float sum4 = (none[0] + none[1]) + (none[2] + none[3]);
    if (__builtin_expect(!__any(sum4 != sum4), 1)) return;
    static_for<0, 8>([&](auto qc) {
        constexpr int q = decltype(qc)::value, lm = lm_of(SET, q), l = lm_l(lm);
        if (e >= p.num_e[l]) return;
        static_for<0, COLS>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            // (weights in operand order: four k at a time, 64 numbers for 16 columns)
            const float* w = p.W + p.w_off[l] + (size_t)type * p.w_type_stride[l] + (size_t)(e * (p.K / 16) + COLS * ct + t) * p.inner[l] * 16 + (lane & 15) * 4;
            f32x4 sum = {0, 0, 0, 0};
#pragma unroll 1
            for (int k = 0; k < p.inner[l]; k += 4) {
                const f32x4 w4 = *reinterpret_cast<const f32x4*>(w + k * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const size_t node = (size_t)node_of(4 * (lane >> 4) + r);
                    f32x4 x4 = *reinterpret_cast<const f32x4*>(p.A + node * p.a_node_stride + p.row_off[lm] + k);
                    if constexpr (SCALED) {
                        const f32x4 f = *reinterpret_cast<const f32x4*>(p.scale + node * p.K + k);
#pragma unroll
                        for (int j = 0; j < 4; ++j) x4[j] *= f[j];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) sum[r] = fmaf(x4[j], w4[j], sum[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (!(fabsf(acc[q][t][r]) <= 3.402823466e38f)) acc[q][t][r] = sum[r];
        });
    });
}

// POLY: linear and contraction (one polynomial per channel, with gradients), both sets of (l, m) in a block; else the linear alone, a
// block per set.
template <int TILES, int COLS, bool POLY, bool SCALED>
__global__ __launch_bounds__(64 * TILES * (POLY ? 2 : 1), 2) void k_linear32(const LinearParams<float> p)
{
    constexpr int WAVES = TILES * (POLY ? 2 : 1), SETS = POLY ? 1 : 2;      // blocks for the sets
    extern __shared__ __align__(16) unsigned char lin_lds[];      // [8 or 16 (l, m)][3 parts][64 lanes][16 bytes]; later the coefficients
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;

    // Block -> (row tile, column block, output block e, set): the blocks that share rows are eight apart, on one die.
    const int cols = p.K / (16 * COLS * TILES), per = cols * p.num_e_max * SETS;
    const int rem = blockIdx.x % (8 * per), tile_index = blockIdx.x / (8 * per) * 8 + rem % 8;
    const int cb = rem / 8 % cols, e = rem / 8 / cols % p.num_e_max;
    const int set = POLY ? wave / TILES : rem / 8 / cols / p.num_e_max;
    int type = 0, tile = tile_index, seg0 = 0, seg_n = p.num_nodes;
    if (p.perm) {
        const RowTile at = row_tile(p.tstart, p.T, tile_index, lane);
        if (at.type < 0) return;
        type = at.type; tile = at.tile; seg0 = at.seg0; seg_n = at.seg_n;
    } else if (tile * 16 >= seg_n) {
        return;
    }
    if (!POLY && (set == 0 ? e >= p.num_e[0] && e >= p.num_e[3] : e >= p.num_e[1] && e >= p.num_e[2])) return;
    // atom a of the tile; beyond the segment the last atom again, whose results are not stored
    auto node_of = [&](int a) {
        const int j = min(tile * 16 + a, seg_n - 1);
        return p.perm ? p.perm[seg0 + j] : j;
    };
    const int tile_in_block = wave % TILES, ct = cb * TILES + tile_in_block, col = ct * 16 * COLS + r16;      // columns of the wavefront, the first one of this lane
    f32x4 acc[8][COLS];
    if (set == 0) {
        SplitProduct<WAVES, COLS, POLY ? 16 : 8, 0, SCALED>::run(p, lin_lds, wave, lane, ct, e, type, node_of, acc);
        plain_sums<COLS, 0, SCALED>(p, lane, ct, e, type, node_of, acc);
    } else {
        SplitProduct<WAVES, COLS, POLY ? 16 : 8, 1, SCALED>::run(p, lin_lds, wave, lane, ct, e, type, node_of, acc);
        plain_sums<COLS, 1, SCALED>(p, lane, ct, e, type, node_of, acc);
    }

    int node[4];
    bool live[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        node[r] = node_of(4 * g + r);
        live[r] = tile * 16 + 4 * g + r < seg_n;
    }
    if constexpr (!POLY) {
        auto store = [&](auto set_c) {
            constexpr int SET = decltype(set_c)::value;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (live[r]) {
                    float* o = p.out + (size_t)node[r] * p.out_node_stride + (size_t)e * p.K + col;
                    static_for<0, 8>([&](auto qc) {
                        constexpr int q = decltype(qc)::value, lm = lm_of(SET, q);
                        if (e < p.num_e[lm_l(lm)]) {
#pragma unroll
                            for (int t = 0; t < COLS; ++t) o[p.out_off[lm] + 16 * t] = acc[q][t][r];
                        }
                    });
                }
        };
        if (set == 0) store(std::integral_constant<int, 0>{});
        else store(std::integral_constant<int, 1>{});
    } else {
        static_assert(COLS == 2, "the exchange below");
        // The two wavefronts of the same columns trade variables: the one ends with all 16 of a lane's atoms 0 and 1, the other with
        // those of atoms 2 and 3.
        float x[2][2][16];       // [columns][atom][variable]
        float* const mine = reinterpret_cast<float*>(lin_lds) + (size_t)wave * 32 * 64 + lane;
        const float* const other = reinterpret_cast<const float*>(lin_lds) + (size_t)(set == 0 ? wave + TILES : wave - TILES) * 32 * 64 + lane;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                mine[(4 * q + 2 * c) * 64] = set == 0 ? acc[q][c][2] : acc[q][c][0];
                mine[(4 * q + 2 * c + 1) * 64] = set == 0 ? acc[q][c][3] : acc[q][c][1];
            }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const float here = set == 0 ? acc[q][c][t] : acc[q][c][2 + t], there = other[(4 * q + 2 * c + t) * 64];
                    x[c][t][lm_of(0, q)] = set == 0 ? here : there;
                    x[c][t][lm_of(1, q)] = set == 0 ? there : here;
                }
        // coefficients of this block's channels: [column tile][16-byte group of monomials][16 channels]
        constexpr int G16 = poly_spec_padded(PolyTable<0>::N) / 4;
        __syncthreads();
        {
            const uint4* src = reinterpret_cast<const uint4*>(p.coef) + ((size_t)type * (p.K / 16) + cb * 2 * TILES) * G16 * 16;
            uint4* dst = reinterpret_cast<uint4*>(lin_lds);
            for (int t = tid; t < 2 * TILES * G16 * 16; t += 64 * WAVES) dst[t] = src[t];
        }
        __syncthreads();
        const int first = set == 0 ? 0 : 2;
#pragma unroll 1
        for (int u = 0; u < 4; ++u) {
            const int c = u >> 1, t = u & 1;
            float v[16], gr[16], f = 0.0f;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                v[q] = u == 0 ? x[0][0][q] : (u == 1 ? x[0][1][q] : (u == 2 ? x[1][0][q] : x[1][1][q]));
                gr[q] = 0.0f;
            }
            const int r = first + t;
            const int nd = r == 0 ? node[0] : (r == 1 ? node[1] : (r == 2 ? node[2] : node[3]));
            const bool lv = r == 0 ? live[0] : (r == 1 ? live[1] : (r == 2 ? live[2] : live[3]));
            const unsigned char* slab = lin_lds + (size_t)(2 * tile_in_block + c) * G16 * 256 + r16 * 16;
            poly_spec_body<float, 0, 0>(slab, 256, v, gr, f, 1.0f);
            if (lv) {
                const int k = col + 16 * c;
                p.M[(size_t)nd * p.K + k] = f;
#pragma unroll
                for (int q = 0; q < 16; ++q) p.M_grad[((size_t)nd * 16 + q) * p.K + k] = gr[q];
            }
        }
    }
}

template <int TILES, int COLS, bool POLY, bool SCALED>
hipError_t launch_linear32_t(const LinearParams<float>& p, hipStream_t s)
{
    constexpr int WAVES = TILES * (POLY ? 2 : 1);
    size_t lds = (size_t)(POLY ? 2 * 16 : 8) * 3072;
    if (POLY) lds = std::max({lds, (size_t)2 * TILES * poly_spec_padded(kPolyTableLen[0]) * 16 * sizeof(float), (size_t)WAVES * 32 * 64 * sizeof(float)});
    const long tiles = ((long)p.num_nodes + 15) / 16 + (p.perm ? p.T : 0);
    const long blocks = (tiles + 7) / 8 * 8 * (p.K / (16 * COLS * TILES)) * p.num_e_max * (POLY ? 1 : 2);
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    if (lds > 64 * 1024) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_linear32<TILES, COLS, POLY, SCALED>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL((k_linear32<TILES, COLS, POLY, SCALED>), dim3((unsigned)blocks), dim3(64 * WAVES), lds, s, p);
    return hipGetLastError();
}

}  // namespace

// 128 channels (and multiples): linears without a contraction always, so that from 512 atoms on, where the launches of row tiles begin, the
// sums of an atom do not depend on the size of the system.  A contraction behind sums of K terms from 2 048 atoms; 96 channels from 1 024.
// k_linear / this, us, launches alone: 128 channels A0 600 atoms 9.9 / 10.7, 1 500 15.8 / 12.4, 10 000 66 / 44, 50 000 310 / 230; its
// adjoint (factors) 600 12.5 / 12.1, 50 000 331 / 250; adjoint of A1, l <= 1, 600 17 / 13, 3 000 52 / 39, 50 000 702 / 532; A1 and its
// contraction, l <= 1, 1 100 36.7 / 38.8, 3 000 54.8 / 41.1, 10 000 145 / 127, 30 000 406 / 357; l = 0 1 100 18.7 / 23.5, 3 000 27.5 /
// 25.1, 20 000 143 / 135.  96 channels adjoint of A0 600 10.1 / 10.9, 1 500 13.9 / 11.6, 3 000 18.9 / 15.2, 20 000 83 / 77; adjoint of
// A1 20 000 206 / 197; with a contraction there is one block of six wavefronts on a CU: 20 000 98 / 110, so that stays with k_linear.
// 64 channels: adjoint of A1 20 000 106 / 106, A1 and its contraction 30 000 145 / 160; 32: 700 7.3 / 7.6: no gain.
bool linear32_ok(const LinearParams<float>& p)
{
    if (!p.W_split) return false;
    // (a contraction of few atoms behind short sums waits for itself here)
    if (p.coef) return p.K % 128 == 0 && (p.split_nodes >= 2048 || p.inner[1] > p.K);
    return p.K % 128 == 0 || (p.K % 96 == 0 && p.split_nodes >= 1024);
}
hipError_t launch_linear32(const LinearParams<float>& p, hipStream_t s)
{
    if (p.K % 32 != 0 || p.T <= 0 || !p.W_split || (p.coef && (p.scale || p.num_e_max != 1 || p.K % 128 != 0))) return hipErrorInvalidValue;
    if (p.coef) return launch_linear32_t<4, 2, true, false>(p, s);
    auto go = [&](auto sc) -> hipError_t {
        constexpr bool SCALED = decltype(sc)::value;
        if (p.K % 128 != 0) return launch_linear32_t<3, 2, false, SCALED>(p, s);
        // 16 columns per wavefront where there are few blocks, us, 16 / 32: A0 600 atoms 10.7 / 12.1, 1 500 12.4 / 13.5, 3 000 17.9 / 18.6,
        // 6 000 28.4 / 26.5, 50 000 242 / 230; adjoint of A1, l <= 1 (three output blocks), 600 13.0 / 14.0, 3 000 42 / 39.
        const long blocks = ((long)p.num_nodes + 15) / 16 * 2 * p.num_e_max;
        if (blocks <= 384) return launch_linear32_t<8, 1, false, SCALED>(p, s);
        return launch_linear32_t<4, 2, false, SCALED>(p, s);
    };
    return p.scale ? go(std::true_type{}) : go(std::false_type{});
}

}  // namespace smx
