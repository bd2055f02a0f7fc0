// Edge kernels for gfx950, general form: fused harmonics + radial splines +
// receiver-segmented aggregation, and the analytic edge-force adjoint, for any
// path list (hidden features up to l = 2) and any number of radial tables.
//
// Work decomposition.  The edge list is receiver-sorted (CSR).  A wavefront owns a
// receiver, or one of two or four parts of a receiver's edges where there are few
// receivers; lane j owns channels j, j + 64, ..., so every table or feature load of
// the wavefront is one contiguous run.  Accumulators (NE per channel) live in
// registers for the whole neighbour loop and parts are added in a fixed order: no
// atomics, bit-reproducible.  Edges are taken in chunks of 16: one lane per edge
// forms direction, harmonics and spline interval; then all 64 lanes share the
// entries of the Clebsch-Gordan-contracted harmonics B (and their gradients in the
// adjoint) of a few edges at a time.
//
// How B meets the channels.  An entry of B multiplies the value of every channel, so
// it has to reach all lanes.  Read from LDS as a broadcast it costs 16 to 64 bytes
// of the LDS pipe's 128 bytes per cycle and lane group, 88 entries of three numbers
// per edge for l <= 1: with that the LDS bounded the adjoint (3 300 cycles per edge and
// wavefront in single precision, 5 400 in double).  Now the wavefront holds the block
// of an edge in a few registers, every lane some of its entries, and the instructions
// that use them do the broadcast:
//   single precision  v_mfma_f32_4x4x1_16b: four rows of B times one value per lane in
//                     8 cycles; the block-broadcast field of the instruction (cbsz = 4,
//                     abid = n) takes the four rows from lanes 4n .. 4n+3, and result row
//                     i of channel j lands in register i of lane j, where the vector code
//                     wants it.  (The matrix pipe does not run beside the vector pipe
//                     here; per multiply-add it costs the same as a vector instruction.)
//   double precision  v_fmac_f64 with the row broadcast of its DPP operand (row_newbcast:n),
//                     at the rate of the plain instruction; every 16-lane row holds the
//                     block.
#include "smx_edge_common.hpp"
#include "smx_paths.hpp"

namespace smx {

namespace {

constexpr int kChunk = 16;   // edges whose geometry is formed together
// Harmonics lie in LDS by entry, a chunk's edges side by side: a lane of block_values reads two edges at once.  Entries are 144
// bytes apart, so that lanes at different entries meet different banks.
constexpr int kEdgeStride = kChunk + 2;

template <int N>
using int_c = std::integral_constant<int, N>;

// The paths that a wavefront takes: all of them (SET 0), those of the sender's components up to l2 = 1 (SET 1) or those of l2 = 2
// (SET 2).
template <int LMAXH, int SET>
struct PathSet {
    using PT = Paths<LMAXH>;
    static constexpr bool in(int p) { return SET == 0 || (PT::l2(p) == 2) == (SET == 2); }
    static constexpr int rank(int p)
    {
        int n = 0;
        for (int q = 0; q < p; ++q) n += in(q);
        return n;
    }
    static constexpr int P = rank(PT::P);
    static constexpr int path(int j)
    {
        for (int p = 0; p < PT::P; ++p)
            if (in(p) && rank(p) == j) return p;
        return -1;
    }
    static constexpr int Q0 = SET == 2 ? 4 : 0, Q1 = SET == 1 ? 4 : PT::NLM;     // components of the sender
};

// Which entry of B[path][m][m2] (and of its two tangential derivatives) every lane and register holds.
//   matrix form:  register g / 16, lanes 4 (g % 16) + i hold row 4 tile + i of group g; a group is one matrix
//                 instruction: (path, row tile, inner index).  Forward: rows m, inner m2; adjoint: rows 3 m2 + t, inner m;
//                 odd rows behind them in DPP form, v = odd_off + m.
//   DPP form:     register v / 16, lane v % 16 of every row: v = 3 (entry_off + m n2 + m2) + t, forward entry_off + m n2 + m2
// CP: a path of the constant harmonic (l1 = 0, so l = l2) has none where it couples like with like only, as an equivariant model
// does: u[m2] = c d[m2] needs no product with a block and has no tangential part.  10 of the 88 rows and columns for l <= 1, 35 of
// 243 for l <= 2; the constants go into the adjoint rows as they are loaded, or into the sums as they are stored.  Evaluations of
// 50 000 atoms, l <= 1, single: 17.2 -> 16.9 ms; 24 999 atoms, double: 12.5 -> 12.1 ms; 3 000 atoms, l <= 2: 1 720 -> 1 658 us.
// In DPP form the pairs that the selection rules exclude have none either (6 of the 78 others, 28 of 208): the adjoint is bound by
// its instructions, us: 24 999 atoms, l <= 1 3 882 -> 3 843, 3 000 463 -> 454; l <= 2, 128 channels 3 000 1 369 -> 1 306, 64 channels
// 5 000 1 184 -> 1 101.  (The matrix form multiplies four rows at a time, of which never all are excluded.)
template <int LMAXH, bool BWD, bool MATRIX, bool CP, int SET>
struct BlockLayout {
    using PT = Paths<LMAXH>;
    static constexpr bool in(int p) { return PathSet<LMAXH, SET>::in(p) && !(CP && PT::l1(p) == 0); }     // whether the path has entries in the block
    static constexpr int n2(int p) { return 2 * PT::l2(p) + 1; }
    static constexpr int nm(int p) { return 2 * PT::l(p) + 1; }
    static constexpr int rows(int p) { return BWD ? 3 * n2(p) : nm(p); }
    static constexpr int inner(int p) { return BWD ? nm(p) : n2(p); }
    // The ninth of nine rows has no tile of its own: a multiply-add with a lane broadcast costs half of a matrix instruction.
    static constexpr bool odd(int p) { return MATRIX && BWD && in(p) && rows(p) > 4 && rows(p) % 4 == 1; }
    static constexpr int tiles(int p) { return in(p) ? (odd(p) ? rows(p) / 4 : (rows(p) + 3) / 4) : 0; }
    static constexpr int odd_off(int p)
    {
        int n = 0;
        for (int q = 0; q < p; ++q) n += odd(q) ? inner(q) : 0;
        return n;
    }
    static constexpr int entry_off(int p)
    {
        int n = 0;
        for (int q = 0; q < p; ++q) n += in(q) ? pairs(q, nm(q), 0) : 0;
        return n;
    }
    static constexpr bool has(int p, int m, int m2) { return MATRIX || !CP || components_couple(PT::l(p), m, PT::l1(p), PT::l2(p), m2); }
    // pairs of path p before (m, m2) that have an entry
    static constexpr int pairs(int p, int m, int m2)
    {
        int n = 0;
        for (int b = 0; b < m * n2(p) + m2; ++b) n += has(p, b / n2(p), b % n2(p));
        return n;
    }
    static constexpr int entry(int p, int m, int m2) { return entry_off(p) + pairs(p, m, m2); }
    static constexpr int tile_off(int p)
    {
        int n = 0;
        for (int q = 0; q < p; ++q) n += tiles(q);
        return n;
    }
    static constexpr int group_off(int p)
    {
        int n = 0;
        for (int q = 0; q < p; ++q) n += tiles(q) * inner(q);
        return n;
    }
    static constexpr int group(int p, int tile, int in) { return group_off(p) + tile * inner(p) + in; }
    static constexpr int TILES = tile_off(PT::P);
    static constexpr int REGS = MATRIX ? (group_off(PT::P) + 15) / 16 : (entry_off(PT::P) * (BWD ? 3 : 1) + 15) / 16;
    static constexpr int LANES = MATRIX ? 64 : 16;      // lanes that hold different entries
    static constexpr int ODD_REGS = (odd_off(PT::P) + 15) / 16;      // of the odd rows: every 16 lanes hold the same
    static constexpr int NV = REGS * LANES + ODD_REGS * 16;
    struct Table {
        short entry[NV];           // index into B, or -1: zero
        unsigned char comp[NV];    // 0: B, 1, 2: derivative along the first, second tangent
    };
    static constexpr Table make()
    {
        Table t{};
        for (int v = 0; v < NV; ++v) { t.entry[v] = -1; t.comp[v] = 0; }
        for (int p = 0; p < PT::P; ++p) {
            if (!in(p)) continue;
            const int N2 = n2(p), NM = nm(p), bo = PT::boff(p), eo = entry_off(p), go = group_off(p), R = rows(p), IN = inner(p);
            if (MATRIX) {
                if (odd(p))
                    for (int in = 0; in < IN; ++in) {
                        const int v = REGS * LANES + odd_off(p) + in;
                        t.entry[v] = (short)(bo + in * N2 + (R - 1) / 3);
                        t.comp[v] = (unsigned char)((R - 1) % 3);
                    }
                for (int tl = 0; tl < tiles(p); ++tl)
                    for (int in = 0; in < IN; ++in)
                        for (int i = 0; i < 4; ++i) {
                            const int row = 4 * tl + i;
                            if (row >= R) continue;
                            const int v = (go + tl * IN + in) * 4 + i;
                            t.entry[v] = (short)(BWD ? bo + in * N2 + row / 3 : bo + row * N2 + in);
                            t.comp[v] = (unsigned char)(BWD ? row % 3 : 0);
                        }
            } else {
                for (int b = 0, e = eo; b < NM * N2; ++b)
                    for (int c = 0; has(p, b / N2, b % N2) && c < (BWD ? 3 : 1); ++c) {
                        const int v = BWD ? 3 * e + c : e;
                        if (c == (BWD ? 2 : 0)) ++e;
                        t.entry[v] = (short)(bo + b);
                        t.comp[v] = (unsigned char)c;
                    }
            }
        }
        return t;
    }
};
template <int LMAXH, bool BWD, bool MATRIX, bool CP, int SET>
__device__ const typename BlockLayout<LMAXH, BWD, MATRIX, CP, SET>::Table block_table = BlockLayout<LMAXH, BWD, MATRIX, CP, SET>::make();

// LDS of a block: the coefficients of the block entries, then a part for each of its four wavefronts
template <typename F, int LMAXH, bool BWD, bool CP, int SET>
struct EdgeLds {
    using BL = BlockLayout<LMAXH, BWD, kMatrix<F>, CP, SET>;
    static constexpr int NY = BWD ? 48 : 16;     // harmonics (and their two tangential derivatives) of an edge
    // edges whose blocks are in LDS at a time: as many as leave room for two thread blocks on a CU
    static constexpr int SUB = BL::NV * (int)sizeof(F) > 2600 ? 2 : (BL::NV * (int)sizeof(F) > 1000 ? 4 : 8);
    static constexpr size_t lists = ((size_t)BL::NV * (2 * sizeof(double) + sizeof(int)) + 15) / 16 * 16;
    static constexpr size_t y_bytes = (size_t)NY * kEdgeStride * sizeof(double);
    static constexpr size_t frame_bytes = BWD ? (size_t)kChunk * 10 * sizeof(double) : 0;    // direction over r, tangents
    static constexpr size_t head_bytes = (size_t)(kChunk + 1) * (sizeof(double) + 2 * sizeof(int)) + 8;  // x, table row, sender row
    static constexpr size_t sum_bytes = BWD ? (size_t)kChunk * 4 * sizeof(F) : 0;
    static constexpr size_t block_bytes = (size_t)SUB * BL::NV * sizeof(F);
    static constexpr size_t per_wave = (y_bytes + frame_bytes + head_bytes + sum_bytes + block_bytes + 15) / 16 * 16;
    static constexpr size_t total = lists + 4 * per_wave;
};

// Three sums over the 64 lanes at once: on return the lanes of row 0 hold the first, of row 2 the second, of rows 1 and 3
// the third (a fixed tree).  Two values swap halves of the wavefront and are added, which sums both over the halves.
template <typename F>
__device__ __forceinline__ F wave_sum3(F s, F g1, F g2)
{
    F zero = g2;
    swap_halves(s, g1);
    const F a = s + g1;              // rows 0, 1: s; rows 2, 3: g1
    swap_halves(g2, zero);
    F x = a, y = g2 + zero;          // every row: g2
    swap_rows(x, y);
    return row_sum_strided<1>(x + y);
}

// The coefficients of the block entries: value v = c0 Y[o0] + c1 Y[o1] (an entry of a real coupling has at most two terms;
// a file with longer ones sets more_terms and pays for a loop), copied to LDS once per thread block.
template <int LMAXH, bool BWD, bool MATRIX, bool CP, int SET, typename F>
__device__ __forceinline__ void block_lists(const AggParams<F>& a, double* coef, int* offs)
{
    using BL = BlockLayout<LMAXH, BWD, MATRIX, CP, SET>;
    for (int v = threadIdx.x; v < BL::NV; v += 256) {
        const int b = block_table<LMAXH, BWD, MATRIX, CP, SET>.entry[v], comp = block_table<LMAXH, BWD, MATRIX, CP, SET>.comp[v];
        double c0 = 0.0, c1 = 0.0;
        int o0 = 0, o1 = 0;
        if (b >= 0) {
            const int s0 = a.B_start[b], s1 = a.B_start[b + 1];
            if (s1 > s0) { c0 = a.B_c[s0]; o0 = a.B_lm1[s0]; }
            if (s1 > s0 + 1) { c1 = a.B_c[s0 + 1]; o1 = a.B_lm1[s0 + 1]; }
        }
        coef[2 * v] = c0; coef[2 * v + 1] = c1;
        offs[v] = (comp * 16 + o0) * kEdgeStride | ((comp * 16 + o1) * kEdgeStride) << 16;
    }
}
template <int LMAXH, bool BWD, bool MATRIX, bool CP, int SET, typename F, int SUB>
__device__ __forceinline__ void block_values(const AggParams<F>& a, const double* coef, const int* offs, const double* Yt, int ns,
                                             F* vals, int lane)
{
    using BL = BlockLayout<LMAXH, BWD, MATRIX, CP, SET>;
#pragma unroll
    for (int j = 0; j < (BL::NV + 63) / 64; ++j) {
        const int v = lane + 64 * j;
        if (BL::NV % 64 == 0 || v < BL::NV) {
            const double2 c = *reinterpret_cast<const double2*>(coef + 2 * v);
            const int o = offs[v], o0 = o & 0xffff, o1 = o >> 16;
            static_assert(SUB % 2 == 0, "pairs of edges");
#pragma unroll
            for (int le = 0; le < SUB; le += 2) {      // (past the chunk's last edge: numbers nobody reads)
                const double2 y0 = *reinterpret_cast<const double2*>(Yt + o0 + le), y1 = *reinterpret_cast<const double2*>(Yt + o1 + le);
                vals[le * BL::NV + v] = (F)(c.x * y0.x + c.y * y1.x);
                vals[(le + 1) * BL::NV + v] = (F)(c.x * y0.y + c.y * y1.y);
            }
        }
    }
    if (a.more_terms) {
        for (int v = lane; v < BL::NV; v += 64) {
            const int b = block_table<LMAXH, BWD, MATRIX, CP, SET>.entry[v];
            if (b < 0) continue;
            for (int le = 0; le < ns; ++le) {
                const double* y = Yt + block_table<LMAXH, BWD, MATRIX, CP, SET>.comp[v] * 16 * kEdgeStride + le;
                double s = 0.0;
                for (int t = a.B_start[b]; t < a.B_start[b + 1]; ++t) s += a.B_c[t] * y[a.B_lm1[t] * kEdgeStride];
                vals[le * BL::NV + v] = (F)s;
            }
        }
    }
}

// Wavefronts that share the paths of a receiver (PathSet).  For l <= 2 a lane holds 71 sums or adjoint rows, and in the adjoint 36
// sums at the components of the sender: too many registers for two wavefronts per SIMD in double precision, and one alone issues a vector instruction
// every six cycles at best.  Two sets of paths hold 40 and 31 rows and read different table entries, so that only the geometry and
// the sums over channels are formed twice.  us, l <= 2, one / two sets: sums of 3 000 atoms double, 128 channels 669 / 586, 64
// channels 366 / 307, single 309 / 291, 172 / 153, 10 000 atoms 943 / 910; adjoint double 1 280 / 1 024, 656 / 528, 400 atoms
// 209 / 148.  Single precision adjoint: sets leave registers for two channels per lane, 652 / 614 (128 channels); up to 64 channels
// there is one in any case, and one set is the better: 346 / 389.
template <typename F, int LMAXH, int CPL, bool BWD>
constexpr int path_sets() { return LMAXH == 2 && (!BWD || sizeof(F) == 8 || CPL == 2) ? 2 : 1; }

// Thread blocks per CU (wavefronts per SIMD) the kernels are compiled for: 168 or 256 registers a lane (none spilled, except 8 by the
// adjoint of l <= 2 in double precision for files that couple outside the selection rules)
template <typename F, int LMAXH, int CPL, bool BWD>
constexpr int agg_blocks()
{
    return sizeof(F) == 4 && CPL == 1 && (LMAXH == 1 || (LMAXH == 2 && !BWD)) ? 3 : 2;
}

// ---------------------------------------------------------------------------
// Forward: out[i, lme, k] = sum over the edges of R_path(r)[k] sum_m2 B[lme, m2] H[sender, m2, k].
// Bound by the coefficient rows: P splines of 16 (32) bytes per channel and edge, 10 KB (20 KB) per edge and wavefront at
// l <= 1, of the 64 bytes per cycle that a CU's vector cache hands out.
template <typename F, int LMAXH, int CPL, bool CP, int SET>
__device__ __forceinline__ void agg_fwd(const AggParams<F>& a, const int parts, const int block, unsigned char* smem)
{
    constexpr bool MX = kMatrix<F>;
    using PT = Paths<LMAXH>;
    using PS = PathSet<LMAXH, SET>;
    using BL = BlockLayout<LMAXH, false, MX, CP, SET>;
    using EL = EdgeLds<F, LMAXH, false, CP, SET>;
    constexpr int NE = PT::NE, P = PS::P, NLM = PT::NLM, SUB = EL::SUB;
    constexpr int W = P <= 5 ? P : 5;     // splines of the ring: requested W paths ahead
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double* coef = reinterpret_cast<double*>(smem);
    int* offs = reinterpret_cast<int*>(coef + 2 * BL::NV);
    unsigned char* base = smem + EL::lists + (size_t)wave * EL::per_wave;
    double* Yt = reinterpret_cast<double*>(base);                                 // [16][kEdgeStride]
    F* vals = reinterpret_cast<F*>(base + EL::y_bytes);                           // [SUB][NV]
    double* xs = reinterpret_cast<double*>(base + EL::y_bytes + EL::block_bytes); // [kChunk + 1]
    int* rows = reinterpret_cast<int*>(xs + kChunk + 1);                          // [kChunk + 1]
    int* grows = rows + kChunk + 1;                                               // [kChunk + 1]

    block_lists<LMAXH, false, MX, CP, SET>(a, coef, offs);
    __syncthreads();

    const unsigned K = (unsigned)a.K;
    // One-dimensional grid, channel group fastest: consecutive blocks go to the dies in turn, so a die only ever
    // works on the channel groups congruent to its number and its L2 holds that share of the spline table alone
    // (half of it at two groups of 64 channels).
    const int groups = (a.K + 64 * CPL - 1) / (64 * CPL);
    const int cgroup = block % groups;
    const int unit = (block / groups) * 4 + wave;
    const int i = __builtin_amdgcn_readfirstlane(unit / parts), part = unit - i * parts;
    const bool real = i < a.num_nodes;
    unsigned k[CPL];
    bool active[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ch = (cgroup * CPL + c) * 64 + lane;
        active[c] = ch < a.K;
        k[c] = active[c] ? (unsigned)ch : 0u;      // lanes beyond the last channel repeat channel 0 and store nothing
    }
    int e0 = 0, e1 = 0, ti = 0;
    if (real) {
        const int b = a.first_neigh[i], n = a.first_neigh[i + 1] - b;
        e0 = b + (int)((long)n * part / parts); e1 = b + (int)((long)n * (part + 1) / parts);
        ti = a.node_types[i];
    }
    e0 = __builtin_amdgcn_readfirstlane(e0); e1 = __builtin_amdgcn_readfirstlane(e1);

    f32x4 tile[MX ? CPL : 1][MX ? BL::TILES : 1];
    F acc[MX ? 1 : CPL][MX ? 1 : NE];
    F same[CPL][NLM];               // CP in matrix form: the sums of the paths of the constant harmonic
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        if constexpr (MX) {
#pragma unroll
            for (int q = 0; q < NLM; ++q) same[c][q] = F(0);
#pragma unroll
            for (int q = 0; q < BL::TILES; ++q) tile[c][q] = f32x4{0, 0, 0, 0};
        } else {
#pragma unroll
            for (int q = 0; q < NE; ++q) acc[c][q] = F(0);
        }
    }

    Vec<F, 4> cf[CPL][W];
    F H[CPL][NLM], Hn[CPL][NLM];
    unsigned k16[CPL], ks[CPL];      // byte offsets of this lane's channels in a table row and in a feature row
    auto offsets = [&]() {
#pragma unroll
        for (int c = 0; c < CPL; ++c) { k16[c] = lane_offset(k[c] * 16); ks[c] = lane_offset(k[c] * (unsigned)sizeof(F)); }
    };
    offsets();
    const unsigned row_bytes = PT::P * K * 4 * sizeof(F), sender_bytes = NLM * K * sizeof(F);
    auto request_spline = [&](const char* row, auto rc) {
        constexpr int rank = decltype(rc)::value, path = PS::path(rank);
#pragma unroll
        for (int c = 0; c < CPL; ++c) cf[c][rank % W] = load_spline<F>(row, path, K, k16[c]);
    };
    auto request_sender = [&](int le) {
        const int grow = grows[le];
#pragma unroll
        for (int q = PS::Q0; q < PS::Q1; ++q) {
            const char* part = reinterpret_cast<const char*>(a.Hsrc) + uniform_offset(grow, sender_bytes, q * (K * (unsigned)sizeof(F)));
#pragma unroll
            for (int c = 0; c < CPL; ++c) Hn[c][q] = load_at<F>(part, ks[c]);
        }
    };
    const char* cur = nullptr;      // table row of the edge under way
    for (int eb = e0; eb < e1; eb += kChunk) {
        const int nE = min(kChunk, e1 - eb);
        wave_lds_sync();
        if (lane <= nE) {
            // lane nE: the first edge of the next chunk, whose features are requested at the end of this one
            // (past the last edge of the part: the last one again)
            const int e = min(eb + lane, e1 - 1);
            double r, x;
            int row, grow;
            edge_head(a, e, ti, r, x, row, grow);
            xs[lane] = x; rows[lane] = row; grows[lane] = grow;
            if (lane < nE) {
                const double dx = a.xyz[3 * (size_t)e], dy = a.xyz[3 * (size_t)e + 1], dz = a.xyz[3 * (size_t)e + 2];
                const double inv = rsqrt_pos(dx * dx + dy * dy + dz * dz);
                double Y[16];
                sph_l3(dz * inv, dx * inv, dy * inv, Y);
#pragma unroll
                for (int q = 0; q < 16; ++q) Yt[q * kEdgeStride + lane] = Y[q];
            }
        }
        wave_lds_sync();
        if (eb == e0) {
            cur = uniform_row(a.tabK, rows[0], row_bytes);
            static_for<0, W>([&](auto qc) { request_spline(cur, qc); });
            request_sender(0);
        }
        for (int sb = 0; sb < nE; sb += SUB) {
            const int ns = min(SUB, nE - sb);
            if (sb) wave_lds_sync();
            block_values<LMAXH, false, MX, CP, SET, F, SUB>(a, coef, offs, Yt + sb, ns, vals, lane);
            wave_lds_sync();
            for (int le = sb; le < sb + ns; ++le) {
                offsets();
                const F x = (F)xs[le];
                F B[BL::REGS];
#pragma unroll
                for (int j = 0; j < BL::REGS; ++j) B[j] = vals[(le - sb) * BL::NV + j * BL::LANES + (lane & (BL::LANES - 1))];
#pragma unroll
                for (int c = 0; c < CPL; ++c)
#pragma unroll
                    for (int q = PS::Q0; q < PS::Q1; ++q) H[c][q] = Hn[c][q];
                request_sender(le + 1);
                const char* next = uniform_row(a.tabK, rows[le + 1], row_bytes);
                static_for<0, P>([&](auto pc) {
                    constexpr int j = decltype(pc)::value, p = PS::path(j), l = PT::l(p), l2 = PT::l2(p), n2 = 2 * l2 + 1;
                    constexpr int lme0 = PT::lme(p, 0), es = PT::num_e(l), t0 = BL::tile_off(p), t1 = t0 + BL::tiles(p);
                    F w[CPL][n2];
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        const Vec<F, 4> k4 = cf[c][j % W];
                        const F R = k4.v[0] + x * (k4.v[1] + x * (k4.v[2] + x * k4.v[3]));
#pragma unroll
                        for (int m2 = 0; m2 < n2; ++m2) w[c][m2] = R * H[c][l2 * l2 + m2];
                    }
                    if constexpr (j + W < P) request_spline(cur, int_c<j + W>{}); else request_spline(next, int_c<j % W>{});
                    if constexpr (!BL::in(p)) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m = 0; m < n2; ++m) {
                                F& s = MX ? same[c][l2 * l2 + m] : acc[MX ? 0 : c][MX ? 0 : lme0 + m * es];
                                s += w[c][m];
                            }
                    } else if constexpr (MX) {
                        static_for<0, n2>([&](auto mc) {
                            static_for<0, BL::tiles(p)>([&](auto tc) {
                                constexpr int g = BL::group(p, decltype(tc)::value, decltype(mc)::value), t = BL::tile_off(p) + decltype(tc)::value;
#pragma unroll
                                for (int c = 0; c < CPL; ++c)
                                    tile[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(B[g / 16], w[c][decltype(mc)::value], tile[c][t], 4, g % 16, 0);
                            });
                        });
                    } else {
                        static_for<0, n2>([&](auto mc) {
                            static_for<0, 2 * l + 1>([&](auto rc) {
                                constexpr int v = BL::entry(p, decltype(rc)::value, decltype(mc)::value);
                                if constexpr (BL::has(p, decltype(rc)::value, decltype(mc)::value)) {
#pragma unroll
                                    for (int c = 0; c < CPL; ++c)
                                        fmac_lane<v % 16>(acc[c][lme0 + decltype(rc)::value * es], B[v / 16], w[c][decltype(mc)::value]);
                                }
                            });
                        });
                    }
                    // path by path
                    if constexpr (MX && !BL::in(p)) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m = 0; m < n2; ++m) pin(same[c][l2 * l2 + m]);
                    } else if constexpr (MX) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int t = t0; t < t1; ++t) pin(tile[c][t]);
                        __builtin_amdgcn_sched_group_barrier(0x002, (3 + n2) * CPL, 0);
                        __builtin_amdgcn_sched_group_barrier(0x008, BL::tiles(p) * n2 * CPL, 0);
                    } else {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m = 0; m < 2 * l + 1; ++m) pin(acc[c][lme0 + m * es]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                cur = next;
            }
        }
    }
    // sum lme of channel c of this lane
    auto value = [&](auto pc, auto mc, int c) -> F& {
        constexpr int p = decltype(pc)::value, m = decltype(mc)::value;
        if constexpr (MX && !BL::in(p)) return same[c][PT::l2(p) * PT::l2(p) + m];
        else if constexpr (MX) return reinterpret_cast<F*>(&tile[c][BL::tile_off(p) + m / 4])[m % 4];
        else return acc[c][PT::lme(p, 0) + m * PT::num_e(PT::l(p))];
    };
    auto every = [&](auto&& f) {      // f(lme, channel slot, sum)
        static_for<0, P>([&](auto pc) {
            constexpr int p = PS::path(decltype(pc)::value);
            static_for<0, 2 * PT::l(p) + 1>([&](auto mc) {
                constexpr int q = PT::lme(p, decltype(mc)::value);
#pragma unroll
                for (int c = 0; c < CPL; ++c) f(q, c, value(int_c<p>{}, mc, c));
            });
        });
    };
    // the parts of a receiver lie in one thread block: the upper half of them hands its sums to the lower half, in LDS
    F* half = reinterpret_cast<F*>(smem);
    for (int h = parts >> 1; h >= 1; h >>= 1) {
        __syncthreads();
        // slot of a receiver's part pair: the sums of the units of a block that give, in order
        const int slot = (wave / parts) * h + part % h;
        F* at = half + (size_t)slot * NE * CPL * 64 + lane;
        if (part >= h && part < 2 * h) every([&](int q, int c, F& v) { at[(size_t)(q * CPL + c) * 64] = v; });
        __syncthreads();
        if (part < h) every([&](int q, int c, F& v) { v += at[(size_t)(q * CPL + c) * 64]; });
    }
    if (!real || part != 0) return;
    if constexpr (CP)
        static_for<0, P>([&](auto pc) {
            constexpr int p = PS::path(decltype(pc)::value);
            if constexpr (!BL::in(p))
                static_for<0, 2 * PT::l(p) + 1>([&](auto mc) {
#pragma unroll
                    for (int c = 0; c < CPL; ++c) value(int_c<p>{}, mc, c) *= (F)a.c_same[PT::l(p) * PT::l(p) + decltype(mc)::value];
                });
        });
    every([&](int q, int c, F& v) {
        if (active[c]) a.out[((size_t)i * NE + q) * K + k[c]] = v;
    });
}

template <typename F, int LMAXH, int CPL, bool CP>
__global__ __launch_bounds__(256, (agg_blocks<F, LMAXH, CPL, false>())) void k_agg_fwd(const AggParams<F> a, const int parts)
{
    extern __shared__ __align__(16) unsigned char smem[];
    if constexpr (path_sets<F, LMAXH, CPL, false>() == 1) agg_fwd<F, LMAXH, CPL, CP, 0>(a, parts, blockIdx.x, smem);
    else if (blockIdx.x % 2 == 0) agg_fwd<F, LMAXH, CPL, CP, 1>(a, parts, blockIdx.x / 2, smem);
    else agg_fwd<F, LMAXH, CPL, CP, 2>(a, parts, blockIdx.x / 2, smem);
}

// ---------------------------------------------------------------------------
// Adjoint: per edge force -dE/dxyz_ij (MACE::reverse_A0, mace.cpp:238-269;
// MACE::reverse_Phi1, mace.cpp:531-574) and the adjoint message to the sender
// row (mace.cpp:579-604), staged per edge for the deterministic sender-side sum.
// With more than one channel group or set of paths each writes its share
// of the force to fpart[share][edge][3]; the caller adds the shares up.
//
// The harmonics depend on the direction only, so their gradient is tangential: two components in a frame (t1, t2)
// orthogonal to the direction carry it.  Per path the rows of B, dB.t1, dB.t2 meet the receiver's adjoint first,
// u[m2][t] = sum_m d[m] (B, dB.t1, dB.t2)[m][m2]; with R and R' of the path they add to four sums per m2,
//   message R u[.][0],  R u[.][1],  R u[.][2],  R' u[.][0],
// and only at the end of the edge these meet the sender feature (radial and two tangential forces).
template <typename F, int LMAXH, int CPL, bool CP, int SET>
__device__ __forceinline__ void agg_bwd(const AggParams<F>& a, const int parts, const int block, unsigned char* smem)
{
    constexpr bool MX = kMatrix<F>;
    using PT = Paths<LMAXH>;
    using PS = PathSet<LMAXH, SET>;
    using BL = BlockLayout<LMAXH, true, MX, CP, SET>;
    using EL = EdgeLds<F, LMAXH, true, CP, SET>;
    constexpr int NE = PT::NE, P = PS::P, NLM = PT::NLM, SUB = EL::SUB;
    constexpr int W = P <= 5 ? P : 5;     // splines of the ring: requested W paths ahead
    constexpr auto first_tangential = [](int l2) {
        for (int p = 0; p < PT::P; ++p)
            if (PT::l2(p) == l2 && BL::in(p)) return p;
        return -1;
    };
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double* coef = reinterpret_cast<double*>(smem);
    int* offs = reinterpret_cast<int*>(coef + 2 * BL::NV);
    unsigned char* base = smem + EL::lists + (size_t)wave * EL::per_wave;
    double* Yt = reinterpret_cast<double*>(base);                                 // [3][16][kEdgeStride]: Y, dY.t1, dY.t2
    double* us = reinterpret_cast<double*>(base + EL::y_bytes);                   // [kChunk][10]: xyz / r, t1, t2, -
    F* vals = reinterpret_cast<F*>(base + EL::y_bytes + EL::frame_bytes);         // [SUB][NV]
    F* sums = vals + (size_t)SUB * BL::NV;                                        // [kChunk][4]: radial, t2, t1, (t2)
    double* xs = reinterpret_cast<double*>(base + EL::y_bytes + EL::frame_bytes + EL::block_bytes + EL::sum_bytes);
    int* rows = reinterpret_cast<int*>(xs + kChunk + 1);
    int* grows = rows + kChunk + 1;

    block_lists<LMAXH, true, MX, CP, SET>(a, coef, offs);
    __syncthreads();

    const unsigned K = (unsigned)a.K;
    // one-dimensional grid, channel group fastest (see k_agg_fwd)
    const int groups = (a.K + 64 * CPL - 1) / (64 * CPL);
    const int cgroup = block % groups;
    const int unit = (block / groups) * 4 + wave;
    const int rel = __builtin_amdgcn_readfirstlane(unit / parts), part = unit - rel * parts, i = a.node_begin + rel;
    if (i >= a.num_nodes) return;
    // Lanes beyond the last channel work on channel 0 with a zero adjoint (all their sums are zero) and skip the
    // message store: no branch on the lane's channel inside the edge loop.
    unsigned k[CPL];
    bool active[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ch = (cgroup * CPL + c) * 64 + lane;
        active[c] = ch < a.K;
        k[c] = active[c] ? (unsigned)ch : 0u;
    }
    const int first = a.first_neigh[i], deg = a.first_neigh[i + 1] - first, ti = a.node_types[i];
    const int e0 = __builtin_amdgcn_readfirstlane(first + (int)((long)deg * part / parts));
    const int e1 = __builtin_amdgcn_readfirstlane(first + (int)((long)deg * (part + 1) / parts));
    const bool shares = groups > 1 || SET > 0;
    double* fout = shares ? a.fpart + (size_t)(SET == 2 ? groups + cgroup : cgroup) * 3 * a.num_edges : a.forces;
    const bool add_forces = !shares && a.accumulate_forces;
    if (e0 >= e1) return;

    F d[CPL][NE];
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int q = 0; q < NE; ++q) {
            const F v = a.d_out[((size_t)i * NE + q) * K + k[c]];
            d[c][q] = active[c] ? v : F(0);
        }
    if constexpr (CP)
        static_for<0, P>([&](auto pc) {
            constexpr int p = PS::path(decltype(pc)::value), l = PT::l(p);
            if constexpr (!BL::in(p))
                static_for<0, 2 * l + 1>([&](auto mc) {
                    constexpr int m = decltype(mc)::value, lme = PT::lme(p, m);
#pragma unroll
                    for (int c = 0; c < CPL; ++c) d[c][lme] *= (F)a.c_same[l * l + m];
                });
        });

    Vec<F, 4> cf[CPL][W];
    unsigned k16[CPL], ks[CPL];      // byte offsets of this lane's channels in a table row and in a feature row
    auto offsets = [&]() {
#pragma unroll
        for (int c = 0; c < CPL; ++c) { k16[c] = lane_offset(k[c] * 16); ks[c] = lane_offset(k[c] * (unsigned)sizeof(F)); }
    };
    offsets();
    const unsigned row_bytes = PT::P * K * 4 * sizeof(F), sender_bytes = NLM * K * sizeof(F);
    auto request_spline = [&](const char* row, auto rc) {
        constexpr int rank = decltype(rc)::value, path = PS::path(rank);
#pragma unroll
        for (int c = 0; c < CPL; ++c) cf[c][rank % W] = load_spline<F>(row, path, K, k16[c]);
    };
    const char* cur = nullptr;      // table row of the edge under way
    for (int eb = e0; eb < e1; eb += kChunk) {
        const int nE = min(kChunk, e1 - eb);
        wave_lds_sync();
        if (lane <= nE) {
            // lane nE: the first edge of the next chunk, whose splines are requested at the end of this one
            // (past the last edge of the part: the last one again)
            const int e = min(eb + lane, e1 - 1);
            double r, x;
            int row, grow;
            edge_head(a, e, ti, r, x, row, grow);
            xs[lane] = x; rows[lane] = row; grows[lane] = grow;
            if (lane < nE) {
                EdgeFrame f;
                edge_frame(a.xyz + 3 * (size_t)e, f);
                const double ir = rcp_pos(r);
                // radial direction as the reference forms it: xyz / r with the caller's r
                double* fr = us + lane * 10;
                fr[0] = f.dx * ir; fr[1] = f.dy * ir; fr[2] = f.dz * ir;
                fr[3] = f.t1x; fr[4] = f.t1y; fr[5] = f.t1z; fr[6] = f.t2x; fr[7] = f.t2y; fr[8] = f.t2z;
                double* y = Yt + lane;
                static_for<0, 16>([&](auto lc) {
                    constexpr int lm = decltype(lc)::value;
                    ylm_tangential<lm>(f, y[lm * kEdgeStride], y[(16 + lm) * kEdgeStride], y[(32 + lm) * kEdgeStride]);
                    if constexpr (lm % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // short live ranges
                });
            }
        }
        wave_lds_sync();
        if (eb == e0) {
            cur = uniform_row(a.tabK, rows[0], row_bytes);
            static_for<0, W>([&](auto qc) { request_spline(cur, qc); });
        }
        for (int sb = 0; sb < nE; sb += SUB) {
            const int ns = min(SUB, nE - sb);
            if (sb) wave_lds_sync();
            block_values<LMAXH, true, MX, CP, SET, F, SUB>(a, coef, offs, Yt + sb, ns, vals, lane);
            wave_lds_sync();
            for (int le = sb; le < sb + ns; ++le) {
                offsets();
                const F x = (F)xs[le];
                // the sender row is met at the end of the edge only: requested here, it has the whole edge to arrive
                F H[CPL][NLM];
                {
                    const int grow = grows[le];
#pragma unroll
                    for (int q = PS::Q0; q < PS::Q1; ++q) {
                        const char* part = reinterpret_cast<const char*>(a.Hsrc) + uniform_offset(grow, sender_bytes, q * (K * (unsigned)sizeof(F)));
#pragma unroll
                        for (int c = 0; c < CPL; ++c) H[c][q] = load_at<F>(part, ks[c]);
                    }
                }
                const char* next = uniform_row(a.tabK, rows[le + 1], row_bytes);
                const F* Bp = vals + (size_t)(le - sb) * BL::NV + (lane & (BL::LANES - 1));
                F B[BL::REGS], Bodd[BL::ODD_REGS + 1];
#pragma unroll
                for (int j = 0; j < BL::REGS; ++j) B[j] = Bp[j * BL::LANES];
#pragma unroll
                for (int j = 0; j < BL::ODD_REGS; ++j) Bodd[j] = vals[(size_t)(le - sb) * BL::NV + BL::REGS * BL::LANES + j * 16 + (lane & 15)];
                F V[CPL][NLM][4];     // message, R u.t1, R u.t2, R' u
                if constexpr (!MX) {
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
#pragma unroll
                        for (int q = PS::Q0; q < PS::Q1; ++q) { V[c][q][1] = F(0); V[c][q][2] = F(0); }
                }
                static_for<0, P>([&](auto pc) {
                    constexpr int j = decltype(pc)::value, p = PS::path(j), l = PT::l(p), l2 = PT::l2(p), n2 = 2 * l2 + 1;
                    constexpr int lme0 = PT::lme(p, 0), es = PT::num_e(l);
                    constexpr bool starts = p == PT::first_with_l2(l2);    // the first path of this l2 starts the sums
                    constexpr bool starts_t = p == first_tangential(l2);   // ... of the tangential parts
                    constexpr bool tangential = BL::in(p);
                    F R[CPL], Rd[CPL];
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        // value and derivative by Horner's rule
                        const Vec<F, 4> k4 = cf[c][j % W];
                        const F q1 = k4.v[2] + x * k4.v[3], d1 = q1 + x * k4.v[3], q2 = k4.v[1] + x * q1;
                        R[c] = k4.v[0] + x * q2;
                        Rd[c] = q2 + x * d1;
                    }
                    if constexpr (j + W < P) request_spline(cur, int_c<j + W>{}); else request_spline(next, int_c<j % W>{});
                    if constexpr (!BL::in(p)) {
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m2 = 0; m2 < n2; ++m2) {
                                const F dm = d[c][lme0 + m2 * es];
                                F* s = V[c][l2 * l2 + m2];
                                s[0] = starts ? R[c] * dm : s[0] + R[c] * dm;
                                s[3] = starts ? Rd[c] * dm : s[3] + Rd[c] * dm;
                            }
                    } else if constexpr (MX) {
                        constexpr int T = BL::tiles(p), R3 = BL::rows(p);
                        constexpr bool ODD = BL::odd(p);
                        f32x4 u[CPL][T];
                        F uodd[CPL];
                        static_for<0, 2 * l + 1>([&](auto mc) {
                            constexpr int m = decltype(mc)::value;
                            static_for<0, T>([&](auto tc) {
                                constexpr int t = decltype(tc)::value, g = BL::group(p, t, m);
#pragma unroll
                                for (int c = 0; c < CPL; ++c)
                                    u[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(B[g / 16], d[c][lme0 + m * es],
                                                                                 m == 0 ? f32x4{0, 0, 0, 0} : u[c][t], 4, g % 16, 0);
                            });
                        });
                        if constexpr (ODD) {
#pragma unroll
                            for (int c = 0; c < CPL; ++c) uodd[c] = F(0);
                            static_for<0, 2 * l + 1>([&](auto mc) {
                                constexpr int m = decltype(mc)::value, v = BL::odd_off(p) + m;
#pragma unroll
                                for (int c = 0; c < CPL; ++c) fmac_lane<v % 16>(uodd[c], Bodd[v / 16], d[c][lme0 + m * es]);
                            });
                        }
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m2 = 0; m2 < n2; ++m2) {
                                F* s = V[c][l2 * l2 + m2];
#pragma unroll
                                for (int t = 0; t < 3; ++t) {
                                    const F uv = ODD && 3 * m2 + t == R3 - 1 ? uodd[c] : u[c][(3 * m2 + t) / 4 < T ? (3 * m2 + t) / 4 : 0][(3 * m2 + t) % 4];
                                    s[t] = (t == 0 ? starts : starts_t) ? R[c] * uv : s[t] + R[c] * uv;
                                    if (t == 0) s[3] = starts ? Rd[c] * uv : s[3] + Rd[c] * uv;
                                }
                            }
                    } else {
                        F u0[CPL][n2];
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m2 = 0; m2 < n2; ++m2) u0[c][m2] = F(0);
                        // the tangential sums take R d: no sums per path for them, except where those are fewer than the components
                        // (24 999 atoms 3 843 -> 3 761 us, 3 000 454 -> 450)
                        constexpr bool PER_PATH = 2 * n2 < 2 * l;
                        F ut[CPL][n2][2];
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m2 = 0; m2 < n2; ++m2) ut[c][m2][0] = ut[c][m2][1] = F(0);
                        static_for<0, 2 * l + 1>([&](auto mc) {
                            constexpr int m = decltype(mc)::value;
#pragma unroll
                            for (int c = 0; c < CPL; ++c) {
                                const F dm = d[c][lme0 + m * es], rd = PER_PATH ? dm : R[c] * dm;
                                static_for<0, n2>([&](auto m2c) {
                                    constexpr int m2 = decltype(m2c)::value, v = 3 * BL::entry(p, m, m2);
                                    if constexpr (BL::has(p, m, m2)) {
                                        fmac_lane<v % 16>(u0[c][m2], B[v / 16], dm);
                                        fmac_lane<(v + 1) % 16>(PER_PATH ? ut[c][m2][0] : V[c][l2 * l2 + m2][1], B[(v + 1) / 16], rd);
                                        fmac_lane<(v + 2) % 16>(PER_PATH ? ut[c][m2][1] : V[c][l2 * l2 + m2][2], B[(v + 2) / 16], rd);
                                    }
                                });
                            }
                        });
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int m2 = 0; m2 < n2; ++m2) {
                                F* s = V[c][l2 * l2 + m2];
                                s[0] = starts ? R[c] * u0[c][m2] : s[0] + R[c] * u0[c][m2];
                                s[3] = starts ? Rd[c] * u0[c][m2] : s[3] + Rd[c] * u0[c][m2];
                                if constexpr (PER_PATH) { s[1] += R[c] * ut[c][m2][0]; s[2] += R[c] * ut[c][m2][1]; }
                            }
                    }
                    // path by path
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
#pragma unroll
                        for (int m2 = 0; m2 < n2; ++m2)
#pragma unroll
                            for (int t = 0; t < 4; ++t)
                                if (tangential || t == 0 || t == 3) pin(V[c][l2 * l2 + m2][t]);
                    if constexpr (MX && BL::in(p)) {
                        // the matrix instructions of a path together: every change between the pipes costs about four cycles
                        __builtin_amdgcn_sched_group_barrier(0x008, BL::tiles(p) * (2 * l + 1) * CPL, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 100, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                cur = next;
                F srad = F(0), g1 = F(0), g2 = F(0);
#pragma unroll
                for (int c = 0; c < CPL; ++c)
#pragma unroll
                    for (int q = PS::Q0; q < PS::Q1; ++q) {
                        const F h = H[c][q];
                        srad += V[c][q][3] * h; g1 += V[c][q][1] * h; g2 += V[c][q][2] * h;
                    }
                if (a.msg) {
                    char* part[NLM];
#pragma unroll
                    for (int q = PS::Q0; q < PS::Q1; ++q)
                        part[q] = reinterpret_cast<char*>(a.msg) + uniform_offset(eb + le - (int)a.msg_edge_begin, sender_bytes, q * (K * (unsigned)sizeof(F)));
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
                        if (active[c]) {
#pragma unroll
                            for (int q = PS::Q0; q < PS::Q1; ++q) store_stream(reinterpret_cast<F*>(part[q] + lane_offset(ks[c])), V[c][q][0]);
                        }
                }
                // sums over the channels of the wavefront, in the feature precision (a fixed tree)
                const F s = wave_sum3(srad, g1, g2);
                if ((lane & 15) == 0) sums[le * 4 + (lane >> 4)] = s;
            }
        }
        wave_lds_sync();
        // the forces of the chunk, put together in double
        if (lane < nE) {
            const double* fr = us + lane * 10;
            const double sr = (double)sums[lane * 4], G2 = (double)sums[lane * 4 + 1], G1 = (double)sums[lane * 4 + 2];
            const double fx = -(fr[0] * sr + fr[3] * G1 + fr[6] * G2);
            const double fy = -(fr[1] * sr + fr[4] * G1 + fr[7] * G2);
            const double fz = -(fr[2] * sr + fr[5] * G1 + fr[8] * G2);
            double* f = fout + 3 * (size_t)(eb + lane);
            if (add_forces) { f[0] += fx; f[1] += fy; f[2] += fz; }
            else { f[0] = fx; f[1] = fy; f[2] = fz; }
        }
    }
}

template <typename F, int LMAXH, int CPL, bool CP>
__global__ __launch_bounds__(256, (agg_blocks<F, LMAXH, CPL, true>())) void k_agg_bwd(const AggParams<F> a, const int parts)
{
    extern __shared__ __align__(16) unsigned char smem[];
    if constexpr (path_sets<F, LMAXH, CPL, true>() == 1) agg_bwd<F, LMAXH, CPL, CP, 0>(a, parts, blockIdx.x, smem);
    else if (blockIdx.x % 2 == 0) agg_bwd<F, LMAXH, CPL, CP, 1>(a, parts, blockIdx.x / 2, smem);
    else agg_bwd<F, LMAXH, CPL, CP, 2>(a, parts, blockIdx.x / 2, smem);
}

template <typename F, int LMAXH, int CPL, bool BWD, bool CP>
hipError_t launch_agg_t(const AggParams<F>& p, hipStream_t s)
{
    constexpr int sets = path_sets<F, LMAXH, CPL, BWD>();
    const int groups = (p.K + 64 * CPL - 1) / (64 * CPL) * sets;
    if (BWD && groups > 1 && !p.fpart) return hipErrorInvalidValue;
    if (!BWD && (p.node_begin != 0 || p.msg_edge_begin != 0)) return hipErrorInvalidValue;
    if (p.node_begin < 0 || p.node_begin > p.num_nodes) return hipErrorInvalidValue;
    const long nodes = p.num_nodes - p.node_begin;
    // the forward sums depend on the parts in their last bits: a call with ghost nodes is split as one without
    // (sets of paths not counted: 1 000 atoms, l <= 2, 128 channels, single 106 / 210 us, counted 129 / 218)
    const int parts = agg_parts<BWD>((long)(BWD ? nodes : p.split_nodes) * (groups / sets));
    const long blocks = (nodes * parts + 3) / 4 * groups;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    dim3 grid((unsigned)blocks);
    void (*kern)(const AggParams<F>, const int);
    size_t lds = sets == 1 ? EdgeLds<F, LMAXH, BWD, CP, 0>::total
                           : std::max(EdgeLds<F, LMAXH, BWD, CP, 1>::total, EdgeLds<F, LMAXH, BWD, CP, 2>::total);
    if constexpr (BWD) kern = k_agg_bwd<F, LMAXH, CPL, CP>;
    else {
        kern = k_agg_fwd<F, LMAXH, CPL, CP>;
        const size_t handed = parts > 1 ? (size_t)2 * Paths<LMAXH>::NE * CPL * 64 * sizeof(F) : 0;   // two givers per block
        lds = lds > handed ? lds : handed;
    }
    if (lds > 64 * 1024) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, p, parts);
    return hipGetLastError();
}

// Channels per lane: two where the registers hold them and more than one half-empty wavefront would result otherwise.
template <typename F, int LMAXH, bool BWD>
int agg_cpl(int K)
{
    return (LMAXH == 0 || (sizeof(F) == 4 && BWD)) && K > 64 ? 2 : 1;
}

template <typename F, int LMAXH, int CPL, bool BWD>
hipError_t launch_agg_cp(const AggParams<F>& p, hipStream_t s)
{
    // (scalar features come here with couplings that the scalar kernels do not take)
    if constexpr (LMAXH > 0) {
        if (p.selected) return launch_agg_t<F, LMAXH, CPL, BWD, true>(p, s);
    }
    return launch_agg_t<F, LMAXH, CPL, BWD, false>(p, s);
}
template <typename F, int LMAXH, bool BWD>
hipError_t launch_agg_sel(const AggParams<F>& p, hipStream_t s)
{
    if constexpr (LMAXH == 0 || (sizeof(F) == 4 && BWD)) {
        if (agg_cpl<F, LMAXH, BWD>(p.K) == 2) return launch_agg_cp<F, LMAXH, 2, BWD>(p, s);
    }
    return launch_agg_cp<F, LMAXH, 1, BWD>(p, s);
}

}  // namespace

template <typename F>
hipError_t launch_agg_fwd(int L_max_H, const AggParams<F>& p, hipStream_t s)
{
    if (L_max_H == 0) return launch_agg_sel<F, 0, false>(p, s);
    if (L_max_H == 1) return launch_agg_sel<F, 1, false>(p, s);
    if (L_max_H == 2) return launch_agg_sel<F, 2, false>(p, s);
    return hipErrorInvalidValue;
}
template <typename F>
hipError_t launch_agg_bwd(int L_max_H, const AggParams<F>& p, hipStream_t s)
{
    if (L_max_H == 0) return launch_agg_sel<F, 0, true>(p, s);
    if (L_max_H == 1) return launch_agg_sel<F, 1, true>(p, s);
    if (L_max_H == 2) return launch_agg_sel<F, 2, true>(p, s);
    return hipErrorInvalidValue;
}
template <typename F, int LMAXH>
int agg_bwd_shares(int K)
{
    if (agg_cpl<F, LMAXH, true>(K) == 2) return (K + 127) / 128 * path_sets<F, LMAXH, 2, true>();
    return (K + 63) / 64 * path_sets<F, LMAXH, 1, true>();
}
template <typename F>
int agg_bwd_groups(int L_max_H, int K)
{
    return L_max_H == 0 ? agg_bwd_shares<F, 0>(K) : (L_max_H == 1 ? agg_bwd_shares<F, 1>(K) : agg_bwd_shares<F, 2>(K));
}
// This file is compiled four times (SMX_EDGE_PART = 0..3), one object per
// precision and direction, so that the instantiations build in parallel.
#ifndef SMX_EDGE_PART
#error "define SMX_EDGE_PART (0: fwd double + helpers, 1: fwd float, 2: bwd double, 3: bwd float)"
#endif
#if SMX_EDGE_PART == 0
template hipError_t launch_agg_fwd<double>(int, const AggParams<double>&, hipStream_t);
#elif SMX_EDGE_PART == 1
template hipError_t launch_agg_fwd<float>(int, const AggParams<float>&, hipStream_t);
#elif SMX_EDGE_PART == 2
template hipError_t launch_agg_bwd<double>(int, const AggParams<double>&, hipStream_t);
template int agg_bwd_groups<double>(int, int);
#else
template hipError_t launch_agg_bwd<float>(int, const AggParams<float>&, hipStream_t);
template int agg_bwd_groups<float>(int, int);
#endif

#if SMX_EDGE_PART == 0

// ---------------------------------------------------------------------------
namespace {
template <typename F, int N>
__device__ __forceinline__ Vec<F, N> ldv(const F* p)
{
    return *reinterpret_cast<const Vec<F, N>*>(p);
}
// of an array that is read once
template <typename F, int N>
__device__ __forceinline__ Vec<F, N> ldv_stream(const F* p)
{
    typedef F VV __attribute__((ext_vector_type(N)));
    const VV t = __builtin_nontemporal_load(reinterpret_cast<const VV*>(p));
    Vec<F, N> v;
#pragma unroll
    for (int c = 0; c < N; ++c) v.v[c] = t[c];
    return v;
}
// V consecutive elements per thread (16-byte accesses when the row width allows); four messages are requested
// before the first is added, the additions keep the ascending edge order
// WINDOW: slist is in ascending order in memory and the messages of the edges [e_lo, e_hi) are taken; otherwise all
// messages of the row are, and the block orders the row's edges in LDS first.
constexpr int SENDER_CAP = 1024;
template <typename F, int V, bool WINDOW>
__global__ void k_sender_reduce(int rows, int width, const int* sstart, int* slist_, int* spare, const F* msg,
                                F* H_adj, int zero_first, long e_lo, long e_hi)
{
    __shared__ __align__(16) int bucket[WINDOW ? 1 : 2 * SENDER_CAP];
    const int j = blockIdx.x;
    int s0 = sstart[j], s1 = sstart[j + 1];
    const int* slist = slist_;
    if constexpr (WINDOW) {
        // narrow to the edges inside [e_lo, e_hi)
        while (s0 < s1 && slist[s0] < e_lo) ++s0;
        while (s1 > s0 && slist[s1 - 1] >= e_hi) --s1;
    } else if (s1 - s0 <= SENDER_CAP) {
        const int n = s1 - s0;
        for (int t = threadIdx.x; t < (n + 3) / 4 * 4; t += blockDim.x) bucket[t] = t < n ? slist[s0 + t] : 0x7fffffff;
        __syncthreads();
        for (int t = threadIdx.x; t < n; t += blockDim.x) {
            const int v = bucket[t];
            bucket[SENDER_CAP + count_below(bucket, n, v)] = v;
        }
        __syncthreads();
        slist = bucket + SENDER_CAP;
        s0 = 0; s1 = n;
    } else {
        if (threadIdx.x < 64) wave_sort_in_memory(slist_, s0, s1 - s0, bucket, threadIdx.x, spare);
        __syncthreads();
    }
    if (s0 == s1 && !zero_first) return;
    for (int q = threadIdx.x * V; q < width; q += blockDim.x * V) {
        Vec<F, V> acc;
        if (zero_first) {
#pragma unroll
            for (int c = 0; c < V; ++c) acc.v[c] = F(0);
        } else {
            acc = ldv<F, V>(H_adj + (size_t)j * width + q);
        }
        int t = s0;
        for (; t + 4 <= s1; t += 4) {
            Vec<F, V> m[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = ldv_stream<F, V>(msg + (size_t)(slist[t + i] - e_lo) * width + q);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < V; ++c) acc.v[c] += m[i].v[c];
        }
        for (; t < s1; ++t) {
            const Vec<F, V> m = ldv_stream<F, V>(msg + (size_t)(slist[t] - e_lo) * width + q);
#pragma unroll
            for (int c = 0; c < V; ++c) acc.v[c] += m.v[c];
        }
        *reinterpret_cast<Vec<F, V>*>(H_adj + (size_t)j * width + q) = acc;
    }
}
}  // namespace

template <typename F>
hipError_t launch_sender_reduce(int rows, int width, const int* sstart, int* slist, int* spare, const F* msg,
                                F* H_adj, int zero_first, bool window, long e_lo, long e_hi, hipStream_t s)
{
    if (rows <= 0) return hipSuccess;
    constexpr int V = 16 / (int)sizeof(F);
    auto go = [&](auto kern, int bs) {
        hipLaunchKernelGGL(kern, dim3(rows), dim3(bs), 0, s, rows, width, sstart, slist, spare, msg, H_adj, zero_first, e_lo, e_hi);
    };
    if (width % V == 0) {
        const int lanes = width / V;
        const int bs = lanes <= 64 ? 64 : (lanes <= 128 ? 128 : 256);
        if (window) go(k_sender_reduce<F, V, true>, bs); else go(k_sender_reduce<F, V, false>, bs);
    } else {
        const int bs = width <= 64 ? 64 : (width <= 128 ? 128 : 256);
        if (window) go(k_sender_reduce<F, 1, true>, bs); else go(k_sender_reduce<F, 1, false>, bs);
    }
    return hipGetLastError();
}
// ---------------------------------------------------------------------------
// The sender-side sum followed by reverse_H1 for scalar hidden features (mace.cpp:402-436 with one block of
// H1): a block of 16 wavefronts sums the messages of 16 consecutive sender rows (wavefront w takes row w, in
// ascending edge order as above), keeps the finished rows in LDS as doubles, and forms
// M0_adj = H1_adj . W^T for them on the matrix cores; wavefront w owns column tile w, its weight operands
// (32 contiguous bytes per lane, k permuted inside groups of 16 on both operands) are requested before the
// sums start.
namespace {
typedef double f64x4_t __attribute__((ext_vector_type(4)));
template <typename F, int KT>
__global__ __launch_bounds__(1024) void k_sender_reduce_linear(int rows, const int* sstart, int* slist_, int* spare,
                                                              const F* msg, F* H_adj, int zero_first, const F* W, F* M_adj)
{
    constexpr int K = 16 * KT, ld = K + 1, V = 16 / (int)sizeof(F);
    constexpr int ROW_CAP = 256;
    __shared__ double X[16 * ld];
    __shared__ __align__(16) int bucket[16][ROW_CAP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16;
    const bool owner = wave < KT;
    f64x4_t wv[KT];
    if (owner) {
#pragma unroll
        for (int j = 0; j < KT; ++j) {
            const Vec<F, 4> t = ldv<F, 4>(W + (size_t)(wave * 16 + r) * K + 16 * j + 4 * g);
#pragma unroll
            for (int c = 0; c < 4; ++c) wv[j][c] = (double)t.v[c];
        }
    }
    {
        const int rr = wave, j = row0 + rr;
        const int q = lane * V;
        const int first = j < rows ? sstart[j] : 0, n = j < rows ? sstart[j + 1] - first : 0;
        const int* slist = wave_sorted_bucket<ROW_CAP>(slist_, first, n, bucket[wave], lane, spare);
        if (q < K) {
            Vec<F, V> acc;
#pragma unroll
            for (int c = 0; c < V; ++c) acc.v[c] = F(0);
            if (j < rows) {
                const int s0 = 0, s1 = n;
                if (!zero_first) acc = ldv<F, V>(H_adj + (size_t)j * K + q);
                int t = s0;
                for (; t + 4 <= s1; t += 4) {
                    Vec<F, V> m[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) m[i] = ldv_stream<F, V>(msg + (size_t)slist[t + i] * K + q);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int c = 0; c < V; ++c) acc.v[c] += m[i].v[c];
                }
                for (; t < s1; ++t) {
                    const Vec<F, V> m = ldv_stream<F, V>(msg + (size_t)slist[t] * K + q);
#pragma unroll
                    for (int c = 0; c < V; ++c) acc.v[c] += m.v[c];
                }
                *reinterpret_cast<Vec<F, V>*>(H_adj + (size_t)j * K + q) = acc;
            }
#pragma unroll
            for (int c = 0; c < V; ++c) X[rr * ld + q + c] = (double)acc.v[c];
        }
    }
    __syncthreads();
    if (owner) {
        f64x4_t acc = {0, 0, 0, 0};
        const double* a = X + r * ld + 4 * g;
#pragma unroll
        for (int j = 0; j < KT; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[16 * j + t], wv[j][t], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = row0 + 4 * q + g;
            if (j < rows) M_adj[(size_t)j * K + wave * 16 + r] = (F)acc[q];
        }
    }
}
}  // namespace

bool sender_reduce_linear_ok(int K) { return K == 32 || K == 48 || K == 64 || K == 96 || K == 128; }

template <typename F>
hipError_t launch_sender_reduce_linear(int rows, int K, const int* sstart, int* slist, int* spare, const F* msg, F* H_adj,
                                       int zero_first, const F* W, F* M_adj, hipStream_t s)
{
    if (!sender_reduce_linear_ok(K)) return hipErrorInvalidValue;
    if (rows <= 0) return hipSuccess;
    const dim3 grid((unsigned)((rows + 15) / 16)), block(1024);
    switch (K / 16) {
    case 2: hipLaunchKernelGGL((k_sender_reduce_linear<F, 2>), grid, block, 0, s, rows, sstart, slist, spare, msg, H_adj, zero_first, W, M_adj); break;
    case 3: hipLaunchKernelGGL((k_sender_reduce_linear<F, 3>), grid, block, 0, s, rows, sstart, slist, spare, msg, H_adj, zero_first, W, M_adj); break;
    case 4: hipLaunchKernelGGL((k_sender_reduce_linear<F, 4>), grid, block, 0, s, rows, sstart, slist, spare, msg, H_adj, zero_first, W, M_adj); break;
    case 6: hipLaunchKernelGGL((k_sender_reduce_linear<F, 6>), grid, block, 0, s, rows, sstart, slist, spare, msg, H_adj, zero_first, W, M_adj); break;
    default: hipLaunchKernelGGL((k_sender_reduce_linear<F, 8>), grid, block, 0, s, rows, sstart, slist, spare, msg, H_adj, zero_first, W, M_adj); break;
    }
    return hipGetLastError();
}
template hipError_t launch_sender_reduce_linear<double>(int, int, const int*, int*, int*, const double*, double*, int, const double*, double*, hipStream_t);
template hipError_t launch_sender_reduce_linear<float>(int, int, const int*, int*, int*, const float*, float*, int, const float*, float*, hipStream_t);

template hipError_t launch_sender_reduce<double>(int, int, const int*, int*, int*, const double*, double*, int, bool, long, long, hipStream_t);
template hipError_t launch_sender_reduce<float>(int, int, const int*, int*, int*, const float*, float*, int, bool, long, long, hipStream_t);

// ---------------------------------------------------------------------------
namespace {
__global__ void k_fpart_reduce(long n3, long stride3, int groups, const double* fpart, double* forces, int accumulate,
                               double* copy, const int* guard)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n3) return;
    double s = accumulate ? forces[t] : 0.0;
    for (int q = 0; q < groups; ++q) s += fpart[(size_t)q * stride3 + t];
    // a skipped evaluation (inputs failed their checks) left nothing in fpart: its forces say so
    if (guard && *guard) s = __builtin_nan("");
    forces[t] = s;
    if (copy) copy[t] = s;
}
}  // namespace
hipError_t launch_fpart_reduce(long edges, long E, int groups, const double* fpart, double* forces, int accumulate,
                               double* copy, hipStream_t s, const int* guard)
{
    const long n3 = 3 * edges;
    if (n3 <= 0 || edges > E) return n3 <= 0 ? hipSuccess : hipErrorInvalidValue;
    hipLaunchKernelGGL(k_fpart_reduce, dim3((unsigned)((n3 + 255) / 256)), dim3(256), 0, s, n3, 3 * E, groups, fpart,
                       forces, accumulate, copy, guard);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
namespace {
// (for callers that ask for the harmonics; spills 6 registers)
__global__ void k_sph_harm(const double* xyz, long E, double* Y, double* Yg)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const double dx = xyz[3 * e], dy = xyz[3 * e + 1], dz = xyz[3 * e + 2];
    const double inv = rsqrt_pos(dx * dx + dy * dy + dz * dz);
    double y[16], G[3][16];
    sph_l3_grad(dz * inv, dx * inv, dy * inv, inv, y, G);
    for (int q = 0; q < 16; ++q) {
        Y[e * 16 + q] = y[q];
        Yg[e * 48 + q] = G[0][q];
        Yg[e * 48 + 16 + q] = G[1][q];
        Yg[e * 48 + 32 + q] = G[2][q];
    }
}

template <typename F>
__global__ void k_radial(int N, const int* first_neigh, const int* node_types, const int* neigh_types,
                         const double* r, const F* tab, const int* pair_table, int T, int nodes, double h,
                         int nspl, double* R)
{
    const int i = blockIdx.x;
    const int ti = node_types[i];
    for (int e = first_neigh[i]; e < first_neigh[i + 1]; ++e) {
        const double rr = r[e];
        int n = (int)(rr / h);
        n = min(max(n, 0), nodes - 2);
        const F x = (F)(rr - h * n);
        const F* row = tab + ((size_t)pair_table[pair_index(T, ti, neigh_types[e])] * (nodes - 1) + n) * 4 * nspl;
        for (int j = threadIdx.x; j < nspl; j += blockDim.x) {
            const F v = row[j] + x * (row[nspl + j] + x * (row[2 * nspl + j] + x * row[3 * nspl + j]));
            R[(size_t)e * nspl + j] = (double)v;
        }
    }
}
}  // namespace

hipError_t launch_sph_harm(const double* xyz, long E, double* Y, double* Y_grad, hipStream_t s)
{
    if (E <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sph_harm, dim3((unsigned)((E + 127) / 128)), dim3(128), 0, s, xyz, E, Y, Y_grad);
    return hipGetLastError();
}

template <typename F>
hipError_t launch_radial(int N, const int* first_neigh, const int* node_types, const int* neigh_types,
                         const double* r, const F* tab, const int* pair_table, int T, int nodes, double h,
                         int nspl, double* R, hipStream_t s)
{
    if (N <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_radial<F>, dim3(N), dim3(128), 0, s, N, first_neigh, node_types, neigh_types, r, tab,
                       pair_table, T, nodes, h, nspl, R);
    return hipGetLastError();
}
template hipError_t launch_radial<double>(int, const int*, const int*, const int*, const double*, const double*, const int*, int, int, double, int, double*, hipStream_t);
template hipError_t launch_radial<float>(int, const int*, const int*, const int*, const double*, const float*, const int*, int, int, double, int, double*, hipStream_t);

#endif  // SMX_EDGE_PART == 0

}  // namespace smx
