// Edge kernels for scalar sender features with a diagonal coupling: layer 0 of every model, layer 1 of models with scalar
// hidden features.  Output lm of a receiver is fed by harmonic lm alone, through the radial spline of order l(lm):
//     out[i, lm, k] = sum over the edges of c_lm Y_lm R_l(r)[k] H[sender, k]
// and the adjoint gives the edge force and the message to the sender row.  Any number of radial tables.
//
// Work decomposition.  A wavefront owns a receiver, or one of two or four parts of its edges.  It works on EW edges at a time,
// 64 / EW lanes and CPL channels per lane each, so that 32, 64, 96 or 128 channels fill whole wavefronts and what an edge
// costs once (its place in the tables, the sums over channels, its forces) is spread over more channels.  Geometry (direction,
// harmonics, tangents, spline interval) is formed for up to 62 edges together, one per lane, in double precision, and left in
// LDS in the feature precision.  How the harmonics reach the channels: as in smx_kernels_edge.hip, by the lane broadcast of
// v_fmac_f64 (DPP) or by v_mfma_f32_4x4x1 with its block broadcast restricted to the lanes of an edge (cbsz = 3 for 32 lanes).
//
// What bounds them: spline coefficients, 4 x 16 (32) bytes per channel and edge, of the 64 bytes per cycle of a CU's vector
// cache.  A variant that kept slices of the table in LDS (one table only, four or eight channels per block) spent its time on
// LDS bank conflicts and on dependent LDS reads at twelve wavefronts per CU, wrote the force of an edge once per slice, and
// copied 130 KB per block first.
#include "smx_edge_common.hpp"

#include <algorithm>

namespace smx {

namespace {

// Wavefronts per SIMD (thread blocks per CU) of the adjoint: what the registers of its channels allow.  20 011 atoms, 96 channels,
// single: adjoints of 275 and 264 us with two, 253 and 237 with three; double, two channels per lane, layer 0: 600 atoms, 64 and 128
// channels 24 / 21 and 33 / 30, 10 000 atoms 243 / 231 and 455 / 441, 24 999 atoms 1 033 / 1 008 (l <= 1), 50 000 atoms 2 828 /
// 2 858 (78 edges an atom; two edges at a time without messages spill one register).  Where messages are stored as well, double and two channels per lane: see launch0.
template <typename F, int CPL>
constexpr int bwd0_blocks() { return CPL <= (sizeof(F) == 8 ? 2 : 3) ? 3 : 2; }
// edges per chunk: one lane each (two are left for a look at the next chunk), as many as leave room for the thread blocks of a CU
template <typename F, bool BWD, int BPC>
constexpr int chunk0()
{
    if (!BWD) return 62;
    if (BPC == 3) return sizeof(F) == 8 ? 30 : 54;
    return sizeof(F) == 8 ? 44 : 62;
}

template <typename F, bool BWD, int BPC>
struct Lds0 {
    static constexpr int CH = chunk0<F, BWD, BPC>();
    static_assert(CH % 2 == 0 && CH + 2 <= 64, "whole iterations, and a lane for every entry");
    static constexpr int NY = BWD ? 48 : 16;          // [lm][3]: harmonic, its two tangential derivatives; or harmonics
    static constexpr size_t val_bytes = ((size_t)CH * NY + 16) * sizeof(F);
    static constexpr size_t head_bytes = (size_t)(CH + 2) * (sizeof(F) + 2 * sizeof(unsigned));
    static constexpr size_t sum_bytes = BWD ? (size_t)(CH + 2) * 4 * sizeof(double) : 0;
    static_assert(val_bytes % 16 == 0, "the sums begin on a 16-byte boundary");
    static constexpr size_t per_wave = (val_bytes + head_bytes + sum_bytes + 15) / 16 * 16;
    static_assert(!BWD || 4 * per_wave * BPC <= 160 * 1024, "the thread blocks of a CU");
};

// ---------------------------------------------------------------------------
template <typename F, int CPL, int EW>
__global__ __launch_bounds__(256, 2) void k_agg0_fwd(const AggParams<F> a, const int parts, const int group_channels)
{
    constexpr bool MX = kMatrix<F>;
    using L = Lds0<F, false, 2>;
    constexpr int LPE = 64 / EW, CH = L::CH, CBSZ = EW == 2 ? 3 : 4;
    constexpr int W = MX || CPL <= 2 ? 4 : 2;          // splines requested ahead
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane / LPE, sl = lane % LPE;
    unsigned char* base = smem + (size_t)wave * L::per_wave;
    F* vals = reinterpret_cast<F*>(base);                       // [CH][16]
    F* xs = reinterpret_cast<F*>(base + L::val_bytes);          // [CH + 2]
    unsigned* toff = reinterpret_cast<unsigned*>(xs + CH + 2);  // [CH + 2]
    unsigned* goff = toff + CH + 2;                             // [CH + 2]

    const unsigned K = (unsigned)a.K;
    const int groups = (a.K + group_channels - 1) / group_channels;
    const int cgroup = blockIdx.x % groups;     // channel group fastest: a die's L2 holds its groups' share of the tables
    const int unit = (blockIdx.x / groups) * 4 + wave;
    const int i = __builtin_amdgcn_readfirstlane(unit / parts), part = unit - i * parts;
    const bool real = i < a.num_nodes;
    unsigned k[CPL];
    bool active[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ch = cgroup * group_channels + c * LPE + sl;
        active[c] = ch < a.K && c * LPE + sl < group_channels;
        k[c] = active[c] ? (unsigned)ch : 0u;
    }
    // Edges of this wavefront: the e1 - e0 from e0 on, or (as_chains: four parts, two edges at a time) two of every eight.
    const bool dealt = a.as_chains;
    int e0 = 0, e1 = 0, ti = 0;
    if (real) {
        const int b = a.first_neigh[i], n = a.first_neigh[i + 1] - b;
        e0 = b + (dealt ? EW * part : (int)((long)n * part / parts));
        e1 = dealt ? e0 + n / (4 * EW) * EW + min(max(n % (4 * EW) - EW * part, 0), EW) : b + (int)((long)n * (part + 1) / parts);
        ti = a.node_types[i];
    }
    e0 = __builtin_amdgcn_readfirstlane(e0); e1 = __builtin_amdgcn_readfirstlane(e1);

    f32x4 tile[MX ? CPL : 1][6];
    F acc[MX ? 1 : CPL][16];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        if constexpr (MX) {
#pragma unroll
            for (int q = 0; q < 6; ++q) tile[c][q] = f32x4{0, 0, 0, 0};
        } else {
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[c][q] = F(0);
        }
    }
    // the entry of an edge's harmonics this lane holds: lane n of every 16, or rows of the six row tiles
    const int pick = MX ? min(lm_of_tile((lane & 31) / 4 < 6 ? (lane & 31) / 4 : 5) + (lane & 3), 15) : (lane & 15);

    Vec<F, 4> cf[CPL][W];
    F H[CPL], Hn[CPL];
    const unsigned row_bytes = 4 * K * 4 * sizeof(F), sender_bytes = K * sizeof(F);
    auto request_spline = [&](unsigned off, int path) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) cf[c][path % W] = load_spline_off<F>(a.tabK, path, K, off + k[c] * 16);
    };
    auto request_sender = [&](unsigned off) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) Hn[c] = load_at<F>(reinterpret_cast<const char*>(a.Hsrc), off + k[c] * (unsigned)sizeof(F));
    };
    unsigned cur = 0;
    for (int eb = e0; eb < e1; eb += CH) {
        const int nE = min(CH, e1 - eb), slots = (nE + EW - 1) / EW * EW;     // edges, and places of whole iterations
        wave_lds_sync();
        if (lane < slots + EW) {
            // the entries from nE on: the first edges of the next chunk (past the last edge of the part: the last one again)
            int e = min(eb + lane, e1 - 1);
            if (dealt) e += (e - e0) / EW * (3 * EW);
            edge_offsets(a, e, ti, row_bytes, sender_bytes, xs, toff, goff, lane);
            if (lane < nE) {
                const double dx = a.xyz[3 * (size_t)e], dy = a.xyz[3 * (size_t)e + 1], dz = a.xyz[3 * (size_t)e + 2];
                const double inv = rsqrt_pos(dx * dx + dy * dy + dz * dz);
                double Y[16];
                sph_l3(dz * inv, dx * inv, dy * inv, Y);
#pragma unroll
                for (int q = 0; q < 16; ++q) vals[lane * 16 + q] = (F)(a.cdiag[q] * Y[q]);
            } else if (lane < slots) {
                // a slot without an edge adds zero
#pragma unroll
                for (int q = 0; q < 16; ++q) vals[lane * 16 + q] = F(0);
            }
        }
        wave_lds_sync();
        if (eb == e0) {
            cur = toff[sub];
            static_for<0, W>([&](auto qc) { request_spline(cur, decltype(qc)::value); });
            request_sender(goff[sub]);
        }
        for (int it = 0; it < slots; it += EW) {
            const int le = it + sub;
            const F x = xs[le], B = vals[le * 16 + pick];
            const unsigned next = toff[le + EW];
#pragma unroll
            for (int c = 0; c < CPL; ++c) H[c] = Hn[c];
            request_sender(goff[le + EW]);
            static_for<0, 4>([&](auto lc) {
                constexpr int l = decltype(lc)::value;
                F w[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    const Vec<F, 4> k4 = cf[c][l % W];
                    w[c] = (k4.v[0] + x * (k4.v[1] + x * (k4.v[2] + x * k4.v[3]))) * H[c];
                }
                if constexpr (l + W < 4) request_spline(cur, l + W); else request_spline(next, l % W);
                if constexpr (MX) {
                    constexpr int t0 = l == 0 ? 0 : (l == 1 ? 1 : (l == 2 ? 2 : 4)), nt = l < 2 ? 1 : 2;
                    static_for<0, nt>([&](auto tc) {
                        constexpr int t = t0 + decltype(tc)::value;
#pragma unroll
                        for (int c = 0; c < CPL; ++c) tile[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(B, w[c], tile[c][t], CBSZ, t, 0);
                    });
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
#pragma unroll
                        for (int t = t0; t < t0 + nt; ++t) pin(tile[c][t]);
                    __builtin_amdgcn_sched_group_barrier(0x002, 4 * CPL, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, nt * CPL, 0);
                } else {
                    static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
#pragma unroll
                        for (int c = 0; c < CPL; ++c) fmac_lane<q>(acc[c][q], B, w[c]);
                    });
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
#pragma unroll
                        for (int q = l * l; q < (l + 1) * (l + 1); ++q) pin(acc[c][q]);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            cur = next;
        }
    }
    // sum lm of channel c
    auto value = [&](auto qc, int c) -> F& {
        constexpr int q = decltype(qc)::value;
        if constexpr (MX) {
            constexpr int t = q < 1 ? 0 : (q < 4 ? 1 : (q < 8 ? 2 : (q < 9 ? 3 : (q < 13 ? 4 : 5))));
            return reinterpret_cast<F*>(&tile[c][t])[q - lm_of_tile(t)];
        } else {
            return acc[c][q];
        }
    };
    // the edges of the two half-wavefronts: sums 2 j and 2 j + 1 trade halves, the lower half ends with the one, the upper with the other
    constexpr int NR = 16 / EW;
    F out[CPL][NR];
    static_for<0, NR>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if constexpr (EW == 2) {
                F lo = value(std::integral_constant<int, 2 * j>{}, c), hi = value(std::integral_constant<int, 2 * j + 1>{}, c);
                swap_halves(lo, hi);
                out[c][j] = lo + hi;
            } else {
                out[c][j] = value(jc, c);
            }
        }
    });
    // the parts of a receiver lie in one thread block: the upper half of them hands its sums to the lower half, in LDS
    F* half = reinterpret_cast<F*>(smem);
    for (int h = parts >> 1; h >= 1; h >>= 1) {
        __syncthreads();
        F* at = half + (size_t)((wave / parts) * h + part % h) * NR * CPL * 64 + lane;
#pragma unroll
        for (int c = 0; c < CPL; ++c)
#pragma unroll
            for (int j = 0; j < NR; ++j)
                if (part >= h && part < 2 * h) at[(j * CPL + c) * 64] = out[c][j];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CPL; ++c)
#pragma unroll
            for (int j = 0; j < NR; ++j)
                if (part < h) out[c][j] += at[(j * CPL + c) * 64];
    }
    if (!real || part != 0) return;
#pragma unroll
    for (int c = 0; c < CPL; ++c)
        if (active[c]) {
#pragma unroll
            for (int j = 0; j < NR; ++j) a.out[((size_t)i * 16 + EW * j + sub) * K + k[c]] = out[c][j];
        }
}

// ---------------------------------------------------------------------------
template <typename F, int CPL, int EW, bool MSG, int BPC>
__global__ __launch_bounds__(256, BPC) void k_agg0_bwd(const AggParams<F> a, const int parts)
{
    constexpr bool MX = kMatrix<F>;
    using L = Lds0<F, true, BPC>;
    constexpr int LPE = 64 / EW, CH = L::CH, CBSZ = EW == 2 ? 3 : 4, GPR = LPE / 4;   // groups of four rows per register
    constexpr int NB = MX ? 16 / GPR : 3;              // registers that hold an edge's harmonics
    constexpr int W = MX || CPL == 1 ? 4 : 2;          // splines requested ahead
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane / LPE, sl = lane % LPE;
    unsigned char* base = smem + (size_t)wave * L::per_wave;
    F* vals = reinterpret_cast<F*>(base);                       // [CH][16][3]
    double* sums = reinterpret_cast<double*>(base + L::val_bytes);    // [CH + 2][4]
    F* xs = reinterpret_cast<F*>(sums + (CH + 2) * 4);          // [CH + 2]
    unsigned* toff = reinterpret_cast<unsigned*>(xs + CH + 2);
    unsigned* goff = toff + CH + 2;

    const unsigned K = (unsigned)a.K;
    const int groups = (a.K + CPL * LPE - 1) / (CPL * LPE);
    const int cgroup = blockIdx.x % groups;
    const int unit = (blockIdx.x / groups) * 4 + wave;
    const int rel = __builtin_amdgcn_readfirstlane(unit / parts), part = unit - rel * parts, i = a.node_begin + rel;
    if (i >= a.num_nodes) return;
    const int first = a.first_neigh[i], deg = a.first_neigh[i + 1] - first, ti = a.node_types[i];
    const int e0 = __builtin_amdgcn_readfirstlane(first + (int)((long)deg * part / parts));
    const int e1 = __builtin_amdgcn_readfirstlane(first + (int)((long)deg * (part + 1) / parts));
    if (e0 >= e1) return;
    double* fout = groups > 1 ? a.fpart + (size_t)cgroup * 3 * a.num_edges : a.forces;
    const bool add_forces = groups == 1 && a.accumulate_forces;
    double* copy = groups == 1 ? a.forces_copy : nullptr;
    // lanes beyond the last channel work on channel 0 with a zero adjoint and store no message
    unsigned k[CPL];
    bool active[CPL];
    F d[CPL][16];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int ch = (cgroup * CPL + c) * LPE + sl;
        active[c] = ch < a.K;
        k[c] = active[c] ? (unsigned)ch : 0u;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const F v = a.d_out[((size_t)i * 16 + q) * K + k[c]];
            d[c][q] = active[c] ? v : F(0);
        }
        d[c][0] *= (F)a.cdiag[0];
    }
    // the entries of an edge's harmonics this lane holds, one per register
    int pick[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) pick[j] = MX ? 3 * (j * GPR + sl / 4) + (lane & 3) : j * 16 + (lane & 15);
    const int out_lane = lane & (LPE - 1);
    const bool writes = EW == 2 ? (out_lane == 0 || out_lane == 8 || out_lane == 16) : (lane == 0 || lane == 16 || lane == 32);
    const int out_slot = EW == 2 ? (out_lane == 0 ? 0 : (out_lane == 16 ? 1 : 2)) : lane / 16;

    Vec<F, 4> cf[CPL][W];
    const unsigned row_bytes = 4 * K * 4 * sizeof(F), sender_bytes = K * sizeof(F);
    auto request_spline = [&](unsigned off, int path) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) cf[c][path % W] = load_spline_off<F>(a.tabK, path, K, off + k[c] * 16);
    };
    unsigned cur = 0;
    for (int eb = e0; eb < e1; eb += CH) {
        const int nE = min(CH, e1 - eb), slots = (nE + EW - 1) / EW * EW;     // edges, and places of whole iterations
        wave_lds_sync();
        if (lane < slots + EW) {
            const int e = min(eb + lane, e1 - 1);
            edge_offsets(a, e, ti, row_bytes, sender_bytes, xs, toff, goff, lane);
            if (lane < nE) {
                EdgeFrame f;
                edge_frame(a.xyz + 3 * (size_t)e, f);
                F* y = vals + lane * 48;
                static_for<0, 16>([&](auto lc) {
                    constexpr int lm = decltype(lc)::value;
                    double Y, g1, g2;
                    ylm_tangential<lm>(f, Y, g1, g2);
                    const double cc = a.cdiag[lm];
                    y[3 * lm] = (F)(cc * Y); y[3 * lm + 1] = (F)(cc * g1); y[3 * lm + 2] = (F)(cc * g2);
                    if constexpr (lm % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // short live ranges
                });
            }
        }
        wave_lds_sync();
        if (eb == e0) {
            cur = toff[sub];
            static_for<0, W>([&](auto qc) { request_spline(cur, decltype(qc)::value); });
        }
        char* mchunk = MSG ? reinterpret_cast<char*>(a.msg) + (unsigned long long)(unsigned)(eb - (int)a.msg_edge_begin) * sender_bytes : nullptr;
        for (int it = 0; it < slots; it += EW) {
            const int le = it + sub;
            const F x = xs[le];
            const unsigned next = toff[le + EW];
            // the sender row is met at the end of the edge only: requested here, it has the whole edge to arrive
            F H[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c) H[c] = load_at<F>(reinterpret_cast<const char*>(a.Hsrc), goff[le] + k[c] * (unsigned)sizeof(F));
            F B[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) B[j] = vals[le * 48 + pick[j]];
            F V[CPL][4];     // message, R u.t1, R u.t2, R' u
            static_for<0, 4>([&](auto lc) {
                constexpr int l = decltype(lc)::value;
                F R[CPL], Rd[CPL];
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    const Vec<F, 4> k4 = cf[c][l % W];
                    const F q1 = k4.v[2] + x * k4.v[3], d1 = q1 + x * k4.v[3], q2 = fma_apart(x, q1, k4.v[1]);
                    R[c] = fma_apart(x, q2, k4.v[0]);
                    Rd[c] = q2 + x * d1;
                }
                if constexpr (l + W < 4) request_spline(cur, l + W); else request_spline(next, l % W);
                if constexpr (l == 0) {
                    // the constant harmonic: its factor is in the adjoint row, and there is no tangential part
#pragma unroll
                    for (int c = 0; c < CPL; ++c) { V[c][0] = R[c] * d[c][0]; V[c][3] = Rd[c] * d[c][0]; }
                } else if constexpr (MX) {
                    f32x4 u[CPL];
                    static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
                            u[c] = __builtin_amdgcn_mfma_f32_4x4x1f32(B[q / GPR], d[c][q], q == l * l ? f32x4{0, 0, 0, 0} : u[c], CBSZ, q % GPR, 0);
                    });
#pragma unroll
                    for (int c = 0; c < CPL; ++c) {
                        V[c][0] += R[c] * u[c][0]; V[c][3] += Rd[c] * u[c][0];
                        V[c][1] = l == 1 ? R[c] * u[c][1] : V[c][1] + R[c] * u[c][1];
                        V[c][2] = l == 1 ? R[c] * u[c][2] : V[c][2] + R[c] * u[c][2];
                    }
                } else {
                    // Sums per order, and the radial function once for each: 2 l - 1 multiplications fewer per channel.  With / without
                    // messages, us: 128 channels, 9 000 atoms 279 -> 274 / 249 -> 242, 9 999 atoms (l <= 1) 433 -> 420, 64 channels,
                    // 20 000 atoms 348 -> 343 / 308 -> 306.  Two channels per lane, three wavefronts and messages have no registers
                    // for three sums side by side (12 spilled, 64 channels, 6 000 atoms 115 -> 137; one by one 113); elsewhere one by
                    // one is slower (249 and 438 us of the 242 and 420 above).
                    constexpr bool ONE = MSG && CPL == 2 && BPC == 3;
                    constexpr int T = ONE ? 1 : 3;
                    static_for<0, 3 / T>([&](auto tc) {
                        constexpr int t0 = decltype(tc)::value * T;
                        F u[CPL][T];
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int t = 0; t < T; ++t) u[c][t] = F(0);
                        static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                            constexpr int q = decltype(qc)::value;
#pragma unroll
                            for (int c = 0; c < CPL; ++c)
                                static_for<0, T>([&](auto uc) {
                                    constexpr int t = decltype(uc)::value, v = 3 * q + t0 + t;
                                    fmac_lane<v % 16>(u[c][t], B[v / 16], d[c][q]);
                                });
                        });
#pragma unroll
                        for (int c = 0; c < CPL; ++c)
#pragma unroll
                            for (int t = 0; t < T; ++t) {
                                F& s = V[c][t0 + t];
                                s = t0 + t > 0 && l == 1 ? R[c] * u[c][t] : s + R[c] * u[c][t];
                                if (t0 + t == 0) V[c][3] += Rd[c] * u[c][t];
                                if constexpr (ONE) pin(s);
                            }
                    });
                }
#pragma unroll
                for (int c = 0; c < CPL; ++c)
#pragma unroll
                    for (int t = MSG ? 0 : 1; t < 4; ++t)
                        if (l > 0 || t == 0 || t == 3) pin(V[c][t]);
                if constexpr (MX && l > 0) {
                    __builtin_amdgcn_sched_group_barrier(0x008, (2 * l + 1) * CPL, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 100, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            cur = next;
            F srad = V[0][3] * H[0], g1 = V[0][1] * H[0], g2 = V[0][2] * H[0];
#pragma unroll
            for (int c = 1; c < CPL; ++c) { srad += V[c][3] * H[c]; g1 += V[c][1] * H[c]; g2 += V[c][2] * H[c]; }
            if constexpr (MSG) {
                if (le < nE) {
                    const unsigned off = (unsigned)le * sender_bytes;
#pragma unroll
                    for (int c = 0; c < CPL; ++c)
                        if (active[c]) store_stream(reinterpret_cast<F*>(mchunk + (off + k[c] * (unsigned)sizeof(F))), V[c][0]);
                }
            }
            const double s = edge_sum3<EW>(srad, g1, g2, lane);
            if (writes) sums[le * 4 + out_slot] = s;
        }
        wave_lds_sync();
        // the forces of the chunk, put together in double
        if (lane < nE) {
            const size_t e = (size_t)(eb + lane);
            EdgeFrame f;
            edge_frame(a.xyz + 3 * e, f);
            const double ir = rcp_pos(a.r[e]);
            const double sr = sums[lane * 4] * ir, G1 = sums[lane * 4 + 1], G2 = sums[lane * 4 + 2];
            double fx = -(f.dx * sr + f.t1x * G1 + f.t2x * G2);
            double fy = -(f.dy * sr + f.t1y * G1 + f.t2y * G2);
            double fz = -(f.dz * sr + f.t1z * G1 + f.t2z * G2);
            double* o = fout + 3 * e;
            if (add_forces) { fx += o[0]; fy += o[1]; fz += o[2]; }
            o[0] = fx; o[1] = fy; o[2] = fz;
            if (copy) { copy[3 * e] = fx; copy[3 * e + 1] = fy; copy[3 * e + 2] = fz; }
        }
    }
}

// Lanes per edge, channels per lane and channels per group.
// Adjoint: two edges per wavefront at 32 lanes each fill the wavefront for every multiple of 32 channels up to 96 (single
// precision: 128); in double precision four channels per lane would need more than 256 registers, and 97 to 128 channels
// take one edge at two channels per lane.  Wider models are cut into groups whose partial forces are added up afterwards.
// Forward: the same for one table and many receivers.  With few receivers (measured at 96 channels: 300 receivers in double
// precision 17.2 us in one group, 13.8 in three; 501 in single 13.4 and 11.8; 3 000 in double 63 and 61) groups of 32
// channels put more wavefronts on the chip.  Tables that do not fit the 4 MB L2 of a die are cut into four groups, so that a
// die, which sees every fourth block, only reads a quarter of them.
template <typename F>
struct Shape0 {
    int cpl, ew, group;
    static Shape0 of(int K)
    {
        if (K <= 32) return {1, 2, 32};
        if (K <= 64) return {2, 2, 64};
        if (K <= 96) return {3, 2, 96};
        return sizeof(F) == 8 ? Shape0{2, 1, 128} : Shape0{4, 2, 128};
    }
    static Shape0 forward(int K, int receivers, size_t table_bytes)
    {
        if (K > 32 && K <= 128 && table_bytes > ((size_t)6 << 20)) return {1, 2, (K + 3) / 4};
        if (receivers <= 3072) return {1, 2, 32};
        return of(K);
    }
};

template <typename F, int CPL, int EW, bool BWD>
hipError_t launch0(const AggParams<F>& p, int group, hipStream_t s)
{
    const int groups = (p.K + group - 1) / group;
    if (group > CPL * 64 / EW) return hipErrorInvalidValue;
    if (BWD && groups > 1 && !p.fpart) return hipErrorInvalidValue;
    if (!BWD && (p.node_begin != 0 || p.msg_edge_begin != 0)) return hipErrorInvalidValue;
    if (p.node_begin < 0 || p.node_begin > p.num_nodes) return hipErrorInvalidValue;
    const long nodes = p.num_nodes - p.node_begin;
    if (!BWD && p.as_chains && EW != 2) return hipErrorInvalidValue;
    const int parts = !BWD && p.as_chains ? 4 : agg_parts<BWD>((long)(BWD ? nodes : p.split_nodes) * groups);
    const long blocks = (nodes * parts + 3) / 4 * groups;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    auto go = [&](auto kern, size_t lds, auto... args) {
        if (lds > 64 * 1024) {
            hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (err != hipSuccess) return err;
        }
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), lds, s, p, args...);
        return hipGetLastError();
    };
    if constexpr (BWD) {
        constexpr int BPC = bwd0_blocks<F, CPL>();
        constexpr size_t lds = 4 * Lds0<F, true, BPC>::per_wave;
        if (!p.msg) return go(k_agg0_bwd<F, CPL, EW, false, BPC>, lds, parts);
        // With messages, double and two channels per lane, the third wavefront costs from where a receiver has one to itself: us, three
        // / two: 64 channels 600 atoms 22 / 24, 6 500 117 / 113, 20 000 352 / 346, 50 000 880 / 840, 128 channels 600 32 / 35,
        // 6 500 215 / 210, 20 000 653 / 620.  (One channel per lane: 50 000 atoms 514 / 550.)
        if constexpr (BPC == 3 && sizeof(F) == 8 && CPL == 2) {
            if (parts == 1) return go(k_agg0_bwd<F, CPL, EW, true, 2>, 4 * Lds0<F, true, 2>::per_wave, parts);
        }
        return go(k_agg0_bwd<F, CPL, EW, true, BPC>, lds, parts);
    } else {
        const size_t handed = parts > 1 ? (size_t)2 * (16 / EW) * CPL * 64 * sizeof(F) : 0;   // two givers per block
        return go(k_agg0_fwd<F, CPL, EW>, std::max(4 * Lds0<F, false, 2>::per_wave, handed), parts, group);
    }
}
template <typename F, bool BWD>
hipError_t launch0_sel(const AggParams<F>& p, hipStream_t s)
{
    const Shape0<F> sh = BWD ? Shape0<F>::of(p.K) : Shape0<F>::forward(p.K, p.split_nodes, p.table_bytes);
    if (sh.ew == 1) {
        if constexpr (sizeof(F) == 8) return launch0<F, 2, 1, BWD>(p, sh.group, s);
    } else {
        switch (sh.cpl) {
        case 1: return launch0<F, 1, 2, BWD>(p, sh.group, s);
        case 2: return launch0<F, 2, 2, BWD>(p, sh.group, s);
        case 3: return launch0<F, 3, 2, BWD>(p, sh.group, s);
        default:
            if constexpr (sizeof(F) == 4) return launch0<F, 4, 2, BWD>(p, sh.group, s);
        }
    }
    return hipErrorInvalidValue;
}

}  // namespace

template <typename F> hipError_t launch_agg0_fwd(const AggParams<F>& p, hipStream_t s) { return launch0_sel<F, false>(p, s); }
template <typename F> hipError_t launch_agg0_bwd(const AggParams<F>& p, hipStream_t s) { return launch0_sel<F, true>(p, s); }
template <typename F> int agg0_bwd_groups(int K)
{
    const int group = Shape0<F>::of(K).group;
    return (K + group - 1) / group;
}
// compiled once per precision
#ifndef SMX_EDGE_PART
#error "define SMX_EDGE_PART (0: double, 1: float)"
#endif
#if SMX_EDGE_PART == 0
typedef double feature_t;
#else
typedef float feature_t;
#endif
template hipError_t launch_agg0_fwd<feature_t>(const AggParams<feature_t>&, hipStream_t);
template hipError_t launch_agg0_bwd<feature_t>(const AggParams<feature_t>&, hipStream_t);
template int agg0_bwd_groups<feature_t>(int);

}  // namespace smx
