// The edges of one receiver with scalar sender features inside a chain (smx_kernels_chain.hip): the aggregation before its node-local
// stages and the adjoint behind them, by all K / 8 wavefronts of a thread block.
//
// 32 lanes and channels an edge, so that a wavefront has two edges at a time and four wavefronts share a group of 32 channels: eight
// edges of the receiver under way.  Geometry is formed once per block, an edge per thread; a kernel of its own forms it for every
// group of channels (smx_kernels_edge0.hip, which also says how the harmonics reach the channels).  Sums over the four wavefronts,
// and of the forces over the channel groups, run in a fixed order through LDS.
#pragma once

#include "smx_edge_common.hpp"

#include <algorithm>

namespace smx {
namespace {

template <typename F, int K>
struct ChainEdges {
    static constexpr bool MX = kMatrix<F>;
    static constexpr int G = K / 32, PARTS = 4, STEP = 2 * PARTS, T = 8 * K;
    static constexpr int CHF = 120, CHB = 80;      // edges at a time, forward and adjoint (whole rounds, and a thread for each)
    static_assert(CHF % STEP == 0 && CHB % STEP == 0 && CHF + STEP <= T, "whole rounds, and a thread for every edge");
    static constexpr size_t heads(int ch) { return (size_t)(ch + STEP) * (sizeof(F) + 2 * sizeof(unsigned)); }
    static constexpr size_t fwd_bytes = std::max((size_t)CHF * 16 * sizeof(F) + heads(CHF), (size_t)PARTS * 16 * K * sizeof(F));
    static constexpr size_t bwd_bytes = (size_t)CHB * (48 * sizeof(F) + G * 4 * sizeof(double)) + heads(CHB);
    static constexpr unsigned row_bytes = 4 * K * 4 * sizeof(F), sender_bytes = K * sizeof(F);

    // what a wavefront and a lane take
    int group, part, sub, sl;
    unsigned k;
    __device__ __forceinline__ ChainEdges(int wave, int lane)
        : group(wave % G), part(wave / G), sub(lane >> 5), sl(lane & 31), k((wave % G) * 32 + (lane & 31)) {}

    __device__ __forceinline__ void splines(const AggParams<F>& a, Vec<F, 4> (&cf)[4], unsigned off, int l) const
    {
        cf[l] = load_spline_off<F>(a.tabK, l, K, off + k * 16);
    }
    __device__ __forceinline__ F sender(const AggParams<F>& a, unsigned off) const
    {
        return load_at<F>(reinterpret_cast<const char*>(a.Hsrc), off + k * (unsigned)sizeof(F));
    }

    // The 16 rows of the receiver: values tid and tid + T of [16][K].  lds: fwd_bytes that nobody reads or writes any more.
    __device__ __forceinline__ void forward(const AggParams<F>& a, int node, int type, unsigned char* lds, int tid, int lane, F (&out)[2]) const
    {
        F* vals = reinterpret_cast<F*>(lds);                        // [CHF][16]
        F* xs = vals + CHF * 16;                                    // [CHF + STEP]
        unsigned* toff = reinterpret_cast<unsigned*>(xs + CHF + STEP);
        unsigned* goff = toff + CHF + STEP;
        const int e0 = a.first_neigh[node], e1 = a.first_neigh[node + 1];
        const int pick = MX ? min(lm_of_tile((lane & 31) / 4 < 6 ? (lane & 31) / 4 : 5) + (lane & 3), 15) : (lane & 15);
        f32x4 tile[6];
        F acc[MX ? 1 : 16];
        if constexpr (MX) {
#pragma unroll
            for (int q = 0; q < 6; ++q) tile[q] = f32x4{0, 0, 0, 0};
        } else {
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[q] = F(0);
        }
        for (int eb = e0; eb < e1; eb += CHF) {
            const int nE = min(CHF, e1 - eb), slots = (nE + STEP - 1) / STEP * STEP;
            if (eb != e0) __syncthreads();
            if (tid < slots + STEP) {
                const int e = min(eb + tid, e1 - 1);
                edge_offsets(a, e, type, row_bytes, sender_bytes, xs, toff, goff, tid);
                if (tid < nE) {
                    const double dx = a.xyz[3 * (size_t)e], dy = a.xyz[3 * (size_t)e + 1], dz = a.xyz[3 * (size_t)e + 2];
                    const double inv = rsqrt_pos(dx * dx + dy * dy + dz * dz);
                    double Y[16];
                    sph_l3(dz * inv, dx * inv, dy * inv, Y);
#pragma unroll
                    for (int q = 0; q < 16; ++q) vals[tid * 16 + q] = (F)(a.cdiag[q] * Y[q]);
                } else if (tid < slots) {
                    // a place without an edge adds zero
#pragma unroll
                    for (int q = 0; q < 16; ++q) vals[tid * 16 + q] = F(0);
                }
            }
            __syncthreads();
            Vec<F, 4> cf[4];
            int le = 2 * part + sub;
            unsigned cur = toff[le];
            static_for<0, 4>([&](auto lc) { splines(a, cf, cur, decltype(lc)::value); });
            F Hn = sender(a, goff[le]);
            for (; le < slots; le += STEP) {
                const F x = xs[le], B = vals[le * 16 + pick], H = Hn;
                const unsigned next = toff[le + STEP];
                Hn = sender(a, goff[le + STEP]);
                static_for<0, 4>([&](auto lc) {
                    constexpr int l = decltype(lc)::value;
                    const Vec<F, 4> k4 = cf[l];
                    const F w = (k4.v[0] + x * (k4.v[1] + x * (k4.v[2] + x * k4.v[3]))) * H;
                    splines(a, cf, next, l);
                    if constexpr (MX) {
                        constexpr int t0 = l == 0 ? 0 : (l == 1 ? 1 : (l == 2 ? 2 : 4)), nt = l < 2 ? 1 : 2;
                        static_for<t0, t0 + nt>([&](auto tc) {
                            constexpr int t = decltype(tc)::value;
                            tile[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(B, w, tile[t], 3, t, 0);
                            pin(tile[t]);
                        });
                    } else {
                        static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                            fmac_lane<decltype(qc)::value>(acc[decltype(qc)::value], B, w);
                            pin(acc[decltype(qc)::value]);
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
        }
        auto value = [&](auto qc) -> F& {
            constexpr int q = decltype(qc)::value;
            if constexpr (MX) {
                constexpr int t = q < 1 ? 0 : (q < 4 ? 1 : (q < 8 ? 2 : (q < 9 ? 3 : (q < 13 ? 4 : 5))));
                return reinterpret_cast<F*>(&tile[t])[q - lm_of_tile(t)];
            } else {
                return acc[q];
            }
        };
        // the edges of the two halves: sums 2 j and 2 j + 1 trade halves, the lower half ends with the one, the upper with the other
        __syncthreads();
        F* red = reinterpret_cast<F*>(lds);                         // [PARTS][16][K]
        static_for<0, 8>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            F lo = value(std::integral_constant<int, 2 * j>{}), hi = value(std::integral_constant<int, 2 * j + 1>{});
            swap_halves(lo, hi);
            red[(part * 16 + 2 * j + sub) * K + k] = lo + hi;
        });
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const F* r = red + tid + j * T;
            out[j] = (r[0] + r[2 * 16 * K]) + (r[16 * K] + r[3 * 16 * K]);      // (as k_agg0_fwd hands them down)
        }
    }

    // Forces of the receiver's edges and (MSG) messages to their senders; d: the adjoint of its 16 rows in LDS, rows `stride` bytes
    // apart.  lds: bwd_bytes that nobody reads or writes any more.
    template <bool MSG>
    __device__ __forceinline__ void adjoint(const AggParams<F>& a, int node, int type, const unsigned char* drow, unsigned stride,
                                            unsigned char* lds, int tid, int lane) const
    {
        double* sums = reinterpret_cast<double*>(lds);              // [G][CHB][4]
        F* vals = reinterpret_cast<F*>(sums + G * CHB * 4);         // [CHB][16][3]
        F* xs = vals + CHB * 48;                                    // [CHB + STEP]
        unsigned* toff = reinterpret_cast<unsigned*>(xs + CHB + STEP);
        unsigned* goff = toff + CHB + STEP;
        constexpr int NB = MX ? 2 : 3;                              // registers that hold an edge's harmonics
        const int e0 = a.first_neigh[node], e1 = a.first_neigh[node + 1];
        if (e0 == e1) return;
        F d[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) d[q] = *reinterpret_cast<const F*>(drow + q * stride + k * sizeof(F));
        d[0] *= (F)a.cdiag[0];
        int pick[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) pick[j] = MX ? 3 * (j * 8 + sl / 4) + (lane & 3) : j * 16 + (lane & 15);
        const bool writes = sl == 0 || sl == 8 || sl == 16;
        const int out_slot = sl == 0 ? 0 : (sl == 16 ? 1 : 2);
        for (int eb = e0; eb < e1; eb += CHB) {
            const int nE = min(CHB, e1 - eb), slots = (nE + STEP - 1) / STEP * STEP;
            if (eb != e0) __syncthreads();
            if (tid < slots + STEP) {
                const int e = min(eb + tid, e1 - 1);
                edge_offsets(a, e, type, row_bytes, sender_bytes, xs, toff, goff, tid);
                if (tid < nE) {
                    EdgeFrame f;
                    edge_frame(a.xyz + 3 * (size_t)e, f);
                    F* y = vals + tid * 48;
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
            __syncthreads();
            Vec<F, 4> cf[4];
            int le = 2 * part + sub;
            unsigned cur = toff[le];
            static_for<0, 4>([&](auto lc) { splines(a, cf, cur, decltype(lc)::value); });
            for (; le < slots; le += STEP) {       // (places without an edge: numbers nobody reads)
                const F x = xs[le];
                const unsigned next = toff[le + STEP];
                const F H = sender(a, goff[le]);
                F B[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) B[j] = vals[le * 48 + pick[j]];
                F V[4];     // message, R u.t1, R u.t2, R' u
                static_for<0, 4>([&](auto lc) {
                    constexpr int l = decltype(lc)::value;
                    const Vec<F, 4> k4 = cf[l];
                    const F q1 = k4.v[2] + x * k4.v[3], d1 = q1 + x * k4.v[3], q2 = fma_apart(x, q1, k4.v[1]);
                    const F R = fma_apart(x, q2, k4.v[0]), Rd = q2 + x * d1;
                    splines(a, cf, next, l);
                    if constexpr (l == 0) {
                        // the constant harmonic: its factor is in the adjoint row, and there is no tangential part
                        V[0] = R * d[0]; V[3] = Rd * d[0];
                    } else if constexpr (MX) {
                        f32x4 u;
                        static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                            constexpr int q = decltype(qc)::value;
                            u = __builtin_amdgcn_mfma_f32_4x4x1f32(B[q / 8], d[q], q == l * l ? f32x4{0, 0, 0, 0} : u, 3, q % 8, 0);
                        });
                        V[0] += R * u[0]; V[3] += Rd * u[0];
                        V[1] = l == 1 ? R * u[1] : V[1] + R * u[1];
                        V[2] = l == 1 ? R * u[2] : V[2] + R * u[2];
                    } else {
                        // as k_agg0_bwd: the sums of an order with the same bits (what follows adds channels in another order there)
                        F u[3] = {F(0), F(0), F(0)};
                        static_for<l * l, (l + 1) * (l + 1)>([&](auto qc) {
                            constexpr int q = decltype(qc)::value, v = 3 * q;
                            fmac_lane<v % 16>(u[0], B[v / 16], d[q]);
                            fmac_lane<(v + 1) % 16>(u[1], B[(v + 1) / 16], d[q]);
                            fmac_lane<(v + 2) % 16>(u[2], B[(v + 2) / 16], d[q]);
                        });
                        V[0] += R * u[0]; V[3] += Rd * u[0];
                        V[1] = l == 1 ? R * u[1] : V[1] + R * u[1];
                        V[2] = l == 1 ? R * u[2] : V[2] + R * u[2];
                    }
#pragma unroll
                    for (int t = MSG ? 0 : 1; t < 4; ++t)
                        if (l > 0 || t == 0 || t == 3) pin(V[t]);
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (MSG) {
                    if (le < nE) store_stream(a.msg + (size_t)(eb + le) * K + k, V[0]);
                }
                const double s = edge_sum3<2>(V[3] * H, V[1] * H, V[2] * H, lane);
                if (writes) sums[(group * CHB + le) * 4 + out_slot] = s;
            }
            __syncthreads();
            // the forces, put together in double
            if (tid < nE) {
                const size_t e = (size_t)(eb + tid);
                EdgeFrame f;
                edge_frame(a.xyz + 3 * e, f);
                double sr = 0.0, G1 = 0.0, G2 = 0.0;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const double* t = sums + (g * CHB + tid) * 4;
                    sr += t[0]; G1 += t[1]; G2 += t[2];
                }
                sr *= rcp_pos(a.r[e]);
                double fx = -(f.dx * sr + f.t1x * G1 + f.t2x * G2);
                double fy = -(f.dy * sr + f.t1y * G1 + f.t2y * G2);
                double fz = -(f.dz * sr + f.t1z * G1 + f.t2z * G2);
                double* o = a.forces + 3 * e;
                if (a.accumulate_forces) { fx += o[0]; fy += o[1]; fz += o[2]; }
                o[0] = fx; o[1] = fy; o[2] = fz;
                if (a.forces_copy) { a.forces_copy[3 * e] = fx; a.forces_copy[3 * e + 1] = fy; a.forces_copy[3 * e + 2] = fz; }
            }
        }
    }
};

}  // namespace
}  // namespace smx
