// One polynomial of the standard product basis in straight-line code: shared by the contraction kernels (smx_kernels_poly.hip,
// smx_kernels_linear.hip).
#pragma once

#include "smx_device.hpp"
#include "smx_poly_shape.hpp"

namespace smx {
namespace {
template <typename F> __device__ __forceinline__ void pin_reg(F& v) { asm volatile("" : "+v"(v)); }
template <typename F> constexpr int spec_group() { return sizeof(F) == 8 ? 4 : 8; }   // coefficients per request

// Coefficients of a polynomial come in small groups, AHEAD of them requested before the one in use: from the LDS one is enough,
// from memory as many as the registers hold (the polynomial is bound by their latency then).  begin() requests the first ones.
template <typename F, int LM, int AHEAD>
struct PolyCoef {
    static constexpr int V = 16 / (int)sizeof(F), N = PolyTable<LM>::N, G = spec_group<F>(), NG = (N + G - 1) / G, RG = G / V;
    static constexpr int ROW0 = poly_spec_offset(LM) / V;   // first 16-byte group of this polynomial in the slab
    typedef F V4 __attribute__((ext_vector_type(V)));
    V4 buf[AHEAD + 1][RG];
    const unsigned char* slab_k;
    int row_stride_bytes;
    __device__ __forceinline__ PolyCoef(const unsigned char* slab, int stride) : slab_k(slab), row_stride_bytes(stride) {}
    template <int GI>
    __device__ __forceinline__ void request()
    {
        if constexpr (GI < NG) {
            constexpr int r0 = GI * RG;
#pragma unroll
            for (int j = 0; j < RG; ++j)
                if ((r0 + j) * V < poly_spec_padded(N))
                    buf[GI % (AHEAD + 1)][j] = *reinterpret_cast<const V4*>(slab_k + (size_t)(ROW0 + r0 + j) * row_stride_bytes);
        }
    }
    template <int FROM = 0>
    __device__ __forceinline__ void begin()
    {
        static_for<FROM, FROM + AHEAD>([&](auto gc) { request<decltype(gc)::value>(); });
    }
};
// Groups of coefficients from which slice `slice` of `slices` of a polynomial begins.
template <typename F, int LM> constexpr int poly_slice(int slice, int slices) { return (PolyTable<LM>::N + spec_group<F>() - 1) / spec_group<F>() * slice / slices; }

// MODE 0: values and gradients (M, M_grad); 1: values only; 2: adjoint, A_adj = sum over the polynomials of
// M_adj[polynomial] * gradient, recomputed from the variables (the coefficient is scaled, the value dropped).
//
// NESTED: the sums in the form below; else monomial by monomial, nearly twice the instructions, which do not wait for each other:
// for a polynomial per thread on an otherwise idle SIMD (24 to 501 atoms: evaluations 1 to 2 % shorter).
// FROM, TO: the groups of coefficients that are taken (monomial by monomial only: their sums do not need each other).
template <typename F, int LM, int MODE, bool NESTED, int AHEAD, int FROM = 0, int TO = PolyCoef<F, LM, AHEAD>::NG>
__device__ __forceinline__ void poly_spec_run(PolyCoef<F, LM, AHEAD>& w16, F (&x)[16], F (&g)[16], F& f, F madj)
{
    using TB = PolyTable<LM>;
    using C = PolyCoef<F, LM, AHEAD>;
    constexpr int V = C::V, G = C::G, NG = C::NG;
    // sum_p x_p Q_p, Q_p = sum_q x_q S_pq, S_pq = w_pq + sum_c w_pqc x_c in the order of the table; the gradient is
    //     g_c += w_pqc x_p x_q,  g_q += x_p S_pq,  g_p += Q_p
    // (the product rule holds as written for repeated indices): two multiply-adds per monomial, three more per pair, two per p,
    // about 300 for the value and gradient of a polynomial of 90 to 112 monomials.  Monomial by monomial they were 530 to 640.
    static_assert(!NESTED || (FROM == 0 && TO == NG), "nested sums are whole ones");
    F tp, pr, S, Q;      // x_p (times M_adj in mode 2), tp x_q
    // The next group is requested before the current one is used; compiler and scheduling barriers keep all groups from being
    // requested at once (the variables would spill).
    static_for<FROM, TO>([&](auto gc) {
        constexpr int gi = decltype(gc)::value;
        if constexpr (gi + AHEAD < TO) w16.template request<gi + AHEAD>();
        asm volatile("" ::: "memory");     // no read of a later group moves above this line
        __builtin_amdgcn_sched_barrier(0);
        constexpr int end = gi * G + G < TB::N ? gi * G + G : TB::N;
        static_for<gi * G, end>([&](auto ic) {
            constexpr int i = decltype(ic)::value, before = i > 0 ? i - 1 : 0, behind = i + 1 < TB::N ? i + 1 : i;
            constexpr int ip = TB::m[i][0], iq = TB::m[i][1], jc = TB::m[i][2];
            constexpr bool new_p = i == 0 || TB::m[before][0] != ip, new_q = new_p || TB::m[before][1] != iq;
            constexpr bool end_p = i + 1 == TB::N || TB::m[behind][0] != ip, end_q = end_p || TB::m[behind][1] != iq;
            const F w = w16.buf[gi % (AHEAD + 1)][(i - gi * G) / V][(i - gi * G) % V];
            if constexpr (!NESTED) {
                const F v = MODE == 2 ? w * madj : w;
                if constexpr (ip == 16) {
                    if constexpr (MODE != 1) g[jc] += v;
                    if constexpr (MODE != 2) f += v * x[jc];
                } else if constexpr (jc == 16) {
                    const F t = v * x[ip];
                    if constexpr (MODE != 1) { g[iq] += t; g[ip] += v * x[iq]; }
                    if constexpr (MODE != 2) f += t * x[iq];
                } else {
                    const F wa = v * x[ip], pbc = x[iq] * x[jc];
                    if constexpr (MODE != 1) { g[ip] += v * pbc; g[iq] += wa * x[jc]; g[jc] += wa * x[iq]; }
                    if constexpr (MODE != 2) f += wa * pbc;
                }
            } else if constexpr (ip == 16) {     // degree 1
                if constexpr (MODE == 0) g[jc] += w;
                if constexpr (MODE == 2) g[jc] += w * madj;
                if constexpr (MODE != 2) f += w * x[jc];
            } else {
                if constexpr (new_p) tp = MODE == 2 ? madj * x[ip] : x[ip];
                if constexpr (jc == 16) {
                    if constexpr (new_q) S = w; else S += w;
                } else {
                    if constexpr (MODE != 1) {
                        if constexpr (new_q) pr = tp * x[iq];
                        g[jc] += w * pr;
                    }
                    if constexpr (new_q) S = w * x[jc]; else S += w * x[jc];
                }
                if constexpr (end_q) {
                    if constexpr (MODE != 1) g[iq] += tp * S;
                    // (the first pair of this p: no entry with the same p and another q before)
                    constexpr int start = [] { int a = i; while (a > 0 && TB::m[a - 1][0] == ip && TB::m[a - 1][1] == iq) --a; return a; }();
                    if constexpr (start == 0 || TB::m[start > 0 ? start - 1 : 0][0] != ip) Q = x[iq] * S; else Q += x[iq] * S;
                }
                if constexpr (end_p) {
                    if constexpr (MODE == 0) g[ip] += Q;
                    if constexpr (MODE == 2) g[ip] += madj * Q;
                    if constexpr (MODE != 2) f += x[ip] * Q;
                }
            }
        });
        if constexpr (NESTED && end < TB::N && TB::m[end < TB::N ? end : 0][0] == TB::m[end - 1][0]) {      // in the middle of a p
            if constexpr (TB::m[end < TB::N ? end : 0][1] == TB::m[end - 1][1]) pin_reg(S); else pin_reg(Q);
        }
        // The sums are final here and the variables are new values for the next group: without this the arithmetic
        // of all groups sinks below the last request (the coefficients of the whole polynomial live at once) and the
        // pairwise products of the variables are hoisted above the first group (over a hundred more live values).
        if constexpr (MODE != 2) pin_reg(f);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            if constexpr (MODE != 1) pin_reg(g[q]);
            pin_reg(x[q]);   // (x is not const for this: its values never change)
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}
// ... with the coefficients in LDS
template <typename F, int LM, int MODE>
__device__ __forceinline__ void poly_spec_body(const unsigned char* slab_k, int row_stride_bytes, F (&x)[16], F (&g)[16], F& f,
                                               F madj)
{
    PolyCoef<F, LM, 1> w16(slab_k, row_stride_bytes);
    w16.begin();
    poly_spec_run<F, LM, MODE, true>(w16, x, g, f, madj);
}

}  // namespace
}  // namespace smx
