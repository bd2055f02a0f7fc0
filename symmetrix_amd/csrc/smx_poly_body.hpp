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
    __device__ __forceinline__ void begin()
    {
        static_for<0, AHEAD>([&](auto gc) { request<decltype(gc)::value>(); });
    }
};

// MODE 0: values and gradients (M, M_grad); 1: values only; 2: adjoint, A_adj = sum over the polynomials of
// M_adj[polynomial] * gradient, recomputed from the variables (the coefficient is scaled, the value dropped).
template <typename F, int LM, int MODE, int AHEAD>
__device__ __forceinline__ void poly_spec_run(PolyCoef<F, LM, AHEAD>& w16, F (&x)[16], F (&g)[16], F& f, F madj)
{
    using TB = PolyTable<LM>;
    using C = PolyCoef<F, LM, AHEAD>;
    constexpr int V = C::V, G = C::G, NG = C::NG;
    // The next group is requested before the current one is used; compiler and scheduling barriers keep all groups from being
    // requested at once (the variables would spill).
    static_for<0, NG>([&](auto gc) {
        constexpr int gi = decltype(gc)::value;
        w16.template request<gi + AHEAD>();
        asm volatile("" ::: "memory");     // no read of a later group moves above this line
        __builtin_amdgcn_sched_barrier(0);
        static_for<gi * G, (gi * G + G < TB::N ? gi * G + G : TB::N)>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            constexpr int ia = TB::m[i][0], ib = TB::m[i][1], jc = TB::m[i][2];
            F w = w16.buf[gi % (AHEAD + 1)][(i - gi * G) / V][(i - gi * G) % V];
            if constexpr (MODE == 2) w *= madj;
            if constexpr (ib == 16) {            // degree 1
                if constexpr (MODE != 1) g[jc] += w;
                if constexpr (MODE != 2) f += w * x[jc];
            } else if constexpr (ia == 16) {     // degree 2
                const F t = w * x[ib];
                if constexpr (MODE != 1) {
                    g[jc] += t;
                    g[ib] += w * x[jc];
                }
                if constexpr (MODE != 2) f += t * x[jc];
            } else {
                const F wa = w * x[ia], pbc = x[ib] * x[jc];
                if constexpr (MODE != 1) {
                    g[ia] += w * pbc;
                    g[ib] += wa * x[jc];
                    g[jc] += wa * x[ib];
                }
                if constexpr (MODE != 2) f += wa * pbc;
            }
        });
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
    poly_spec_run<F, LM, MODE>(w16, x, g, f, madj);
}

}  // namespace
}  // namespace smx
