// One polynomial of the standard product basis in straight-line code: shared by the contraction kernels (smx_kernels_poly.hip,
// smx_kernels_linear.hip).
#pragma once

#include "smx_device.hpp"
#include "smx_poly_shape.hpp"

namespace smx {
namespace {
template <typename F> __device__ __forceinline__ void pin_reg(F& v) { asm volatile("" : "+v"(v)); }
template <typename F> constexpr int spec_group() { return sizeof(F) == 8 ? 4 : 8; }   // coefficients per request

// MODE 0: values and gradients (M, M_grad); 1: values only; 2: adjoint, A_adj = sum over the polynomials of
// M_adj[polynomial] * gradient, recomputed from the variables (the coefficient is scaled, the value dropped).
template <typename F, int LM, int MODE>
__device__ __forceinline__ void poly_spec_body(const unsigned char* slab_k, int row_stride_bytes, F (&x)[16], F (&g)[16], F& f,
                                               F madj)
{
    using TB = PolyTable<LM>;
    constexpr int V = 16 / (int)sizeof(F);
    typedef F V4 __attribute__((ext_vector_type(V)));
    constexpr int row0 = poly_spec_offset(LM) / V;   // first 16-byte group of this polynomial in the slab
    // Coefficients come in small groups: the next group is requested before the current one is used; compiler
    // and scheduling barriers keep all groups from being requested at once (the variables would spill).
    constexpr int G = spec_group<F>(), NG = (TB::N + G - 1) / G, RG = G / V;
    V4 wbuf[2][RG];
    auto request = [&](auto gc, V4 (&w)[RG]) {
        constexpr int r0 = decltype(gc)::value * RG;
#pragma unroll
        for (int j = 0; j < RG; ++j)
            if ((r0 + j) * V < poly_spec_padded(TB::N))
                w[j] = *reinterpret_cast<const V4*>(slab_k + (size_t)(row0 + r0 + j) * row_stride_bytes);
    };
    request(std::integral_constant<int, 0>{}, wbuf[0]);
    static_for<0, NG>([&](auto gc) {
        constexpr int gi = decltype(gc)::value;
        if constexpr (gi + 1 < NG) request(std::integral_constant<int, gi + 1>{}, wbuf[(gi + 1) & 1]);
        asm volatile("" ::: "memory");     // no read of a later group moves above this line
        __builtin_amdgcn_sched_barrier(0);
        static_for<gi * G, (gi * G + G < TB::N ? gi * G + G : TB::N)>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            constexpr int ia = TB::m[i][0], ib = TB::m[i][1], jc = TB::m[i][2];
            F w = wbuf[gi & 1][(i - gi * G) / V][(i - gi * G) % V];
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

}  // namespace
}  // namespace smx
