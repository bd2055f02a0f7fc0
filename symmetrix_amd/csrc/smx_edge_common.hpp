// What the edge kernels share: loads of spline and feature rows, lane broadcasts, sums over lanes, edge geometry, and how many
// wavefronts work on a receiver.
#pragma once

#include "smx_device.hpp"
#include "smx_kernels.hpp"

namespace smx {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename F>
constexpr bool kMatrix = sizeof(F) == 4;

// Lane-broadcast multiply-add of the double-precision kernels: acc += (b of lane N of the lane's 16-lane row) * v.  The
// instruction reads b through DPP, which needs two wait states after a vector instruction that wrote b.  Here b comes from LDS;
// that the compiler puts no move, spill or accumulator read of b in front of it is checked in the built code
// (check_device_code.py: the build fails otherwise).  Its own form of the move from another lane is an instruction by itself,
// not joined with the multiply-add: twice the instructions of these kernels' inner loops.
template <int N>
__device__ __forceinline__ void fmac_lane(double& acc, double b, double v)
{
    asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(b), "v"(v), "n"(N));
}
template <int N>
__device__ __forceinline__ void fmac_lane(float& acc, float b, float v)
{
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(b), "v"(v), "n"(N));
}

// Loads and stores of a wavefront's rows: an address that is the same for all lanes, held in scalar registers, plus a 32-bit
// offset per lane.
template <typename T>
__device__ __forceinline__ T load_at(const char* row, unsigned lane_bytes)
{
    return *reinterpret_cast<const T*>(row + lane_bytes);
}
// The four coefficients of one spline: 16 bytes in single precision, two halves of 16 bytes in double (a table row is
// [path][half][K][16 bytes], so that every load instruction of a wavefront covers 1 KB without gaps).
template <typename F>
__device__ __forceinline__ Vec<F, 4> load_spline(const char* row, int path, unsigned K, unsigned k16)
{
    if constexpr (sizeof(F) == 4) return load_at<Vec<F, 4>>(row + path * (K * 16), k16);
    else {
        Vec<F, 4> c;
        const Vec<F, 2> lo = load_at<Vec<F, 2>>(row + 2 * path * (K * 16), k16);
        const Vec<F, 2> hi = load_at<Vec<F, 2>>(row + (2 * path + 1) * (K * 16), k16);
        c.v[0] = lo.v[0]; c.v[1] = lo.v[1]; c.v[2] = hi.v[0]; c.v[3] = hi.v[1];
        return c;
    }
}
// The same for a row whose byte offset from the start of the array the lane holds (lanes of one wavefront on different rows).
template <typename F>
__device__ __forceinline__ Vec<F, 4> load_spline_off(const F* tab, int path, unsigned K, unsigned off)
{
    const char* t = reinterpret_cast<const char*>(tab);
    if constexpr (sizeof(F) == 4) return load_at<Vec<F, 4>>(t + path * (K * 16), off);
    else {
        Vec<F, 4> c;
        const Vec<F, 2> lo = load_at<Vec<F, 2>>(t + 2 * path * (K * 16), off), hi = load_at<Vec<F, 2>>(t + (2 * path + 1) * (K * 16), off);
        c.v[0] = lo.v[0]; c.v[1] = lo.v[1]; c.v[2] = hi.v[0]; c.v[3] = hi.v[1];
        return c;
    }
}
// row n of an array of rows of that many bytes, n the same in all lanes
__device__ __forceinline__ const char* uniform_row(const void* base, int n, unsigned row_bytes)
{
    return reinterpret_cast<const char*>(base) + (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane(n) * row_bytes;
}
// The byte offset of a lane, formed anew: the address of a load is then scalar registers plus 32 bits per lane.  An offset that
// stays the same is widened to 64 bits outside the loop otherwise, and every load pays for a 64-bit addition per lane (26 to 32
// of 590 instructions per edge in the general adjoint; without them 50 000 atoms, l <= 1, single precision 17.6 -> 17.2 ms).
__device__ __forceinline__ unsigned lane_offset(unsigned bytes)
{
    asm volatile("" : "+v"(bytes));
    return bytes;
}
// Where row n (the same in all lanes) of an array begins, in bytes, plus `part`: an offset that stays in scalar registers (or the
// compiler adds the part to every lane's address).
__device__ __forceinline__ unsigned long long uniform_offset(int n, unsigned row_bytes, unsigned part)
{
    unsigned long long at = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane(n) * row_bytes + part;
    asm volatile("" : "+s"(at));
    return at;
}
// The value is final here: keeps the compiler from collecting the arithmetic of several paths, whose operands would all stay
// live (it moves plain arithmetic across scheduling fences).
template <typename F>
__device__ __forceinline__ void pin(F& v)
{
    asm volatile("" : "+v"(v));
}

// The upper 32 lanes of a trade places with the lower 32 of b (swap_rows: the odd 16-lane rows of a with the even rows of b).
// Added up afterwards, that sums both values over the halves (rows), the first in the lower and the second in the upper lanes.
template <typename F>
__device__ __forceinline__ void swap_halves(F& a, F& b)
{
    if constexpr (sizeof(F) == 4) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
    } else {
        const unsigned long long x = __double_as_longlong(a), y = __double_as_longlong(b);
        const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
        a = __longlong_as_double(((unsigned long long)hi[0] << 32) | lo[0]);
        b = __longlong_as_double(((unsigned long long)hi[1] << 32) | lo[1]);
    }
}
template <typename F>
__device__ __forceinline__ void swap_rows(F& a, F& b)
{
    if constexpr (sizeof(F) == 4) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
    } else {
        const unsigned long long x = __double_as_longlong(a), y = __double_as_longlong(b);
        const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
        a = __longlong_as_double(((unsigned long long)hi[0] << 32) | lo[0]);
        b = __longlong_as_double(((unsigned long long)hi[1] << 32) | lo[1]);
    }
}
// What the lanes need of an edge before its features: spline interval and argument, table row, sender row.
template <typename F>
__device__ __forceinline__ void edge_head(const AggParams<F>& a, int e, int ti, double& r, double& x, int& row, int& grow)
{
    r = a.r[e];
    const int n = spline_interval(r, a.spl_inv_h, a.spl_nodes - 2);
    x = r - a.spl_h * n;
    row = a.pair_table[pair_index(a.T, ti, a.neigh_types[e])] * (a.spl_nodes - 1) + n;
    grow = a.gather[e];
}

// Direction of an edge and a frame orthogonal to it.  The harmonics depend on the direction only, so their gradient is
// tangential: the derivative along a tangent is that of the homogeneous form over the length.
struct EdgeFrame {
    double dx, dy, dz, inv;              // edge vector, 1 / length
    double nx, ny, nz;                   // direction
    double t1x, t1y, t1z, t2x, t2y, t2z; // tangents
};
__device__ __forceinline__ void edge_frame(const double* xyz, EdgeFrame& f)
{
    f.dx = xyz[0]; f.dy = xyz[1]; f.dz = xyz[2];
    f.inv = rsqrt_pos(f.dx * f.dx + f.dy * f.dy + f.dz * f.dz);
    f.nx = f.dx * f.inv; f.ny = f.dy * f.inv; f.nz = f.dz * f.inv;
    // t1 = n x a / |n x a| with a the axis the direction n is least aligned with (|n x a|^2 >= 2/3), t2 = n x t1
    const double ax = fabs(f.nx), ay = fabs(f.ny), az = fabs(f.nz);
    if (ax <= ay && ax <= az) { f.t1x = 0.0; f.t1y = f.nz; f.t1z = -f.ny; }
    else if (ay <= az) { f.t1x = -f.nz; f.t1y = 0.0; f.t1z = f.nx; }
    else { f.t1x = f.ny; f.t1y = -f.nx; f.t1z = 0.0; }
    const double tn = rsqrt_pos(f.t1x * f.t1x + f.t1y * f.t1y + f.t1z * f.t1z);
    f.t1x *= tn; f.t1y *= tn; f.t1z *= tn;
    f.t2x = f.ny * f.t1z - f.nz * f.t1y; f.t2y = f.nz * f.t1x - f.nx * f.t1z; f.t2z = f.nx * f.t1y - f.ny * f.t1x;
}
// harmonic LM and its derivatives along the two tangents (the harmonics' axes are the permuted ones: z, x, y)
template <int LM>
__device__ __forceinline__ void ylm_tangential(const EdgeFrame& f, double& Y, double& d1, double& d2)
{
    double g0, g1, g2;
    ylm_g<LM>(f.nz, f.nx, f.ny, Y, g0, g1, g2);
    d1 = (g0 * f.t1z + g1 * f.t1x + g2 * f.t1y) * f.inv;
    d2 = (g0 * f.t2z + g1 * f.t2x + g2 * f.t2y) * f.inv;
}

// ---- scalar sender features (smx_kernels_edge0.hip, smx_kernels_chain.hip)
// a b + c into a register of its own.  Left alone, the compiler copies c first and accumulates in the copy where the registers of c
// belong to the next load: 24 copies among the 218 instructions of the single-precision adjoint for 96 channels.
__device__ __forceinline__ float fma_apart(float a, float b, float c)
{
    float r;
    asm("v_fma_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ double fma_apart(double a, double b, double c) { return fma(a, b, c); }

constexpr int lm_of_tile(int t) { return t == 0 ? 0 : (t == 1 ? 1 : (t == 2 ? 4 : (t == 3 ? 8 : (t == 4 ? 9 : 13)))); }

// interval, argument and rows of an edge; offsets of its table and sender rows in bytes (32 bits: launch_agg0_ok)
template <typename F>
__device__ __forceinline__ void edge_offsets(const AggParams<F>& a, int e, int ti, unsigned row_bytes, unsigned sender_bytes, F* xs,
                                             unsigned* toff, unsigned* goff, int slot)
{
    double r, x;
    int row, grow;
    edge_head(a, e, ti, r, x, row, grow);
    xs[slot] = (F)x; toff[slot] = (unsigned)row * row_bytes; goff[slot] = (unsigned)grow * sender_bytes;
}

// Three sums over the lanes of each half-wavefront (EW = 2) or over all lanes (EW = 1).  On return lane 0 of the half
// holds s, lane 16 g1, lane 8 g2.  In single precision two lanes (up to eight channels) are added as they are, everything beyond
// in double: the forces come from sums over all channels, which cancel.
template <int EW, typename F>
__device__ __forceinline__ double edge_sum3(F s, F g1, F g2, int lane)
{
    if constexpr (EW == 1) {
        static_assert(sizeof(F) == 8, "half-wavefronts in single precision");
        F t = g2;
        swap_halves(s, t);
        F a = s + t;                     // lower half s, upper half g2
        F u = g1;
        swap_halves(g1, u);
        F b = g1 + u;                    // g1 in both
        swap_rows(a, b);                 // rows 0, 2: a, rows 1, 3: b
        F x = a + b;
        x = row_sum_strided<1>(x);       // row 0: s, row 1: g1, row 2: g2, row 3: g1
        return x;
    } else {
        F t = g2;
        swap_rows(s, g1);
        swap_rows(g2, t);
        F x = s + g1, y = g2 + t;        // rows 0, 2: s; rows 1, 3: g1; y: g2 in every row
        const F mine = (lane & 8) ? y : x, other = (lane & 8) ? x : y;      // the lane eight further on wants the other one
        double z = (double)mine + (double)row_rotate<8>(other);
        z += half_mirror(z); z += lane_xor1(z); z += lane_xor2(z);
        return z;
    }
}

// Messages to the senders: 0.1 to 5 GB written once, and read once by the next launch.  As ordinary stores they drove the
// spline tables and feature rows out of the L2s.
template <typename T>
__device__ __forceinline__ void store_stream(T* to, T v)
{
    __builtin_nontemporal_store(v, to);
}

// How many wavefronts share a receiver, of `units` receivers times channel groups.  A wavefront takes 0.5 to 2 us per edge,
// and about 2 048 of them are in flight: fewer units leave SIMDs idle, up to three rounds of them leave the last round
// nearly empty.  The adjoint gains up to three rounds (K = 128, l <= 1, single precision, 1 500 receivers: 214, 194, 157 us
// for one, two and four wavefronts); the forward kernel, which has to add the parts, only where the chip is not full
// (500 receivers: 52, 38, 41 us; 3 000: 153, 160, 163).
template <bool BWD>
int agg_parts(long units)
{
    if (BWD) return units <= 2048 ? 4 : (units <= 6144 ? 2 : 1);
    return units <= 512 ? 4 : (units <= 3072 ? 2 : 1);
}

}  // namespace
}  // namespace smx
