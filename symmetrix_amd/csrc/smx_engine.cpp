// Host orchestration and C ABI of the MACE energy+forces engine.
//
// Pipeline (the stage list of MACE::compute_node_energies_forces,
// libsymmetrix/source/mace.cpp:17-64), one HIP kernel or one batched MFMA
// launch per stage, all on one stream, nothing computed on the host:
//
//   prep        CSR offsets, sender lists, species groups        (integers only)
//   agg0_fwd    Phi0 = sum_j R0 Y H0                             mace.cpp:158-178
//   A0_lin      A0 = Phi0 . A0_weights[type][l]        (MFMA)    mace.cpp:180-199
//   M0          symmetric contraction + gradient                 mace.cpp:348-370
//   H1          H1 = M0 . H1_weights[l]                (MFMA)    mace.cpp:397-423
//   agg1_fwd    Phi1 = CG . sum_j R1 Y H1[j]                     mace.cpp:453-502
//   A1          A1 = Phi1 . A1_weights[l]              (MFMA)    mace.cpp:607-642
//   M1          symmetric contraction + gradient                 mace.cpp:759-777
//   H2          H2 = H1[l=0].W[type] + M1.W            (MFMA)    mace.cpp:796-832
//   readout     energies, H1_adj seed, H2_adj          (MFMA)    mace.cpp:876-903
//   rev_H2, rev_M1, rev_A1, agg1_bwd, sender_reduce, rev_H1, rev_M0,
//   rev_A0_lin, agg0_bwd                                         mace.cpp:54-63
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/symmetrix_amd.h"
#include "smx_host_model.hpp"
#include "smx_internal.hpp"
#include "smx_json.hpp"
#include "smx_kernels.hpp"
#include "smx_paths.hpp"

namespace smx {

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

static thread_local std::string g_last_error;

#define HIPCHK(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            throw ::smx::Error(e_ == hipErrorOutOfMemory ? SMX_ENOMEM : SMX_EHIP,                      \
                        std::string(#expr) + ": " + hipGetErrorString(e_));                            \
    } while (0)

// growable device array with std::vector::resize semantics (contents kept, new tail zeroed)
template <typename T>
struct DVec {
    T* p = nullptr;
    size_t n = 0, cap = 0;
    ~DVec() { if (p) (void)hipFree(p); }
    DVec() = default;
    DVec(const DVec&) = delete;
    DVec& operator=(const DVec&) = delete;
    void reserve(size_t m, hipStream_t s, bool keep)
    {
        if (m <= cap) return;
        // headroom against regrowth when the edge count drifts: an eighth, a sixty-fourth for buffers beyond 1 GiB
        const size_t newcap = m + (m * sizeof(T) > ((size_t)1 << 30) ? m / 64 : m / 8) + 64;
        T* q = nullptr;
        if (p && !(keep && n)) {
            // nothing to carry over: release first, so that the two sizes never coexist
            HIPCHK(hipStreamSynchronize(s));
            HIPCHK(hipFree(p));
            p = nullptr; cap = 0; n = 0;
        }
        HIPCHK(hipMalloc(&q, newcap * sizeof(T)));
        if (p) {
            HIPCHK(hipMemcpyAsync(q, p, n * sizeof(T), hipMemcpyDeviceToDevice, s));
            HIPCHK(hipStreamSynchronize(s));
            HIPCHK(hipFree(p));
        }
        p = q;
        cap = newcap;
    }
    // size to m elements; previous contents are undefined afterwards
    void size_to(size_t m, hipStream_t s) { reserve(m ? m : 1, s, false); n = m; }
    // std::vector::resize
    void resize(size_t m, hipStream_t s)
    {
        reserve(m ? m : 1, s, true);
        if (m > n) HIPCHK(hipMemsetAsync(p + n, 0, (m - n) * sizeof(T), s));
        n = m;
    }
    void upload(const T* host, size_t m, hipStream_t s)
    {
        size_to(m, s);
        if (m) HIPCHK(hipMemcpyAsync(p, host, m * sizeof(T), hipMemcpyHostToDevice, s));
    }
};

// Growable pinned host array: copies between it and the device are asynchronous and go through no staging of the runtime's.
// Whoever fills it again has waited for the last copy from or to it.
template <typename T>
struct HostBuf {
    T* p = nullptr;
    size_t cap = 0;
    ~HostBuf() { if (p) (void)hipHostFree(p); }
    HostBuf() = default;
    HostBuf(const HostBuf&) = delete;
    HostBuf& operator=(const HostBuf&) = delete;
    T* room(size_t m)
    {
        if (m > cap) {
            const size_t newcap = m + m / 8 + 64;
            if (p) { HIPCHK(hipHostFree(p)); p = nullptr; cap = 0; }
            HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&p), newcap * sizeof(T)));
            cap = newcap;
        }
        return p;
    }
};
// Host to device in pieces through a ring of pinned slots: the copy of one piece runs while the next is being filled.
struct Uploader {
    static constexpr size_t SLOT = (size_t)2 << 20;
    static constexpr int SLOTS = 4;
    HostBuf<char> ring;
    hipEvent_t done[SLOTS] = {};
    bool busy[SLOTS] = {};
    int slot = 0;
    size_t fill = 0;          // bytes of the current slot taken
    ~Uploader() { for (auto& e : done) if (e) (void)hipEventDestroy(e); }
    void put(char* dst, const void* src_, size_t n, hipStream_t s)
    {
        const char* src = static_cast<const char*>(src_);
        ring.room(SLOT * SLOTS);
        while (n > 0) {
            if (fill == 0 && busy[slot]) { HIPCHK(hipEventSynchronize(done[slot])); busy[slot] = false; }
            const size_t m = std::min(n, SLOT - fill);
            char* at = ring.p + (size_t)slot * SLOT + fill;
            std::memcpy(at, src, m);
            HIPCHK(hipMemcpyAsync(dst, at, m, hipMemcpyHostToDevice, s));
            dst += m; src += m; n -= m; fill += (m + 255) / 256 * 256;
            if (fill >= SLOT) next(s);
        }
    }
    // n bytes of an empty slot, to be filled and copied by the caller
    char* take(size_t n)
    {
        ring.room(SLOT * SLOTS);
        if (busy[slot]) { HIPCHK(hipEventSynchronize(done[slot])); busy[slot] = false; }
        fill = n;
        return ring.p + (size_t)slot * SLOT;
    }
    // the current slot is not written again before its copies are done
    void next(hipStream_t s)
    {
        if (fill == 0) return;
        if (!done[slot]) HIPCHK(hipEventCreateWithFlags(&done[slot], hipEventDisableTiming));
        HIPCHK(hipEventRecord(done[slot], s));
        busy[slot] = true;
        slot = (slot + 1) % SLOTS;
        fill = 0;
    }
};

template <typename T, typename S>
static void upload_as(DVec<T>& d, const std::vector<S>& h, hipStream_t s)
{
    std::vector<T> tmp(h.begin(), h.end());
    d.upload(tmp.data(), tmp.size(), s);
    HIPCHK(hipStreamSynchronize(s));  // tmp goes out of scope
}

// the bf16 number nearest to x, as its bits, and back
static unsigned short bf16_of(float x)
{
    unsigned u;
    std::memcpy(&u, &x, 4);
    if (x != x) return 0x7fc0;
    return (unsigned short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
static float float_of_bf16(unsigned short h)
{
    const unsigned u = (unsigned)h << 16;
    float x;
    std::memcpy(&x, &u, 4);
    return x;
}

static const char* kStageNames =
    "prep;agg0_fwd;A0_lin;M0;H1;agg1_fwd;A1;M1;H2;readout;rev_H2;rev_M1;rev_A1;agg1_bwd;sender_reduce;"
    "rev_H1;rev_M0;rev_A0_lin;agg0_bwd;force_sum1;force_sum0";
enum Stage { ST_PREP, ST_AGG0F, ST_A0LIN, ST_M0, ST_H1, ST_AGG1F, ST_A1, ST_M1, ST_H2, ST_READOUT, ST_REVH2,
             ST_REVM1, ST_REVA1, ST_AGG1B, ST_SRED, ST_REVH1, ST_REVM0, ST_REVA0LIN, ST_AGG0B, ST_FSUM1, ST_FSUM0, ST_COUNT };

struct EngineBase {
    virtual ~EngineBase()
    {
        for (int i = 0; i < ST_COUNT; ++i) {
            if (ev0[i]) (void)hipEventDestroy(ev0[i]);
            if (ev1[i]) (void)hipEventDestroy(ev1[i]);
        }
    }
    HostModel hm;
    int precision = 0;
    int poly_tables = 0;            // bit 0 / bit 1: layer 0 / layer 1 contraction runs the table-specialised kernel
    int contraction_tables() const { return poly_tables; }
    int edges_in_chains = 0;        // bit 0 / bit 1: the chains of the last evaluation took the aggregation of layer 0 / layer 1 along
    int device = 0;                 // ordinal of the GPU the model was loaded on
    hipStream_t stream = nullptr;   // stream of the current call
    bool profiling = false;
    hipEvent_t ev0[ST_COUNT] = {}, ev1[ST_COUNT] = {};
    bool ev_used[ST_COUNT] = {};
    int H1_rows_override = -1;
    size_t msg_limit_bytes = (size_t)32 << 30;   // staging buffer of the layer-1 adjoint messages

    virtual void compute(int N, const int* node_types, const int* num_neigh, const int* neigh_indices,
                         const int* neigh_types, const double* xyz, const double* r, long E, bool on_device,
                         double* d_energies, double* d_forces, int N_local, long E_local) = 0;
    virtual void stage(const char* name, int N, const int* node_types, const int* num_neigh,
                       const int* neigh_indices, const int* neigh_types, const double* xyz, const double* r,
                       long E, int flag_a, int flag_b) = 0;
    virtual void get_array(const char* name, double* out, long cap, long* n) = 0;
    virtual void set_array(const char* name, const double* in, long n) = 0;
    virtual void fill_array(const char* name, long n, double value) = 0;
    virtual void forces_view(ForcesView* v) = 0;
    virtual void check_device_status(bool on_device) = 0;   // the stream has been waited for
    virtual void finish_host_call() = 0;                    // waits; an evaluation of host arrays that was refused raises
    virtual void evaluate_list(int N, const int* node_types, const int* num_neigh, const int* neigh_indices,
                               const int* neigh_types, const double* xyz, const double* r, long E, double* energies,
                               double* forces, double* virial) = 0;
    virtual void reduce_forces(int num_atoms, const int* sender_atom, const int* receiver_atom,
                               double* atom_forces, double* virial, bool sender_on_device) = 0;

    void stage_begin(int st)
    {
        if (!profiling) return;
        if (!ev0[st]) { HIPCHK(hipEventCreate(&ev0[st])); HIPCHK(hipEventCreate(&ev1[st])); }
        HIPCHK(hipEventRecord(ev0[st], stream));
    }
    void stage_end(int st)
    {
        if (!profiling) return;
        HIPCHK(hipEventRecord(ev1[st], stream));
        ev_used[st] = true;
    }
    // a stage without a launch of its own: another one's does its work, or there is none
    void stage_absent(int st) { ev_used[st] = false; }
};

template <typename F>
struct Engine : EngineBase {
    // ---- model on device
    DVec<F> tab0, tab1, tabK0, tabK1, H0, A0w, H1w, A1w;
    DVec<F> linA0, linA0T, linA1, linA1T;    // the same weights in operand order (operand_weights)
    DVec<unsigned short> splitA0, splitA0T, splitA1, splitA1T;    // ... and in single precision in three bf16 parts (split_weights)
    DVec<F> H1wT;                            // transposes, for the kernels that take a chain of stages
    DVec<int> pair_table0, pair_table1;
    DVec<int> B0_start, B0_lm1, B1_start, B1_lm1;
    DVec<double> B0_c, B1_c;
    std::vector<long> A1w_off;   // per l
    int num_cus = 0;
    int more_terms1 = 0;       // an entry of layer 1's coupling list has more than two terms
    int split_nodes = 0;       // receivers that are not ghosts, of the evaluation under way
    bool diagonal1 = false;    // scalar hidden features, and output lm of layer 1 is fed by cdiag1[lm] Y_lm alone
    double cdiag1[16] = {};
    bool selected1 = false;            // layer 1 couples by the selection rules only; with the constant harmonic, by these factors
    double c_same1[9] = {};
    DVec<double> fpart;
    DVec<double> H2w_H1, H2w_M1, H2v_H1, H2v_M1, ro1, ro2_w1, ro2_w2, E0;
    struct DevPoly {
        DVec<int> packed, chunks;
        DVec<F> coef;
        int num_entries = 0;
    };
    std::vector<std::unique_ptr<DevPoly>> P0;
    DevPoly P1;
    // pointer tables for the polynomial kernel: [0..num_LM) = P0, then P1
    DVec<const int4*> pp_packed;
    DVec<const int*> pp_chunks;
    DVec<const F*> pp_coef;
    DVec<F> M0_slabs, M1_slabs;   // contraction coefficients by column tile (smx_poly_shape.hpp)
    DVec<int> pp_nent;
    bool M0_tables = false, M1_tables = false;   // every polynomial of the layer maps onto its compile-time table

    // ---- geometry of the current edge list (device)
    DVec<int> g_node_types, g_num_neigh, g_neigh_indices, g_neigh_types;
    DVec<char> g_in;               // host arrays of a whole-pipeline call, one behind the other
    Uploader uploader;
    HostBuf<char> host_out;        // results on their way to the caller
    HostBuf<int> sticky;           // failed input checks not yet reported: [0] device-resident calls, [1] host-array calls
    DVec<double> g_xyz, g_r;
    const int *node_types = nullptr, *num_neigh = nullptr, *neigh_indices = nullptr, *neigh_types = nullptr;
    const double *xyz = nullptr, *r = nullptr;
    long E = 0;
    long E1 = 0;   // leading edges whose receivers take part in layer 1 (all of them unless ghost nodes follow)
    int N_geo = 0;
    long geo_edges = 0;   // edges of the N_geo receivers
    DVec<int> first_neigh, scan_tmp, s_count, s_start, s_list, t_count, t_start, t_cursor, t_perm, flags;
    int sender_rows = 0;
    long sender_edges = -1;        // edges that s_start / s_list cover
    bool guarded = false;          // offsets and lists are those of a whole-pipeline call, emptied if its checks failed (flags[3])
    bool evaluating = false;       // a whole-pipeline call has begun to replace what the one before left
    bool refused = false;          // the last one failed: there are no forces until something else makes some
    bool senders_differ = false;   // a caller's sender atoms were not the senders of the evaluation before
    // pair terms: ZBL constants per species pair, density-normalisation splines, divisors of the last forward pass
    DVec<double> zbl_a, zbl_rmax, zbl_zz, A0spl, A1spl, div0, div1;
    ZblParams zbl_params() const
    {
        ZblParams z{};
        z.T = hm.T; z.a_pair = zbl_a.p; z.rmax_pair = zbl_rmax.p; z.zz_pair = zbl_zz.p;
        for (int q = 0; q < 4; ++q) z.c[q] = hm.zbl_c[q];
        z.p = hm.zbl_p;
        return z;
    }
    PairSpline scale_spline(int layer) const
    {
        PairSpline sp{};
        sp.c = layer == 0 ? A0spl.p : A1spl.p;
        sp.h = layer == 0 ? hm.A0_spline_h : hm.A1_spline_h;
        sp.nodes = layer == 0 ? hm.A0_spline_nodes : hm.A1_spline_nodes;
        return sp;
    }
    // caller's output arrays of the running whole-pipeline call; the kernel that forms the final values writes
    // them too and clears the pointer, otherwise a copy is enqueued at the end
    double* energies_copy = nullptr;
    double* forces_copy = nullptr;
    bool senders_counted = false;   // the sender histogram (and s_rank) was formed by the fused node-list launch
    DVec<int> s_rank;               // place of every edge inside its sender's bucket, until the buckets are filled; then scratch
    long counters_clean = 0;        // leading entries of s_count known to be zero (every sender-list build leaves them so)
    long rf_clean = 0;              // the same for rf_count

    // ---- state (mace.hpp members)
    DVec<F> dPhi0;     // adjoint of Phi0 where Phi0 stays (separate_dPhi0), else it takes Phi0's place
    DVec<F> Phi0, A0, A0_adj, M0, M0_grad, M0_adj, H1, H1_adj, Phi1, dPhi1, A1, A1_adj, M1, M1_grad, M1_adj, msg;
    DVec<double> H2, H2_adj, node_energies, node_forces, scratch_d;

    int K() const { return hm.K; }
    int NLM() const { return hm.num_LM; }
    int NE() const { return hm.num_lme; }

    explicit Engine(HostModel&& m, int prec)
    {
        hm = std::move(m);
        precision = prec;
        HIPCHK(hipGetDevice(&device));
        hipStream_t s = nullptr;
        auto cat = [](const std::vector<std::vector<double>>& t) {
            std::vector<double> out;
            for (auto& v : t) out.insert(out.end(), v.begin(), v.end());
            return out;
        };
        upload_as(tab0, cat(hm.tables0), s);
        upload_as(tab1, cat(hm.tables1), s);
        upload_as(pair_table0, hm.pair_table0, s);
        upload_as(pair_table1, hm.pair_table1, s);
        upload_as(H0, hm.H0_weights, s);
        upload_as(A0w, hm.A0_weights, s);
        upload_as(H1w, hm.H1_weights, s);
        {
            std::vector<double> all;
            for (auto& w : hm.A1_weights) { A1w_off.push_back((long)all.size()); all.insert(all.end(), w.begin(), w.end()); }
            upload_as(A1w, all, s);
        }
        // layer 1 with scalar hidden features: whether every output lm is fed by harmonic lm alone
        diagonal1 = hm.L_max == 0 && hm.num_B == 16;
        for (int b = 0; diagonal1 && b < 16; ++b) {
            cdiag1[b] = 0.0;
            for (int t = hm.B_start[b]; t < hm.B_start[b + 1]; ++t) {
                if (hm.B_lm1[t] != b) diagonal1 = false;
                else cdiag1[b] += hm.B_c[t];
            }
        }
        // the edge kernels read the tables as [interval][path][channel][4 coefficients], in double in two halves of 16 bytes
        // per channel: one load instruction of a wavefront (one path, consecutive channels) then covers contiguous memory
        auto regroup = [&](const std::vector<std::vector<double>>& tables, int nspl, DVec<F>& dst) {
            const int R = hm.spl_nodes - 1, Kc = hm.K, Pn = nspl / Kc;
            std::vector<double> out((size_t)tables.size() * R * nspl * 4);
            constexpr int V = 16 / sizeof(F);      // coefficients of 16 bytes stay together
            size_t o = 0;
            for (auto& t : tables)
                for (int n = 0; n < R; ++n)
                    for (int pth = 0; pth < Pn; ++pth)
                        for (int h = 0; h < 4; h += V)
                            for (int k = 0; k < Kc; ++k)
                                for (int q = h; q < h + V; ++q) out[o++] = t[((size_t)n * 4 + q) * nspl + pth * Kc + k];
            upload_as(dst, out, s);
        };
        regroup(hm.tables0, hm.nspl0, tabK0);
        regroup(hm.tables1, hm.nspl1, tabK1);
        // layer 0 couples Y_lm straight into output slot lm
        {
            std::vector<int> st(17), lm(16);
            std::vector<double> c(16, 1.0);
            for (int q = 0; q < 16; ++q) { st[q] = q; lm[q] = q; }
            st[16] = 16;
            upload_as(B0_start, st, s); upload_as(B0_lm1, lm, s); upload_as(B0_c, c, s);
        }
        upload_as(B1_start, hm.B_start, s);
        upload_as(B1_lm1, hm.B_lm1, s);
        upload_as(B1_c, hm.B_c, s);
        selected1 = true;
        for (int pth = 0, b0 = 0; pth < hm.num_paths; ++pth) {
            const int l = hm.Phi1_l[pth], l1 = hm.Phi1_l1[pth], l2 = hm.Phi1_l2[pth], n = 2 * l + 1, n2 = 2 * l2 + 1;
            for (int m = 0; m < n; ++m)
                for (int m2 = 0; m2 < n2; ++m2) {
                    const int b = b0 + m * n2 + m2;
                    double c = 0.0;
                    for (int t = hm.B_start[b]; t < hm.B_start[b + 1]; ++t) {
                        selected1 = selected1 && (l1 != 0 || hm.B_lm1[t] == 0) && (components_couple(l, m, l1, l2, m2) || hm.B_c[t] == 0.0);
                        c += hm.B_c[t];
                    }
                    if (l1 == 0 && m == m2) c_same1[l * l + m] = c;
                }
            b0 += n * n2;
        }
        for (int b = 0; b < hm.num_B; ++b) more_terms1 |= hm.B_start[b + 1] - hm.B_start[b] > 2;
        upload_as(H2w_H1, hm.H2_weights_for_H1, s);
        upload_as(H2w_M1, hm.H2_weights_for_M1, s);
        {
            // first layer of the readout network times the transposed weights of H2: the gradient of H2 has rank 16
            auto through_readout = [&](const std::vector<double>& w, auto& dst) {
                const size_t Kc = hm.K, n = w.size() / (Kc * Kc);
                std::vector<double> out(n * 16 * Kc);
                for (size_t b = 0; b < n; ++b)
                    for (size_t h = 0; h < 16; ++h)
                        for (size_t i = 0; i < Kc; ++i) {
                            double sum = 0.0;
                            for (size_t j = 0; j < Kc; ++j) sum += hm.readout_2_w1[h * Kc + j] * w[(b * Kc + i) * Kc + j];
                            out[(b * 16 + h) * Kc + i] = sum;
                        }
                upload_as(dst, out, s);
            };
            if (tail_fused_ok(hm.K)) { through_readout(hm.H2_weights_for_H1, H2v_H1); through_readout(hm.H2_weights_for_M1, H2v_M1); }
        }
        upload_as(ro1, hm.readout_1_weights, s);
        upload_as(ro2_w1, hm.readout_2_w1, s);
        upload_as(ro2_w2, hm.readout_2_w2, s);
        upload_as(E0, hm.atomic_energies, s);
        if (hm.has_zbl) {
            // zbl.cpp:22-35: screening length and envelope radius of every ordered species pair
            const int T = hm.T;
            std::vector<double> a((size_t)T * T), rm((size_t)T * T), zz((size_t)T * T);
            for (int i = 0; i < T; ++i)
                for (int j = 0; j < T; ++j) {
                    const int Zi = hm.atomic_numbers[i], Zj = hm.atomic_numbers[j];
                    if (Zi < 0 || Zj < 0 || Zi >= (int)hm.zbl_covalent_radii.size() || Zj >= (int)hm.zbl_covalent_radii.size())
                        throw Error(SMX_EFILE, "model file: zbl_covalent_radii does not cover the atomic numbers of the model");
                    a[(size_t)i * T + j] = hm.zbl_a_prefactor * 0.529 / (std::pow((double)Zi, hm.zbl_a_exp) + std::pow((double)Zj, hm.zbl_a_exp));
                    rm[(size_t)i * T + j] = hm.zbl_covalent_radii[Zi] + hm.zbl_covalent_radii[Zj];
                    zz[(size_t)i * T + j] = (double)Zi * (double)Zj;
                }
            upload_as(zbl_a, a, s); upload_as(zbl_rmax, rm, s); upload_as(zbl_zz, zz, s);
        }
        if (hm.A0_scaled) upload_as(A0spl, hm.A0_spline_c, s);
        if (hm.A1_scaled) upload_as(A1spl, hm.A1_spline_c, s);
        auto up_poly = [&](DevPoly& d, const PolySpec& p) {
            upload_as(d.packed, p.packed, s); upload_as(d.chunks, p.chunks, s);
            upload_as(d.coef, p.coef, s);
            d.num_entries = p.num_entries;
        };
        std::vector<const int4*> vpk;
        std::vector<const int*> vch;
        std::vector<const F*> vco;
        std::vector<int> vne;
        auto reg = [&](DevPoly& d) {
            vpk.push_back(reinterpret_cast<const int4*>(d.packed.p)); vch.push_back(d.chunks.p);
            vco.push_back(d.coef.p); vne.push_back(d.num_entries);
        };
        for (int LM = 0; LM < hm.num_LM; ++LM) {
            P0.emplace_back(new DevPoly());
            up_poly(*P0.back(), hm.P0[LM]);
            reg(*P0.back());
        }
        up_poly(P1, hm.P1);
        reg(P1);
        pp_packed.upload(vpk.data(), vpk.size(), s); pp_chunks.upload(vch.data(), vch.size(), s);
        pp_coef.upload(vco.data(), vco.size(), s);
        pp_nent.upload(vne.data(), vne.size(), s);
        M0_tables = hm.num_LM == 1 || hm.num_LM == 4 || hm.num_LM == 9;
        for (int LM = 0; LM < hm.num_LM; ++LM) M0_tables = M0_tables && hm.P0[LM].table == LM;
        M1_tables = hm.P1.table == 0;
        M0_tables = M0_tables && poly_spec_shape((int)sizeof(F), hm.K, hm.num_LM).CB > 0;
        M1_tables = M1_tables && poly_spec_shape((int)sizeof(F), hm.K, 1).CB > 0;
        // slabs of the straight-line polynomials: [species][column tile][monomial / V][16][V]
        auto slabs = [&](DVec<F>& dst, const PolySpec* polys, int NP) {
            constexpr int V = 16 / (int)sizeof(F);
            const size_t tiles = (size_t)(hm.K + 15) / 16, slab = (size_t)poly_spec_offset(NP) * 16;
            std::vector<F> h((size_t)hm.T * tiles * slab, F(0));
            for (int P = 0; P < NP; ++P) {
                const int tn = kPolyTableLen[polys[P].table], m0 = poly_spec_offset(P);
                for (int t = 0; t < hm.T; ++t)
                    for (int i = 0; i < tn; ++i)
                        for (int k = 0; k < hm.K; ++k) {
                            const int m = m0 + i;
                            h[((size_t)t * tiles + k / 16) * slab + ((size_t)(m / V) * 16 + k % 16) * V + m % V] =
                                (F)polys[P].table_coef[((size_t)t * tn + i) * hm.K + k];
                        }
            }
            dst.upload(h.data(), h.size(), s);
            HIPCHK(hipStreamSynchronize(s));   // h goes out of scope
        };
        if (num_cus == 0) {
            hipDeviceProp_t prop;
            HIPCHK(hipGetDeviceProperties(&prop, device));
            num_cus = prop.multiProcessorCount;
        }
        if (M0_tables) slabs(M0_slabs, hm.P0.data(), hm.num_LM);
        if (M1_tables) slabs(M1_slabs, &hm.P1, 1);
        if (linear_ok(hm.K)) {
            const bool chain = chain_ok(hm.K) && M0_tables && M1_tables;
            operand_weights(s);
            if (sizeof(F) == 4 && (hm.K % 128 == 0 || hm.K % 96 == 0)) split_weights(s);
            if (chain) {
                auto transposed = [&](const std::vector<double>& w, auto& dst) {
                    const size_t Kc = hm.K, n = w.size() / (Kc * Kc);
                    std::vector<double> out(w.size());
                    for (size_t b = 0; b < n; ++b)
                        for (size_t i = 0; i < Kc; ++i)
                            for (size_t j = 0; j < Kc; ++j) out[(b * Kc + j) * Kc + i] = w[(b * Kc + i) * Kc + j];
                    upload_as(dst, out, s);
                };
                transposed(hm.H1_weights, H1wT);
            }
        }
        poly_tables = (M0_tables ? 1 : 0) | (M1_tables ? 2 : 0);
        flags.resize(8, s);
        sticky.room(2); sticky.p[0] = sticky.p[1] = 0;
        HIPCHK(hipStreamSynchronize(s));
    }

    // Every matrix of the A-basis linears and of their adjoints, in the order [l][type][output block]: f(inner size, B(k, n)); done(i)
    // after the last one of an array: 0 A0, 1 its transpose, 2 A1, 3 its transpose.
    template <typename Block, typename Done>
    void linear_weights(Block&& block, Done&& done)
    {
        const int K = hm.K;
        for (int pass = 0; pass < 2; ++pass) {
            for (int l = 0; l < 4; ++l)
                for (int t = 0; t < hm.T; ++t) {
                    const double* w = hm.A0_weights.data() + ((size_t)t * 4 + l) * K * K;
                    block(K, [&](int k, int n) { return pass ? w[(size_t)n * K + k] : w[(size_t)k * K + n]; });
                }
            done(pass);
        }
        for (int l = 0; l < 4; ++l) {
            const double* w = hm.A1_weights[l].data();
            block(hm.num_e[l] * K, [&](int k, int n) { return w[(size_t)k * K + n]; });
        }
        done(2);
        for (int l = 0; l < 4; ++l)
            for (int eb = 0; eb < hm.num_e[l]; ++eb) {
                const double* w = hm.A1_weights[l].data();
                block(K, [&](int k, int n) { return w[((size_t)eb * K + n) * K + k]; });
            }
        done(3);
    }
    // ... in the operand order of k_linear and of the chains, [column tile][step][64][V]
    void operand_weights(hipStream_t s)
    {
        constexpr int V = 16 / (int)sizeof(F);
        std::vector<double> out;
        linear_weights([&](int inner, auto&& B) {
            for (int ct = 0; ct < hm.K / 16; ++ct)
                for (int st = 0; st < inner / (4 * V); ++st)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int v = 0; v < V; ++v) out.push_back(B(4 * V * st + lane / 16 * V + v, ct * 16 + lane % 16));
        }, [&](int i) {
            DVec<F>* const to[4] = {&linA0, &linA0T, &linA1, &linA1T};
            upload_as(*to[i], out, s);
            out.clear();
        });
    }
    // ... of k_linear32: [column tile][piece of 32 terms][part][64][8], w kSplitScale = part 0 + part 1 + part 2 in bf16, rounded to nearest
    void split_weights(hipStream_t s)
    {
        std::vector<unsigned short> out;
        linear_weights([&](int inner, auto&& B) {
            for (int ct = 0; ct < hm.K / 16; ++ct)
                for (int st = 0; st < inner / 32; ++st) {
                    const size_t at = out.size();
                    out.resize(at + 3 * 512);
                    for (int i = 0; i < 512; ++i) {
                        float rest = (float)B(32 * st + i / 128 * 8 + i % 8, ct * 16 + i / 8 % 16) * kSplitScale;
                        for (int part = 0; part < 3; ++part) {
                            const unsigned short h = bf16_of(rest);
                            out[at + part * 512 + i] = h;
                            rest -= float_of_bf16(h);
                        }
                    }
                }
        }, [&](int i) {
            DVec<unsigned short>* const to[4] = {&splitA0, &splitA0T, &splitA1, &splitA1T};
            to[i]->upload(out.data(), out.size(), s);
            HIPCHK(hipStreamSynchronize(s));   // out changes
            out.clear();
        });
    }

    // ---- input checks of an evaluation.  flags[0]: stage-level calls (read back at once); flags[2]: the word the checks
    // of the running evaluation raise; flags[3]: its copy for the kernels after the list preparation ("live": raised ->
    // energies and forces are NaN); flags[4]: ticket of the list preparation, flags[5]: of the virial (both zero between launches).  The evaluation clears flags[2] again in its
    // readout launch, after the last reader, so every evaluation, eager or a replayed graph, starts from a clean word.
    // sticky: what failed and has not been reported, in host memory, written by the list preparation and read by the next
    // call that waits for the stream (a host-array call reports at its own end).
    int* guard_status = nullptr;   // check word of the running evaluation
    bool guard_clear_enqueued = false;   // ... and a launch that clears it again is in the stream
    bool guard_on_device = false;
    const int* guard_live() const { return guard_status ? flags.p + 3 : nullptr; }
    InputGuard input_guard(int N)
    {
        InputGuard g;
        if (!guard_status) return g;
        g.status = guard_status;
        g.live = flags.p + 3;
        g.sticky = sticky.p + (guard_on_device ? 0 : 1);
        g.first_neigh = first_neigh.p; g.n_first = N + 1;
        g.tstart = t_start.p; g.n_tstart = hm.T + 1;
        return g;
    }
    void check_device_status(bool on_device) override
    {
        volatile int* w = sticky.p + (on_device ? 0 : 1);
        const int f = *w;
        if (!f) return;
        *w = 0;
        const std::string what = on_device ? "a device-resident evaluation was skipped: " : "";
        const std::string then = on_device ? " (its node energies and forces are NaN)" : "";
        if (f & 1)
            throw Error(SMX_EINVAL, what + "node_types / neigh_types / neigh_indices hold an index outside the model or the node range" +
                                    (on_device ? ", or num_neigh does not add up to the number of edges" : "") + then);
        throw Error(SMX_ERANGE, what + "an edge length lies outside (0, r_cut): the radial spline tables do not cover it" + then);
    }

    // ------------------------------------------------------------------
    // geometry handling

    // What a failed evaluation leaves is not used again: unchecked indices on the device, emptied lists, forces that were never
    // computed.  Stage calls then need their inputs anew, and there is nothing to reduce.
    void forget_evaluation()
    {
        node_types = num_neigh = neigh_indices = neigh_types = nullptr;
        xyz = r = nullptr;
        E = E1 = geo_edges = 0; N_geo = 0;
        sender_rows = -1; sender_edges = -1; guarded = false;
        node_forces.n = node_energies.n = 0;
        pending_A1_adj = pending_A0_adj = pending_A1 = pending_A0 = pending_M0_grad = -1;
        refused = true;
    }
    bool has_forces() const { return !refused || node_forces.n > 0; }
    // word that tells whether the evaluation whose lists are in place was skipped
    const int* skipped_word() const { return guarded ? flags.p + 3 : nullptr; }
    void finish_host_call() override
    {
        HIPCHK(hipStreamSynchronize(stream));
        try {
            check_device_status(false);
        } catch (...) {
            forget_evaluation();
            throw;
        }
    }
    void set_geometry_ptrs(int N, const int* nt, const int* nn, const int* ni, const int* nty, const double* x,
                           const double* rr, long E_, bool on_device)
    {
        hipStream_t s = stream;
        if (on_device) {
            if (nt) node_types = nt;
            if (nn) num_neigh = nn;
            if (ni) neigh_indices = ni;
            if (nty) neigh_types = nty;
            if (x) xyz = x;
            if (rr) r = rr;
        } else {
            if (nt) { g_node_types.upload(nt, N, s); node_types = g_node_types.p; }
            if (nn) { g_num_neigh.upload(nn, N, s); num_neigh = g_num_neigh.p; }
            if (ni) { g_neigh_indices.upload(ni, E_, s); neigh_indices = g_neigh_indices.p; }
            if (nty) { g_neigh_types.upload(nty, E_, s); neigh_types = g_neigh_types.p; }
            if (x) { g_xyz.upload(x, 3 * E_, s); xyz = g_xyz.p; }
            if (rr) { g_r.upload(rr, E_, s); r = g_r.p; }
        }
        if (E_ >= 0) { E = E_; E1 = E_; }
    }
    // the host arrays of a whole-pipeline call
    void upload_inputs(int N, const int* nt, const int* nn, const int* ni, const int* nty, const double* x, const double* rr, long E_)
    {
        auto up = [](size_t n) { return (n + 255) / 256 * 256; };
        const size_t n4 = up((size_t)N * 4), e4 = up((size_t)E_ * 4), e8 = up((size_t)E_ * 8), e24 = up((size_t)E_ * 24);
        g_in.size_to(2 * n4 + 2 * e4 + e8 + e24, stream);
        char* d = g_in.p;
        const bool one = g_in.n <= Uploader::SLOT;   // small: the arrays laid out in one slot, one copy
        char* h = one ? uploader.take(g_in.n) : nullptr;
        auto put = [&](const void* src, size_t bytes, size_t room) {
            char* at = d;
            if (bytes && one) std::memcpy(h + (at - g_in.p), src, bytes);
            else if (bytes) uploader.put(at, src, bytes, stream);
            d += room;
            return at;
        };
        node_types = reinterpret_cast<int*>(put(nt, (size_t)N * 4, n4));
        num_neigh = reinterpret_cast<int*>(put(nn, (size_t)N * 4, n4));
        neigh_indices = reinterpret_cast<int*>(put(ni, (size_t)E_ * 4, e4));
        neigh_types = reinterpret_cast<int*>(put(nty, (size_t)E_ * 4, e4));
        r = reinterpret_cast<double*>(put(rr, (size_t)E_ * 8, e8));
        xyz = reinterpret_cast<double*>(put(x, (size_t)E_ * 24, e24));
        if (one && g_in.n) HIPCHK(hipMemcpyAsync(g_in.p, h, g_in.n, hipMemcpyHostToDevice, stream));
        uploader.next(stream);
        E = E_; E1 = E_;
    }
    void build_first_neigh(int N)
    {
        hipStream_t s = stream;
        first_neigh.size_to((size_t)N + 1, s);
        scan_tmp.size_to((size_t)N / 1024 + 2, s);
        HIPCHK(launch_scan_exclusive(num_neigh, first_neigh.p, N, scan_tmp.p, s));
        N_geo = N;
    }
    void build_type_groups(int N)
    {
        hipStream_t s = stream;
        const int T = hm.T;
        if (N > 0) need(node_types, "node_types");
        t_count.size_to(T, s); t_start.size_to((size_t)T + 1, s); t_cursor.size_to(T, s); t_perm.size_to(N, s);
        scan_tmp.size_to((size_t)std::max(N, T) / 1024 + 2, s);
        HIPCHK(launch_type_groups(node_types, N, T, t_count.p, t_start.p, t_cursor.p, t_perm.p, scan_tmp.p, s));
    }
    // counters that a list build finds at zero
    void clean_counters(DVec<int>& c, long rows, long& clean)
    {
        const int* before = c.p;
        c.size_to((size_t)rows, stream);
        if (c.p != before) clean = 0;
        if (clean < rows) { HIPCHK(launch_fill<int>(c.p, rows, 0, stream)); clean = rows; }
    }
    void build_sender_lists(int rows)
    {
        hipStream_t s = stream;
        if (!senders_counted) clean_counters(s_count, rows, counters_clean);
        s_start.size_to((size_t)rows + 1, s);
        s_list.size_to((size_t)E1, s); s_rank.size_to((size_t)E1, s);
        scan_tmp.size_to((size_t)rows / 1024 + 2, s);
        HIPCHK(launch_sender_lists(neigh_indices, E1, rows, s_count.p, s_rank.p, s_start.p, s_list.p, scan_tmp.p,
                                   senders_counted, nullptr, s, input_guard(N_geo)));
        senders_counted = false;
        sender_rows = rows; sender_edges = E1;
    }
    // stage-level calls: check whichever integer arrays this call brought
    void validate_stage_inputs(int N, bool have_nt, bool have_ni, bool have_nty, bool have_r)
    {
        hipStream_t s = stream;
        HIPCHK(hipMemsetAsync(flags.p, 0, sizeof(int), s));
        if (have_nt) HIPCHK(launch_check_range(node_types, N, hm.T, flags.p, s));
        if (have_nty) HIPCHK(launch_check_range(neigh_types, E, hm.T, flags.p, s));
        if (have_ni) {
            const size_t rows_now = H1.n / ((size_t)hm.num_LM * hm.K);
            HIPCHK(launch_check_range(neigh_indices, E, (int)std::max<size_t>(rows_now, (size_t)N), flags.p, s));
        }
        if (have_r) HIPCHK(launch_check_r(r, E, hm.r_cut, flags.p, s));
        int f = 0;
        HIPCHK(hipMemcpyAsync(&f, flags.p, sizeof(int), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        if (f & 1) throw Error(SMX_EINVAL, "node_types / neigh_types / neigh_indices hold an index outside the model or the node range");
        if (f & 2) throw Error(SMX_ERANGE, "an edge length lies outside (0, r_cut): the radial spline tables do not cover it");
    }
    int edges_from_counts_check(int N, const int* host_num_neigh, long E_)
    {
        long tot = 0;
        for (int i = 0; i < N; ++i) {
            if (host_num_neigh[i] < 0) throw Error(SMX_EINVAL, "negative num_neigh entry");
            tot += host_num_neigh[i];
        }
        if (tot != E_) throw Error(SMX_EINVAL, "sum(num_neigh) does not match the number of edges");
        return 0;
    }

    // ------------------------------------------------------------------
    AggParams<F> agg_params(int layer, int N)
    {
        AggParams<F> p{};
        p.num_nodes = N; p.K = hm.K;
        p.first_neigh = first_neigh.p; p.node_types = node_types; p.neigh_types = neigh_types;
        p.xyz = xyz; p.r = r; p.T = hm.T; p.spl_nodes = hm.spl_nodes; p.spl_h = hm.spl_h; p.spl_inv_h = 1.0 / hm.spl_h;
        p.num_edges = E; p.split_nodes = split_nodes > 0 ? split_nodes : N;
        p.table_bytes = (layer == 0 ? tabK0.n : tabK1.n) * sizeof(F);
        for (int q = 0; q < 16; ++q) p.cdiag[q] = layer == 0 ? 1.0 : cdiag1[q];
        p.selected = layer == 1 && selected1;
        for (int q = 0; q < 9; ++q) p.c_same[q] = c_same1[q];
        if (layer == 0) {
            p.gather = neigh_types; p.Hsrc = H0.p; p.tab = tab0.p; p.tabK = tabK0.p; p.pair_table = pair_table0.p;
            p.B_start = B0_start.p; p.B_lm1 = B0_lm1.p; p.B_c = B0_c.p;
        } else {
            p.gather = neigh_indices; p.Hsrc = H1.p; p.tab = tab1.p; p.tabK = tabK1.p; p.pair_table = pair_table1.p;
            p.B_start = B1_start.p; p.B_lm1 = B1_lm1.p; p.B_c = B1_c.p; p.more_terms = more_terms1;
        }
        return p;
    }
    void need(const void* p, const char* what)
    {
        if (!p) throw Error(SMX_EINVAL, std::string("stage called before its inputs exist: ") + what);
    }
    // offsets and species of the edges of N receivers
    void need_edges(int N)
    {
        need(first_neigh.p, "num_neigh");
        if (N > N_geo) throw Error(SMX_EINVAL, "stage called for more nodes than the last num_neigh");
        if (N > 0) need(node_types, "node_types");
        if (E > 0) need(neigh_types, "neigh_types");
    }

    // Whether a layer's aggregation and adjoint take the kernels for scalar sender features: a diagonal coupling, and byte
    // offsets into the tables and the sender rows (`rows` of them) that fit 32 bits.
    bool scalar_edges(int layer, size_t rows) const
    {
        if (layer == 1 && !diagonal1) return false;
        const size_t tables = layer == 0 ? hm.tables0.size() : hm.tables1.size();
        const size_t row = (size_t)hm.K * sizeof(F), limit = (size_t)1 << 32;
        return tables * (hm.spl_nodes - 1) * 16 * row < limit && rows * row < limit;
    }
    hipError_t agg_fwd(int layer, int N, F* out)
    {
        auto p = agg_params(layer, N);
        p.out = out;
        p.as_chains = layer == 0 && ghosts_apart(N);
        if (scalar_edges(layer, layer == 0 ? hm.T : H1.n / hm.K)) return launch_agg0_fwd<F>(p, stream);
        return launch_agg_fwd<F>(layer == 0 ? 0 : hm.L_max, p, stream);
    }
    int agg_bwd_groups(int layer) const
    {
        if (scalar_edges(layer, layer == 0 ? hm.T : H1.n / hm.K)) return agg0_bwd_groups<F>(hm.K);
        return smx::agg_bwd_groups<F>(layer == 0 ? 0 : hm.L_max, hm.K);
    }
    hipError_t agg_bwd(int layer, const AggParams<F>& p)
    {
        if (scalar_edges(layer, layer == 0 ? hm.T : H1.n / hm.K)) return launch_agg0_bwd<F>(p, stream);
        return launch_agg_bwd<F>(layer == 0 ? 0 : hm.L_max, p, stream);
    }

    // ---- stages ------------------------------------------------------
    void st_agg0_fwd(int N)
    {
        need(xyz, "xyz (compute_Y)"); need(r, "r (compute_R0)"); need_edges(N);
        Phi0.size_to((size_t)N * 16 * K(), stream);
        HIPCHK(agg_fwd(0, N, Phi0.p));
    }
    template <typename TA, typename TC, typename CT>
    GemmParams<TA, TC, CT> gemm_base(int N, bool typed)
    {
        GemmParams<TA, TC, CT> g{};
        g.num_nodes = N;
        if (typed) { need(t_perm.p, "species groups"); g.perm = t_perm.p; g.tstart = t_start.p; g.T = hm.T; }
        return g;
    }
    template <typename TA, typename TC, typename CT>
    static GemmProb<TA, TC, CT> gemm_prob(const TA* A, long a_node_stride, long a_off, long a_sub_stride, TC* C,
                                          long c_node_stride, long c_off, long c_sub_stride, const CT* W,
                                          long w_type_stride, long w_off, int transW, int accumulate, int Kd, int Nn,
                                          int sub)
    {
        GemmProb<TA, TC, CT> q{};
        q.A = A; q.a_node_stride = a_node_stride; q.a_off = a_off; q.a_sub_stride = a_sub_stride;
        q.C = C; q.c_node_stride = c_node_stride; q.c_off = c_off; q.c_sub_stride = c_sub_stride;
        q.W = W; q.w_type_stride = w_type_stride; q.w_off = w_off; q.transW = transW; q.accumulate = accumulate;
        q.Kd = Kd; q.Nn = Nn; q.sub = sub;
        return q;
    }
    LinearParams<F> linear_A0(int N, bool reverse)
    {
        const int k = K();
        LinearParams<F> q{};
        need(t_perm.p, "species groups");
        q.num_nodes = N; q.K = k; q.T = hm.T; q.perm = t_perm.p; q.tstart = t_start.p;
        q.W = reverse ? linA0T.p : linA0.p; q.W_split = reverse ? splitA0T.p : splitA0.p;
        q.split_nodes = deciding_nodes(N);
        q.a_node_stride = q.out_node_stride = 16L * k; q.num_e_max = 1;
        for (int lm = 0; lm < 16; ++lm) q.row_off[lm] = q.out_off[lm] = lm * k;
        for (int l = 0; l < 4; ++l) {
            q.inner[l] = k; q.num_e[l] = 1;
            q.w_off[l] = (size_t)l * hm.T * k * k; q.w_type_stride[l] = (size_t)k * k;
        }
        return q;
    }
    // (`groups`: the contraction behind it depends on the species)
    LinearParams<F> linear_A1(int N, bool reverse, bool groups)
    {
        const int k = K(), ne = NE();
        LinearParams<F> q{};
        q.num_nodes = N; q.K = k; q.T = hm.T;
        if (groups) { need(t_perm.p, "species groups"); q.perm = t_perm.p; q.tstart = t_start.p; }
        q.W = reverse ? linA1T.p : linA1.p; q.W_split = reverse ? splitA1T.p : splitA1.p;
        q.split_nodes = deciding_nodes(N);
        (reverse ? q.out_node_stride : q.a_node_stride) = (long)ne * k;
        (reverse ? q.a_node_stride : q.out_node_stride) = 16L * k;
        size_t off = 0;
        int lme = 0;
        q.num_e_max = 1;
        for (int l = 0; l < 4; ++l) {
            const int nel = hm.num_e[l];
            q.inner[l] = reverse ? k : nel * k; q.num_e[l] = reverse ? nel : 1;
            q.num_e_max = std::max(q.num_e_max, q.num_e[l]);
            q.w_off[l] = off;
            off += (size_t)nel * k * k;
            for (int m = 0; m < 2 * l + 1; ++m) {
                const int lm = l * l + m;
                (reverse ? q.out_off : q.row_off)[lm] = (lme + m * nel) * k;
                (reverse ? q.row_off : q.out_off)[lm] = lm * k;
            }
            lme += (2 * l + 1) * nel;
        }
        return q;
    }
    // Whether the A-basis linears of N nodes take k_linear, and with the contraction behind them: it streams its operands
    // through blocks of 16 atoms, and with few atoms the latency of that stream is longer than the row-streaming kernel (and a
    // contraction launch) take.  Measured, us: linear and contraction 501 atoms 96 channels fp32 21 against 22, 1 000 fp64 32
    // against 30, 2 000 34 against 40, 500 and 1 000 of the l <= 1 model fp64 65, 68 against 57, 88; adjoint linears alone 500
    // fp32 17 against 16, fp64 24 against 33, l <= 1 24 and 31 against 32 and 57.  The local nodes decide, so that a call with ghost
    // nodes gives the bits of one without.
    int deciding_nodes(int N) const { return split_nodes > 0 ? split_nodes : N; }
    bool use_linear(int N) const { return linear_ok(K()) && deciding_nodes(N) >= 512; }
    bool fused_contraction(int layer, int N) const
    {
        return linear_ok(K()) && deciding_nodes(N) >= 1024 &&
               (layer == 0 ? M0_tables && NLM() == 1 && !hm.A0_scaled : M1_tables && !hm.A1_scaled);
    }
    // Whether the node-local stages of an evaluation of N nodes run as chains (smx_kernels_chain.hip).  A chain reads all weights
    // once per atom, the row tiles once per 16 atoms, and both gain from wider rows, so the line is one of atoms times channels.
    // Whole evaluations, us, launches per stage against chains: one l, double, 96 channels 1 024 atoms 285 / 260, 1 536 atoms 339 /
    // 366, 128 channels 768 atoms 322 / 279, 1 024 atoms 342 / 338, single, 96 channels 1 536 atoms 240 / 233; l <= 1, 128 channels
    // double 512 atoms 514 / 444, single 768 atoms 410 / 399, 96 channels 348 / 325, 64 channels double 1 024 atoms 457 / 396;
    // l <= 2, 128 channels double 400 atoms 759 / 686, 64 channels single 768 atoms 386 / 337.  Times of the stages are those of
    // launches of their own, so an evaluation that takes them has these.
    // Ghost nodes take a block each in the chains of layer 0 and none in that of layer 1, so that all nodes have a line of their
    // own: local / all nodes, us as above: one l, double, 96 channels 400 / 1 117 263 / 231, 600 / 1 547 285 / 301; single, 128
    // channels 400 / 1 100 225 / 204, 600 / 1 547 243 / 270, 96 channels 600 / 1 547 195 / 189, 768 / 1 866 212 / 211; l <= 1, 128
    // channels double 400 / 1 100 508 / 496, single 341 / 321, 600 / 1 474 366 / 416, 64 channels double 768 / 1 776 382 / 376,
    // 1 000 / 2 181 430 / 439, 96 channels single 400 / 1 634 354 / 343, 600 / 2 182 416 / 452; l <= 2, 64 channels double 768 /
    // 1 776 636 / 632.
    bool use_chains(int N) const
    {
        static const long most[3] = {98304, 65536, 49152}, most_nodes = sizeof(F) == 8 ? 139264 : 163840;
        return !profiling && split_nodes > 0 && chain_ok(K()) && M0_tables && M1_tables && !hm.A0_scaled && !hm.A1_scaled &&
               (long)split_nodes * K() <= most[hm.L_max] && (long)N * K() <= most_nodes;
    }
    // The layer-0 adjoint linear writes over Phi0, unless the evaluation keeps Phi0 to form A0 from it on request.
    bool separate_dPhi0(int N) const { return fused_contraction(0, N) || (use_chains(N) && NLM() == 1); }
    ChainParams<F> chain_params(int N)
    {
        ChainParams<F> p{};
        need(t_perm.p, "species groups");
        p.N = N; p.K = K(); p.T = hm.T; p.perm = t_perm.p; p.tstart = t_start.p;
        return p;
    }
    // A0, M0 and H1, with chain_edges the layer-0 aggregation before them
    void st_chain0(int N)
    {
        const size_t k = K(), nlm = NLM();
        const bool edges = chain_edges(0, N);
        if (edges) {
            need(xyz, "xyz"); need(r, "r"); need_edges(N);
            Phi0.size_to((size_t)N * 16 * k, stream);
        }
        A0.size_to((size_t)N * 16 * k, stream);
        M0.size_to((size_t)N * nlm * k, stream);
        if (nlm == 1) M0_grad.size_to((size_t)N * 16 * k, stream);
        if (H1.n != M0.n) H1.resize(M0.n, stream);   // mace.cpp:400
        auto p = chain_params(N);
        p.Phi = Phi0.p; p.W = linA0.p; p.WH1 = H1w.p; p.coef = M0_slabs.p;
        p.A = A0.p; p.M = M0.p; p.M_grad = M0_grad.p; p.H1 = H1.p;
        auto agg = agg_params(0, N);
        agg.out = Phi0.p;
        HIPCHK(with_channels(K(), [&](auto kc) { return launch_chain0<F, decltype(kc)::value>(p, edges ? &agg : nullptr, hm.L_max, stream); }));
        if (nlm == 1) pending_A0 = N;
    }
    // Whether the chains of a layer, of N nodes, take its aggregation and the adjoint of it along (scalar features): not where a CU
    // holds one block and there are more blocks than CUs, whose aggregations as launches of their own spread better.  Whole
    // evaluations, us, separate / along: one l, double, 96 channels 24 atoms 87 / 78, 256 102 / 86, 300 135 / 142, 1 000 246 / 267, 128
    // channels 256 118 / 105, 300 167 / 182, 64 channels 200 76 / 61, 1 500 213 / 203, 32 channels 1 000 99 / 88, 2 000 158 / 143,
    // 3 000 194 / 197; single, 96 channels 24 71 / 60, 501 96 / 87, 1 000 165 / 152, 128 channels 256 88 / 77, 400 125 / 129, 64
    // channels 1 500 156 / 144, 32 channels 3 000 149 / 141; l <= 1 (layer 0 only), 128 channels double 107 201 / 198, 256 250 / 242,
    // 500 442 / 443, single 200 150 / 142, 96 channels 600 303 / 309, 64 channels 1 000 258 / 253; l <= 2, 128 channels double 24 228 / 227,
    // 128 292 / 288, 256 449 / 447, single 24 183 / 172, 256 268 / 255, 96 channels double 24 190 / 187, 256 382 / 377, single 250 222 / 208, 64
    // channels double 24 161 / 154, 700 558 / 545, single 700 337 / 328.
    // Ghost nodes have blocks in layer 0 only, so that all nodes have a line of their own there: local / all nodes, us as above
    // (separate in the order of the chains): one l, double, 96 channels 230 / 748 190 / 183, 256 / 850 209 / 212, 128 channels
    // 100 / 405 159 / 160, 150 / 591 203 / 213, 200 / 686 212 / 220, 250 / 842 256 / 271, 32 channels 1 850 / 3 721 211 / 211, 2 048 / 3 959
    // 215 / 220; single, 128 channels 230 / 748 155 / 153, 256 / 850 171 / 179, 64 channels (l <= 1) 200 / 798 156 / 144; l <= 1, double, 96
    // channels 170 / 659 314 / 312, 200 / 798 350 / 366, 128 channels 96 / 469 272 / 275, 120 / 561 322 / 335, 200 / 798 428 / 458, single, 128
    // channels 170 / 659 228 / 226, 200 / 798 254 / 267, 96 channels 256 / 913 237 / 229; l <= 2, 128 channels double 120 / 561 430 / 445,
    // single 170 / 659 328 / 321, 200 / 798 368 / 380, 96 channels double 200 / 798 501 / 502, single 256 / 913 340 / 331.
    bool chain_edges(int layer, int N) const
    {
        if (!scalar_edges(layer, layer == 0 ? hm.T : H1.n / hm.K) || (layer == 1 && NLM() > 1)) return false;
        if (sizeof(F) == 4 && (hm.K <= 64 || (hm.K == 96 && NLM() == 1))) return true;
        if (sizeof(F) == 8 && hm.K <= 64) return split_nodes <= 2048 && N <= 3840;
        return split_nodes <= num_cus && N <= (sizeof(F) == 8 ? (hm.K == 96 ? 3 : 2) : (hm.K == 96 ? 6 : 3)) * num_cus;
    }
    // Chains whose layer-0 aggregation is a launch of its own for the ghost nodes' sake: the sums over the edges of a receiver run in
    // the order of the chains, so that a call with ghost nodes gives the bits of one without.
    bool ghosts_apart(int N) const { return use_chains(N) && !chain_edges(0, N) && chain_edges(0, split_nodes); }
    bool chain1_messages(int N) const { return chain_edges(1, N) && (size_t)E1 * hm.K * sizeof(F) <= msg_limit_bytes; }
    // A1, M1, the tail and the adjoints back to dPhi1, the aggregation before and its adjoint behind them where that is so
    void st_chain1(int N, bool zero_energies, bool zero_forces)
    {
        const size_t k = K();
        if (chain_edges(1, N)) {
            need(xyz, "xyz"); need(r, "r"); need(neigh_indices, "neigh_indices"); need_edges(N);
            Phi1.size_to((size_t)N * NE() * k, stream);
        }
        messages_left = chain1_messages(N);
        if (messages_left) msg.size_to((size_t)E1 * k, stream);
        A1.size_to((size_t)N * 16 * k, stream);
        M1.size_to((size_t)N * k, stream); M1_grad.size_to((size_t)N * 16 * k, stream);
        dPhi1.size_to(Phi1.n, stream);
        auto p = chain_params(N);
        p.Phi = Phi1.p; p.W = linA1.p; p.Wt = linA1T.p; p.coef = M1_slabs.p;
        p.M = M1.p; p.M_grad = M1_grad.p; p.out = dPhi1.p;
        const auto q = tail_params(N, zero_energies);
        auto agg = agg_params(1, N);
        agg.out = Phi1.p; agg.msg = messages_left ? msg.p : nullptr; agg.forces = node_forces.p; agg.accumulate_forces = zero_forces ? 0 : 1;
        HIPCHK(with_channels(K(), [&](auto kc) { return launch_chain1<F, decltype(kc)::value>(p, q, chain_edges(1, N) ? &agg : nullptr, hm.L_max, stream); }));
        if (guard_status && q.rows > 0) guard_clear_enqueued = true;
        energies_copy = nullptr;
        pending_A1 = N; pending_A1_adj = N;
    }
    // the messages (`add_messages`: those of the last layer-1 adjoint are not in H1_adj yet), M0_adj, A0_adj, dPhi0, and with chain_edges
    // the adjoint of the layer-0 aggregation, which writes the caller's copy of the forces as well
    void st_chain2(int N, bool add_messages)
    {
        const size_t k = K();
        M0_adj.size_to(M0.n, stream);
        DVec<F>& to = separate_dPhi0(N) ? dPhi0 : Phi0;
        to.size_to((size_t)N * 16 * k, stream);
        if (add_messages && sender_rows != N) build_sender_lists(N);
        auto p = chain_params(N);
        p.Wt = linA0T.p; p.WH1 = H1wT.p; p.coef = M0_slabs.p; p.A = A0.p; p.M = M0_adj.p; p.M_grad = M0_grad.p; p.out = to.p;
        p.msg = add_messages ? msg.p : nullptr; p.H1_adj = H1_adj.p; p.sstart = s_start.p; p.slist = s_list.p; p.spare = s_rank.p;
        auto agg = agg_params(0, N);
        agg.forces = node_forces.p; agg.accumulate_forces = 1; agg.forces_copy = forces_copy;
        const bool edges = chain_edges(0, N);
        HIPCHK(with_channels(K(), [&](auto kc) { return launch_chain2<F, decltype(kc)::value>(p, edges ? &agg : nullptr, hm.L_max, stream); }));
        if (edges) forces_copy = nullptr;
        pending_A0_adj = N;
    }
    // A0 (or A1) and its contraction in one launch
    void st_linear_contraction(int layer, int N)
    {
        const size_t k = K();
        DVec<F>& M = layer == 0 ? M0 : M1;
        DVec<F>& M_grad = layer == 0 ? M0_grad : M1_grad;
        (layer == 0 ? A0 : A1).size_to((size_t)N * 16 * k, stream);
        M.size_to((size_t)N * k, stream); M_grad.size_to((size_t)N * 16 * k, stream);
        auto q = layer == 0 ? linear_A0(N, false) : linear_A1(N, false, true);
        q.A = layer == 0 ? Phi0.p : Phi1.p; q.coef = layer == 0 ? M0_slabs.p : M1_slabs.p;
        q.M = M.p; q.M_grad = M_grad.p;
        HIPCHK(launch_linear<F>(q, stream));
        (layer == 0 ? pending_A0 : pending_A1) = N;
    }
    // A0[i, l-block] = Phi0[i, l-block] . A0_weights[type_i][l]  (reverse: transposed weights)
    // `from_M0`: the adjoint product takes M0_grad . M0_adj (one polynomial per channel) as its operand
    // instead of a stored A0_adj
    void st_A0_lin(int N, bool reverse, bool from_M0 = false)
    {
        const int k = K();
        const F* src = reverse ? (from_M0 ? M0_grad.p : A0_adj.p) : Phi0.p;
        DVec<F>& to = reverse ? (separate_dPhi0(N) ? dPhi0 : Phi0) : A0;
        to.size_to((size_t)N * 16 * k, stream);
        F* dst = to.p;
        if (use_linear(N)) {
            auto q = linear_A0(N, reverse);
            q.A = src; q.out = dst; q.scale = from_M0 ? M0_adj.p : nullptr;
            HIPCHK(launch_linear<F>(q, stream));
            return;
        }
        auto g = gemm_base<F, F, F>(N, true);
        g.nprob = 4;
        for (int l = 0; l < 4; ++l) {
            g.prob[l] = gemm_prob<F, F, F>(src, 16L * k, (long)l * l * k, k, dst, 16L * k, (long)l * l * k, k, A0w.p,
                                           4L * k * k, (long)l * k * k, reverse ? 1 : 0, 0, k, k, 2 * l + 1);
            if (from_M0) { g.prob[l].Ascale = M0_adj.p; g.prob[l].ascale_node_stride = k; }
        }
        HIPCHK((launch_gemm<F, F, F>(g, stream)));
    }
    // density normalisation of A0 / A1 and its adjoint; no-ops for models without it (mace.cpp:280, 688)
    void st_scale(int layer, int N, bool reverse)
    {
        if (!(layer == 0 ? hm.A0_scaled : hm.A1_scaled)) return;
        need(r, "r"); need_edges(N);
        DVec<double>& dv = layer == 0 ? div0 : div1;
        DVec<F>& A = layer == 0 ? A0 : A1;
        DVec<F>& Aa = layer == 0 ? A0_adj : A1_adj;
        const int width = 16 * K();
        if (A.n < (size_t)N * width) throw Error(SMX_EINVAL, "density normalisation called before its A-basis exists");
        if (!reverse) {
            dv.size_to((size_t)N, stream);
            HIPCHK(launch_scale_fwd<F>(N, first_neigh.p, node_types, neigh_types, r, scale_spline(layer), hm.T, A.p, width,
                                       dv.p, flags.p, stream));
        } else {
            need(xyz, "xyz");
            if (dv.n < (size_t)N || Aa.n < (size_t)N * width)
                throw Error(SMX_EINVAL, "adjoint of the density normalisation called before its forward pass");
            node_forces.resize((size_t)3 * E, stream);
            HIPCHK(launch_scale_bwd<F>(N, first_neigh.p, node_types, neigh_types, xyz, r, scale_spline(layer), hm.T, A.p,
                                       Aa.p, width, dv.p, node_forces.p, flags.p, stream));
        }
    }
    void check_spline_flag()
    {
        int f = 0;
        HIPCHK(hipMemcpyAsync(&f, flags.p, sizeof(int), hipMemcpyDeviceToHost, stream));
        HIPCHK(hipStreamSynchronize(stream));
        if (f & 4) {
            HIPCHK(hipMemsetAsync(flags.p, 0, sizeof(int), stream));
            throw Error(SMX_ERANGE, "Out of bounds in CubicSpline::evaluate.");
        }
    }
    void st_zbl(int N)
    {
        if (!hm.has_zbl) return;
        HIPCHK(launch_zbl(N, first_neigh.p, node_types, neigh_types, xyz, r, zbl_params(), node_energies.p,
                          node_forces.p, stream));
    }
    // Layer 0 with several polynomials per channel and the standard product basis: the evaluation keeps no
    // gradients (16 numbers per polynomial and channel: four times the variables at l <= 1, nine times at l <= 2,
    // written once and read once); the adjoint stage evaluates them again from the variables instead.
    bool recompute_M0_grad() const { return M0_tables && NLM() > 1; }
    // mode 0: values and gradients; 1: values only; 2: layer-0 adjoint from the variables (A0_adj from A0, M0_adj)
    void st_poly(int N, bool layer1, int mode = 0)
    {
        PolyParams<F> p{};
        p.num_nodes = N; p.K = K(); p.mode = mode;
        const int off = layer1 ? NLM() : 0;
        p.NP = layer1 ? 1 : NLM();
        if (layer1) {
            M1.size_to((size_t)N * K(), stream); M1_grad.size_to((size_t)N * 16 * K(), stream);
            p.A = A1.p; p.M = M1.p; p.M_grad = M1_grad.p;
        } else if (mode == 2) {
            p.A = A0.p; p.M_adj = M0_adj.p; p.A_adj = A0_adj.p;
        } else {
            M0.size_to((size_t)N * NLM() * K(), stream);
            if (mode == 0) M0_grad.size_to((size_t)N * NLM() * 16 * K(), stream);
            p.A = A0.p; p.M = M0.p; p.M_grad = mode == 0 ? M0_grad.p : nullptr;
        }
        p.packed = pp_packed.p + off; p.chunks = pp_chunks.p + off; p.coef = pp_coef.p + off; p.num_entries = pp_nent.p + off;
        p.table_slabs = (layer1 ? M1_tables : M0_tables) ? (layer1 ? M1_slabs.p : M0_slabs.p) : nullptr;
        p.num_cus = num_cus;
        need(t_perm.p, "species groups");
        p.perm = t_perm.p; p.tstart = t_start.p; p.T = hm.T;
        HIPCHK(launch_poly<F>(p, stream));
    }
    void st_H1(int N, bool reverse)
    {
        const int k = K(), nlm = NLM();
        if (reverse) M0_adj.size_to(M0.n, stream);
        else if (H1.n != M0.n) H1.resize(M0.n, stream);   // mace.cpp:400
        const F* src = reverse ? H1_adj.p : M0.p;
        F* dst = reverse ? M0_adj.p : H1.p;
        auto g = gemm_base<F, F, F>(N, false);
        g.nprob = hm.L_max + 1;
        for (int l = 0; l <= hm.L_max; ++l)
            g.prob[l] = gemm_prob<F, F, F>(src, (long)nlm * k, (long)l * l * k, k, dst, (long)nlm * k, (long)l * l * k, k,
                                           H1w.p, 0, (long)l * k * k, reverse ? 1 : 0, 0, k, k, 2 * l + 1);
        HIPCHK((launch_gemm<F, F, F>(g, stream)));
    }
    void st_agg1_fwd(int N)
    {
        need(xyz, "xyz (compute_Y)"); need(r, "r (compute_R1)"); need(neigh_indices, "neigh_indices"); need_edges(N);
        Phi1.size_to((size_t)N * NE() * K(), stream);
        HIPCHK(agg_fwd(1, N, Phi1.p));
    }
    void st_A1(int N, bool reverse, bool from_M1 = false)
    {
        const int k = K(), ne = NE();
        if (reverse) dPhi1.size_to(Phi1.n, stream); else A1.size_to((size_t)N * 16 * k, stream);
        if (use_linear(N)) {
            auto q = linear_A1(N, reverse, false);
            q.A = reverse ? (from_M1 ? M1_grad.p : A1_adj.p) : Phi1.p; q.out = reverse ? dPhi1.p : A1.p;
            q.scale = from_M1 ? M1_adj.p : nullptr;
            HIPCHK(launch_linear<F>(q, stream));
            return;
        }
        long lme_off = 0;
        auto g = gemm_base<F, F, F>(N, false);
        g.nprob = 4;
        for (int l = 0; l < 4; ++l) {
            const int nel = hm.num_e[l];
            if (!reverse)
                g.prob[l] = gemm_prob<F, F, F>(Phi1.p, (long)ne * k, lme_off * k, (long)nel * k, A1.p, 16L * k,
                                               (long)l * l * k, k, A1w.p, 0, A1w_off[l], 0, 0, nel * k, k, 2 * l + 1);
            else
            {
                g.prob[l] = gemm_prob<F, F, F>(from_M1 ? M1_grad.p : A1_adj.p, 16L * k, (long)l * l * k, k, dPhi1.p, (long)ne * k,
                                               lme_off * k, (long)nel * k, A1w.p, 0, A1w_off[l], 1, 0, k, nel * k, 2 * l + 1);
                if (from_M1) { g.prob[l].Ascale = M1_adj.p; g.prob[l].ascale_node_stride = k; }
            }
            lme_off += (2 * l + 1) * nel;
        }
        HIPCHK((launch_gemm<F, F, F>(g, stream)));
    }
    // H2 = H1[l=0] . W_H1[type] + M1 . W_M1 in one launch (mace.cpp:820-845)
    void st_H2(int N)
    {
        const int k = K(), nlm = NLM();
        H2.size_to((size_t)N * k, stream);
        auto g = gemm_base<F, double, double>(N, true);
        g.nprob = 1;
        g.prob[0] = gemm_prob<F, double, double>(H1.p, (long)nlm * k, 0, 0, H2.p, k, 0, 0, H2w_H1.p, (long)k * k, 0, 0, 0,
                                                 k, k, 1);
        g.prob[0].A2 = M1.p; g.prob[0].a2_node_stride = k; g.prob[0].W2 = H2w_M1.p; g.prob[0].w2_type_stride = 0;
        g.prob[0].transW2 = 0; g.prob[0].Kd2 = k;
        HIPCHK((launch_gemm<F, double, double>(g, stream)));
    }
    // H1_adj[l=0] += H2_adj . W_H1[type]^T and M1_adj = H2_adj . W_M1^T in one launch
    void st_reverse_H2(int N, bool zero_H1_adj)
    {
        const int k = K(), nlm = NLM();
        H1_adj.resize(H1.n, stream); M1_adj.size_to(M1.n, stream);
        if (zero_H1_adj) HIPCHK(hipMemsetAsync(H1_adj.p, 0, H1_adj.n * sizeof(F), stream));
        auto g = gemm_base<double, F, double>(N, true);
        g.nprob = 2;
        g.prob[0] = gemm_prob<double, F, double>(H2_adj.p, k, 0, 0, H1_adj.p, (long)nlm * k, 0, 0, H2w_H1.p, (long)k * k,
                                                 0, 1, 1, k, k, 1);
        g.prob[1] = gemm_prob<double, F, double>(H2_adj.p, k, 0, 0, M1_adj.p, k, 0, 0, H2w_M1.p, 0, 0, 1, 0, k, k, 1);
        HIPCHK((launch_gemm<double, F, double>(g, stream)));
    }
    // H2, readouts and reverse_H2 of the full pipeline in one launch (they touch one atom's rows only)
    TailParams<F> tail_params(int N, bool zero_energies)
    {
        const int k = K(), nlm = NLM();
        need(t_perm.p, "species groups");
        H2.size_to((size_t)N * k, stream); H2_adj.size_to((size_t)N * k, stream);
        node_energies.resize((size_t)N, stream);
        H1_adj.size_to(H1.n, stream); M1_adj.size_to(M1.n, stream);
        const int rows = (int)(H1.n / ((size_t)nlm * k));
        if (rows < N || M1.n < (size_t)N * k) throw Error(SMX_EINVAL, "readouts called before H1 and M1 exist for these nodes");
        TailParams<F> p{};
        p.N = N; p.rows = rows; p.K = k; p.num_LM = nlm; p.T = hm.T; p.num_cus = num_cus;
        p.perm = t_perm.p; p.tstart = t_start.p;
        p.E0 = E0.p; p.w1 = ro1.p; p.W1 = ro2_w1.p; p.w2 = ro2_w2.p; p.scale = hm.readout_2_scale;
        p.H1 = H1.p; p.M1 = M1.p; p.W_H1 = H2w_H1.p; p.W_M1 = H2w_M1.p; p.V_H1 = H2v_H1.p; p.V_M1 = H2v_M1.p;
        p.H2 = H2.p; p.H2_adj = H2_adj.p; p.H1_adj = H1_adj.p; p.M1_adj = M1_adj.p;
        p.node_energies = node_energies.p; p.zero_energies = zero_energies ? 1 : 0; p.energies_copy = energies_copy;
        p.guard = guard_live(); p.guard_clear = guard_status;
        p.guard_forces = guard_status ? node_forces.p : nullptr; p.guard_copy = guard_status ? forces_copy : nullptr; p.guard_forces_n = guard_status ? (long)node_forces.n : 0;
        return p;
    }
    void st_tail(int N, bool zero_energies)
    {
        const auto p = tail_params(N, zero_energies);
        HIPCHK(launch_tail_fused<F>(p, stream));
        if (guard_status && p.rows > 0) guard_clear_enqueued = true;
        energies_copy = nullptr;
    }
    void st_readouts(int N, bool zero_energies)
    {
        const int k = K(), nlm = NLM();
        if (N > 0) need(node_types, "node_types");
        node_energies.resize((size_t)N, stream);
        H1_adj.size_to(H1.n, stream);
        H2_adj.size_to(H2.n, stream);
        const int rows = (int)(H1.n / ((size_t)nlm * k));
        if (rows < N || H2.n < (size_t)N * k) throw Error(SMX_EINVAL, "readouts called before H1 and H2 exist for these nodes");
        HIPCHK(launch_readout_fused<F>(N, rows, k, nlm, node_types, E0.p, ro1.p, ro2_w1.p, ro2_w2.p, hm.readout_2_scale,
                                       H1.p, H2.p, H2_adj.p, H1_adj.p, node_energies.p, zero_energies ? 1 : 0,
                                       energies_copy, guard_live(), guard_status, guard_status ? node_forces.p : nullptr,
                                       guard_status ? forces_copy : nullptr, guard_status ? (long)node_forces.n : 0, stream));
        if (guard_status && rows > 0) guard_clear_enqueued = true;
        energies_copy = nullptr;
    }
    // node counts for which compute() left A1_adj / A0_adj unwritten (-1: they are current)
    int pending_A1_adj = -1, pending_A0_adj = -1;
    int pending_A1 = -1, pending_A0 = -1;       // the same for A1 and A0 (st_linear_contraction)
    int pending_M0_grad = -1;   // compute() kept no layer-0 gradients for this many nodes: formed when somebody asks
    void materialise_A()
    {
        if (pending_A0 >= 0) { const int n = pending_A0; pending_A0 = -1; if (n > 0) st_A0_lin(n, false); }
        if (pending_A1 >= 0) { const int n = pending_A1; pending_A1 = -1; if (n > 0) st_A1(n, false); }
    }
    void materialise_adjoints(bool gradients)
    {
        if (gradients) materialise_A();
        if (pending_A1_adj >= 0) { st_reverse_M1(pending_A1_adj); pending_A1_adj = -1; }
        if (pending_A0_adj >= 0) { st_reverse_M0(pending_A0_adj); pending_A0_adj = -1; }
        if (gradients && pending_M0_grad >= 0) {
            const int n = pending_M0_grad;
            pending_M0_grad = -1;
            // (the species groups of the evaluation are still in place: compute() leaves them built for all its nodes,
            // and every call that rebuilds them comes through here first; the caller's arrays are not read again)
            if (n > 0) st_poly(n, false, 0);
        }
    }
    void st_reverse_M1(int N)
    {
        A1_adj.size_to(A1.n, stream);
        HIPCHK(launch_poly_reverse<F>(N, 1, K(), M1_grad.p, M1_adj.p, A1_adj.p, stream));
    }
    void st_reverse_M0(int N)
    {
        A0_adj.size_to(A0.n, stream);
        if (A0.n > (size_t)N * 16 * K())
            HIPCHK(hipMemsetAsync(A0_adj.p, 0, A0_adj.n * sizeof(F), stream));  // mace.cpp:376-377
        if (pending_M0_grad >= 0) {
            need(t_perm.p, "species groups");
            st_poly(N, false, 2);
        } else {
            HIPCHK(launch_poly_reverse<F>(N, NLM(), K(), M0_grad.p, M0_adj.p, A0_adj.p, stream));
        }
    }
    void st_agg1_bwd(int N, bool zero_dxyz, bool zero_H1_adj)
    {
        need(xyz, "xyz"); need(r, "r"); need(neigh_indices, "neigh_indices"); need_edges(N);
        const int k = K(), nlm = NLM();
        node_forces.resize((size_t)3 * E, stream);
        H1_adj.resize(H1.n, stream);
        const int rows = (int)(H1.n / ((size_t)nlm * k));
        const size_t row_bytes = (size_t)nlm * k * sizeof(F);
        if ((size_t)E1 * row_bytes > msg_limit_bytes) {
            agg1_bwd_chunked(N, rows, zero_dxyz, zero_H1_adj);
            return;
        }
        msg.size_to((size_t)E1 * nlm * k, stream);
        auto p = agg_params(1, N);
        p.d_out = dPhi1.p; p.forces = node_forces.p; p.accumulate_forces = zero_dxyz ? 0 : 1; p.msg = msg.p;
        agg_bwd_stage(1, p, E1, ST_AGG1B, ST_FSUM1);
        if (chain_messages) { messages_left = true; stage_absent(ST_SRED); return; }
        stage_begin(ST_SRED);
        if (sender_rows != rows) build_sender_lists(rows);
        if (fuse_reverse_H1 && nlm == 1 && sender_reduce_linear_ok(k) && M0.n == (size_t)rows * k) {
            // scalar hidden features: reverse_H1 of the summed rows in the same launch
            M0_adj.size_to(M0.n, stream);
            HIPCHK(launch_sender_reduce_linear<F>(rows, k, s_start.p, s_list.p, s_rank.p, msg.p, H1_adj.p, zero_H1_adj ? 1 : 0, H1w.p,
                                                  M0_adj.p, stream));
            reverse_H1_done = true;
        } else {
            HIPCHK(launch_sender_reduce<F>(rows, nlm * k, s_start.p, s_list.p, s_rank.p, msg.p, H1_adj.p, zero_H1_adj ? 1 : 0,
                                           false, 0, E1, stream));
        }
        stage_end(ST_SRED);
    }
    bool chain_messages = false;    // compute() leaves the sender-side sum to the chain behind the layer-1 adjoint
    bool messages_left = false;     // ... and the stage did so
    bool fuse_reverse_H1 = false;   // compute() wants reverse_H1 folded into the sender-side sum
    bool reverse_H1_done = false;   // ... and the stage did it
    // The same stage for edge lists whose messages do not fit the staging buffer: receivers are taken in
    // chunks, each chunk's messages are added to the sender rows before the next chunk overwrites them.  Every
    // sender still receives its messages in ascending edge order, so the result does not depend on the chunking.
    void agg1_bwd_chunked(int N, int rows, bool zero_dxyz, bool zero_H1_adj)
    {
        const int k = K(), nlm = NLM();
        const size_t row_bytes = (size_t)nlm * k * sizeof(F);
        const long max_rows = (long)std::max<size_t>(msg_limit_bytes / row_bytes, 1);
        // receiver boundaries: equal receiver counts, then halved until every chunk's edges fit (read back from the CSR)
        int nchunks = (int)std::min<long>(N, (E1 + max_rows - 1) / max_rows + 1);
        std::vector<int> bnd, fe;
        for (;;) {
            bnd.assign((size_t)nchunks + 1, 0); fe.assign((size_t)nchunks + 1, 0);
            for (int c = 0; c <= nchunks; ++c) {
                bnd[c] = (int)((long)N * c / nchunks);
                HIPCHK(hipMemcpyAsync(&fe[c], first_neigh.p + bnd[c], sizeof(int), hipMemcpyDeviceToHost, stream));
            }
            HIPCHK(hipStreamSynchronize(stream));
            long worst = 0;
            for (int c = 0; c < nchunks; ++c) worst = std::max<long>(worst, (long)fe[c + 1] - fe[c]);
            if (worst <= max_rows || nchunks >= N) {
                if (worst > max_rows)
                    throw Error(SMX_ENOMEM, "one receiver's messages exceed the staging limit (smx_set_staging_limit)");
                msg.size_to((size_t)worst * nlm * k, stream);
                break;
            }
            nchunks = (int)std::min<long>(N, 2L * nchunks);
        }
        const int groups = agg_bwd_groups(1);
        if (groups > 1) fpart.size_to((size_t)groups * 3 * E, stream);
        if (sender_rows != rows) build_sender_lists(rows);
        HIPCHK(launch_sort_buckets(s_start.p, rows, s_list.p, s_rank.p, stream));   // the windows below need the order in memory
        stage_begin(ST_AGG1B);
        for (int c = 0; c < nchunks; ++c) {
            auto p = agg_params(1, bnd[c + 1]);
            p.node_begin = bnd[c]; p.msg_edge_begin = fe[c];
            p.d_out = dPhi1.p; p.forces = node_forces.p; p.accumulate_forces = zero_dxyz ? 0 : 1; p.msg = msg.p;
            p.fpart = groups > 1 ? fpart.p : nullptr;
            HIPCHK(agg_bwd(1, p));
            HIPCHK(launch_sender_reduce<F>(rows, nlm * k, s_start.p, s_list.p, s_rank.p, msg.p, H1_adj.p,
                                           (c == 0 && zero_H1_adj) ? 1 : 0, true, fe[c], fe[c + 1], stream));
        }
        stage_end(ST_AGG1B);
        stage_absent(ST_SRED);
        if (groups == 1) { stage_absent(ST_FSUM1); return; }
        stage_begin(ST_FSUM1);
        HIPCHK(launch_fpart_reduce(E1, E, groups, fpart.p, node_forces.p, zero_dxyz ? 0 : 1, nullptr, stream, guard_live()));
        stage_end(ST_FSUM1);
    }
    void st_agg0_bwd(int N)
    {
        need(xyz, "xyz"); need(r, "r"); need_edges(N);
        node_forces.resize((size_t)3 * E, stream);
        auto p = agg_params(0, N);
        p.d_out = separate_dPhi0(N) ? dPhi0.p : Phi0.p; p.forces = node_forces.p; p.accumulate_forces = 1; p.msg = nullptr;
        agg_bwd_stage(0, p, E, ST_AGG0B, ST_FSUM0);
    }
    // Adjoint of an aggregation; wide models are cut into channel groups whose partial forces are added in order.  The last
    // one of an evaluation (layer 0) writes the caller's copy of the forces as well.
    void agg_bwd_stage(int layer, AggParams<F>& p, long edges, int st_kernel, int st_sum)
    {
        const int groups = agg_bwd_groups(layer);
        double* copy = layer == 0 ? forces_copy : nullptr;
        if (groups > 1) {
            fpart.size_to((size_t)groups * 3 * E, stream);
            p.fpart = fpart.p;
        } else if (copy && scalar_edges(0, hm.T)) {
            p.forces_copy = copy;
            forces_copy = nullptr;
        }
        stage_begin(st_kernel);
        HIPCHK(agg_bwd(layer, p));
        stage_end(st_kernel);
        if (groups == 1) { stage_absent(st_sum); return; }
        stage_begin(st_sum);
        HIPCHK(launch_fpart_reduce(edges, E, groups, fpart.p, node_forces.p, p.accumulate_forces, copy, stream, guard_live()));
        if (copy) forces_copy = nullptr;
        stage_end(st_sum);
    }

    // ------------------------------------------------------------------
    void compute(int N, const int* nt, const int* nn, const int* ni, const int* nty, const double* x,
                 const double* rr, long E_, bool on_device, double* d_energies, double* d_forces, int N_local,
                 long E_local) override
    {
        try {
            compute_impl(N, nt, nn, ni, nty, x, rr, E_, on_device, d_energies, d_forces, N_local, E_local);
        } catch (...) {
            // whatever was half built is not trusted by the next call
            senders_counted = false; counters_clean = 0; sender_rows = -1;
            energies_copy = nullptr; forces_copy = nullptr;
            fuse_reverse_H1 = chain_messages = false;
            // checks of the failed call may have raised the word that only its readout launch would have cleared
            if (guard_status && !guard_clear_enqueued) (void)launch_fill<int>(guard_status, 1, 0, stream);
            (void)launch_fill<int>(flags.p + 4, 2, 0, stream);
            guard_status = nullptr;
            if (evaluating) forget_evaluation();
            evaluating = false;
            throw;
        }
        guard_status = nullptr;
        evaluating = refused = false;
    }
    void compute_impl(int N, const int* nt, const int* nn, const int* ni, const int* nty, const double* x,
                      const double* rr, long E_, bool on_device, double* d_energies, double* d_forces, int N_local,
                      long E_local)
    {
        edges_in_chains = 0;
        if (N < 0 || E_ < 0) throw Error(SMX_EINVAL, "negative num_nodes or num_edges");
        if (E_ > 2147483647L) throw Error(SMX_EINVAL, "more than 2^31 - 1 edges: edge offsets are 32-bit");
        // ghost nodes (the last N - N1 nodes and their edges) go through layer 0 only: their H1 rows feed the
        // local receivers, their adjoint comes back through H1_adj (pair_symmetrix_mace.cpp:662-698)
        const int N1 = N_local < 0 ? N : N_local;
        if (N1 > N || E_local > E_) throw Error(SMX_EINVAL, "more local nodes or edges than nodes or edges");
        if (N1 < N && E_local < 0) {
            if (on_device) throw Error(SMX_EINVAL, "the number of local edges is needed with ghost nodes");
            E_local = 0;
            for (int i = 0; i < N1; ++i) E_local += nn[i];
        }
        if (!on_device) edges_from_counts_check(N, nn, E_);
        if (N == 0) {
            if (E_ != 0) throw Error(SMX_EINVAL, "edges without nodes");
            E = 0; N_geo = 0; geo_edges = 0; sender_rows = -1; guarded = false;
            node_energies.size_to(0, stream); node_forces.size_to(0, stream);
            return;
        }
        evaluating = true;
        stage_begin(ST_PREP);
        if (on_device) set_geometry_ptrs(N, nt, nn, ni, nty, x, rr, E_, true);
        else upload_inputs(N, nt, nn, ni, nty, x, rr, E_);
        if (N1 < N) E1 = E_local;
        geo_edges = E_; split_nodes = N1; guarded = true;
        // Range checks come before any kernel that uses these integers as indices: inside the list preparation, whose last
        // launch empties the lists when a check failed (input_guard).  Host arrays are checked the same way and the result
        // is looked at when the call waits for the stream anyway.
        guard_status = flags.p + 2; guard_clear_enqueued = false; guard_on_device = on_device;
        if (!on_device && (hm.A0_scaled || hm.A1_scaled)) HIPCHK(launch_fill<int>(flags.p, 1, 0, stream));
        if (N <= 65536) {
            // one launch for first_neigh, species groups, the sender histogram and the sender offsets
            hipStream_t s = stream;
            first_neigh.size_to((size_t)N + 1, s);
            t_start.size_to((size_t)hm.T + 1, s); t_perm.size_to((size_t)N, s);
            clean_counters(s_count, N, counters_clean);
            s_start.size_to((size_t)N + 1, s);
            s_rank.size_to((size_t)E1, s);
            InputChecks chk;
            chk.status = guard_status; chk.neigh_types = neigh_types; chk.r = r; chk.r_cut = hm.r_cut; chk.num_edges = E;
            chk.num_local_nodes = N1;
            HIPCHK(launch_node_lists_count(num_neigh, N, first_neigh.p, node_types, hm.T, t_start.p, t_perm.p,
                                           neigh_indices, E1, N, s_count.p, s_rank.p, s_start.p, flags.p + 4, chk, s));
            N_geo = N;
            senders_counted = true;
        } else {
            build_first_neigh(N);
            HIPCHK(launch_check_counts(num_neigh, N, first_neigh.p, N1, E, E1, guard_status, stream));
            HIPCHK(launch_check_range(node_types, N, hm.T, guard_status, stream));
            HIPCHK(launch_check_range(neigh_types, E, hm.T, guard_status, stream));
            HIPCHK(launch_check_range(neigh_indices, E1, N, guard_status, stream));
            HIPCHK(launch_check_r(r, E, hm.r_cut, guard_status, stream));
            build_type_groups(N);
        }
        sender_rows = -1;
        build_sender_lists(N);
        stage_end(ST_PREP);

        node_energies.size_to((size_t)N1, stream);
        node_forces.size_to((size_t)3 * E, stream);
        if (N == 0) return;

        energies_copy = d_energies; forces_copy = d_forces;
        // Terms that add to the forces before the layer-1 adjoint writes them (mace.cpp:27-35, 56): with any of
        // them the force array starts at zero and every later stage accumulates.
        const bool early_forces = hm.has_zbl || hm.A1_scaled || N1 < N;
        if (early_forces) HIPCHK(launch_fill<double>(node_forces.p, 3 * E, 0.0, stream));
        if (hm.has_zbl) {
            HIPCHK(launch_fill<double>(node_energies.p, (long)N1, 0.0, stream));
            st_zbl(N1);
        }
        const bool chain = use_chains(N);
        if (chain && chain_edges(0, N)) edges_in_chains = 1;
        if (edges_in_chains) stage_absent(ST_AGG0F);
        else { stage_begin(ST_AGG0F); st_agg0_fwd(N); stage_end(ST_AGG0F); }
        pending_A0 = pending_A1 = -1;
        pending_M0_grad = recompute_M0_grad() ? N : -1;
        if (chain) {
            stage_begin(ST_A0LIN); st_chain0(N); stage_end(ST_A0LIN);
            stage_absent(ST_M0); stage_absent(ST_H1);
        } else if (fused_contraction(0, N)) {
            stage_begin(ST_A0LIN); st_linear_contraction(0, N); stage_end(ST_A0LIN);
            stage_absent(ST_M0);
        } else {
            stage_begin(ST_A0LIN); st_A0_lin(N, false); stage_end(ST_A0LIN);
            st_scale(0, N, false);
            stage_begin(ST_M0); st_poly(N, false, pending_M0_grad >= 0 ? 1 : 0); stage_end(ST_M0);
        }
        if (!chain) { stage_begin(ST_H1); st_H1(N, false); stage_end(ST_H1); }
        // the species groups cover the nodes of the current stages
        if (N1 < N) build_type_groups(N1);
        if (chain) {
            if (chain_edges(1, N1)) { edges_in_chains |= 2; stage_absent(ST_AGG1F); }
            else { stage_begin(ST_AGG1F); st_agg1_fwd(N1); stage_end(ST_AGG1F); }
            stage_begin(ST_A1); st_chain1(N1, !hm.has_zbl, !early_forces); stage_end(ST_A1);
            for (int st : {ST_M1, ST_H2, ST_READOUT, ST_REVH2, ST_REVM1, ST_REVA1}) stage_absent(st);
            if (messages_left) {
                for (int st : {ST_AGG1B, ST_FSUM1, ST_SRED}) stage_absent(st);
            } else {
                chain_messages = true;
                st_agg1_bwd(N1, !early_forces, false);
                chain_messages = false;
            }
            if (N1 < N) build_type_groups(N);
            stage_begin(ST_REVA0LIN); st_chain2(N, messages_left); stage_end(ST_REVA0LIN);
            for (int st : {ST_REVH1, ST_REVM0}) stage_absent(st);
            if (!chain_edges(0, N)) st_agg0_bwd(N);
            else for (int st : {ST_AGG0B, ST_FSUM0}) stage_absent(st);
            finish_evaluation(N1, on_device);
            return;
        }
        stage_begin(ST_AGG1F); st_agg1_fwd(N1); stage_end(ST_AGG1F);
        if (fused_contraction(1, N1)) {
            stage_begin(ST_A1); st_linear_contraction(1, N1); stage_end(ST_A1);
            stage_absent(ST_M1);
        } else {
            stage_begin(ST_A1); st_A1(N1, false); stage_end(ST_A1);
            st_scale(1, N1, false);
            stage_begin(ST_M1); st_poly(N1, true); stage_end(ST_M1);
        }
        if (tail_fused_ok(K())) {
            stage_begin(ST_H2); st_tail(N1, !hm.has_zbl); stage_end(ST_H2);
            stage_absent(ST_READOUT); stage_absent(ST_REVH2);
        } else {
            stage_begin(ST_H2); st_H2(N1); stage_end(ST_H2);
            stage_begin(ST_READOUT); st_readouts(N1, !hm.has_zbl); stage_end(ST_READOUT);
            stage_begin(ST_REVH2); st_reverse_H2(N1, false); stage_end(ST_REVH2);
        }
        // Without density normalisation nothing between reverse_M and the adjoint linear reads A_adj: the
        // linear then forms M_grad . M_adj itself while loading its rows (one polynomial per channel) and
        // A_adj is only written if somebody asks for it (get_array).
        const bool scaled_operand = use_linear(N) || gemm_scaled_operand_ok(K(), K(), sizeof(F));
        const bool fuse1 = !hm.A1_scaled && scaled_operand, fuse0 = !hm.A0_scaled && NLM() == 1 && scaled_operand;
        if (fuse1) stage_absent(ST_REVM1);
        else { stage_begin(ST_REVM1); st_reverse_M1(N1); stage_end(ST_REVM1); }
        pending_A1_adj = fuse1 ? N1 : -1;
        st_scale(1, N1, true);
        stage_begin(ST_REVA1); st_A1(N1, true, fuse1); stage_end(ST_REVA1);
        fuse_reverse_H1 = N1 == N; reverse_H1_done = false;
        st_agg1_bwd(N1, !early_forces, false);
        fuse_reverse_H1 = false;
        if (N1 < N) build_type_groups(N);
        if (reverse_H1_done) stage_absent(ST_REVH1);
        else { stage_begin(ST_REVH1); st_H1(N, true); stage_end(ST_REVH1); }
        if (fuse0) stage_absent(ST_REVM0);
        else { stage_begin(ST_REVM0); st_reverse_M0(N); stage_end(ST_REVM0); }
        pending_A0_adj = fuse0 ? N : -1;
        st_scale(0, N, true);
        stage_begin(ST_REVA0LIN); st_A0_lin(N, true, fuse0); stage_end(ST_REVA0LIN);
        st_agg0_bwd(N);
        finish_evaluation(N1, on_device);
    }
    // the layer-0 adjoint, and what the caller's arrays still lack
    void finish_evaluation(int N1, bool on_device)
    {
        // (a skipped evaluation: the readout launch has filled the forces with NaN, and every sum of partial forces
        // after it looks at the guard itself)
        if (guard_status && !guard_clear_enqueued) HIPCHK(launch_fill<int>(guard_status, 1, 0, stream));

        if (energies_copy) HIPCHK(hipMemcpyAsync(energies_copy, node_energies.p, (size_t)N1 * sizeof(double), hipMemcpyDeviceToDevice, stream));
        if (forces_copy && E) HIPCHK(hipMemcpyAsync(forces_copy, node_forces.p, (size_t)3 * E * sizeof(double), hipMemcpyDeviceToDevice, stream));
        energies_copy = nullptr; forces_copy = nullptr;
        // the reference throws from CubicSpline::evaluate for an edge beyond the normalisation spline
        // (cubic_spline.cpp:19-20); callers of the device-resident variant vouch for their edge lengths
        if (!on_device && (hm.A0_scaled || hm.A1_scaled)) check_spline_flag();
    }

    // stage-level entry points (host arrays)
    void stage(const char* name, int N, const int* nt, const int* nn, const int* ni, const int* nty,
               const double* x, const double* rr, long E_, int fa, int fb) override
    {
        const std::string s(name);
        energies_copy = nullptr; forces_copy = nullptr;
        fuse_reverse_H1 = false; guard_status = nullptr; split_nodes = 0;
        materialise_adjoints(true);
        if (N < 0) throw Error(SMX_EINVAL, "negative num_nodes");
        // A stage may cover the leading nodes of a longer edge list (the pair style runs layer 1 on its local
        // nodes with the arrays of local + ghost nodes, pair_symmetrix_mace.cpp:681-693): the edge arrays keep
        // their full length, the stage's own edges are the first sum(num_neigh[0..N)).
        long own_edges = -1;
        if (nn) {
            own_edges = 0;
            for (int i = 0; i < N; ++i) {
                if (nn[i] < 0) throw Error(SMX_EINVAL, "negative num_neigh entry");
                own_edges += nn[i];
            }
            const long have = E_ >= 0 ? E_ : E;
            if (own_edges > have) throw Error(SMX_EINVAL, "sum(num_neigh) exceeds the number of edges");
        }
        if (guarded) {
            // (a device-resident evaluation before this call: were its arrays fit for use?)
            int skipped = 0;
            HIPCHK(hipMemcpyAsync(&skipped, flags.p + 3, sizeof(int), hipMemcpyDeviceToHost, stream));
            HIPCHK(hipStreamSynchronize(stream));
            if (skipped) forget_evaluation();
        }
        set_geometry_ptrs(N, nt, nn, ni, nty, x, rr, E_, false);
        if (nn) {
            build_first_neigh(N); E1 = own_edges; geo_edges = own_edges;
            if (guarded) { sender_edges = -1; guarded = false; }
        }
        try {
            validate_stage_inputs(N, nt != nullptr, ni != nullptr, nty != nullptr, rr != nullptr);
        } catch (...) {
            // arrays that failed their checks are not there for the next call
            if (nt) node_types = nullptr;
            if (ni) neigh_indices = nullptr;
            if (nty) neigh_types = nullptr;
            if (rr) r = nullptr;
            throw;
        }
        if (s == "Y" || s == "R0" || s == "R1") return;  // geometry remembered; evaluated inside the fused kernels
        if (s == "A0") { build_type_groups(N); st_agg0_fwd(N); st_A0_lin(N, false); }
        else if (s == "reverse_A0") { build_type_groups(N); st_A0_lin(N, true); st_agg0_bwd(N); }
        else if (s == "A0_scaled") { st_scale(0, N, false); if (hm.A0_scaled) check_spline_flag(); }
        else if (s == "reverse_A0_scaled") { st_scale(0, N, true); if (hm.A0_scaled) check_spline_flag(); }
        else if (s == "A1_scaled") { st_scale(1, N, false); if (hm.A1_scaled) check_spline_flag(); }
        else if (s == "reverse_A1_scaled") {
            if (hm.A1_scaled) {
                node_forces.resize((size_t)3 * E, stream);
                if (fa) HIPCHK(launch_fill<double>(node_forces.p, 3 * E, 0.0, stream));
            }
            st_scale(1, N, true);
            if (hm.A1_scaled) check_spline_flag();
        }
        else if (s == "M0") { build_type_groups(N); st_poly(N, false); }
        else if (s == "reverse_M0") st_reverse_M0(N);
        else if (s == "H1") st_H1(N, false);
        else if (s == "reverse_H1") st_H1(N, true);
        else if (s == "Phi1") { need(node_types, "node_types (compute_R1)"); st_agg1_fwd(N); }
        else if (s == "reverse_Phi1") { sender_rows = -1; st_agg1_bwd(N, fa != 0, fb != 0); }
        else if (s == "A1") st_A1(N, false);
        else if (s == "reverse_A1") st_A1(N, true);
        else if (s == "M1") { build_type_groups(N); st_poly(N, true); }
        else if (s == "reverse_M1") st_reverse_M1(N);
        else if (s == "H2") { build_type_groups(N); st_H2(N); }
        else if (s == "reverse_H2") { build_type_groups(N); st_reverse_H2(N, fa != 0); }
        else if (s == "readouts") st_readouts(N, false);
        else if (s == "ZBL") {
            // zbl.cpp:96-125 adds to the caller's node_energies / node_forces: here to the engine's arrays, which
            // grow like std::vector::resize (new entries zero) when the edge list changed
            if (hm.has_zbl) {
                need(xyz, "xyz"); need(r, "r"); need_edges(N);
                node_energies.resize((size_t)N, stream);
                node_forces.resize((size_t)3 * E, stream);
                st_zbl(N);
            }
        }
        else throw Error(SMX_EINVAL, "unknown stage " + s);
    }

    // ------------------------------------------------------------------
    struct Named { DVec<F>* f; DVec<double>* d; };
    Named find(const std::string& n)
    {
        if (n == "A0") return {&A0, nullptr};
        if (n == "A0_adj") return {&A0_adj, nullptr};
        if (n == "M0") return {&M0, nullptr};
        if (n == "M0_grad") return {&M0_grad, nullptr};
        if (n == "M0_adj") return {&M0_adj, nullptr};
        if (n == "H1") return {&H1, nullptr};
        if (n == "H1_adj") return {&H1_adj, nullptr};
        if (n == "Phi0") return {&Phi0, nullptr};
        if (n == "Phi1") return {&Phi1, nullptr};
        if (n == "Phi1_adj" || n == "dPhi1") return {&dPhi1, nullptr};
        if (n == "A1") return {&A1, nullptr};
        if (n == "A1_adj") return {&A1_adj, nullptr};
        if (n == "M1") return {&M1, nullptr};
        if (n == "M1_grad") return {&M1_grad, nullptr};
        if (n == "M1_adj") return {&M1_adj, nullptr};
        if (n == "H0_weights") return {&H0, nullptr};
        if (n == "H2") return {nullptr, &H2};
        if (n == "H2_adj") return {nullptr, &H2_adj};
        if (n == "node_energies") return {nullptr, &node_energies};
        if (n == "node_forces") return {nullptr, &node_forces};
        return {nullptr, nullptr};
    }
    // entries of a named array as get_array would copy them
    size_t array_length(const std::string& s)
    {
        if (s == "Y") return (size_t)E * 16;
        if (s == "Y_grad") return (size_t)E * 48;
        if (s == "R0") return (size_t)E * hm.nspl0;
        if (s == "R1") return (size_t)E * hm.nspl1;
        if (s == "M0_grad" && pending_M0_grad >= 0) return (size_t)pending_M0_grad * NLM() * 16 * K();
        if (s == "A1_adj" && pending_A1_adj >= 0) return A1.n;
        if (s == "A0_adj" && pending_A0_adj >= 0) return A0.n;
        Named v = find(s);
        if (!v.f && !v.d) throw Error(SMX_EINVAL, "unknown array '" + s + "'");
        return v.d ? v.d->n : v.f->n;
    }
    void get_array(const char* name, double* out, long cap, long* n) override
    {
        const std::string s(name);
        hipStream_t st = stream;
        const size_t len = array_length(s);
        if (n) *n = (long)len;
        if (s == "Y" || s == "Y_grad") need(xyz, "xyz (compute_Y)");
        if (s == "R0" || s == "R1") { need(r, "r (compute_R0/R1)"); need_edges(N_geo); }
        if (!out) return;
        // (arrays the evaluation left unwritten are formed when they are asked for; the others do not wait for that)
        if (s == "A1_adj" || s == "A0_adj" || s == "M0_grad") materialise_adjoints(s == "M0_grad");
        if (s == "A0" || s == "A1") materialise_A();
        const double* src = nullptr;
        if (s == "Y" || s == "Y_grad") {
            scratch_d.size_to((size_t)E * 64, st);
            HIPCHK(launch_sph_harm(xyz, E, scratch_d.p, scratch_d.p + (size_t)E * 16, st));
            src = s == "Y" ? scratch_d.p : scratch_d.p + (size_t)E * 16;
        } else if (s == "R0" || s == "R1") {
            const bool l1 = s == "R1";
            scratch_d.size_to(len, st);
            HIPCHK(launch_radial<F>(N_geo, first_neigh.p, node_types, neigh_types, r, l1 ? tab1.p : tab0.p,
                                    l1 ? pair_table1.p : pair_table0.p, hm.T, hm.spl_nodes, hm.spl_h, l1 ? hm.nspl1 : hm.nspl0,
                                    scratch_d.p, st));
            src = scratch_d.p;
        } else {
            Named v = find(s);
            if (v.d) src = v.d->p;
            else if (std::is_same<F, double>::value) src = reinterpret_cast<const double*>(v.f->p);
            else {
                scratch_d.size_to(len, st);
                HIPCHK((launch_convert<F, double>(v.f->p, scratch_d.p, (long)len, st)));
                src = scratch_d.p;
            }
        }
        if (cap > 0 && len > 0) download(out, src, std::min((size_t)cap, len) * sizeof(double));
        else HIPCHK(hipStreamSynchronize(st));
    }
    // device to caller's memory, and the stream waited for: through pinned memory while that is small (the runtime's own
    // staging of pageable memory costs 30 us a copy)
    void download(void* out, const void* src, size_t bytes)
    {
        if (bytes > ((size_t)32 << 20)) {
            HIPCHK(hipMemcpyAsync(out, src, bytes, hipMemcpyDeviceToHost, stream));
            HIPCHK(hipStreamSynchronize(stream));
            return;
        }
        char* h = host_out.room(bytes);
        HIPCHK(hipMemcpyAsync(h, src, bytes, hipMemcpyDeviceToHost, stream));
        HIPCHK(hipStreamSynchronize(stream));
        std::memcpy(out, h, bytes);
    }
    void set_array(const char* name, const double* in, long n) override
    {
        const std::string s(name);
        hipStream_t st = stream;
        if (n < 0) throw Error(SMX_EINVAL, "negative length");
        materialise_adjoints(true);
        Named v = find(s);
        if (s == "R0" || s == "R1")
            throw Error(SMX_EUNSUPPORTED, "unsupported: '" + s + "' is evaluated from r inside the edge kernels and never "
                        "stored; call compute_" + s + " with the edge lengths instead of assigning it");
        if ((!v.f && !v.d) || s == "M0_grad" || s == "M1_grad")
            throw Error(SMX_EINVAL, "array '" + s + "' cannot be set");
        if (s == "H0_weights" && (size_t)n != (size_t)hm.T * hm.K)
            throw Error(SMX_EINVAL, "H0_weights holds num_elements * num_channels values");
        if (v.d) { v.d->upload(in, (size_t)n, st); }
        else if (std::is_same<F, double>::value) { reinterpret_cast<DVec<double>*>(v.f)->upload(in, (size_t)n, st); }
        else {
            scratch_d.upload(in, (size_t)n, st);
            v.f->size_to((size_t)n, st);
            HIPCHK((launch_convert<double, F>(scratch_d.p, v.f->p, n, st)));
        }
        HIPCHK(hipStreamSynchronize(st));
    }

    void forces_view(ForcesView* v) override
    {
        v->node_forces = has_forces() ? node_forces.p : nullptr; v->forces_len = (long)node_forces.n; v->xyz = xyz;
        v->first_neigh = first_neigh.p; v->skipped = skipped_word();
        v->num_edges = E; v->receiver_edges = geo_edges; v->num_receivers = N_geo; v->device = device;
    }
    // size a named array to n entries, all equal to `value`, without a host copy
    void fill_array(const char* name, long n, double value) override
    {
        const std::string s(name);
        if (n < 0) throw Error(SMX_EINVAL, "negative length");
        materialise_adjoints(true);
        Named v = find(s);
        if ((!v.f && !v.d) || s == "H0_weights" || s == "M0_grad" || s == "M1_grad")
            throw Error(SMX_EINVAL, "array '" + s + "' cannot be set");
        if (v.d) { v.d->size_to((size_t)n, stream); HIPCHK(launch_fill<double>(v.d->p, n, value, stream)); }
        else { v.f->size_to((size_t)n, stream); HIPCHK(launch_fill<F>(v.f->p, n, (F)value, stream)); }
    }

    // ------------------------------------------------------------------
    DVec<int> rf_send, rf_nodes, rf_count, rf_rank, rf_sstart, rf_slist;
    HostBuf<int> rf_nodes_host;
    DVec<double> rf_out, rf_part;   // rf_out: see fetch_reduction
    static constexpr size_t RF_HEAD = 8;
    double* reduction_room(size_t values)
    {
        const double* before = rf_out.p;
        rf_out.size_to(RF_HEAD + values, stream);
        if (rf_out.p != before) HIPCHK(launch_fill<double>(rf_out.p, RF_HEAD, 0.0, stream));
        return rf_out.p;
    }
    void reduce_forces(int num_atoms, const int* sender_atom, const int* receiver_atom, double* atom_forces,
                       double* virial, bool sender_on_device) override
    {
        hipStream_t s = stream;
        need(node_forces.p, "node_forces");
        if (!has_forces()) throw Error(SMX_EINVAL, "the last evaluation was refused: there are no forces to reduce");
        if (node_forces.n != (size_t)3 * E) throw Error(SMX_EINVAL, "node_forces does not match the current edge list");
        if (!atom_forces && !virial) return;
        if (virial && E > 0) need(xyz, "xyz");
        if (geo_edges > E) throw Error(SMX_EINVAL, "num_neigh of the last call covers more edges than there are");
        ForceGather g{};
        g.num_nodes = N_geo; g.first_neigh = first_neigh.p; g.node_edges = geo_edges; g.num_edges = E; g.forces = node_forces.p; g.xyz = xyz;
        g.skipped = skipped_word();
        int atoms = N_geo;
        if (atom_forces) {
            atoms = num_atoms;
            if (num_atoms <= 0) throw Error(SMX_EINVAL, "num_atoms must be positive");
            if (!sender_atom && E > 0) throw Error(SMX_EINVAL, "sender_atom is required");
            if (receiver_atom) {
                // receiver_atom[i] = atom row of receiver block i: the blocks of every atom, in ascending order
                if (geo_edges != E) throw Error(SMX_EINVAL, "num_neigh of the last call does not cover every edge");
                int* start = rf_nodes_host.room((size_t)num_atoms + 1 + N_geo);
                int* list = start + num_atoms + 1;
                std::fill(start, start + num_atoms + 1, 0);
                for (int i = 0; i < N_geo; ++i) {
                    if (receiver_atom[i] < 0 || receiver_atom[i] >= num_atoms) throw Error(SMX_EINVAL, "receiver_atom out of range");
                    ++start[receiver_atom[i]];
                }
                int acc = 0;
                for (int a = 0; a <= num_atoms; ++a) { const int c = start[a]; start[a] = acc; acc += c; }
                for (int i = 0; i < N_geo; ++i) list[start[receiver_atom[i]]++] = i;
                for (int a = num_atoms; a > 0; --a) start[a] = start[a - 1];
                start[0] = 0;
                rf_nodes.upload(start, (size_t)num_atoms + 1 + N_geo, s);
                g.node_start = rf_nodes.p; g.node_list = rf_nodes.p + num_atoms + 1;
            } else if (num_atoms < N_geo) {
                throw Error(SMX_EINVAL, "num_atoms is smaller than the number of receivers");
            }
        } else if (receiver_atom && geo_edges != E) {
            throw Error(SMX_EINVAL, "num_neigh of the last call does not cover every edge");
        }
        double* out = reduction_room(atom_forces ? (size_t)3 * num_atoms : 0);
        // The senders of the evaluation's own lists, as a rule: those lists are used then, and compared with the caller's
        // array on the way.  (Lists made anew from it: three launches, 30 us of a 230 us step at 501 atoms.)
        const bool same_senders = atom_forces && !receiver_atom && !senders_differ && num_atoms == N_geo && sender_rows == num_atoms &&
                                  sender_edges == E && geo_edges == E && E > 0;
        auto device_senders = [&] {
            if (sender_on_device) return sender_atom;
            rf_send.size_to((size_t)E, s);
            uploader.put(reinterpret_cast<char*>(rf_send.p), sender_atom, (size_t)E * sizeof(int), s);
            uploader.next(s);
            return (const int*)rf_send.p;
        };
        if (same_senders) {
            g.senders = device_senders(); g.differ = reinterpret_cast<int*>(out + 1);
            g.send_start = s_start.p; g.send_list = s_list.p; g.send_spare = s_rank.p;
            g.atom_forces = out + RF_HEAD;
            gather_forces(g, atoms, virial ? out + 2 : nullptr);
            if (fetch_reduction(num_atoms, atom_forces, virial, nullptr)) return;
            senders_differ = true;
            g.senders = nullptr; g.differ = nullptr;
        }
        int* flag = reinterpret_cast<int*>(out);
        if (atom_forces) {
            const int* send = device_senders();
            clean_counters(rf_count, num_atoms, rf_clean);
            rf_rank.size_to((size_t)E, s);
            rf_sstart.size_to((size_t)num_atoms + 1, s); rf_slist.size_to((size_t)E, s);
            scan_tmp.size_to((size_t)num_atoms / 1024 + 2, s);
            HIPCHK(launch_sender_lists(send, E, num_atoms, rf_count.p, rf_rank.p, rf_sstart.p, rf_slist.p, scan_tmp.p, false,
                                       flag, s));
            g.send_start = rf_sstart.p; g.send_list = rf_slist.p; g.send_spare = rf_rank.p;
            g.atom_forces = out + RF_HEAD;
        }
        gather_forces(g, atoms, virial ? out + 2 : nullptr);
        fetch_reduction(num_atoms, atom_forces, virial, nullptr);
    }
    void gather_forces(ForceGather& g, int atoms, double* d_virial)
    {
        g.num_atoms = atoms;
        if (d_virial) {
            rf_part.size_to((size_t)6 * force_gather_blocks(atoms), stream);
            g.partial = rf_part.p;
            g.ticket = flags.p + 5;
        }
        HIPCHK(launch_force_gather(g, d_virial, stream));
    }
    // The sums, [RF_HEAD: range flag, differ, virial[6]][num_atoms][3][energies], in one copy; false: the senders differed.
    bool fetch_reduction(int num_atoms, double* atom_forces, double* virial, double* energies)
    {
        const size_t nf = atom_forces ? (size_t)3 * num_atoms : 0, total = RF_HEAD + nf + (energies ? num_atoms : 0);
        double* h = reinterpret_cast<double*>(host_out.room(total * sizeof(double)));
        HIPCHK(hipMemcpyAsync(h, rf_out.p, total * sizeof(double), hipMemcpyDeviceToHost, stream));
        HIPCHK(hipStreamSynchronize(stream));
        const bool differ = *reinterpret_cast<const int*>(h + 1) != 0, range = *reinterpret_cast<const int*>(h) != 0;
        if (differ || range) HIPCHK(launch_fill<double>(rf_out.p, 2, 0.0, stream));
        if (differ) return false;
        if (range) throw Error(SMX_EINVAL, "sender_atom out of range");
        if (atom_forces) std::memcpy(atom_forces, h + RF_HEAD, nf * sizeof(double));
        if (virial) std::memcpy(virial, h + 2, 6 * sizeof(double));
        if (energies) std::memcpy(energies, h + RF_HEAD + nf, (size_t)num_atoms * sizeof(double));
        return true;
    }
    // Evaluation and reduction of one list on the device (receiver i and sender index are atoms) with the results in the
    // caller's memory: the sender lists of the evaluation serve the reduction too, and everything comes back together.
    void evaluate_list(int N, const int* nt, const int* nn, const int* ni, const int* nty, const double* x, const double* rr,
                       long E_, double* energies, double* forces, double* virial) override
    {
        double* out = reduction_room((size_t)4 * N);
        compute(N, nt, nn, ni, nty, x, rr, E_, true, out + RF_HEAD + (size_t)3 * N, nullptr, -1, -1);
        ForceGather g{};
        g.num_nodes = N; g.first_neigh = first_neigh.p; g.node_edges = geo_edges; g.num_edges = E; g.forces = node_forces.p; g.xyz = xyz;
        g.skipped = skipped_word();
        g.send_start = s_start.p; g.send_list = s_list.p; g.send_spare = s_rank.p;
        g.atom_forces = out + RF_HEAD;
        gather_forces(g, N, out + 2);
        fetch_reduction(N, forces, virial, energies);
    }
};

void set_last_error(const std::string& msg) { g_last_error = msg; }

}  // namespace smx

// ===========================================================================
struct smx_model {
    std::unique_ptr<smx::EngineBase> eng;
};

namespace smx {
int engine_forces_view(smx_model* m, ForcesView* out, std::string* err)
{
    if (!m || !m->eng) { if (err) *err = "null model"; return SMX_EINVAL; }
    m->eng->forces_view(out);
    return SMX_OK;
}
}  // namespace smx

namespace {

template <typename Fn>
int guarded(Fn&& fn)
{
    try {
        fn();
        return SMX_OK;
    } catch (const smx::Error& e) {
        smx::g_last_error = e.what();
        return e.code;
    } catch (const smx::JsonError& e) {
        smx::g_last_error = e.what();
        return SMX_EFILE;
    } catch (const std::bad_alloc&) {
        smx::g_last_error = "out of host memory";
        return SMX_ENOMEM;
    } catch (const std::exception& e) {
        const std::string w = e.what();
        smx::g_last_error = w;
        return w.rfind("unsupported:", 0) == 0 ? SMX_EUNSUPPORTED : SMX_EINVAL;
    }
}

void require_device()
{
    static thread_local int checked = -1;   // ordinal this thread has looked at already
    int cur = -1;
    if (checked >= 0 && hipGetDevice(&cur) == hipSuccess && cur == checked) return;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0)
        throw smx::Error(SMX_ENODEVICE, "no HIP device available: this engine has no CPU path");
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) throw smx::Error(SMX_ENODEVICE, "hipGetDevice failed");
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) throw smx::Error(SMX_ENODEVICE, "hipGetDeviceProperties failed");
    if (std::string(prop.gcnArchName).rfind("gfx950", 0) != 0)
        throw smx::Error(SMX_ENODEVICE, std::string("kernels are built for gfx950 only; found ") + prop.gcnArchName);
    checked = dev;
}

// A stage call leaves the arrays it does not take (nullptr here) as they were.  An array without an element may come as a null
// pointer (an empty vector's): it is there, and empty.
template <typename T>
const T* given(const T* p, long n)
{
    static const T none{};
    return p || n != 0 ? p : &none;
}
std::nullptr_t given(std::nullptr_t, long) { return nullptr; }

smx::EngineBase& E(smx_model* m)
{
    if (!m || !m->eng) throw smx::Error(SMX_EINVAL, "null model");
    return *m->eng;
}

}  // namespace

// ---------------------------------------------------------------------------
// Device neighbour list (canonical order; see smx_kernels_nlist.hip)
namespace smx {
struct NeighborList {
    DVec<double> part, xyz, r;
    DVec<char> in_dev;        // [shift vectors][shift integers] and, for host inputs, [positions][species]
    DVec<int> atom_bin, bin_count, bin_start, bin_atoms, count, cfirst, first, num_neigh, neigh_indices,
        neigh_types, neigh_shift, scan_tmp;
    DVec<long long> keys, sorted;
    HostBuf<char> in_host;    // the same on its way there; every call waits for the stream before it returns
    HostBuf<int> totals;
    DVec<unsigned long long> chain_sums;
    HostBuf<unsigned long long> chain_total;
    unsigned launches = 0;    // tag of the last chained launch
    int chain_rounds = NL_CHAIN_ROUNDS;
    bool wait = true;         // false: a build from host positions returns when the number of edges is known (smx_nlist_set_wait)
    const double* shift_vec = nullptr;
    const int* shift_int = nullptr;
    double* pos_dev = nullptr;     // copies of host inputs (smx_nlist_build_host / smx_nlist_update_host)
    int* types_dev = nullptr;
    int host_atoms = -1;           // number of them, -1: none
    int N = 0, num_shifts = 0;
    long E = 0, num_candidates = 0;
    double r_list = 0.0;
    double density = 0.0;          // atoms and images considered by the last build, per volume

    static constexpr size_t BRING_BYTES = (size_t)64 << 10;    // inputs brought by a kernel

    // Lists of up to this many atoms try every atom as a sender: the three launches that bin the atoms take longer.
    static constexpr int ALL_ATOMS = 512;

    NlEdgeArrays edge_arrays(const int* d_types)
    {
        NlEdgeArrays a;
        a.types = d_types; a.shift_int = shift_int; a.first = first.p; a.num_neigh = num_neigh.p;
        a.neigh_indices = neigh_indices.p; a.neigh_types = neigh_types.p; a.neigh_shift = neigh_shift.p; a.xyz = xyz.p; a.r = r.p;
        return a;
    }
    void edge_room(size_t n, hipStream_t s)
    {
        neigh_indices.size_to(n, s); neigh_types.size_to(n, s); neigh_shift.size_to(3 * n, s);
        xyz.size_to(3 * n, s); r.size_to(n, s);
    }
    long edge_capacity() const
    {
        return (long)std::min({neigh_indices.cap, neigh_types.cap, neigh_shift.cap / 3, xyz.cap / 3, r.cap});
    }
    static size_t up(size_t n) { return (n + 255) / 256 * 256; }
    // shifts (and host inputs) to the device in one copy
    void send_inputs(const double* h_pos, const int* h_types, const int* h_shift_int, const double* h_shift_vec, hipStream_t s)
    {
        const size_t bv = up((size_t)24 * num_shifts), bi = up((size_t)12 * num_shifts), bp = h_pos ? up((size_t)24 * N) : 0;
        const size_t total = bv + bi + bp + (h_pos ? up((size_t)4 * N) : 0);
        in_dev.size_to(total, s);
        char* h = in_host.room(total);
        std::memcpy(h, h_shift_vec, (size_t)24 * num_shifts);
        std::memcpy(h + bv, h_shift_int, (size_t)12 * num_shifts);
        if (h_pos && N > 0) {
            std::memcpy(h + bv + bi, h_pos, (size_t)24 * N);
            std::memcpy(h + bv + bi + bp, h_types, (size_t)4 * N);
        }
        if (total <= BRING_BYTES) HIPCHK(launch_bring(in_dev.p, h, total, s));
        else HIPCHK(hipMemcpyAsync(in_dev.p, h, total, hipMemcpyHostToDevice, s));
        shift_vec = reinterpret_cast<const double*>(in_dev.p);
        shift_int = reinterpret_cast<const int*>(in_dev.p + bv);
        pos_dev = h_pos ? reinterpret_cast<double*>(in_dev.p + bv + bi) : nullptr;
        types_dev = h_pos ? reinterpret_cast<int*>(in_dev.p + bv + bi + bp) : nullptr;
        host_atoms = h_pos ? N : -1;
    }
    void bounding_box(const double* d_pos, const double* h_pos, double* lo, double* hi, hipStream_t s)
    {
        for (int k = 0; k < 3; ++k) { lo[k] = 1e300; hi[k] = -1e300; }
        if (h_pos) {
            for (int i = 0; i < N; ++i)
                for (int k = 0; k < 3; ++k) {
                    const double v = h_pos[3 * (size_t)i + k];
                    if (!(std::fabs(v) < 1e300)) throw Error(SMX_EINVAL, "neighbour list: positions are not finite");
                    lo[k] = std::min(lo[k], v); hi[k] = std::max(hi[k], v);
                }
        } else {
            // per-block partials, finished on the host
            const int nblk = std::min(256, (N + 255) / 256);
            part.size_to((size_t)nblk * 6, s);
            HIPCHK(launch_nl_bbox(d_pos, N, part.p, nblk, s));
            std::vector<double> hp((size_t)nblk * 6);
            HIPCHK(hipMemcpyAsync(hp.data(), part.p, hp.size() * sizeof(double), hipMemcpyDeviceToHost, s));
            HIPCHK(hipStreamSynchronize(s));
            for (int k = 0; k < 3; ++k)
                for (int b = 0; b < nblk; ++b) { lo[k] = std::min(lo[k], hp[(size_t)b * 6 + k]); hi[k] = std::max(hi[k], hp[(size_t)b * 6 + 3 + k]); }
        }
        for (int k = 0; k < 3; ++k)
            if (!(lo[k] <= hi[k]) || !(hi[k] - lo[k] < 1e300)) throw Error(SMX_EINVAL, "neighbour list: positions are not finite");
    }

    double image_density(const NlGrid& g, const double* h_shift_vec) const
    {
        double volume = 1.0;
        for (int k = 0; k < 3; ++k) {
            double lo = 0.0, hi = 0.0;
            for (int q = 0; q < num_shifts; ++q) { lo = std::min(lo, h_shift_vec[3 * q + k]); hi = std::max(hi, h_shift_vec[3 * q + k]); }
            volume *= g.hi[k] - g.lo[k] + hi - lo;
        }
        return volume > 0.0 ? (double)N * num_shifts / volume : 0.0;
    }
    // Pairs to make room for when an object has none: as many as a homogeneous system of this density has within r, between 64
    // and 256 per atom (an eighth is added where the memory is taken).  Too little costs a second search: 64 for all, as this
    // was, were too few for an fcc alloy at 6 A (78) and for water at 5 A with a skin of 0.6 A (73).
    size_t first_room(double r) const
    {
        const double pairs = 4.0 / 3.0 * 3.14159265358979 * r * r * r * density;
        return (size_t)N * (size_t)std::min(std::max(pairs, 64.0), 256.0);
    }

    NlChain next_chain(hipStream_t s)
    {
        if (chain_sums.cap == 0) {
            chain_sums.size_to((size_t)nl_blocks(NL_CHAIN_ATOMS), s);
            HIPCHK(hipMemsetAsync(chain_sums.p, 0, chain_sums.n * sizeof(unsigned long long), s));
        }
        unsigned long long* total = chain_total.room(1);
        if (++launches == 0) {      // (the tags begin again)
            HIPCHK(hipMemsetAsync(chain_sums.p, 0, chain_sums.n * sizeof(unsigned long long), s));
            launches = 1;
        }
        NlChain c;
        c.sums = chain_sums.p; c.tag = (unsigned long long)launches << 32; c.host_total = total; c.rounds = chain_rounds;
        *total = 0;
        return c;
    }
    // The total of a chained launch: after the stream has finished, or (early) as soon as the launch has written it, which is
    // before its entries are complete.  The wait ends with the launch, whose blocks do not wait without a bound: the stream is
    // asked now and then whether it has failed, or finished without a total.
    long chained_total(const NlChain& c, bool early, hipStream_t s)
    {
        const volatile unsigned long long* word = c.host_total;
        if (!early) HIPCHK(hipStreamSynchronize(s));
        for (unsigned n = 1; *word >> 32 != c.tag >> 32; ++n) {
            if (n % 4096) { __builtin_ia32_pause(); continue; }
            const hipError_t state = hipStreamQuery(s);
            if (state == hipErrorNotReady) continue;
            HIPCHK(state);
            if (*word >> 32 != c.tag >> 32) throw Error(SMX_EHIP, "neighbour list: the launch left no total");
        }
        const unsigned long long total = *word & 0xffffffffull;
        if (total > 0x7fffffffull) throw Error(SMX_EINVAL, "neighbour list: more than 2^31 candidate pairs");
        return (long)total;
    }

    // Candidates: every (receiver, sender, image) closer than r_list, ordered per receiver.  Edges: those closer than r_cut.
    // Everything is enqueued with the room that is there; the host waits once, for the totals, and where the room did not
    // suffice it makes more and repeats the part that did not fit (kernels that lack room write nothing).
    long build(int N_, const double* d_pos, const double* h_pos, const int* d_types, const int* h_types, int num_shifts_,
               const int* h_shift_int, const double* h_shift_vec, double r_list_, double r_cut, hipStream_t s)
    {
        if (N_ < 0 || num_shifts_ <= 0 || !(r_list_ > 0.0) || !h_shift_int || !h_shift_vec || (N_ > 0 && !d_pos && !h_pos))
            throw Error(SMX_EINVAL, "neighbour list: bad arguments");
        int zero_shift = -1;
        for (int q = 0; q < num_shifts_; ++q)
            if (h_shift_int[3 * q] == 0 && h_shift_int[3 * q + 1] == 0 && h_shift_int[3 * q + 2] == 0) zero_shift = q;
        N = N_; num_shifts = num_shifts_; r_list = r_list_; E = 0; num_candidates = 0;
        cfirst.size_to((size_t)N + 1, s); first.size_to((size_t)N + 1, s); num_neigh.size_to((size_t)N, s);
        totals.room(2);
        send_inputs(h_pos, h_types, h_shift_int, h_shift_vec, s);
        if (h_pos) { d_pos = pos_dev; d_types = types_dev; }
        if (N == 0) {
            edge_room(0, s);
            HIPCHK(hipMemsetAsync(first.p, 0, sizeof(int), s));
            HIPCHK(hipStreamSynchronize(s));
            return 0;
        }
        NlGrid g{};
        bounding_box(d_pos, h_pos, g.lo, g.hi, s);
        const bool all = N <= ALL_ATOMS;
        scan_tmp.size_to((size_t)N / 1024 + 2, s);
        if (!all) {
            long nbins = 1;
            for (int k = 0; k < 3; ++k) {
                const double ext = g.hi[k] - g.lo[k];
                int nb = (int)std::floor(std::min(ext / r_list, 1e6));
                nb = std::max(1, std::min(nb, 128));
                g.nb[k] = nb;
                g.inv_bs[k] = ext > 0.0 ? nb / ext : 0.0;
                nbins *= nb;
            }
            atom_bin.size_to((size_t)N, s); bin_count.size_to((size_t)2 * nbins, s); bin_start.size_to((size_t)nbins + 1, s);
            bin_atoms.size_to((size_t)N, s); scan_tmp.size_to((size_t)std::max<long>(nbins, N) / 1024 + 2, s);
            HIPCHK(launch_fill<int>(bin_count.p, 2 * nbins, 0, s));
            HIPCHK(launch_nl_bins(d_pos, N, g, atom_bin.p, bin_count.p, s));
            HIPCHK(launch_scan_exclusive(bin_count.p, bin_start.p, (int)nbins, scan_tmp.p, s));
            HIPCHK(launch_nl_bin_fill(N, atom_bin.p, bin_start.p, bin_count.p + nbins, bin_atoms.p, s));
        }
        const int* bs = all ? nullptr : bin_start.p;
        const int* ba = all ? nullptr : bin_atoms.p;
        const bool direct = r_list == r_cut;   // no skin: the candidates are the edges
        const bool chained = N <= NL_CHAIN_ATOMS;
        density = image_density(g, h_shift_vec);
        if (sorted.cap == 0) { keys.size_to(first_room(r_list), s); sorted.size_to(first_room(r_list), s); }
        if (edge_capacity() == 0) edge_room(first_room(r_cut), s);
        if (!chained) {
            count.size_to((size_t)N, s);
            HIPCHK(launch_nl_search(false, d_pos, N, g, bs, ba, num_shifts, shift_vec, zero_shift, r_list, count.p, nullptr, 0,
                                    nullptr, nullptr, nullptr, nullptr, s));
            HIPCHK(launch_scan_exclusive(count.p, cfirst.p, N, scan_tmp.p, s));
        }
        for (;;) {
            const long room = (long)std::min(keys.cap, sorted.cap);
            const NlEdgeArrays edges = edge_arrays(d_types);
            NlChain chain{};
            if (chained) chain = next_chain(s);
            HIPCHK(launch_nl_search(true, d_pos, N, g, bs, ba, num_shifts, shift_vec, zero_shift, r_list, nullptr, cfirst.p,
                                    direct ? std::min(room, edge_capacity()) : room, keys.p, sorted.p, direct ? &edges : nullptr,
                                    chained ? &chain : nullptr, s));
            long total;
            if (chained) {
                total = chained_total(chain, !direct || (h_pos && !wait), s);
            } else {
                HIPCHK(hipMemcpyAsync(totals.p, cfirst.p + N, sizeof(int), hipMemcpyDeviceToHost, s));
                HIPCHK(hipStreamSynchronize(s));
                total = totals.p[0];
                if (total < 0) throw Error(SMX_EINVAL, "neighbour list: more than 2^31 candidate pairs");
            }
            num_candidates = total;
            if (total <= room && (!direct || total <= edge_capacity())) break;
            keys.size_to((size_t)total, s); sorted.size_to((size_t)total, s);
            if (direct) edge_room((size_t)total, s);
        }
        E = direct ? num_candidates : filter(d_pos, d_types, r_cut, num_candidates, s);
        edge_room((size_t)E, s);
        return E;
    }

    // edges: the candidates closer than r_cut at the given positions, in candidate order (`room`: what the candidate arrays hold)
    long filter(const double* d_pos, const int* d_types, double r_cut, long room, hipStream_t s)
    {
        if (edge_capacity() == 0) edge_room(first_room(r_cut), s);
        const bool chained = N <= NL_CHAIN_ATOMS;
        if (!chained) {
            totals.room(2);
            HIPCHK(launch_nl_filter(false, d_pos, N, cfirst.p, sorted.p, room, num_shifts, shift_vec, r_cut, num_neigh.p, nullptr, 0,
                                    nullptr, nullptr, s));
            HIPCHK(launch_scan_exclusive(num_neigh.p, first.p, N, scan_tmp.p, s));
        }
        for (;;) {
            const long cap = edge_capacity();
            const NlEdgeArrays edges = edge_arrays(d_types);
            NlChain chain{};
            if (chained) chain = next_chain(s);
            HIPCHK(launch_nl_filter(true, d_pos, N, cfirst.p, sorted.p, room, num_shifts, shift_vec, r_cut, num_neigh.p, first.p, cap,
                                    &edges, chained ? &chain : nullptr, s));
            long total;
            if (chained) {
                total = chained_total(chain, false, s);
            } else {
                HIPCHK(hipMemcpyAsync(totals.p + 1, first.p + N, sizeof(int), hipMemcpyDeviceToHost, s));
                HIPCHK(hipStreamSynchronize(s));
                total = totals.p[1];
            }
            if (total <= cap) return total;
            edge_room((size_t)total, s);
        }
    }
    long update(const double* d_pos, const int* d_types, double r_cut, hipStream_t s)
    {
        if (!(r_cut > 0.0) || r_cut > r_list || (N > 0 && !d_pos))
            throw Error(SMX_EINVAL, "neighbour list: the cutoff must be positive and no larger than the radius of the last build");
        E = 0;
        first.size_to((size_t)N + 1, s); num_neigh.size_to((size_t)N, s);
        if (N == 0) {
            HIPCHK(hipMemsetAsync(first.p, 0, sizeof(int), s));
            return 0;
        }
        E = filter(d_pos, d_types, r_cut, num_candidates, s);
        edge_room((size_t)E, s);
        return E;
    }
    // positions of an orthorhombic cell folded into it along the periodic axes (in place) with the lattice offsets taken
    // off, and the image shifts that cover r_list: the arithmetic of wrap_positions / image_shifts of
    // symmetrix_amd/neighbors.py for such cells, operation by operation.  Returns whether an offset is not zero.
    static bool fold_box(int N, const double* pos, const double* cell, const int* pbc, double* folded, long long* off)
    {
        bool any = false;
        const double inv[3] = {1.0 / cell[0], 1.0 / cell[1], 1.0 / cell[2]};
        for (long i = 0; i < 3L * N; ++i) {
            const int k = (int)(i % 3);
            const double f = pos[i] * inv[k];
            if (!std::isfinite(f)) throw Error(SMX_EINVAL, "positions are not finite");
            const double o = pbc[k] ? std::floor(f) : 0.0;
            off[i] = (long long)o;
            any = any || o != 0.0;
            folded[i] = pos[i] - o * cell[k];
        }
        return any;
    }
    static void box_shifts(const double* cell, const int* pbc, double r_list, std::vector<int>& si, std::vector<double>& sv)
    {
        int n[3];
        for (int k = 0; k < 3; ++k) n[k] = pbc[k] ? (int)std::ceil(r_list / cell[k]) : 0;
        for (int a = -n[0]; a <= n[0]; ++a)
            for (int b = -n[1]; b <= n[1]; ++b)
                for (int c = -n[2]; c <= n[2]; ++c) {
                    si.insert(si.end(), {a, b, c});
                    sv.insert(sv.end(), {a * cell[0], b * cell[1], c * cell[2]});
                }
    }
};
}  // namespace smx

extern "C" {

const char* smx_last_error(void) { return smx::g_last_error.c_str(); }

int smx_model_load(const char* json_path, int flags, smx_model** out)
{
    return guarded([&] {
        if (!json_path || !out) throw smx::Error(SMX_EINVAL, "null argument");
        if (flags != SMX_FP64 && flags != SMX_FP32_FEATURES) throw smx::Error(SMX_EINVAL, "unknown precision flag");
        *out = nullptr;
        smx::HostModel hm = smx::load_host_model(json_path);
        require_device();
        {
            // the scratch array of the entry point that does not allocate: its address on this device, once
            std::string err;
            const int rc = smx::noalloc_setup_current_device(&err);
            if (rc != SMX_OK) throw smx::Error(rc, err);
        }
        std::unique_ptr<smx_model> m(new smx_model());
        if (flags == SMX_FP64) m->eng.reset(new smx::Engine<double>(std::move(hm), flags));
        else m->eng.reset(new smx::Engine<float>(std::move(hm), flags));
        *out = m.release();
    });
}

void smx_model_free(smx_model* m)
{
    if (!m) return;
    (void)hipDeviceSynchronize();
    delete m;
}

int smx_model_get_int(const smx_model* m, const char* key, int* out)
{
    return guarded([&] {
        if (!m || !key || !out) throw smx::Error(SMX_EINVAL, "null argument");
        const smx::HostModel& h = m->eng->hm;
        const std::string k(key);
        if (k == "num_elements") *out = h.T;
        else if (k == "num_channels") *out = h.K;
        else if (k == "l_max") *out = h.l_max;
        else if (k == "num_lm") *out = h.num_lm;
        else if (k == "L_max") *out = h.L_max;
        else if (k == "num_LM") *out = h.num_LM;
        else if (k == "has_zbl") *out = h.has_zbl ? 1 : 0;
        else if (k == "num_lme") *out = h.num_lme;
        else if (k == "num_lelm1lm2") *out = h.num_lelm1lm2;
        else if (k == "precision") *out = m->eng->precision;
        else if (k == "num_radial_tables_0") *out = (int)h.tables0.size();
        else if (k == "num_radial_tables_1") *out = (int)h.tables1.size();
        else if (k == "contraction_tables") *out = m->eng->contraction_tables();
        else if (k == "edges_in_chains") *out = m->eng->edges_in_chains;
        else throw smx::Error(SMX_EINVAL, "unknown integer key '" + k + "'");
    });
}

int smx_model_get_double(const smx_model* m, const char* key, double* out)
{
    return guarded([&] {
        if (!m || !key || !out) throw smx::Error(SMX_EINVAL, "null argument");
        const std::string k(key);
        if (k == "r_cut") *out = m->eng->hm.r_cut;
        else throw smx::Error(SMX_EINVAL, "unknown double key '" + k + "'");
    });
}

int smx_model_get_atomic_numbers(const smx_model* m, int* out, int cap, int* n)
{
    return guarded([&] {
        if (!m) throw smx::Error(SMX_EINVAL, "null model");
        const auto& v = m->eng->hm.atomic_numbers;
        if (n) *n = (int)v.size();
        for (int i = 0; out && i < cap && i < (int)v.size(); ++i) out[i] = v[i];
    });
}
int smx_model_get_atomic_energies(const smx_model* m, double* out, int cap, int* n)
{
    return guarded([&] {
        if (!m) throw smx::Error(SMX_EINVAL, "null model");
        const auto& v = m->eng->hm.atomic_energies;
        if (n) *n = (int)v.size();
        for (int i = 0; out && i < cap && i < (int)v.size(); ++i) out[i] = v[i];
    });
}

int smx_compute_node_energies_forces(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh,
                                     const int* neigh_indices, const int* neigh_types, const double* xyz,
                                     const double* r, long num_edges)
{
    return guarded([&] {
        auto& e = E(m);
        if (num_nodes > 0 && (!node_types || !num_neigh)) throw smx::Error(SMX_EINVAL, "null node array");
        if (num_edges > 0 && (!neigh_indices || !neigh_types || !xyz || !r)) throw smx::Error(SMX_EINVAL, "null edge array");
        e.stream = nullptr;
        e.compute(num_nodes, node_types, num_neigh, neigh_indices, neigh_types, xyz, r, num_edges, false, nullptr, nullptr, -1, -1);
        e.finish_host_call();
    });
}

int smx_compute_device(smx_model* m, int num_nodes, const int* d_node_types, const int* d_num_neigh,
                       const int* d_neigh_indices, const int* d_neigh_types, const double* d_xyz, const double* d_r,
                       long num_edges, double* d_node_energies, double* d_node_forces, void* stream)
{
    return guarded([&] {
        auto& e = E(m);
        if (num_nodes > 0 && (!d_node_types || !d_num_neigh)) throw smx::Error(SMX_EINVAL, "null node array");
        if (num_edges > 0 && (!d_neigh_indices || !d_neigh_types || !d_xyz || !d_r)) throw smx::Error(SMX_EINVAL, "null edge array");
        e.stream = static_cast<hipStream_t>(stream);
        e.compute(num_nodes, d_node_types, d_num_neigh, d_neigh_indices, d_neigh_types, d_xyz, d_r, num_edges, true,
                  d_node_energies, d_node_forces, -1, -1);
    });
}

int smx_compute_ghosted(smx_model* m, int num_local_nodes, int num_ghost_nodes, const int* node_types,
                        const int* num_neigh, const int* neigh_indices, const int* neigh_types, const double* xyz,
                        const double* r, long num_edges)
{
    return guarded([&] {
        auto& e = E(m);
        if (num_local_nodes < 0 || num_ghost_nodes < 0) throw smx::Error(SMX_EINVAL, "negative node count");
        const int n = num_local_nodes + num_ghost_nodes;
        if (n > 0 && (!node_types || !num_neigh)) throw smx::Error(SMX_EINVAL, "null node array");
        if (num_edges > 0 && (!neigh_indices || !neigh_types || !xyz || !r)) throw smx::Error(SMX_EINVAL, "null edge array");
        e.stream = nullptr;
        e.compute(n, node_types, num_neigh, neigh_indices, neigh_types, xyz, r, num_edges, false, nullptr, nullptr,
                  num_local_nodes, -1);
        e.finish_host_call();
    });
}

int smx_compute_ghosted_device(smx_model* m, int num_local_nodes, int num_ghost_nodes, const int* d_node_types,
                               const int* d_num_neigh, const int* d_neigh_indices, const int* d_neigh_types,
                               const double* d_xyz, const double* d_r, long num_edges, long num_local_edges,
                               double* d_node_energies, double* d_node_forces, void* stream)
{
    return guarded([&] {
        auto& e = E(m);
        if (num_local_nodes < 0 || num_ghost_nodes < 0 || num_local_edges < 0) throw smx::Error(SMX_EINVAL, "negative count");
        const int n = num_local_nodes + num_ghost_nodes;
        if (n > 0 && (!d_node_types || !d_num_neigh)) throw smx::Error(SMX_EINVAL, "null node array");
        if (num_edges > 0 && (!d_neigh_indices || !d_neigh_types || !d_xyz || !d_r)) throw smx::Error(SMX_EINVAL, "null edge array");
        e.stream = static_cast<hipStream_t>(stream);
        e.compute(n, d_node_types, d_num_neigh, d_neigh_indices, d_neigh_types, d_xyz, d_r, num_edges, true,
                  d_node_energies, d_node_forces, num_local_nodes, num_local_edges);
    });
}

int smx_set_num_H1_rows(smx_model* m, int rows)
{
    return guarded([&] { E(m).H1_rows_override = rows; });
}

#define SMX_STAGE(fn, name, NT, NN, NI, NTY, XYZ, R, EE, FA, FB) \
    return guarded([&] { auto& e = E(m); e.stream = nullptr; e.stage(name, num_nodes, given(NT, num_nodes), given(NN, num_nodes), given(NI, EE), \
        given(NTY, EE), given(XYZ, EE), given(R, EE), EE, FA, FB); HIPCHK(hipStreamSynchronize(e.stream)); })

int smx_compute_Y(smx_model* m, const double* xyz, long n3)
{
    const int num_nodes = 0;
    if (n3 % 3) { smx::g_last_error = "xyz length is not a multiple of 3"; return SMX_EINVAL; }
    SMX_STAGE(smx_compute_Y, "Y", nullptr, nullptr, nullptr, nullptr, xyz, nullptr, n3 / 3, 0, 0);
}
int smx_compute_R0(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh, const int* neigh_types,
                   const double* r, long num_edges)
{
    SMX_STAGE(smx_compute_R0, "R0", node_types, num_neigh, nullptr, neigh_types, nullptr, r, num_edges, 0, 0);
}
int smx_compute_R1(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh, const int* neigh_types,
                   const double* r, long num_edges)
{
    SMX_STAGE(smx_compute_R1, "R1", node_types, num_neigh, nullptr, neigh_types, nullptr, r, num_edges, 0, 0);
}
int smx_compute_A0(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh, const int* neigh_types,
                   long num_edges)
{
    SMX_STAGE(smx_compute_A0, "A0", node_types, num_neigh, nullptr, neigh_types, nullptr, nullptr, num_edges, 0, 0);
}
int smx_reverse_A0(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh, const int* neigh_types,
                   const double* xyz, const double* r, long num_edges)
{
    SMX_STAGE(smx_reverse_A0, "reverse_A0", node_types, num_neigh, nullptr, neigh_types, xyz, r, num_edges, 0, 0);
}
int smx_compute_A0_scaled(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh,
                          const int* neigh_types, const double* r, long num_edges)
{
    SMX_STAGE(smx_compute_A0_scaled, "A0_scaled", node_types, num_neigh, nullptr, neigh_types, nullptr, r, num_edges, 0, 0);
}
int smx_reverse_A0_scaled(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh,
                          const int* neigh_types, const double* xyz, const double* r, long num_edges)
{
    SMX_STAGE(smx_reverse_A0_scaled, "reverse_A0_scaled", node_types, num_neigh, nullptr, neigh_types, xyz, r, num_edges, 0, 0);
}
int smx_compute_A1_scaled(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh,
                          const int* neigh_types, const double* r, long num_edges)
{
    SMX_STAGE(smx_compute_A1_scaled, "A1_scaled", node_types, num_neigh, nullptr, neigh_types, nullptr, r, num_edges, 0, 0);
}
int smx_reverse_A1_scaled(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh,
                          const int* neigh_types, const double* xyz, const double* r, long num_edges, int zero_dxyz)
{
    SMX_STAGE(smx_reverse_A1_scaled, "reverse_A1_scaled", node_types, num_neigh, nullptr, neigh_types, xyz, r, num_edges,
              zero_dxyz, 0);
}
int smx_compute_M0(smx_model* m, int num_nodes, const int* node_types)
{
    SMX_STAGE(smx_compute_M0, "M0", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_reverse_M0(smx_model* m, int num_nodes, const int* node_types)
{
    SMX_STAGE(smx_reverse_M0, "reverse_M0", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_compute_H1(smx_model* m, int num_nodes)
{
    SMX_STAGE(smx_compute_H1, "H1", nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_reverse_H1(smx_model* m, int num_nodes)
{
    SMX_STAGE(smx_reverse_H1, "reverse_H1", nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_compute_Phi1(smx_model* m, int num_nodes, const int* num_neigh, const int* neigh_indices, long num_edges)
{
    SMX_STAGE(smx_compute_Phi1, "Phi1", nullptr, num_neigh, neigh_indices, nullptr, nullptr, nullptr, num_edges, 0, 0);
}
int smx_reverse_Phi1(smx_model* m, int num_nodes, const int* num_neigh, const int* neigh_indices, const double* xyz,
                     const double* r, long num_edges, int zero_dxyz, int zero_H1_adj)
{
    SMX_STAGE(smx_reverse_Phi1, "reverse_Phi1", nullptr, num_neigh, neigh_indices, nullptr, xyz, r, num_edges, zero_dxyz, zero_H1_adj);
}
int smx_compute_A1(smx_model* m, int num_nodes)
{
    SMX_STAGE(smx_compute_A1, "A1", nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_reverse_A1(smx_model* m, int num_nodes)
{
    SMX_STAGE(smx_reverse_A1, "reverse_A1", nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_compute_M1(smx_model* m, int num_nodes, const int* node_types)
{
    SMX_STAGE(smx_compute_M1, "M1", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_reverse_M1(smx_model* m, int num_nodes, const int* node_types)
{
    SMX_STAGE(smx_reverse_M1, "reverse_M1", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_compute_H2(smx_model* m, int num_nodes, const int* node_types)
{
    SMX_STAGE(smx_compute_H2, "H2", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}
int smx_reverse_H2(smx_model* m, int num_nodes, const int* node_types, int zero_H1_adj)
{
    SMX_STAGE(smx_reverse_H2, "reverse_H2", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, zero_H1_adj, 0);
}
int smx_compute_readouts(smx_model* m, int num_nodes, const int* node_types)
{
    SMX_STAGE(smx_compute_readouts, "readouts", node_types, nullptr, nullptr, nullptr, nullptr, nullptr, -1, 0, 0);
}

int smx_compute_ZBL(smx_model* m, int num_nodes, const int* node_types, const int* num_neigh, const int* neigh_types,
                    const double* r, const double* xyz, long num_edges)
{
    SMX_STAGE(smx_compute_ZBL, "ZBL", node_types, num_neigh, nullptr, neigh_types, xyz, r, num_edges, 0, 0);
}

int smx_get_array(smx_model* m, const char* name, double* out, long cap, long* n)
{
    return guarded([&] {
        if (!name) throw smx::Error(SMX_EINVAL, "null name");
        E(m).get_array(name, out, cap, n);
        if (out) E(m).check_device_status(true);
    });
}
int smx_set_array(smx_model* m, const char* name, const double* in, long n)
{
    return guarded([&] {
        if (!name || (!in && n > 0)) throw smx::Error(SMX_EINVAL, "null argument");
        E(m).set_array(name, in, n);
    });
}

int smx_fill_array(smx_model* m, const char* name, long n, double value)
{
    return guarded([&] {
        if (!name) throw smx::Error(SMX_EINVAL, "null name");
        auto& e = E(m);
        e.fill_array(name, n, value);
        HIPCHK(hipStreamSynchronize(e.stream));
    });
}

int smx_set_profiling(smx_model* m, int enabled)
{
    return guarded([&] {
        auto& e = E(m);
        e.profiling = enabled != 0;
        for (int i = 0; i < smx::ST_COUNT; ++i) e.ev_used[i] = false;
    });
}
int smx_set_staging_limit(smx_model* m, long bytes)
{
    return guarded([&] {
        if (bytes <= 0) throw smx::Error(SMX_EINVAL, "the staging limit must be positive");
        E(m).msg_limit_bytes = (size_t)bytes;
    });
}
const char* smx_stage_names(void) { return smx::kStageNames; }
int smx_get_stage_times(smx_model* m, float* ms, int cap, int* n)
{
    return guarded([&] {
        auto& e = E(m);
        HIPCHK(hipStreamSynchronize(e.stream));
        if (n) *n = smx::ST_COUNT;
        for (int i = 0; ms && i < cap && i < smx::ST_COUNT; ++i) {
            ms[i] = 0.f;
            if (e.ev_used[i]) HIPCHK(hipEventElapsedTime(&ms[i], e.ev0[i], e.ev1[i]));
        }
    });
}
int smx_synchronize(smx_model* m)
{
    return guarded([&] {
        auto& e = E(m);
        HIPCHK(hipStreamSynchronize(e.stream));
        e.check_device_status(true);
    });
}
int smx_reduce_forces(smx_model* m, int num_atoms, const int* sender_atom, const int* receiver_atom,
                      double* atom_forces, double* virial)
{
    return guarded([&] {
        E(m).reduce_forces(num_atoms, sender_atom, receiver_atom, atom_forces, virial, false);
        E(m).check_device_status(true);   // forces of a skipped device-resident evaluation are NaN: say why
    });
}
int smx_reduce_forces_device(smx_model* m, int num_atoms, const int* d_sender_atom, double* atom_forces, double* virial)
{
    return guarded([&] {
        E(m).reduce_forces(num_atoms, d_sender_atom, nullptr, atom_forces, virial, true);
        E(m).check_device_status(true);
    });
}

int smx_evaluate_list(smx_model* m, smx_nlist* nl, double* energies, double* atom_forces, double* virial)
{
    return guarded([&] {
        auto& e = E(m);
        if (!nl || !energies || !atom_forces || !virial) throw smx::Error(SMX_EINVAL, "null argument");
        auto& n = *reinterpret_cast<smx::NeighborList*>(nl);
        if (n.host_atoms != n.N) throw smx::Error(SMX_EINVAL, "smx_evaluate_list needs a list built from host positions");
        e.stream = nullptr;
        if (n.N == 0) { for (int q = 0; q < 6; ++q) virial[q] = 0.0; return; }
        e.evaluate_list(n.N, n.types_dev, n.num_neigh.p, n.neigh_indices.p, n.neigh_types.p, n.xyz.p, n.r.p, n.E, energies,
                        atom_forces, virial);
        e.check_device_status(true);
    });
}

smx_nlist* smx_nlist_create(void)
{
    smx_nlist* out = nullptr;
    guarded([&] { out = reinterpret_cast<smx_nlist*>(new smx::NeighborList()); });
    return out;
}
int smx_nlist_set_wait(smx_nlist* nl, int wait)
{
    return guarded([&] {
        if (!nl) throw smx::Error(SMX_EINVAL, "null argument");
        reinterpret_cast<smx::NeighborList*>(nl)->wait = wait != 0;
    });
}
int smx_nlist_set_chain_rounds(smx_nlist* nl, int rounds)
{
    return guarded([&] {
        if (!nl || rounds < 0) throw smx::Error(SMX_EINVAL, "null list or negative number of rounds");
        reinterpret_cast<smx::NeighborList*>(nl)->chain_rounds = rounds;
    });
}
void smx_nlist_free(smx_nlist* nl) { delete reinterpret_cast<smx::NeighborList*>(nl); }
int smx_nlist_build(smx_nlist* nl, int num_atoms, const double* d_positions, const int* d_types, int num_shifts,
                    const int* shift_int, const double* shift_vec, double r_list, double r_cut, void* stream,
                    long* num_edges)
{
    return guarded([&] {
        if (!nl || !shift_int || !shift_vec || (num_atoms > 0 && !d_positions)) throw smx::Error(SMX_EINVAL, "null argument");
        if (!(r_cut > 0.0) || r_cut > r_list) throw smx::Error(SMX_EINVAL, "neighbour list: need 0 < r_cut <= r_list");
        const long e = reinterpret_cast<smx::NeighborList*>(nl)->build(num_atoms, d_positions, nullptr, d_types, nullptr,
            num_shifts, shift_int, shift_vec, r_list, r_cut, (hipStream_t)stream);
        if (num_edges) *num_edges = e;
    });
}
int smx_nlist_update(smx_nlist* nl, const double* d_positions, const int* d_types, double r_cut, void* stream,
                     long* num_edges)
{
    return guarded([&] {
        if (!nl) throw smx::Error(SMX_EINVAL, "null argument");
        const long e = reinterpret_cast<smx::NeighborList*>(nl)->update(d_positions, d_types, r_cut, (hipStream_t)stream);
        if (num_edges) *num_edges = e;
    });
}
int smx_nlist_build_host(smx_nlist* nl, int num_atoms, const double* positions, const int* types, int num_shifts,
                         const int* shift_int, const double* shift_vec, double r_list, double r_cut, long* num_edges)
{
    return guarded([&] {
        if (!nl || !shift_int || !shift_vec || num_atoms < 0 || (num_atoms > 0 && (!positions || !types)))
            throw smx::Error(SMX_EINVAL, "null argument");
        if (!(r_cut > 0.0) || r_cut > r_list) throw smx::Error(SMX_EINVAL, "neighbour list: need 0 < r_cut <= r_list");
        require_device();
        const long e = reinterpret_cast<smx::NeighborList*>(nl)->build(num_atoms, nullptr, positions ? positions : shift_vec,
            nullptr, types, num_shifts, shift_int, shift_vec, r_list, r_cut, nullptr);
        if (num_edges) *num_edges = e;
    });
}
int smx_nlist_build_box(smx_nlist* nl, int num_atoms, const double* positions, const int* types, const double* cell,
                        const int* pbc, double r_list, double r_cut, long long* offsets, int* folded, long* num_edges)
{
    return guarded([&] {
        if (!nl || !cell || !pbc || !offsets || num_atoms < 0 || (num_atoms > 0 && (!positions || !types)))
            throw smx::Error(SMX_EINVAL, "null argument");
        if (!(r_cut > 0.0) || r_cut > r_list) throw smx::Error(SMX_EINVAL, "neighbour list: need 0 < r_cut <= r_list");
        for (int k = 0; k < 3; ++k)
            if (!(cell[k] > 0.0) || !std::isfinite(cell[k])) throw smx::Error(SMX_EINVAL, "neighbour list: cell lengths must be positive");
        require_device();
        std::vector<double> pos((size_t)3 * num_atoms + 3), sv;
        std::vector<int> si;
        const bool any = smx::NeighborList::fold_box(num_atoms, positions, cell, pbc, pos.data(), offsets);
        smx::NeighborList::box_shifts(cell, pbc, r_list, si, sv);
        const long e = reinterpret_cast<smx::NeighborList*>(nl)->build(num_atoms, nullptr, pos.data(), nullptr, types,
            (int)(si.size() / 3), si.data(), sv.data(), r_list, r_cut, nullptr);
        if (folded) *folded = any ? 1 : 0;
        if (num_edges) *num_edges = e;
    });
}
int smx_nlist_update_host(smx_nlist* nl, const double* positions, double r_cut, long* num_edges)
{
    return guarded([&] {
        if (!nl) throw smx::Error(SMX_EINVAL, "null argument");
        auto& n = *reinterpret_cast<smx::NeighborList*>(nl);
        if (n.host_atoms != n.N || (n.N > 0 && !positions))
            throw smx::Error(SMX_EINVAL, "neighbour list: update from host positions needs a build from host positions first");
        if (n.N > 0) {
            char* h = n.in_host.room((size_t)24 * n.N);
            std::memcpy(h, positions, (size_t)24 * n.N);
            HIPCHK(hipMemcpyAsync(n.pos_dev, h, (size_t)24 * n.N, hipMemcpyHostToDevice, nullptr));
        }
        const long e = n.update(n.pos_dev, n.types_dev, r_cut, nullptr);
        HIPCHK(hipStreamSynchronize(nullptr));
        if (num_edges) *num_edges = e;
    });
}
int smx_nlist_inputs(smx_nlist* nl, const double** d_positions, const int** d_types)
{
    return guarded([&] {
        if (!nl) throw smx::Error(SMX_EINVAL, "null argument");
        auto& n = *reinterpret_cast<smx::NeighborList*>(nl);
        if (d_positions) *d_positions = n.pos_dev;
        if (d_types) *d_types = n.types_dev;
    });
}
int smx_nlist_arrays(smx_nlist* nl, const int** num_neigh, const int** first_neigh, const int** neigh_indices,
                     const int** neigh_types, const int** neigh_shift, const double** xyz, const double** r)
{
    return guarded([&] {
        if (!nl) throw smx::Error(SMX_EINVAL, "null argument");
        auto& n = *reinterpret_cast<smx::NeighborList*>(nl);
        if (num_neigh) *num_neigh = n.num_neigh.p;
        if (first_neigh) *first_neigh = n.first.p;
        if (neigh_indices) *neigh_indices = n.neigh_indices.p;
        if (neigh_types) *neigh_types = n.neigh_types.p;
        if (neigh_shift) *neigh_shift = n.neigh_shift.p;
        if (xyz) *xyz = n.xyz.p;
        if (r) *r = n.r.p;
    });
}
int smx_nlist_copy_to_host(smx_nlist* nl, int* num_neigh, int* neigh_indices, int* neigh_types, int* neigh_shift,
                           double* xyz, double* r)
{
    return guarded([&] {
        if (!nl) throw smx::Error(SMX_EINVAL, "null argument");
        auto& n = *reinterpret_cast<smx::NeighborList*>(nl);
        const size_t E = (size_t)n.E, N = (size_t)n.N;
        if (num_neigh && N) HIPCHK(hipMemcpy(num_neigh, n.num_neigh.p, N * sizeof(int), hipMemcpyDeviceToHost));
        if (neigh_indices && E) HIPCHK(hipMemcpy(neigh_indices, n.neigh_indices.p, E * sizeof(int), hipMemcpyDeviceToHost));
        if (neigh_types && E) HIPCHK(hipMemcpy(neigh_types, n.neigh_types.p, E * sizeof(int), hipMemcpyDeviceToHost));
        if (neigh_shift && E) HIPCHK(hipMemcpy(neigh_shift, n.neigh_shift.p, 3 * E * sizeof(int), hipMemcpyDeviceToHost));
        if (xyz && E) HIPCHK(hipMemcpy(xyz, n.xyz.p, 3 * E * sizeof(double), hipMemcpyDeviceToHost));
        if (r && E) HIPCHK(hipMemcpy(r, n.r.p, E * sizeof(double), hipMemcpyDeviceToHost));
    });
}

}  // extern "C"
