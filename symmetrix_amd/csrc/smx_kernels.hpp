// Launch interface of the gfx950 kernels (definitions in smx_kernels_*.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "smx_poly_shape.hpp"

namespace smx {

// ---------------------------------------------------------------------------
// Edge aggregation (forward) and its adjoint.  One templated pair of kernels
// serves layer 0 (MACE::compute_A0 / reverse_A0 without the channel-mixing
// linear, libsymmetrix/source/mace.cpp:158-178, 238-269) and layer 1
// (compute_Phi1 / reverse_Phi1, mace.cpp:453-605): per edge
//     out[i, lme, k] += R_path(lme)[k](r_ij) * sum_m2 B_ij[lme, m2] * H[g_ij, l2^2+m2, k]
// with B_ij[.,.] = sum_m1 C * Y_m1(r_ij) the Clebsch-Gordan-contracted
// harmonics of the edge, H the gathered sender row (H0_weights[type_j] for
// layer 0, H1[neigh_index] for layer 1) and R the radial spline set of the
// species pair.  Y, B and R are recomputed per edge inside the kernels and
// never stored.
template <typename F>
struct AggParams {
    int num_nodes;
    int K;
    const int* first_neigh;   // [num_nodes+1] CSR offsets of the receiver-sorted edge list
    const int* node_types;    // [num_nodes]
    const int* neigh_types;   // [E]
    const int* gather;        // [E] row of Hsrc per edge
    const double* xyz;        // [E][3]
    const double* r;          // [E]
    const F* Hsrc;            // [rows][NLM][K]
    const F* tab;             // [table][nodes-1][4][P*K]
    const F* tabK;            // the same numbers for the general edge kernels: [table][nodes-1][P][K][4], in double [table][nodes-1][P][2][K][2]
    size_t table_bytes;       // of tabK, all tables
    const int* pair_table;    // [T(T+1)/2] -> table
    int T;
    int spl_nodes;
    double spl_h;
    double spl_inv_h;         // 1 / spl_h
    const int* B_start;       // [NB+1] rows of the coupling list
    const int* B_lm1;
    const double* B_c;
    F* out;                   // fwd: [num_nodes][NE][K]
    const F* d_out;           // bwd: adjoint of out
    double* forces;           // bwd: [E][3]
    int accumulate_forces;    // bwd: add to forces instead of overwriting
    F* msg;                   // bwd: [E][NLM][K] adjoint message to the sender row, or null
    double* fpart;            // bwd: [shares][E][3] partial forces, needed when agg_bwd_groups() > 1
    double* forces_copy;      // bwd, scalar kernels, one channel group: receives the forces as well (or null)
    long num_edges;
    double cdiag[16];         // scalar kernels: output lm is fed by cdiag[lm] Y_lm
    // components couple by the selection rules only (components_couple); like with like through the constant harmonic (l1 = 0),
    // component l^2 + m with this factor
    int selected;
    double c_same[9];
    int more_terms;           // some entry of the coupling list has more than two terms
    int split_nodes;          // fwd, general kernel: receivers that decide how many wavefronts share one (the local nodes of a call with ghosts)
    int as_chains;            // fwd, scalar kernels: four wavefronts per receiver, sums in the order of the chains (smx_chain_edges.hpp)
    // bwd, general kernel only: receivers [node_begin, num_nodes) are processed and the message of edge e goes to
    // row e - msg_edge_begin of msg (edge lists too long for one staging buffer are taken in receiver chunks)
    int node_begin;
    long msg_edge_begin;
};

template <typename F> hipError_t launch_agg_fwd(int L_max_H, const AggParams<F>& p, hipStream_t s);
template <typename F> hipError_t launch_agg_bwd(int L_max_H, const AggParams<F>& p, hipStream_t s);
// shares of a force, one per channel group and set of paths that launch_agg_bwd splits the work into; with more than one, the
// forces come out as fpart[share][E][3] and launch_fpart_reduce adds them up
template <typename F> int agg_bwd_groups(int L_max_H, int K);

// The same two stages for scalar sender features (path list of L_max = 0) whose coupling is diagonal (cdiag), with tables and
// sender rows of less than 4 GiB.
template <typename F> hipError_t launch_agg0_fwd(const AggParams<F>& p, hipStream_t s);
template <typename F> hipError_t launch_agg0_bwd(const AggParams<F>& p, hipStream_t s);
template <typename F> int agg0_bwd_groups(int K);

// forces (+)= sum over the shares in fpart, added in ascending order
// (`copy`, if not null, receives the same sums: the caller's output array of the whole-pipeline call;
// `guard`, if not null and raised, makes every force NaN instead: the evaluation was skipped)
hipError_t launch_fpart_reduce(long edges, long E, int groups, const double* fpart, double* forces, int accumulate,
                               double* copy, hipStream_t s, const int* guard = nullptr);

// H_adj[j] (+)= sum of msg[e - e_lo] over the edges e of sender j, in ascending edge order; window: over those with
// e_lo <= e < e_hi, and slist is in ascending order already (launch_sort_buckets).  spare, here and below: scratch as long as
// slist (the ranks of the list build have served), for rows whose edges do not fit the LDS
template <typename F>
hipError_t launch_sender_reduce(int rows, int width, const int* sstart, int* slist, int* spare, const F* msg, F* H_adj,
                                int zero_first, bool window, long e_lo, long e_hi, hipStream_t s);
// The same sum for rows of K scalar features, followed by M_adj[rows][K] = H_adj . W^T (W [K][K], row n holding
// the weights of input channel n: reverse_H1 of an L_max = 0 model) in the same launch; K as sender_reduce_linear_ok
bool sender_reduce_linear_ok(int K);
template <typename F>
hipError_t launch_sender_reduce_linear(int rows, int K, const int* sstart, int* slist, int* spare, const F* msg, F* H_adj,
                                       int zero_first, const F* W, F* M_adj, hipStream_t s);

// ---------------------------------------------------------------------------
// Neighbour list on the device (smx_kernels_nlist.hip)
struct NlGrid {
    double lo[3], hi[3];     // bounding box of the positions
    double inv_bs[3];        // 1 / bin size
    int nb[3];               // bins per axis
};
// n bytes (a multiple of 16) of pinned host memory into device memory by a kernel: a few KB before a launch that needs them
// arrive sooner than by a copy command, whose completion the launch waits for (24 atoms: 14 us).
hipError_t launch_bring(void* to, const void* from_host, size_t n, hipStream_t s);
hipError_t launch_nl_bbox(const double* pos, int N, double* part, int nblocks, hipStream_t s);
hipError_t launch_nl_bins(const double* pos, int N, const NlGrid& g, int* atom_bin, int* bin_count, hipStream_t s);
hipError_t launch_nl_bin_fill(int N, const int* atom_bin, const int* bin_start, int* bin_cursor, int* bin_atoms,
                              hipStream_t s);
// edge arrays that the list kernels fill; first and num_neigh are written by a search that emits edges
struct NlEdgeArrays {
    const int* types;          // species of the atoms, or null
    const int* shift_int;      // [num_shifts][3]
    int* first;
    int* num_neigh;
    int* neigh_indices;
    int* neigh_types;
    int* neigh_shift;
    double* xyz;
    double* r;
};
// Offsets found inside the launch that uses them (chained_offset): one slot per block, a tag in the upper 32 bits that no
// earlier launch on these slots had, a word in host memory for tag | total (0xffffffff: too many), and how many times a block
// looks at the slots before it counts for itself what it misses (0: it does not look).
struct NlChain {
    unsigned long long* sums;
    unsigned long long tag;
    unsigned long long* host_total;
    int rounds;
};
constexpr int NL_CHAIN_ROUNDS = 4096;     // several milliseconds, where a launch on an idle chip waits for microseconds
// Up to this many atoms: a block reads the slots of all blocks before it (2 048 at most).  Beyond, launches for counting and
// for the prefix sum are a small part of the whole.
constexpr int NL_CHAIN_ATOMS = 8192;
inline int nl_blocks(int N) { return (N + 3) / 4; }
// bin_start == nullptr: every atom is tried, no bins (with a chain only).  fill: the ordered keys go to `sorted` (keys: scratch
// of the same size), and with `edges` every candidate is written as an edge; offsets are read from `first`, or with a chain
// found and written there.  Nothing is written past `capacity`.
hipError_t launch_nl_search(bool fill, const double* pos, int N, const NlGrid& g, const int* bin_start,
                            const int* bin_atoms, int num_shifts, const double* shift_vec, int zero_shift,
                            double r_cut, int* count, int* first, long capacity, long long* keys, long long* sorted,
                            const NlEdgeArrays* edges, const NlChain* chain, hipStream_t s);
// `room`: keys that `sorted` holds; with more candidates than that there are no edges.  fill with a chain counts as well.
hipError_t launch_nl_filter(bool fill, const double* pos, int N, const int* cfirst, const long long* sorted, long room, int num_shifts,
                            const double* shift_vec, double r_cut, int* count, int* first, long capacity,
                            const NlEdgeArrays* edges, const NlChain* chain, hipStream_t s);

// ---------------------------------------------------------------------------
// Pair terms of the edge length alone (smx_kernels_pair.hip)
struct ZblParams {
    int T;
    const double* a_pair;      // [T][T] screening length of the species pair
    const double* rmax_pair;   // [T][T] envelope radius: sum of the covalent radii
    const double* zz_pair;     // [T][T] Z_i * Z_j
    double c[4];
    int p;
};
struct PairSpline {
    const double* c;           // [pairs][nodes-1][4], unordered pairs (a <= b) row-major upper triangle
    double h;
    int nodes;
};
// node_energies[i] += sum_j V(r_ij), node_forces[ij] -= V'(r_ij) xyz_ij / r_ij      (zbl.cpp:96-125)
hipError_t launch_zbl(int N, const int* first_neigh, const int* node_types, const int* neigh_types, const double* xyz,
                      const double* r, const ZblParams& z, double* energies, double* forces, hipStream_t s);
// A[i] /= 1 + sum_j s(r_ij), divisor kept (mace.cpp:273-297, 681-705); bit 4 of *flags: r outside the spline
template <typename F>
hipError_t launch_scale_fwd(int N, const int* first_neigh, const int* node_types, const int* neigh_types, const double* r,
                            const PairSpline& sp, int T, F* A, int width, double* divisor, int* flags, hipStream_t s);
// adjoint of the above (mace.cpp:299-346, 707-757): forces += ..., A_adj /= divisor
template <typename F>
hipError_t launch_scale_bwd(int N, const int* first_neigh, const int* node_types, const int* neigh_types,
                            const double* xyz, const double* r, const PairSpline& sp, int T, const F* A, F* A_adj,
                            int width, const double* divisor, double* forces, int* flags, hipStream_t s);

// ---------------------------------------------------------------------------
// Integer list preparation
hipError_t launch_scan_exclusive(const int* in, int* out, int n, int* block_sums, hipStream_t s);  // out[n] = total
// Guard of an evaluation, carried by the last launch of the sender-list build: when the checks of this evaluation
// raised the status word, first_neigh[n_first], tstart[n_tstart] and the sender offsets are zeroed (no edges, no species
// groups: the kernels that follow then touch no unchecked index) and the status is ORed into the sticky word the
// host reads later.  Raised or not, the status is copied into the `live` word, which the kernels after this launch
// read (energies and forces become NaN); the status word itself is cleared again by the readout kernel of the same
// evaluation, after every reader of it has run, so that a replayed graph starts clean.  status == nullptr: no guard.
struct InputGuard {
    const int* status = nullptr;
    int* live = nullptr;
    int* sticky = nullptr;
    int* first_neigh = nullptr; int n_first = 0;
    int* tstart = nullptr; int n_tstart = 0;
};
// What launch_node_lists_count checks besides the sender rows when status is not null: species of nodes and edges,
// edge lengths inside (0, r_cut), no negative count, counts adding up to num_edges (all nodes) and to the key
// count (the first num_local_nodes nodes).  Bits: 1 = index or count, 2 = edge length.
struct InputChecks {
    int* status = nullptr;
    const int* neigh_types = nullptr;
    const double* r = nullptr;
    double r_cut = 0.0;
    long num_edges = 0;
    int num_local_nodes = 0;
};
// Edges by sender: sstart[rows + 1] offsets, slist[E] the edges of every row in no particular order (readers order a
// bucket as they read it; launch_sort_buckets does it in memory).  count[rows] must be zero on entry and is zero again
// when the launches have run; rank[E] is scratch.  counted: histogram, ranks and offsets came with
// launch_node_lists_count.  range_flag (or null): bit 1 raised where a key is outside [0, rows).
hipError_t launch_sender_lists(const int* gather, long E, int rows, int* count, int* rank, int* sstart, int* slist,
                               int* block_sums, bool counted, int* range_flag, hipStream_t s,
                               const InputGuard& guard = InputGuard());
hipError_t launch_sort_buckets(const int* start, int rows, int* list, int* spare, hipStream_t s);
hipError_t launch_check_counts(const int* num_neigh, int N, const int* first_neigh, int num_local_nodes, long num_edges,
                               long num_local_edges, int* status, hipStream_t s);
// first_neigh, species groups, the sender histogram count[rows] of `key[n]` with rank[n] = the place each
// entry took in its bucket, and the sender offsets sstart[rows + 1], in one launch (N, rows <= 65536).  The counters and
// *ticket must be zero on entry (every sender-list build leaves them so).
hipError_t launch_node_lists_count(const int* num_neigh, int N, int* first_neigh, const int* node_types, int T,
                                   int* tstart, int* perm, const int* key, long n, int rows, int* count, int* rank,
                                   int* sstart, int* ticket, const InputChecks& chk, hipStream_t s);
hipError_t launch_type_groups(const int* node_types, int N, int T, int* tcount, int* tstart, int* cursor,
                              int* perm, int* block_sums, hipStream_t s);
// flags[0] |= 1 if any index is outside [0, limit)
hipError_t launch_check_range(const int* v, long n, int limit, int* flags, hipStream_t s);
hipError_t launch_check_r(const double* r, long n, double r_cut, int* flags, hipStream_t s);

// ---------------------------------------------------------------------------
// Symmetric contraction (MACE::compute_M0 / compute_M1, mace.cpp:348-370, 759-777):
// value and gradient of NP polynomials of the 16 A_lm of one channel.
template <typename F>
struct PolyParams {
    int num_nodes, K, NP;              // NP polynomials (num_LM for M0, 1 for M1)
    const F* A;                        // [N][16][K]
    F* M;                              // [N][NP][K]
    F* M_grad;                         // [N][NP][16][K]
    // per polynomial (device arrays of length NP): per-variable entry lists, packed
    // mono | fa << 16 | fb << 24 in chunks of four (padding entries address the
    // all-zero row `num_entries`), and the chunk counts [32] = (v, first part), (v, rest)
    const int4* const* packed;
    const int* const* chunks;
    const F* const* coef;              // coef[p]: [T][num_entries + 1][K]
    const int* num_entries;            // monomials per polynomial
    const int* perm; const int* tstart; int T;   // atoms grouped by species
    // Standard product basis: when every polynomial p of the launch has its monomials inside compile-time table p
    // (smx_poly_tables.inc), the coefficients as [T][channel blocks] slabs in the layout of poly_spec_shape and the
    // straight-line kernel runs; else null.
    const F* table_slabs;
    int num_cus;
    // with table_slabs only: 0 values and gradients; 1 values only (M_grad unused); 2 adjoint,
    // A_adj[N][16][K] = sum_p M_adj[N][NP][K] * dM_p/dA recomputed from A (M and M_grad unused)
    int mode;
    const F* M_adj;
    F* A_adj;
};

template <typename F> hipError_t launch_poly(const PolyParams<F>& p, hipStream_t s);
// the table_slabs branch of launch_poly (smx_kernels_poly.hip)
template <typename F> hipError_t launch_poly_spec(const PolyParams<F>& p, hipStream_t s);

// A_adj[i,lm,k] = sum_LM M_grad[i,LM,lm,k] * M_adj[i,LM,k]   (reverse_M0 / reverse_M1)
template <typename F>
hipError_t launch_poly_reverse(int N, int NP, int K, const F* M_grad, const F* M_adj, F* A_adj, hipStream_t s);

// ---------------------------------------------------------------------------
// Dense channel mixing on the matrix cores.  A launch holds up to four
// independent products (blockIdx.z), each
//   C[row(node,s)][n] (+)= sum_k A[row(node,s)][k] * W[type(node)][k][n]   (or W^T)
//                          (+ sum_k A2[node][k] * W2[type(node)][k][n] when A2 is set)
// rows are (node, s) with s < sub; row (node,s) of A starts at
// A + node*a_node_stride + a_off + s*a_sub_stride and is Kd long.
template <typename TA, typename TC, typename CT>
struct GemmProb {
    const TA* A; long a_node_stride, a_off, a_sub_stride;
    TC* C; long c_node_stride, c_off, c_sub_stride;
    const CT* W; long w_type_stride, w_off;   // w_type_stride 0: one matrix for all species
    int transW;              // 0: W block is [Kd][Nn]; 1: W block is [Nn][Kd]
    int accumulate;          // 1: C += ...
    int Kd, Nn, sub;         // inner size, output columns, rows per node
    // optional second product into the same rows (sub must be 1): row of A2 starts at A2 + node*a2_node_stride
    const TA* A2; long a2_node_stride;
    // optional per-node factor of the first operand: A[row(node,s)][k] * Ascale[node*ascale_node_stride + k]
    // (row-streaming kernel only; not together with A2)
    const TA* Ascale; long ascale_node_stride;
    const CT* W2; long w2_type_stride;
    int transW2, Kd2;
};
template <typename TA, typename TC, typename CT>
struct GemmParams {
    int num_nodes;
    const int* perm;         // [num_nodes] nodes grouped by species, or null when no weight depends on the species
    const int* tstart;       // [T+1]
    int T;
    int nprob;
    int vec_ok;              // set by launch_gemm: every offset and size is a multiple of four elements
    GemmProb<TA, TC, CT> prob[4];
};
template <typename TA, typename TC, typename CT>
hipError_t launch_gemm(const GemmParams<TA, TC, CT>& p, hipStream_t s);
// whether a product with inner size Kd, Nn output columns and elements of `elem` bytes can take Ascale
bool gemm_scaled_operand_ok(int Kd, int Nn, size_t elem);

// ---------------------------------------------------------------------------
// Channel-mixing linears of the 16 (l, m) rows of an atom, with the contraction behind them (smx_kernels_linear.hip):
//     out[node][lm (, e)][K] = sum over inner[l] of A[node][lm][.] W_l(, e)[.][K]   (times scale[node][.] on the operand)
// Weights in operand order, [type][e][column tile of 16][inner / (4 V)][64 lanes][V], V = 16 bytes: lane 16 q + c holds
// k = 4 V step + q V + (0 .. V - 1) of column c.  With `coef` the polynomial of output slot 0 (one per channel) follows, and M and
// M_grad are written instead of out: coefficients [type][column tile][monomials / V][16][V], padded as in smx_poly_shape.hpp.
template <typename F>
struct LinearParams {
    int num_nodes, K, T;
    const int* perm; const int* tstart;      // species groups, or null when nothing depends on the species
    const F* A; long a_node_stride;
    const F* scale;                          // [num_nodes][K] factor of the operand rows, or null
    int inner[4], num_e[4], num_e_max;       // inner size and output blocks per l
    int row_off[16];                         // of (l, m) in an operand row, elements
    const F* W; size_t w_off[4], w_type_stride[4];
    const unsigned short* W_split;           // single precision: the weights times kSplitScale as three bf16 parts, offsets and strides
                                             // three times those of W, or null
    int split_nodes;                         // nodes that decide which kernel it is (the local ones of a call with ghosts)
    F* out; long out_node_stride; int out_off[16];
    const F* coef; F* M; F* M_grad;
};
inline bool linear_ok(int K) { return K % 32 == 0; }     // whole pieces of a row, and column tiles in pairs
template <typename F> hipError_t launch_linear(const LinearParams<F>& p, hipStream_t s);
// the part of launch_linear that runs on bf16 parts of the numbers (smx_kernels_linear32.hip)
constexpr float kSplitScale = 16777216.0f;
bool linear32_ok(const LinearParams<float>& p);
hipError_t launch_linear32(const LinearParams<float>& p, hipStream_t s);

// ---------------------------------------------------------------------------
// Readout tail (MACE::compute_readouts, mace.cpp:876-903) in one launch: node_energies[i] (+)= E0[type] +
// w1 . H1[i, l=0] + MLP_{K->16->1}(H2[i]) with W1[16][K], H2_adj = gradient of the network, H1_adj[rows][num_LM][K]
// seeded with w1 in the scalar block of the first N rows and zero elsewhere.  guard / guard_clear / guard_forces: as
// in TailParams below.
template <typename F>
hipError_t launch_readout_fused(int N, int rows, int K, int num_LM, const int* node_types, const double* atomic_energies,
                                const double* w1, const double* W1, const double* w2, double scale, const F* H1,
                                const double* H2, double* H2_adj, F* H1_adj, double* node_energies, int zero_energies,
                                double* energies_copy, const int* guard, int* guard_clear, double* guard_forces, double* guard_copy,
                                long guard_forces_n, hipStream_t s);
// H2 (mace.cpp:820-845), the readout tail and reverse_H2 (mace.cpp:847-874) in one launch; K a multiple of 16
// up to 128 (tail_fused_ok).  Atoms grouped by species (perm, tstart); H1_adj [rows][num_LM][K] is written
// whole (seed plus the adjoint of H2 in the scalar block, zero elsewhere), M1_adj [N][K] too.
template <typename F>
struct TailParams {
    int N, rows, K, num_LM, T;
    const int* perm; const int* tstart;
    const double* E0; const double* w1; const double* W1; const double* w2; double scale;
    const F* H1; const F* M1;
    const double* W_H1;      // [T][K][K]
    const double* W_M1;      // [K][K]
    const double* V_H1;      // [T][16][K]: W1 . W_H1^T
    const double* V_M1;      // [16][K]: W1 . W_M1^T
    double* H2; double* H2_adj; F* H1_adj; F* M1_adj;
    double* node_energies; int zero_energies; double* energies_copy;
    const int* guard;        // live status of a device-resident evaluation (or null): raised -> energies are NaN
    int* guard_clear;        // the word the input checks of the next evaluation raise (or null): cleared here
    double* guard_forces;    // raised guard: these guard_forces_n edge-force components become NaN as well (the
    double* guard_copy;      // (and those of the caller's array, if not null)
    long guard_forces_n;     // adjoint kernels of a skipped evaluation see no edges and write none)
    int num_cus;             // of the device: how many blocks run at once
};
bool tail_fused_ok(int K);
template <typename F> hipError_t launch_tail_fused(const TailParams<F>& p, hipStream_t s);

// ---------------------------------------------------------------------------
// The node-local stages between two aggregations in one launch each (smx_kernels_chain.hip), a block per atom: A0, M0, H1; A1,
// M1, the readout tail and their adjoints (with the arrays of the tail in q); messages, M0_adj, A0_adj, dPhi0.  Standard product
// basis in both layers, no density normalisation, with_channels(K).
template <typename F>
struct ChainParams {
    int N, K, T;
    const int* perm; const int* tstart;
    const F* Phi;            // rows of the aggregation (0, 1), where it is not in the same launch
    const F* W; const F* Wt; // A-basis weights in operand order (0, 1), transposed ones (1, 2)
    const F* WH1;            // [L_max + 1][K][K] of H1 (0), its transposes (2)
    const F* coef;           // contraction coefficients by column tile: [species][column tile][monomials / V][16][V]
    F* A;                    // A-basis: written (0) or read (2) where layer 0 has several polynomials per channel
    F* M; F* M_grad;         // polynomials and gradients: written (0, 1); M0_adj is written, M0_grad read (2)
    F* H1;                   // (0)
    F* out;                  // dPhi1 (1), dPhi0 (2)
    const F* msg; F* H1_adj; const int* sstart; int* slist; int* spare;     // (2)
    unsigned lds_front, lds_part, lds_edges;    // set by the launchers
};
inline bool chain_ok(int K) { return K == 32 || K == 64 || K == 96 || K == 128; }
template <typename F, int K> hipError_t launch_chain0(ChainParams<F> p, const AggParams<F>* agg, int L_max, hipStream_t s);
template <typename F, int K> hipError_t launch_chain1(ChainParams<F> p, const TailParams<F>& q, const AggParams<F>* agg, int L_max, hipStream_t s);
template <typename F, int K> hipError_t launch_chain2(ChainParams<F> p, const AggParams<F>* agg, int L_max, hipStream_t s);
// f(K as a constant) for the numbers of channels above
template <typename Fn>
hipError_t with_channels(int K, Fn&& f)
{
    switch (K) {
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 96: return f(std::integral_constant<int, 96>{});
    case 128: return f(std::integral_constant<int, 128>{});
    default: return hipErrorInvalidValue;
    }
}
template <typename T> hipError_t launch_fill(T* p, long n, T v, hipStream_t s);
template <typename TS, typename TD> hipError_t launch_convert(const TS* src, TD* dst, long n, hipStream_t s);

// Y[E][16], Y_grad[E][3][16] as the reference stores them (mace.cpp:118-148); inspection only
hipError_t launch_sph_harm(const double* xyz, long E, double* Y, double* Y_grad, hipStream_t s);
// R[E][nspl] spline values (mace.cpp:66-116); inspection only
template <typename F>
hipError_t launch_radial(int N, const int* first_neigh, const int* node_types, const int* neigh_types,
                         const double* r, const F* tab, const int* pair_table, int T, int nodes, double h,
                         int nspl, double* R, hipStream_t s);

// atom_forces[j] += f_e, atom_forces[i] -= f_e in a fixed order per atom; virial[6] = sum xyz (x) f, in LAMMPS order
struct ForceGather {
    int num_atoms;
    const int* send_start; int* send_list;           // edges by sender atom (null: no sender side)
    int* send_spare;                                 // as long as send_list, for buckets that do not fit the LDS
    const int* node_start; const int* node_list;     // nodes whose edges count as received by the atom; null: node i is atom i
    int num_nodes;
    const int* first_neigh;                          // [num_nodes + 1], or null without nodes
    long node_edges, num_edges;                      // edges of the nodes, all: those behind have no receiver here, but send and
                                                     // are part of the virial
    const double* forces; const double* xyz;         // [E][3] (xyz for the virial only)
    double* atom_forces;                             // [num_atoms][3] or null
    double* partial;                                 // [force_gather_blocks][6], needed for the virial, else null
    int* ticket;                                     // with partial: a word that is zero, and is zero again afterwards
    const int* flag;                                 // raised, or ...
    const int* skipped;                              // ... this one: the outputs are NaN (each may be null)
    const int* senders;                              // sender atom of every edge, where send_list is another array's: compared,
    int* differ;                                     // ... and set to 1 where they are not the same (null: not compared)
};
int force_gather_blocks(int num_atoms);             // at least one: edges may be there without an atom
hipError_t launch_force_gather(const ForceGather& g, double* virial, hipStream_t s);

}  // namespace smx
