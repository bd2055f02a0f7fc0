#!/usr/bin/env python3
"""Benchmark of the MACE energy+forces hot path on one MI355X.

One "step" = one evaluation of node energies and per-edge forces
(MACE::compute_node_energies_forces, libsymmetrix/source/mace.cpp:17-64) for a
fixed synthetic atomic configuration whose edge arrays are already resident in
HBM.  Metric: atom-steps/s = atoms / seconds per step.

Prints ONE JSON line.  Besides the driver's fields it carries
  roofline      the slowest edge kernel of the step against the HBM roofline
                (algorithmic bytes per launch / HIP-event duration of that kernel's stage)
  roofline_stages   the same figures for every edge stage (aggregations, their adjoints, the sender-side sum)
  mfma          the dense channel-mixing stages against the matrix-core peak (algorithmic flops / stage time), with the
                matrix-pipe busy share rocprofv3 counted for the stage's kernel (profiles/)
  contraction   the two symmetric contractions against the vector-arithmetic peak (flops of the nested polynomials / stage
                time) and their HBM side (variables in, values and gradients out)
  cpu_baseline  the CPU oracle (serial fp64 restatement of the reference path)
                timed on this host on the same workload
  stages_ms     HIP-event time of every stage of the pipeline
  other_precision   the same workload in the other precision mode
  second_config     (default run) the metric's second configuration: 50 000-atom alloy, K = 128, l <= 1 hidden
                    features, float32 features, with its own roofline
  pair_dependent_tables   (default run) the headline workload with one radial table per species pair
  capacity_config   (default run) the capacity configuration: a million-atom water box, MD-style steps with the
                    neighbour list searched and filtered on the device
"""
from __future__ import annotations

import argparse
import json
import os
import re
import sys
import tempfile
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

HBM_PEAK = 8.0e12  # bytes/s, MI355X HBM3E

# kernel behind each edge stage: kernels for scalar sender features / general kernels
SCALAR_KERNEL = {"agg0_fwd": "k_agg0_fwd", "agg1_fwd": "k_agg0_fwd", "agg1_bwd": "k_agg0_bwd", "agg0_bwd": "k_agg0_bwd",
                 "sender_reduce": "k_sender_reduce_linear"}
GENERAL_KERNEL = {"agg1_fwd": "k_agg_fwd", "agg1_bwd": "k_agg_bwd", "sender_reduce": "k_sender_reduce"}
EDGE_STAGES = ["agg0_fwd", "agg1_fwd", "agg1_bwd", "sender_reduce", "agg0_bwd"]


def stage_kernel(stage, L_max):
    """Name of the kernel that runs an edge stage for this kind of model."""
    return (SCALAR_KERNEL if stage.startswith("agg0") or L_max == 0 else GENERAL_KERNEL)[stage]


def measured_traffic(workload, dtype, stage, kernel):
    """HBM bytes per launch of `kernel` in `stage`, from the rocprofv3 counter summary kept under profiles/
    (FETCH_SIZE and WRITE_SIZE runs scaled by a copy of known size; the file says how it was made).  None when
    the file holds no line for this kernel, stage and precision, e.g. after a kernel was renamed."""
    path = os.path.join(HERE, "profiles", f"edge_kernels_{workload}_hbm_traffic.txt")
    if not os.path.exists(path):
        return None
    tag = "<double" if dtype == "float64" else "<float"
    for line in open(path):
        cols = line.split()
        if len(cols) >= 6 and line.startswith(kernel + tag) and stage in cols:
            k = cols.index(stage)
            try:
                return float(cols[k + 3]) * 1e6      # columns after the stage: fetch MB, write MB, traffic MB
            except (ValueError, IndexError):
                return None
    return None


MFMA_PEAK = {"float64": 78.6e12, "float32": 157.3e12}   # dense matrix-core peaks of MI355X, flop/s
# k_linear32 forms a single-precision product from six bfloat16 ones (dense peak 2.5 Pflop/s)
MFMA_PEAK_BF16_PARTS = 2.5e15 / 6
# kernel behind each dense stage (as the kernel trace names it) when it runs in feature precision F
DENSE_KERNEL = {"A0_lin": r"{L}{one}, false(, (true|false))?>", "A1": r"{L}true, false(, (true|false))?>",
                "H1": r"k_gemm_rows<{F}, {F}, {F}, \d, false", "H2": r"k_tail_fused<{F}",
                "rev_A1": r"{L}false, true(, true)?>", "rev_A0_lin": r"{L}false, {one}(, (true|false))?>",
                "rev_H1": r"k_gemm_rows<{F}, {F}, {F}, \d, false"}   # {one}: one polynomial per channel in layer 0
# {L}: the linears' kernels up to their arguments (with a contraction, with factors)
LINEARS = {"float64": r"k_linear<double, \d, ", "float32": r"(k_linear<float, \d, |k_linear32<\d, \d, )"}


def dense_peak(stage, dtype, N, K, L_max, contraction):
    """Matrix-core peak behind a dense stage.  The linears of the A-basis take k_linear32 by its dispatch's rule (N: local nodes;
    contraction: the symmetric contraction is in the same launch, behind sums of K terms in layer 0 and for scalar hidden features)."""
    if stage == "H2":      # the tail works in double whatever the feature precision
        return MFMA_PEAK["float64"]
    if dtype == "float32" and stage in ("A0_lin", "A1", "rev_A1", "rev_A0_lin") and N >= 512:
        if K % 128 == 0 and (not contraction or N >= 2048 or (stage == "A1" and L_max > 0)):
            return MFMA_PEAK_BF16_PARTS
        if K % 96 == 0 and not contraction and N >= 1024:
            return MFMA_PEAK_BF16_PARTS
    return MFMA_PEAK[dtype]


def dense_flops(stage, N, K, n_LM, n_e):
    """Flops per evaluation of a dense stage: 2 x rows x K x K multiply-adds per atom for the products (A0 linear: 16 rows;
    H1: n_LM; A1: n_e rows of K into 16 / n_e, i.e. 2 n_e K^2), as much again for each adjoint; H2 and the tail behind it
    two K x K products, and four with the 16 hidden units (the units, and the three adjoints of rank 16)."""
    per_atom = {
        "A0_lin": 32 * K * K, "rev_A0_lin": 32 * K * K,
        "H1": 2 * n_LM * K * K, "rev_H1": 2 * n_LM * K * K,
        "A1": 2 * n_e * K * K, "rev_A1": 2 * n_e * K * K,
        "H2": 4 * K * K + 128 * K,      # H2, readout network with its gradient, reverse_H2: one launch
    }
    return per_atom[stage] * N


# vector multiply-add peaks of MI355X, flop/s (32-bit multiply-adds issue in half the cycles of 64-bit ones)
VALU_PEAK = {"float64": 78.6e12, "float32": 157.3e12}


def nested_tables():
    """The monomials of the polynomials of the standard product basis in the nested order of the contraction kernels."""
    import importlib.util
    spec = importlib.util.spec_from_file_location("gen_poly_tables", os.path.join(HERE, "symmetrix_amd", "csrc", "gen_poly_tables.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)
    return [gen.nested(t) for t in gen.tables()]


def contraction_work(n_atoms, K, L_max, layer, s_bytes, mode="both"):
    """Arithmetic and HBM bytes of one symmetric-contraction launch, with the monomial lists of the standard product basis
    (harmonics up to l = 3, correlation 3) in the nested form sum_p x_p sum_q x_q (w_pq + sum_c w_pqc x_c) that the kernels
    evaluate.  Flops per atom and channel: a monomial of degree three a multiply-add for the value of its pair and one for
    the gradient, of degree two an addition, of degree one a multiply-add for the value and one operation for the gradient; a
    pair (p, q) a product and two multiply-adds, a p a multiply-add for the value and one operation for the gradient ("both";
    "value" leaves the gradients away, and "adjoint", which forms them again times the polynomial's adjoint, the values).  Bytes:
    the 16 variables in; out, per polynomial, the value ("both", "value") and its 16 gradient components ("both"); the adjoint
    reads the polynomials' adjoints and writes 16 sums."""
    gradient, value = mode != "value", mode != "adjoint"
    polys = (L_max + 1) ** 2 if layer == 0 else 1
    flops_per = 0
    for table in nested_tables()[:polys]:
        one = 16      # the constant
        flops_per += sum((2 if c != one else 1) + (2 if gradient and c != one else 0) for p, q, c in table if p != one)
        flops_per += sum((2 if value else 0) + ((1 if value else 2) if gradient else 0) for p, q, c in table if p == one)
        flops_per += (2 + (3 if gradient else 0)) * len({(p, q) for p, q, c in table if p != one})
        flops_per += ((2 if value else 0) + ((1 if value else 3) if gradient else 0)) * len({p for p, q, c in table if p != one})
    words = {"both": 16 + 17 * polys, "value": 16 + polys, "adjoint": 32 + polys}[mode]
    return flops_per * n_atoms * K, words * K * s_bytes * n_atoms


def edge_valu_flops(stage, E, K, L_max):
    """Multiply-adds the edge stages need by the algorithm (2 flops each), per evaluation: 2 * 16 * K per edge for
    the layer-0 aggregation, 2 * n_r * K for layer 1 (n_r products of a harmonic with a sender component: 16, 88 or
    243 for hidden features up to l = 0, 1, 2), and about 3.5 times as much for each adjoint (edge force and sender
    message).  Radial splines and harmonics come on top and are not counted."""
    n_r = {0: 16, 1: 88, 2: 243}[L_max]
    per_edge = {"agg0_fwd": 2 * 16 * K, "agg1_fwd": 2 * n_r * K, "agg0_bwd": 7 * 16 * K, "agg1_bwd": 7 * n_r * K}
    return per_edge.get(stage, 0) * E


def measured_mfma_busy(workload, dtype, stage, L_max):
    """Matrix-pipe busy share of the kernel behind a dense stage (SQ_VALU_MFMA_BUSY_CYCLES over SIMD cycles), from
    the rocprofv3 counter summary kept under profiles/; None when the file has no line for that kernel."""
    path = os.path.join(HERE, "profiles", f"bench_{workload}_shader_counters.txt")
    if not os.path.exists(path) or stage not in DENSE_KERNEL:
        return None
    name = re.compile(DENSE_KERNEL[stage].format(F="double" if dtype == "float64" else "float", L=LINEARS[dtype],
                                                 one="true" if L_max == 0 else "false"))
    for line in open(path):
        if name.match(line) and line.rstrip().endswith("%"):
            try:
                return float(line.split()[-1].rstrip("%")) / 100.0
            except ValueError:
                return None
    return None


def algorithmic_bytes(stage, N, E, K, s, n_LM, n_e):
    """Per-evaluation algorithmic HBM bytes of the edge kernels.

    Spline, weight and coupling tables are cache resident and not counted;
    every per-edge gather is.  36 = xyz 24 + r 8 + neighbour type 4; 40 adds the
    neighbour index; 24 is the force write, 48 a force read-modify-write.
    """
    table = {
        "agg0_fwd": 36 * E + (8 + 16 * K * s) * N,
        "agg1_fwd": (40 + n_LM * K * s) * E + (8 + n_e * K * s) * N,
        "agg1_bwd": (64 + 2 * n_LM * K * s) * E + n_e * K * s * N,
        "sender_reduce": (4 + n_LM * K * s) * E + 2 * n_LM * K * s * N,
        "agg0_bwd": 84 * E + 16 * K * s * N,
    }
    return table.get(stage)


def run_capacity(args):
    """Capacity run: the l <= 1 water model on a box of about --atoms atoms, MD-style steps.

    Every step moves all atoms by N(0, 0.01^2) on the device, refreshes the edge list on the device (a new search
    with a skin every --rebuild-every steps, the cutoff filter of the remembered pairs otherwise) and evaluates
    energies and edge forces.  Nothing but the edge count crosses to the host.  The box is a small random water box
    repeated 4 x 4 x 4 times, so that before the first move every copy of an atom must get the same energy and
    force: that is checked at full size and reported.
    """
    import torch
    from symmetrix_amd import modelgen, neighbors, systems
    from symmetrix_amd.mace import MACE

    dev = torch.device("cuda:0")
    cfg = dict(modelgen.CONFIGS["off_medium"])
    cfg["pair_dependent_radial"] = False
    model_path = os.path.join(args.model_dir, "smx_bench_off_medium.json")
    if not os.path.exists(model_path):
        modelgen.write_model(model_path, **cfg)
    reps = 4
    n_mol = max(4, -(-args.atoms // (3 * reps ** 3)))
    bpos, bcell, bsp = systems.water_box(n_mol, seed=0)
    nb = len(bpos)
    offs = np.array([[a, b, c] for a in range(reps) for b in range(reps) for c in range(reps)], dtype=np.float64) * bcell
    pos = (offs[:, None, :] + bpos[None, :, :]).reshape(-1, 3)
    species = np.tile(bsp, reps ** 3).astype(np.int32)
    cell = bcell * reps
    N = len(pos)
    r_cut, skin = cfg["r_cut"], args.skin
    dpos = torch.from_numpy(np.ascontiguousarray(pos)).to(dev)
    dty = torch.from_numpy(species).to(dev)
    del pos
    eng = MACE(model_path, args.dtype)
    if args.staging_gb > 0:
        eng.set_staging_limit(int(args.staging_gb * 1e9))
    nl = neighbors.DeviceNeighborList()
    stream = torch.cuda.current_stream().cuda_stream
    out_E = torch.zeros(N, dtype=torch.float64, device=dev)
    out_F = None

    def evaluate(E):
        nonlocal out_F
        if out_F is None or out_F.numel() < 3 * E:
            out_F = torch.zeros(int(3 * E * 1.05), dtype=torch.float64, device=dev)
        p = nl.ptr
        eng.compute_device(N, dty.data_ptr(), p["num_neigh"], p["neigh_indices"], p["neigh_types"], p["xyz"], p["r"], E,
                           out_E.data_ptr(), out_F.data_ptr(), stream)

    # ---- before any move: all 64 copies of the small box must agree
    E = nl.build(N, dpos.data_ptr(), dty.data_ptr(), cell, r_cut, skin=skin)
    evaluate(E)
    torch.cuda.synchronize()
    num_neigh = torch.empty(N, dtype=torch.int32, device=dev)
    neigh = torch.empty(E, dtype=torch.int32, device=dev)

    class DeviceInts:   # zero-copy view of a device array of the list object
        def __init__(self, ptr, n):
            self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i4", data=(ptr, False), version=2)

    num_neigh.copy_(torch.as_tensor(DeviceInts(nl.ptr["num_neigh"], N), device=dev))
    neigh.copy_(torch.as_tensor(DeviceInts(nl.ptr["neigh_indices"], E), device=dev))
    recv = torch.repeat_interleave(torch.arange(N, device=dev), num_neigh.long())
    f = out_F[:3 * E].view(E, 3)
    fa = torch.zeros(N, 3, dtype=torch.float64, device=dev)
    fa.index_add_(0, neigh.long(), f)
    fa.index_add_(0, recv, -f)
    e_rep = out_E.view(reps ** 3, nb)
    f_rep = fa.view(reps ** 3, nb, 3)
    e_dev = float((e_rep - e_rep[0]).abs().max().item())
    f_dev = float((f_rep - f_rep[0]).abs().max().item())
    e_scale = float(e_rep[0].abs().max().item())
    f_scale = float(f_rep[0].abs().max().item())
    energy0 = float(out_E.sum().item())
    del num_neigh, neigh, recv, fa, f, e_rep, f_rep
    torch.cuda.empty_cache()

    # ---- MD-style steps
    gen = torch.Generator(device=dev)
    gen.manual_seed(0)
    t_list_build, t_list_update, t_eval, t_step = [], [], [], []
    edges = []
    total = args.warmup + args.steps
    for it in range(total):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        dpos.add_(torch.randn(dpos.shape, dtype=torch.float64, device=dev, generator=gen), alpha=0.01)
        rebuild = it % args.rebuild_every == 0
        if rebuild:
            E = nl.build(N, dpos.data_ptr(), dty.data_ptr(), cell, r_cut, skin=skin)
        else:
            E = nl.update(dpos.data_ptr(), dty.data_ptr(), r_cut)
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        evaluate(E)
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        if it >= args.warmup:
            (t_list_build if rebuild else t_list_update).append(t1 - t0)
            t_eval.append(t2 - t1)
            t_step.append(t2 - t0)
            edges.append(E)
        if it % 10 == 0:
            print(f"[capacity] step {it}/{total} edges={E} step={1e3 * (t2 - t0):.1f} ms", file=sys.stderr, flush=True)
    free_b, total_b = torch.cuda.mem_get_info()
    ms = 1e3 * float(np.mean(t_step))
    K, L_max = cfg["num_channels"], cfg["L_max"]
    # stage times of two more evaluations on the last list (HIP events on the kernels' stream)
    eng.set_profiling(True)
    acc = {}
    for _ in range(2):
        evaluate(E)
        for k, v in eng.stage_times().items():
            acc[k] = acc.get(k, 0.0) + v / 2
    eng.set_profiling(False)
    n_LM, n_e, s_b = (L_max + 1) ** 2, {0: 16, 1: 40, 2: 71}[L_max], 8 if args.dtype == "float64" else 4
    # When the adjoint messages exceed the staging buffer, the layer-1 adjoint and the sender-side sum alternate per
    # receiver chunk inside one stage: the roofline then prices both kernels' bytes against the stage's time.
    chunked = acc.get("sender_reduce", 0.0) < 0.01 * acc.get("agg1_bwd", 1.0)
    b_bwd = algorithmic_bytes("agg1_bwd", N, E, K, s_b, n_LM, n_e) + (algorithmic_bytes("sender_reduce", N, E, K, s_b, n_LM, n_e) if chunked else 0)
    t_bwd = acc.get("agg1_bwd", 0.0) * 1e-3
    ach = b_bwd / t_bwd / 1e9 if t_bwd > 0 else 0.0
    line = {
        "metric": "atom-steps/s per MI355X (energy+forces)", "value": N / (ms * 1e-3), "unit": "atom-steps/s",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None,
        "dtype": "f64" if args.dtype == "float64" else "f32-features/f64-accumulation", "data": "synthetic",
        "config": {
            "workload": f"water_capacity: {N} atoms ({reps}^3 copies of a {nb}-atom water box, moved by N(0, 0.01^2) A every "
                        f"step), about {int(np.mean(edges))} edges, K={K}, L_max={L_max}, r_cut={r_cut}, device neighbour list "
                        f"with skin {skin} A searched anew every {args.rebuild_every} steps and filtered every step",
            "atoms": N, "edges_mean": float(np.mean(edges)), "channels": K, "L_max": L_max,
        },
        "step_breakdown_ms": {
            "evaluation": 1e3 * float(np.mean(t_eval)),
            "move_and_list_search": 1e3 * float(np.mean(t_list_build)) if t_list_build else None,
            "move_and_list_filter": 1e3 * float(np.mean(t_list_update)) if t_list_update else None,
            "list_searches_timed": len(t_list_build), "list_filters_timed": len(t_list_update),
        },
        "evaluation_only_value": N / float(np.mean(t_eval)),
        "hbm_in_use_GB": (total_b - free_b) / 1e9,
        "copies_check": {"energy_max_abs_diff": e_dev, "energy_scale": e_scale, "atom_force_max_abs_diff": f_dev, "atom_force_scale": f_scale,
                         "note": "64 periodic copies of the small box before the first move: equal up to summation order"},
        "energy_first": energy0,
        "stages_ms": acc,
        "roofline": {"bound": "hbm", "kernel": "k_agg_bwd" + (" + k_sender_reduce, alternating per receiver chunk" if chunked else ""),
                     "stage": "agg1_bwd", "achieved": ach, "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": ach / (HBM_PEAK / 1e9),
                     "traffic": None, "algorithmic_bytes_per_launch": b_bwd, "kernel_ms": acc.get("agg1_bwd", 0.0)},
    }
    del eng, nl, out_E, out_F, dpos, dty
    torch.cuda.empty_cache()
    return line


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default="off_small", choices=["tiny", "off_small", "off_medium", "off_medium_l2", "mp_medium", "water_capacity"])
    ap.add_argument("--atoms", type=int, default=1000000, help="water_capacity: target atom count")
    ap.add_argument("--rebuild-every", type=int, default=10, help="water_capacity: steps between neighbour searches")
    ap.add_argument("--staging-gb", type=float, default=0.0,
                    help="water_capacity: bound for the adjoint message buffer in GB (0 = the library's default)")
    ap.add_argument("--skin", type=float, default=0.6, help="water_capacity: list radius minus cutoff (Angstrom)")
    ap.add_argument("--scale", type=float, default=1.0, help="shrink the atom count (tests)")
    ap.add_argument("--dtype", default=None, choices=["float64", "float32"],
                    help="default: float64, and float32 features for water_capacity")
    ap.add_argument("--ghosts", action="store_true",
                    help="periodic images as explicit ghost nodes that go through layer 0 only (the pair style's "
                         "no_mpi_message_passing layout on one rank) instead of senders mapped to their owners")
    ap.add_argument("--pair-tables", action="store_true",
                    help="a radial table of its own for every species pair (several distinct tables take the "
                         "general edge kernels)")
    ap.add_argument("--no-second", action="store_true",
                    help="default workload only: skip the second configuration of the metric (mp_medium, float32 features) "
                         "and the pair-dependent-table variant that ride along")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--cpu-atoms", type=int, default=0, help="atoms in the CPU sample (0 = whole workload)")
    ap.add_argument("--model-dir", default=tempfile.gettempdir())
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also launch one device-to-device copy of 1 GiB (a kernel of known traffic for counter runs)")
    args = ap.parse_args()
    if args.dtype is None:
        args.dtype = "float32" if args.workload == "water_capacity" else "float64"
    if args.gpus != 1:
        print("bench.py: this build runs on exactly one GPU (no collectives exist in it); use --gpus 1", file=sys.stderr)
        sys.exit(2)

    import torch
    from symmetrix_amd import modelgen, neighbors, systems
    from symmetrix_amd.mace import MACE

    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(1)
    dev = torch.device("cuda:0")
    if args.workload == "water_capacity":
        print(json.dumps(run_capacity(args)))
        return

    def measure(workload, dtype, steps, warmup, pair_tables=False, ghosts=False, scale=1.0, both=True, host_leg=True):
        """One workload in one precision (and, with `both`, in the other): model file, synthetic system, timing."""
        cfg = dict(modelgen.CONFIGS[workload])
        # plain MACE has a species-independent radial network: every pair table of the file is equal;
        # pair_tables gives every species pair its own table (as a distance transform does)
        cfg["pair_dependent_radial"] = bool(pair_tables)
        model_path = os.path.join(args.model_dir, f"smx_bench_{workload}{'_pairs' if pair_tables else ''}.json")
        if not os.path.exists(model_path):
            modelgen.write_model(model_path, **cfg)
        pos, cell, species = systems.config_system(workload, seed=0, scale=scale)
        nl = neighbors.neighbor_list(pos, cell, cfg["r_cut"])
        ea = neighbors.edge_arrays(nl, species)
        N, E = int(ea["num_nodes"]), int(len(ea["r"]))
        N_ghost, E_local = 0, E
        if ghosts:
            ea = neighbors.ghost_edge_arrays(nl, species)
            N, N_ghost = int(ea["num_local_nodes"]), int(ea["num_ghost_nodes"])
            E_local, E = int(ea["num_neigh"][:N].sum()), int(len(ea["r"]))

        def to_dev(a, dt):
            return torch.from_numpy(np.ascontiguousarray(a)).to(dev, dtype=dt)

        d = dict(
            node_types=to_dev(ea["node_types"], torch.int32), num_neigh=to_dev(ea["num_neigh"], torch.int32),
            neigh_indices=to_dev(ea["neigh_indices"], torch.int32), neigh_types=to_dev(ea["neigh_types"], torch.int32),
            xyz=to_dev(ea["xyz"], torch.float64), r=to_dev(ea["r"], torch.float64),
        )
        out_E = torch.zeros(N, dtype=torch.float64, device=dev)
        out_F = torch.zeros(3 * E, dtype=torch.float64, device=dev)

        def run_mode(dtype, steps, warmup):
            eng = MACE(model_path, dtype)
            stream = torch.cuda.current_stream().cuda_stream

            def step():
                if ghosts:
                    eng.compute_ghosted_device(N, N_ghost, d["node_types"].data_ptr(), d["num_neigh"].data_ptr(),
                                               d["neigh_indices"].data_ptr(), d["neigh_types"].data_ptr(), d["xyz"].data_ptr(),
                                               d["r"].data_ptr(), E, E_local, out_E.data_ptr(), out_F.data_ptr(), stream)
                else:
                    eng.compute_device(N, d["node_types"].data_ptr(), d["num_neigh"].data_ptr(), d["neigh_indices"].data_ptr(),
                                       d["neigh_types"].data_ptr(), d["xyz"].data_ptr(), d["r"].data_ptr(), E,
                                       out_E.data_ptr(), out_F.data_ptr(), stream)

            for _ in range(warmup):
                step()
            torch.cuda.synchronize()
            # timed region: exactly `steps` evaluations as asynchronous enqueues between two synchronisations
            t0 = time.perf_counter()
            for _ in range(steps):
                step()
            torch.cuda.synchronize()
            dt_async = time.perf_counter() - t0
            # the same number of steps with per-stage HIP events on the stream the kernels run on (the events are per
            # model and reused every step, so they are read back after every step)
            eng.set_profiling(True)
            acc = {}
            t0 = time.perf_counter()
            for _ in range(steps):
                step()
                for k, v in eng.stage_times().items():
                    acc[k] = acc.get(k, 0.0) + v
            torch.cuda.synchronize()
            dt = time.perf_counter() - t0
            eng.set_profiling(False)
            res = dict(ms_sync=1e3 * dt / steps, ms=1e3 * dt_async / steps, stages={k: v / steps for k, v in acc.items()},
                       tables=eng._int("num_radial_tables_0"), contraction_tables=eng._int("contraction_tables"))
            if host_leg:
                # the same evaluation through the host-array entry point (upload, range checks, download included)
                hsteps = max(3, min(10, steps // 4))

                def host_step():
                    if ghosts:
                        eng.compute_ghosted(N, N_ghost, ea["node_types"], ea["num_neigh"], ea["neigh_indices"],
                                            ea["neigh_types"], ea["xyz"], ea["r"])
                    else:
                        eng.compute_node_energies_forces(N, ea["node_types"], ea["num_neigh"], ea["neigh_indices"],
                                                         ea["neigh_types"], ea["xyz"], ea["r"])
                host_step()
                t0 = time.perf_counter()
                for _ in range(hsteps):
                    host_step()
                    _ = eng.node_energies, eng.node_forces
                res["ms_host"] = 1e3 * (time.perf_counter() - t0) / hsteps
                step()
                torch.cuda.synchronize()
            res["energy"] = float(out_E.sum().item())
            res["forces"] = out_F.cpu().numpy().copy()
            del eng
            return res

        res = run_mode(dtype, steps, warmup)
        K, L_max = cfg["num_channels"], cfg["L_max"]
        n_LM = (L_max + 1) ** 2
        n_e = {0: 16, 1: 40, 2: 71}[L_max]
        s_bytes = 8 if dtype == "float64" else 4

        def stage_bytes(k):   # layer-0 stages run over all nodes and edges, layer-1 stages over the local ones
            if k.startswith("agg0"):
                return algorithmic_bytes(k, N + N_ghost, E, K, s_bytes, n_LM, n_e)
            return algorithmic_bytes(k, N, E_local, K, s_bytes, n_LM, n_e)

        dom = max(EDGE_STAGES, key=lambda k: res["stages"].get(k, 0.0))
        dom_bytes = stage_bytes(dom)
        dom_s = res["stages"][dom] * 1e-3
        achieved = dom_bytes / dom_s / 1e9 if dom_s > 0 else 0.0
        total_bytes = sum(stage_bytes(k) for k in EDGE_STAGES) + (32 * E + 24 * N)
        kernel = stage_kernel(dom, L_max)
        prof_name = workload + ("_pairs" if pair_tables else "")
        profiled = scale == 1.0 and not ghosts
        stages_rl = {}
        for k in EDGE_STAGES:
            ms_k = res["stages"].get(k, 0.0)
            if ms_k <= 0.0:
                continue
            b_k = stage_bytes(k)
            kern_k = stage_kernel(k, L_max)
            ach = b_k / (ms_k * 1e-3) / 1e9
            stages_rl[k] = {"kernel": kern_k, "algorithmic_bytes": b_k, "kernel_ms": ms_k, "achieved": ach,
                            "frac": ach / (HBM_PEAK / 1e9),
                            "traffic": measured_traffic(prof_name, dtype, k, kern_k) if profiled else None}
            fl = edge_valu_flops(k, E if k.startswith("agg0") else E_local, K, L_max)
            if fl:
                # the same stage against the vector arithmetic it cannot do without (the bound that bites: about
                # 20 bytes of HBM data per edge and channel against one to several hundred multiply-adds)
                stages_rl[k]["valu"] = {"flops": fl, "achieved_tflops": fl / (ms_k * 1e-3) / 1e12,
                                        "peak_tflops": VALU_PEAK[dtype] / 1e12, "frac": fl / (ms_k * 1e-3) / VALU_PEAK[dtype]}
        mfma = {}
        for k in ("A0_lin", "H1", "A1", "H2", "rev_A1", "rev_H1", "rev_A0_lin"):
            ms_k = res["stages"].get(k, 0.0)
            n_k = (N + N_ghost) if k in ("A0_lin", "H1", "rev_H1", "rev_A0_lin") else N
            fl = dense_flops(k, n_k, K, n_LM, n_e)
            # (a stage folded into another launch has no time of its own)
            peak = dense_peak(k, dtype, N, K, L_max, res["stages"].get({"A0_lin": "M0", "A1": "M1"}.get(k), 1.0) == 0.0)
            if ms_k == 0.0:
                mfma[k] = {"flops": fl, "note": "folded into another launch (sender_reduce carries reverse_H1 for scalar hidden features)"}
                continue
            mfma[k] = {"flops": fl, "kernel_ms": ms_k, "achieved_tflops": fl / (ms_k * 1e-3) / 1e12, "peak_tflops": peak / 1e12,
                       "frac": fl / (ms_k * 1e-3) / peak,
                       "mfma_busy_profiled": measured_mfma_busy(workload, dtype, k, L_max) if profiled and not pair_tables else None}
        # the symmetric contractions: vector arithmetic against the vector peak, and their HBM side
        contraction = {}
        # (layer 0 with several polynomials per channel and the standard basis keeps no gradients: values in M0,
        # the gradient formed again in rev_M0)
        split0 = bool(res["contraction_tables"] & 1) and n_LM > 1
        for k, layer, n_k, mode in (("M0", 0, N + N_ghost, "value" if split0 else "both"), ("M1", 1, N, "both"),
                                    ("rev_M0", 0, N + N_ghost, "adjoint")):
            ms_k = res["stages"].get(k, 0.0)
            if k == "rev_M0" and not split0:
                continue
            fl, by = contraction_work(n_k, K, L_max, layer, s_bytes, mode)
            if ms_k == 0.0:
                contraction[k] = {"flops": fl, "note": "evaluated in the launch of the layer's A-basis linear"}
                continue
            vpeak = VALU_PEAK[dtype]
            contraction[k] = {"kernel": "k_poly_spec" if res["contraction_tables"] & (1 << layer) else "k_poly", "mode": mode,
                              "flops": fl, "kernel_ms": ms_k, "achieved_tflops": fl / (ms_k * 1e-3) / 1e12,
                              "peak_tflops": vpeak / 1e12, "valu_frac": fl / (ms_k * 1e-3) / vpeak,
                              "algorithmic_bytes": by, "hbm_frac": by / (ms_k * 1e-3) / HBM_PEAK}
        out = dict(
            cfg=cfg, model_path=model_path, ea=ea, N=N, E=E, N_ghost=N_ghost, E_local=E_local, res=res,
            value=N / (res["ms"] * 1e-3),
            workload=f"{workload}: {N} atoms, {E} edges, K={K}, L_max={L_max}, r_cut={cfg['r_cut']}, random-init symmetrix "
                     f"JSON model (seed 0), " + ("one radial table per species pair" if pair_tables else
                                                 "species-independent radial tables"),
            roofline={
                "bound": "hbm", "kernel": kernel, "stage": dom, "achieved": achieved, "peak": HBM_PEAK / 1e9, "unit": "GB/s",
                "frac": achieved / (HBM_PEAK / 1e9),
                "traffic": measured_traffic(prof_name, dtype, dom, kernel) if profiled else None,
                "algorithmic_bytes_per_launch": dom_bytes, "kernel_ms": res["stages"][dom],
                "whole_step_algorithmic_bytes": total_bytes,
                "whole_step_frac": (total_bytes / HBM_PEAK) / (res["ms"] * 1e-3),
            },
            roofline_stages=stages_rl, mfma=mfma, contraction=contraction,
        )
        if both:
            other = "float32" if dtype == "float64" else "float64"
            out["other"] = (other, run_mode(other, max(5, steps // 2), warmup))
        return out

    if args.calibrate_copy:
        src = torch.ones(1 << 28, dtype=torch.float32, device=dev)   # 1 GiB read + 1 GiB written
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst

    if args.ghosts:
        args.no_cpu = True     # the CPU leg times the plain layout
    m = measure(args.workload, args.dtype, args.steps, args.warmup, pair_tables=args.pair_tables, ghosts=args.ghosts,
                scale=args.scale)
    res, cfg, N, E = m["res"], m["cfg"], m["N"], m["E"]
    other, res_other = m["other"]
    line = {
        "metric": "atom-steps/s per MI355X (energy+forces)",
        "value": m["value"],
        "unit": "atom-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": res["ms"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if args.dtype == "float64" else "f32-features/f64-accumulation",
        "data": "synthetic",
        "config": {
            "workload": m["workload"], "atoms": N, "edges": E, "channels": cfg["num_channels"], "L_max": cfg["L_max"],
            "scale": args.scale, "ghost_nodes": m["N_ghost"], "edges_of_local_receivers": m["E_local"],
        },
        "roofline": m["roofline"],
        "roofline_stages": m["roofline_stages"],
        "mfma": m["mfma"],
        "contraction": m["contraction"],
        "stages_ms": res["stages"],
        "ms_per_step_with_event_readback": res["ms_sync"],
        "host_arrays": {"ms_per_step": res["ms_host"], "value": N / (res["ms_host"] * 1e-3),
                        "note": "numpy arrays in, numpy energies and forces out: PCIe transfers and input checks included"},
        "energy": res["energy"],
        "other_precision": {"dtype": other, "ms_per_step": res_other["ms"], "value": N / (res_other["ms"] * 1e-3),
                            "energy": res_other["energy"], "stages_ms": res_other["stages"]},
    }
    default_run = args.workload == "off_small" and args.scale == 1.0 and not args.ghosts and not args.pair_tables
    if default_run and not args.no_second:
        # the metric is quoted on two configurations: the second one (50 000-atom alloy, K = 128, hidden features up
        # to l = 1, float32 features) rides along with its own figures; fewer steps, no CPU leg
        s2 = max(5, args.steps // 5)
        m2 = measure("mp_medium", "float32", s2, 2, both=False, host_leg=False)
        line["second_config"] = {
            "workload": m2["workload"], "dtype": "f32-features/f64-accumulation", "steps": s2, "warmup": 2,
            "ms_per_step": m2["res"]["ms"], "value": m2["value"], "unit": "atom-steps/s", "roofline": m2["roofline"],
            "roofline_stages": m2["roofline_stages"], "mfma": m2["mfma"], "contraction": m2["contraction"],
            "stages_ms": m2["res"]["stages"], "energy": m2["res"]["energy"],
        }
        # the headline workload with one radial table per species pair (ten tables for four species)
        m3 = measure("off_small", args.dtype, max(5, args.steps // 2), args.warmup, pair_tables=True, both=False, host_leg=False)
        line["pair_dependent_tables"] = {
            "workload": m3["workload"], "dtype": line["dtype"], "ms_per_step": m3["res"]["ms"], "value": m3["value"],
            "unit": "atom-steps/s", "roofline": m3["roofline"], "roofline_stages": m3["roofline_stages"],
            "stages_ms": m3["res"]["stages"],
        }
        # the capacity configuration at its size, a short MD-style loop (two list searches); freed before the CPU leg
        del m2, m3
        torch.cuda.empty_cache()
        free_b, _ = torch.cuda.mem_get_info()
        if free_b > 200e9 and not args.no_cpu:
            cargs = argparse.Namespace(**vars(args))
            cargs.steps, cargs.warmup, cargs.dtype, cargs.rebuild_every = 20, 2, "float32", 10
            line["capacity_config"] = run_capacity(cargs)
        else:
            line["capacity_config"] = {"skipped": f"needs about 185 GB of free HBM, {free_b / 1e9:.0f} GB are free"}

    # ---- CPU baseline: the oracle (serial fp64 port of the reference path) on this host
    if not args.no_cpu:
        from oracle.oracle import OracleMACE
        ea = m["ea"]
        orc = OracleMACE(m["model_path"])
        if args.cpu_atoms and args.cpu_atoms < N:
            p2, c2, s2_ = systems.config_system(args.workload, seed=0, scale=args.scale * args.cpu_atoms / N)
            nl2 = neighbors.neighbor_list(p2, c2, cfg["r_cut"])
            ea2 = neighbors.edge_arrays(nl2, s2_)
            sample = f"{ea2['num_nodes']} atoms / {len(ea2['r'])} edges sub-box of the workload (same density, same model), 1 evaluation"
        else:
            ea2 = ea
            sample = f"the whole workload ({N} atoms, {E} edges), 1 evaluation"
        # repeated until about 10 s of CPU time have been spent (at most 5 evaluations); the best time counts
        times = []
        while len(times) < 5 and sum(times) < 10.0:
            t0 = time.perf_counter()
            orc.compute_node_energies_forces(ea2["num_nodes"], ea2["node_types"], ea2["num_neigh"], ea2["neigh_indices"],
                                             ea2["neigh_types"], ea2["xyz"], ea2["r"])
            times.append(time.perf_counter() - t0)
        dt = min(times)
        sample += f" x {len(times)} (best taken)"
        cpu_value = ea2["num_nodes"] / dt
        line["cpu_baseline"] = {"value": cpu_value, "unit": "atom-steps/s", "cores": 1, "kind": "port",
                                "sample": sample, "seconds": dt, "host_cores": os.cpu_count(),
                                "gpu_over_cpu_1core": m["value"] / cpu_value}
        if ea2 is ea:
            Ecpu = float(orc.node_energies.sum())
            line["cpu_baseline"]["energy_rel_diff_vs_gpu"] = abs(Ecpu - res["energy"]) / abs(Ecpu)
            line["cpu_baseline"]["force_max_abs_diff_vs_gpu"] = float(np.abs(orc.node_forces - res["forces"]).max())
    print(json.dumps(line))


if __name__ == "__main__":
    main()
