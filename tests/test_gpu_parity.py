"""GPU parity tests proper (run on an MI355X with -m gpu).

Every check goes through the C ABI (symmetrix_amd.mace.MACE is a ctypes face of
include/symmetrix_amd.h) and compares the HIP engine with the CPU oracle on the
same seeded inputs.  Tolerances are the ones the task states:
  fp64 mode           energy rel <= 1e-10, forces max-abs <= 1e-8 eV/A
  fp32-feature mode   energy rel <= 1e-5,  forces max-abs <= 1e-4 eV/A
"""
import json
import os

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")
TOL = {"float64": dict(E=1e-10, F=1e-8, inter=1e-11), "float32": dict(E=1e-5, F=1e-4, inter=2e-5)}
INTERMEDIATES = ["Y", "Y_grad", "R0", "R1", "A0", "M0", "H1", "Phi1", "A1", "M1", "H2", "H2_adj", "M1_adj",
                 "A1_adj", "Phi1_adj", "H1_adj", "M0_adj", "A0_adj", "M1_grad", "M0_grad"]
# (M0_grad last: with several polynomials per channel an evaluation keeps no layer-0 gradients, the adjoint forms
# them again from A0; asking for the array evaluates them from the A0 the evaluation left)


@pytest.fixture(scope="module")
def gpu():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU box"
    from symmetrix_amd.mace import MACE
    return MACE


def _oracle():
    from oracle.oracle import OracleMACE
    return OracleMACE


def _compare(orc, eng, dtype, names=INTERMEDIATES):
    tol = TOL[dtype]
    for name in names:
        a = getattr(orc, name); b = getattr(eng, name)
        assert a.shape == b.shape, name
        scale = max(1.0, np.abs(a).max()) if len(a) else 1.0
        assert np.abs(a - b).max(initial=0.0) <= tol["inter"] * scale * 10, name
    Eo, Eg = orc.node_energies.sum(), eng.node_energies.sum()
    assert abs(Eo - Eg) <= tol["E"] * abs(Eo)
    assert np.abs(orc.node_energies - eng.node_energies).max() <= tol["E"] * max(1.0, np.abs(orc.node_energies).max()) * 10
    assert np.abs(orc.node_forces - eng.node_forces).max(initial=0.0) <= tol["F"]


CASES = [
    # K, L_max, atoms, pair-dependent radial
    (32, 0, 40, True), (32, 1, 40, True), (96, 0, 48, False), (128, 1, 36, True), (48, 1, 24, True),
    (20, 0, 17, True), (64, 1, 30, False), (128, 0, 30, True),
    # wider than one block of channels: several channel groups and column tiles
    (256, 0, 20, False), (192, 1, 16, False),
    # hidden features up to l = 2 (128x0e+128x1o+128x2e and the like): 17 paths, 9 polynomials
    (16, 2, 30, True), (128, 2, 20, False), (40, 2, 26, True),
]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max,natoms,pair", CASES)
def test_pipeline_matches_oracle(gpu, tmp_models, K, L_max, natoms, pair, dtype):
    model = H.tiny_model(K=K, L_max=L_max, n_pts=64, seed=K + L_max, pair=pair)
    path = H.write_model(model, tmp_models / f"m_{K}_{L_max}_{int(pair)}.json")
    orc = _oracle()(model)
    eng = gpu(path, dtype)
    pos, cell, sp = H.small_system(natoms, seed=natoms)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"case K={K} L_max={L_max} atoms={natoms} edges={len(ea['r'])} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)
    # bit-reproducible: no atomics on floats anywhere
    f1, e1 = eng.node_forces, eng.node_energies
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(f1, eng.node_forces) and np.array_equal(e1, eng.node_energies)
    # caller-side reduction, symmetrix_calc.py:93-102 / pair_symmetrix_mace.cpp:334-368
    F, V = eng.reduce_forces(len(pos), nl["j"], virial=True)
    assert np.allclose(F, H.atom_forces(nl, orc.node_forces, len(pos)), atol=TOL[dtype]["F"] * 10)
    f = orc.node_forces.reshape(-1, 3); x = ea["xyz"].reshape(-1, 3)
    W = x.T @ f
    Vref = np.array([W[0, 0], W[1, 1], W[2, 2], 0.5 * (W[0, 1] + W[1, 0]), 0.5 * (W[0, 2] + W[2, 0]), 0.5 * (W[1, 2] + W[2, 1])])
    assert np.allclose(V, Vref, atol=TOL[dtype]["F"] * 100)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max,natoms,layers", [(32, 0, 40, (0, 1)), (33, 1, 25, (0, 1)), (96, 0, 48, (1,)),
                                                   (20, 1, 30, (0,)), (16, 2, 22, (0, 1)), (128, 1, 20, (0, 1))])
def test_monomials_outside_the_standard_basis_take_the_general_kernel(gpu, tmp_models, K, L_max, natoms, layers, dtype):
    """The symmetric contraction has a kernel compiled for the monomial lists of the standard product basis (every
    other model in this file runs it) and a general one that walks whatever lists the file holds.  Files with one
    more monomial in the polynomials of layer 0, of layer 1 or of both: the loader must send exactly those layers to
    the general kernel, and all intermediates, energies and forces must still match the oracle."""
    model = H.add_foreign_monomials(H.tiny_model(K=K, L_max=L_max, n_pts=64, seed=K + L_max, pair=False), layers, seed=K)
    path = H.write_model(model, tmp_models / f"foreign_{K}_{L_max}_{len(layers)}_{layers[0]}.json")
    orc = _oracle()(model)
    eng = gpu(path, dtype)
    assert eng._int("contraction_tables") == 3 - sum(1 << l for l in layers)
    pos, cell, sp = H.small_system(natoms, seed=natoms)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"case K={K} L_max={L_max} atoms={natoms} edges={len(ea['r'])} foreign monomials in layers {layers} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,natoms", [(20, 70), (96, 200), (33, 9)])
def test_two_species_three_radial_tables(gpu, tmp_models, K, natoms, dtype):
    """Scalar hidden features with a few distinct pair tables: the scalar edge kernels choose the table per edge."""
    model = H.tiny_model(K=K, L_max=0, T=(1, 8), n_pts=50, seed=K, pair=True)
    path = H.write_model(model, tmp_models / f"two_{K}.json")
    orc = _oracle()(model)
    eng = gpu(path, dtype)
    pos, cell, sp = H.small_system(natoms, probs=(0.6, 0.4), seed=natoms)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"case K={K} atoms={natoms} edges={len(ea['r'])} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,natoms", [(24, 60), (7, 33)])
def test_long_spline_tables(gpu, tmp_models, K, natoms, dtype):
    """One radial table with 400 nodes (the other cases have 24 to 256)."""
    model = H.tiny_model(K=K, L_max=0, n_pts=400, seed=K, pair=False)
    path = H.write_model(model, tmp_models / f"long_{K}.json")
    orc = _oracle()(model)
    eng = gpu(path, dtype)
    pos, cell, sp = H.small_system(natoms, seed=natoms)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"case K={K} atoms={natoms} edges={len(ea['r'])} {dtype} 400 spline nodes", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)
    f1, e1 = eng.node_forces, eng.node_energies
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(f1, eng.node_forces) and np.array_equal(e1, eng.node_energies)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,natoms", [(6, 41), (7, 33), (20, 52)])
def test_channel_counts_that_leave_lanes_idle(gpu, tmp_models, K, natoms, dtype):
    """Scalar hidden features and a channel count below the 32 lanes that an edge has: lanes beyond the last channel work
    on another one with a zero adjoint, add nothing to the sums and store nothing."""
    model = H.tiny_model(K=K, L_max=0, n_pts=64, seed=100 + K, pair=False)
    path = H.write_model(model, tmp_models / f"partial_{K}.json")
    orc = _oracle()(model)
    eng = gpu(path, dtype)
    pos, cell, sp = H.small_system(natoms, seed=natoms)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"case K={K} atoms={natoms} edges={len(ea['r'])} {dtype} idle lanes", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)
    f1, e1 = eng.node_forces, eng.node_energies
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(f1, eng.node_forces) and np.array_equal(e1, eng.node_energies)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_golden_fixture(gpu, dtype):
    z = np.load(os.path.join(GOLD, "tiny_case.npz"))
    eng = gpu(os.path.join(GOLD, "tiny_model.json"), dtype)
    eng.compute_node_energies_forces(len(z["node_types"]), z["node_types"], z["num_neigh"], z["neigh_indices"],
                                     z["neigh_types"], z["xyz"], z["r"])
    tol = TOL[dtype]
    E = z["node_energies"].sum()
    assert abs(eng.node_energies.sum() - E) <= tol["E"] * abs(E)
    assert np.abs(eng.node_forces - z["node_forces"]).max() <= tol["F"]
    for name in ("A0", "M0", "H1", "Phi1", "A1", "M1", "H2", "H1_adj", "A0_adj"):
        assert np.abs(getattr(eng, name) - z[name]).max() <= tol["inter"] * 10 * max(1.0, np.abs(z[name]).max()), name


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max,natoms,zbl,density", [(32, 0, 40, True, False), (96, 0, 48, True, True),
                                                        (48, 1, 30, True, True), (128, 1, 24, False, True),
                                                        (32, 2, 22, True, True)])
def test_pair_terms_match_oracle(gpu, tmp_models, K, L_max, natoms, zbl, density, dtype):
    """Models with ZBL repulsion and / or density-normalised layers (mace.cpp:27-35, 273-346, 681-757)."""
    model = H.tiny_model(K=K, L_max=L_max, n_pts=64, seed=K + L_max, pair=(K != 96), zbl=zbl, density=density)
    path = H.write_model(model, tmp_models / f"p_{K}_{L_max}_{int(zbl)}{int(density)}.json")
    orc = _oracle()(model)
    eng = gpu(path, dtype)
    pos, cell, sp = H.small_system(natoms, seed=natoms + 1)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"case K={K} L_max={L_max} atoms={natoms} zbl={zbl} density={density} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)
    f1, e1 = eng.node_forces, eng.node_energies
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(f1, eng.node_forces) and np.array_equal(e1, eng.node_energies)


def test_density_normalisation_stage_calls(gpu, tmp_models):
    """compute_A0_scaled / reverse_A0_scaled and their layer-1 twins called stage by stage, as test_mace.py does."""
    model = H.tiny_model(K=8, L_max=1, n_pts=40, seed=9, density=True)
    path = H.write_model(model, tmp_models / "stage_scaled.json")
    orc = _oracle()(model)
    eng = gpu(path)
    pos, cell, sp = H.small_system(10, seed=3)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, nt, nn, ni, nty, xyz, r = H.call_args(ea)
    rng = np.random.default_rng(1)
    for m in (orc, eng):
        m.compute_Y(xyz); m.compute_R0(N, nt, nn, nty, r); m.compute_A0(N, nt, nn, nty)
        m.compute_A0_scaled(N, nt, nn, nty, r)
    assert np.allclose(orc.A0, eng.A0, atol=1e-12)
    adj = rng.normal(size=len(orc.A0))
    for m in (orc, eng):
        m.A0_adj = adj
        m.node_forces = np.zeros(len(xyz))
        m.reverse_A0_scaled(N, nt, nn, nty, xyz, r)
    assert np.allclose(orc.A0_adj, eng.A0_adj, atol=1e-12)
    assert np.allclose(orc.node_forces, eng.node_forces, atol=1e-11)
    A1 = rng.normal(size=N * 16 * 8)
    for m in (orc, eng):
        m.A1 = A1
        m.compute_A1_scaled(N, nt, nn, nty, r)
        m.A1_adj = adj[:len(A1)]
        m.reverse_A1_scaled(N, nt, nn, nty, xyz, r, True)
    assert np.allclose(orc.A1, eng.A1, atol=1e-12) and np.allclose(orc.A1_adj, eng.A1_adj, atol=1e-12)
    assert np.allclose(orc.node_forces, eng.node_forces, atol=1e-11)


def test_stage_level_calls_follow_the_reference_test_method(gpu, tmp_models):
    """symmetrix/test/test_mace.py drives the evaluator stage by stage and overwrites
    intermediates between calls (e.g. :246-249).  Same here, against the oracle."""
    model = H.tiny_model(K=8, L_max=1, n_pts=40, seed=9)
    path = H.write_model(model, tmp_models / "stage.json")
    orc = _oracle()(model)
    eng = gpu(path)
    pos, cell, sp = H.small_system(10, seed=3)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, nt, nn, ni, nty, xyz, r = H.call_args(ea)
    rng = np.random.default_rng(0)
    for m in (orc, eng):
        m.compute_Y(xyz)
        m.compute_R0(N, nt, nn, nty, r)
        m.compute_A0(N, nt, nn, nty)
    assert np.allclose(orc.A0, eng.A0, atol=1e-12)
    assert np.allclose(orc.R0, eng.R0, atol=1e-12) and np.allclose(orc.Y, eng.Y, atol=1e-13)
    A0 = rng.normal(size=len(orc.A0))
    for m in (orc, eng):
        m.A0 = A0
        m.compute_M0(N, nt)
        m.M0_adj = np.ones(len(m.M0))
        m.reverse_M0(N, nt)
    assert np.allclose(orc.M0, eng.M0, atol=1e-11) and np.allclose(orc.A0_adj, eng.A0_adj, atol=1e-10)
    for m in (orc, eng):
        m.compute_H1(N)
        m.H1_adj = np.ones(len(m.H1))
        m.reverse_H1(N)
    assert np.allclose(orc.H1, eng.H1, atol=1e-11) and np.allclose(orc.M0_adj, eng.M0_adj, atol=1e-11)
    for m in (orc, eng):
        m.compute_R1(N, nt, nn, nty, r)
        m.compute_Phi1(N, nn, ni)
        m.Phi1_adj = np.ones(len(m.Phi1))
        m.reverse_Phi1(N, nn, ni, xyz, r, True, True)
    assert np.allclose(orc.Phi1, eng.Phi1, atol=1e-11)
    assert np.allclose(orc.node_forces, eng.node_forces, atol=1e-10)
    assert np.allclose(orc.H1_adj, eng.H1_adj, atol=1e-10)
    for m in (orc, eng):
        m.compute_A1(N)
        m.A1_adj = np.ones(len(m.A1))
        m.reverse_A1(N)
    assert np.allclose(orc.A1, eng.A1, atol=1e-12) and np.allclose(orc.Phi1_adj, eng.Phi1_adj, atol=1e-12)
    for m in (orc, eng):
        m.compute_M1(N, nt)
        m.M1_adj = np.ones(len(m.M1))
        m.reverse_M1(N, nt)
    assert np.allclose(orc.M1, eng.M1, atol=1e-12) and np.allclose(orc.A1_adj, eng.A1_adj, atol=1e-11)
    for m in (orc, eng):
        m.compute_H2(N, nt)
        m.H2_adj = np.ones(len(m.H2))
        m.reverse_H2(N, nt, True)
    assert np.allclose(orc.H2, eng.H2, atol=1e-12)
    assert np.allclose(orc.M1_adj, eng.M1_adj, atol=1e-12) and np.allclose(orc.H1_adj, eng.H1_adj, atol=1e-12)
    for m in (orc, eng):
        m.node_energies = np.zeros(N)
        m.compute_readouts(N, nt)
    assert np.allclose(orc.node_energies, eng.node_energies, atol=1e-12)
    assert np.allclose(orc.H2_adj, eng.H2_adj, atol=1e-12) and np.allclose(orc.H1_adj, eng.H1_adj, atol=1e-13)
    # reverse_A0 accumulates into node_forces (mace.cpp:237)
    for m in (orc, eng):
        m.A0_adj = np.ones(len(m.A0))
        m.node_forces = np.zeros(len(xyz))
        m.reverse_A0(N, nt, nn, nty, xyz, r)
    assert np.allclose(orc.node_forces, eng.node_forces, atol=1e-10)


def test_edge_cases(gpu, tmp_models):
    model = H.tiny_model(K=8, L_max=0, n_pts=32, seed=2)
    path = H.write_model(model, tmp_models / "edge.json")
    orc = _oracle()(model)
    eng = gpu(path)
    # no nodes at all
    eng.compute_node_energies_forces(0, [], [], [], [], [], [])
    assert len(eng.node_energies) == 0 and len(eng.node_forces) == 0
    # isolated atoms only: E_i = E0[type]
    eng.compute_node_energies_forces(3, [0, 2, 1], [0, 0, 0], [], [], [], [])
    assert np.allclose(eng.node_energies, np.array(model["atomic_energies"])[[0, 2, 1]], atol=1e-14)
    # ragged degrees, including zero-degree receivers in the middle
    rng = np.random.default_rng(4)
    nn = np.array([3, 0, 5, 1, 0, 2], dtype=np.int32)
    E = int(nn.sum())
    nt = rng.integers(0, 3, size=6).astype(np.int32)
    ni = rng.integers(0, 6, size=E).astype(np.int32)
    nty = nt[ni]
    xyz = rng.normal(size=(E, 3)); xyz *= (rng.uniform(0.8, 3.9, size=(E, 1)) / np.linalg.norm(xyz, axis=1, keepdims=True))
    r = np.linalg.norm(xyz, axis=1)
    args = (6, nt, nn, ni, nty, xyz.reshape(-1), r)
    orc.compute_node_energies_forces(*args); eng.compute_node_energies_forces(*args)
    _compare(orc, eng, "float64")
    # a receiver with more edges than one LDS chunk, several times over
    nn = np.array([70, 1], dtype=np.int32); E = 71
    ni = rng.integers(0, 2, size=E).astype(np.int32); nt = np.array([0, 1], dtype=np.int32); nty = nt[ni]
    xyz = rng.normal(size=(E, 3)); xyz *= (rng.uniform(0.8, 3.9, size=(E, 1)) / np.linalg.norm(xyz, axis=1, keepdims=True))
    args = (2, nt, nn, ni, nty, xyz.reshape(-1), np.linalg.norm(xyz, axis=1))
    orc.compute_node_energies_forces(*args); eng.compute_node_energies_forces(*args)
    _compare(orc, eng, "float64")


def test_invalid_inputs_raise(gpu, tmp_models):
    model = H.tiny_model(K=8, L_max=0, n_pts=32, seed=2)
    eng = gpu(H.write_model(model, tmp_models / "inv.json"))
    xyz = np.array([[1.0, 0, 0], [-1.0, 0, 0]]).reshape(-1)
    ok = (2, [0, 1], [1, 1], [1, 0], [1, 0], xyz, [1.0, 1.0])
    eng.compute_node_energies_forces(*ok)
    with pytest.raises(ValueError):      # beyond the spline table (cubic_spline_set.cpp:54 would read past it)
        eng.compute_node_energies_forces(2, [0, 1], [1, 1], [1, 0], [1, 0], xyz * 5, [5.0, 5.0])
    with pytest.raises(ValueError):      # species index outside the model
        eng.compute_node_energies_forces(2, [0, 7], [1, 1], [1, 0], [1, 0], xyz, [1.0, 1.0])
    with pytest.raises(ValueError):      # sender outside the node range
        eng.compute_node_energies_forces(2, [0, 1], [1, 1], [5, 0], [1, 0], xyz, [1.0, 1.0])
    with pytest.raises(ValueError):      # counts do not add up
        eng.compute_node_energies_forces(2, [0, 1], [2, 1], [1, 0], [1, 0], xyz, [1.0, 1.0])
    eng.compute_node_energies_forces(*ok)   # still usable afterwards


@pytest.mark.parametrize("workload", ["off_small", "mp_medium"])
def test_full_size_properties(gpu, tmp_models, workload):
    """At the benchmark's full size: properties that do not need the oracle."""
    from symmetrix_amd import modelgen, neighbors, systems
    cfg = dict(modelgen.CONFIGS[workload]); cfg["pair_dependent_radial"] = False
    path = str(tmp_models / f"{workload}.json")
    modelgen.write_model(path, **cfg)
    pos, cell, sp = systems.config_system(workload)
    nl = neighbors.neighbor_list(pos, cell, cfg["r_cut"]); ea = neighbors.edge_arrays(nl, sp)
    e64 = gpu(path, "float64")
    e64.compute_node_energies_forces(*H.call_args(ea))
    E64, f64 = e64.node_energies.sum(), e64.node_forces
    F = e64.reduce_forces(len(pos), nl["j"])
    assert np.abs(F.sum(0)).max() < 1e-9                       # Newton's third law
    assert np.allclose(F, H.atom_forces(nl, f64, len(pos)), atol=1e-10)
    # relabelling the atoms permutes the answers
    perm = np.random.default_rng(0).permutation(len(pos))
    nl2 = neighbors.neighbor_list(pos[perm], cell, cfg["r_cut"]); ea2 = neighbors.edge_arrays(nl2, sp[perm])
    e64.compute_node_energies_forces(*H.call_args(ea2))
    assert abs(e64.node_energies.sum() - E64) <= 1e-10 * abs(E64)
    assert np.allclose(e64.reduce_forces(len(pos), nl2["j"]), F[perm], atol=1e-9)
    # fp32-feature mode against fp64 mode
    e32 = gpu(path, "float32")
    e32.compute_node_energies_forces(*H.call_args(ea))
    assert abs(e32.node_energies.sum() - E64) <= 1e-5 * abs(E64)
    assert np.abs(e32.node_forces - f64).max() <= 1e-4


def test_calculator_energy_forces_stress(gpu, tmp_models):
    """The calculator face (symmetrix_calc.py:72-102): forces are -dE/dx and the
    stress is dE/d(strain)/V, both checked by central differences of the engine's own energy."""
    from symmetrix_amd.calc import SymmetrixCalculator
    model = H.tiny_model(K=16, L_max=1, n_pts=64, seed=21)
    path = H.write_model(model, tmp_models / "calc.json")
    calc = SymmetrixCalculator(path, species=["H", "C", "O"], num_spline_points=64)   # conversion keywords are accepted
    # a file that is no symmetrix JSON: RuntimeError, as the reference's loader raises before it converts
    # (symmetrix_calc.py:54-56); the message names the conversion to run
    bad = tmp_models / "checkpoint.model"
    bad.write_bytes(b"PK\x03\x04 not json")
    with pytest.raises(RuntimeError, match="symmetrix_extract_mace"):
        SymmetrixCalculator(str(bad))
    pos, cell, sp = H.small_system(14, density=0.09, seed=8)
    Z = np.array(model["atomic_numbers"])[sp]
    res = calc.compute(pos, cell, Z)
    orc = _oracle()(model)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    orc.compute_node_energies_forces(*H.call_args(ea))
    assert res["energy"] == pytest.approx(orc.node_energies.sum(), rel=1e-10)
    assert np.allclose(res["forces"], H.atom_forces(nl, orc.node_forces, len(pos)), atol=1e-8)
    # the list built on the device (default) and the numpy builder give the same bits
    res_h = SymmetrixCalculator(path, neighbor_list="host").compute(pos, cell, Z)
    assert res_h["energy"] == res["energy"] and np.array_equal(res_h["energies"], res["energies"])
    assert np.array_equal(res_h["forces"], res["forces"]) and np.array_equal(res_h["stress"], res["stress"])
    F, e0 = res["forces"].copy(), res["energy"]
    h = 1e-5
    for a, c in ((0, 0), (3, 1), (7, 2)):
        p = pos.copy(); p[a, c] += h; ep = calc.compute(p, cell, Z)["energy"]
        p[a, c] -= 2 * h; em = calc.compute(p, cell, Z)["energy"]
        assert -(ep - em) / (2 * h) == pytest.approx(F[a, c], abs=1e-6)
    stress = calc.compute(pos, cell, Z)["stress"]
    V = float(np.prod(cell))
    voigt = [(0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1)]
    for q, (a, b) in enumerate(voigt):
        def strained(eps):
            S = np.eye(3); S[a, b] += eps / 2; S[b, a] += eps / 2
            return calc.compute(pos @ S.T, np.diag(cell) @ S.T, Z)["energy"]
        d = (strained(h) - strained(-h)) / (2 * h) / V
        assert d == pytest.approx(stress[q], abs=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["ortho", "triclinic", "small_cell", "open", "empty"])
def test_device_neighbor_list_is_bit_identical_to_the_host_builder(case):
    """Edge order, integer arrays, xyz and r of the device builder against symmetrix_amd.neighbors.neighbor_list."""
    import torch
    from symmetrix_amd import neighbors
    rng = np.random.default_rng(11)
    pbc = (True, True, True)
    if case == "ortho":
        cell = np.array([13.0, 11.0, 12.5]); pos = rng.uniform(0, 1, size=(300, 3)) * cell; rc = 4.5
    elif case == "triclinic":
        cell = np.array([[9.0, 0.0, 0.0], [2.5, 8.0, 0.0], [-1.5, 2.0, 10.0]])
        pos = rng.uniform(0, 1, size=(150, 3)) @ cell; rc = 5.0
    elif case == "small_cell":
        cell = np.array([3.1, 3.3, 2.9]); pos = rng.uniform(0, 1, size=(5, 3)) * cell; rc = 5.0   # several images per pair
    elif case == "open":
        cell = np.array([30.0, 30.0, 30.0]); pos = rng.uniform(5, 12, size=(60, 3)); rc = 4.0; pbc = (False, True, False)
    else:
        cell = np.array([10.0, 10.0, 10.0]); pos = np.zeros((0, 3)); rc = 4.0
    types = rng.integers(0, 3, size=len(pos)).astype(np.int32)
    ref = neighbors.neighbor_list(pos, cell, rc, pbc)
    dpos = torch.from_numpy(np.ascontiguousarray(pos)).cuda()
    dty = torch.from_numpy(types).cuda()
    dnl = neighbors.DeviceNeighborList()
    print(f"case {case} atoms={len(pos)} edges={len(ref['r'])}", flush=True)
    E = dnl.build(len(pos), dpos.data_ptr(), dty.data_ptr(), cell, rc, pbc)
    got = dnl.to_host()
    assert E == len(ref["r"])
    assert np.array_equal(got["i"], ref["i"]) and np.array_equal(got["j"], ref["j"])
    assert np.array_equal(got["S"], ref["S"].reshape(-1, 3))
    assert np.array_equal(got["xyz"], ref["xyz"].reshape(-1, 3)) and np.array_equal(got["r"], ref["r"])
    assert np.array_equal(got["first_neigh"], ref["first_neigh"])
    assert np.array_equal(got["neigh_types"], types[ref["j"]])


@pytest.mark.gpu
def test_device_neighbor_list_update_equals_fresh_build():
    """Skin list + per-step cutoff filter at moved positions against a fresh host build at the moved positions."""
    import torch
    from symmetrix_amd import neighbors
    rng = np.random.default_rng(3)
    cell = np.array([[12.0, 0.0, 0.0], [1.0, 11.0, 0.0], [0.5, -1.0, 12.5]])
    pos = rng.uniform(0, 1, size=(400, 3)) @ cell
    types = rng.integers(0, 4, size=len(pos)).astype(np.int32)
    rc, skin = 4.5, 1.0
    dnl = neighbors.DeviceNeighborList()
    dty = torch.from_numpy(types).cuda()
    dpos = torch.from_numpy(pos).cuda()
    dnl.build(len(pos), dpos.data_ptr(), dty.data_ptr(), cell, rc, skin=skin)
    for step in range(3):
        pos = pos + rng.uniform(-0.15, 0.15, size=pos.shape)      # total drift stays below skin / 2
        dpos = torch.from_numpy(pos).cuda()
        print(f"update step {step}", flush=True)
        E = dnl.update(dpos.data_ptr(), dty.data_ptr(), rc)
        # the list keeps the frame of its build: atoms that drifted out of the cell are not folded back in
        got, ref = dnl.to_host(), neighbors.neighbor_list(pos, cell, rc, offsets=np.zeros((len(pos), 3), dtype=int))
        assert E == len(ref["r"])
        for k in ("i", "j", "S", "xyz", "r", "first_neigh"):
            assert np.array_equal(got[k], ref[k].reshape(got[k].shape)), k
    with pytest.raises(ValueError):
        dnl.update(dpos.data_ptr(), dty.data_ptr(), rc + 2 * skin)
    # the same through host arrays
    hnl = neighbors.DeviceNeighborList()
    hnl.build_host(pos, types, cell, rc, skin=skin)
    pos2 = pos + rng.uniform(-0.1, 0.1, size=pos.shape)
    E = hnl.update_host(pos2, rc)
    got, ref = hnl.to_host(), neighbors.neighbor_list(pos2, cell, rc, offsets=hnl.offsets)
    assert hnl.offsets.any()                   # some atoms had left the cell before this build
    assert E == len(ref["r"]) and np.array_equal(got["j"], ref["j"]) and np.array_equal(got["r"], ref["r"])
    assert np.array_equal(got["S"], ref["S"]) and np.array_equal(got["xyz"], ref["xyz"])
    far = pos2 + rng.integers(-2, 3, size=pos2.shape) @ cell      # whole lattice vectors away: same edges
    E2 = hnl.build_host(far, types, cell, rc)
    got2, ref2 = hnl.to_host(), neighbors.neighbor_list(far, cell, rc)
    assert E2 == len(ref2["r"]) == len(neighbors.neighbor_list(pos2, cell, rc)["r"])
    for k in ("i", "j", "S", "xyz", "r"):
        assert np.array_equal(got2[k], ref2[k].reshape(got2[k].shape)), k
    assert np.array_equal(got["neigh_types"], types[ref["j"]])


@pytest.mark.gpu
@pytest.mark.parametrize("atoms,volume", [(1, 1.0), (3, 10.0), (4, 10.0), (5, 10.0), (40, 10.0), (512, 12.0), (513, 12.0),
                                          (4097, 12.0), (8192, 14.0), (8193, 14.0)])
def test_list_sizes_at_which_the_search_changes(atoms, volume):
    """Bins or all atoms, offsets found inside the launch or by a prefix sum, more edges than there is room for at first and
    more keys per receiver than fit the LDS (40 atoms in a wide cutoff): host builder's list, with and without a skin."""
    from symmetrix_amd import neighbors
    rng = np.random.default_rng(atoms)
    cell = np.full(3, (atoms * volume) ** (1.0 / 3.0))
    pos = rng.uniform(0, 1, size=(atoms, 3)) * cell
    types = rng.integers(0, 3, size=atoms).astype(np.int32)
    rc = 9.9 if atoms == 40 else 3.3
    nl = neighbors.DeviceNeighborList()
    for wait, skin in ((True, 0.0), (True, 0.7), (False, 0.0), (False, 0.7)):
        nl.set_wait(wait)
        print(f"atoms {atoms} wait {wait} skin {skin}", flush=True)
        E = nl.build_host(pos, types, cell, rc, skin=skin)
        ref = neighbors.neighbor_list(pos, cell, rc)
        got = nl.to_host()
        assert E == len(ref["r"])
        for k in ("i", "j", "S", "xyz", "r", "first_neigh"):
            assert np.array_equal(got[k], ref[k].reshape(got[k].shape)), k
        if skin:
            moved = pos + rng.uniform(-0.15, 0.15, size=pos.shape)
            E = nl.update_host(moved, rc)
            got, ref = nl.to_host(), neighbors.neighbor_list(moved, cell, rc, offsets=np.zeros((atoms, 3), dtype=int))
            assert E == len(ref["r"])
            for k in ("i", "j", "S", "xyz", "r", "first_neigh"):
                assert np.array_equal(got[k], ref[k].reshape(got[k].shape)), k


@pytest.mark.gpu
def test_device_resident_loop_positions_to_forces(gpu, tmp_models):
    """positions on the device -> device neighbour list -> compute_device -> per-atom forces, against the host path."""
    import torch
    from symmetrix_amd import neighbors
    model = H.tiny_model(K=16, L_max=1, n_pts=48, seed=5)
    path = H.write_model(model, tmp_models / "loop.json")
    eng = gpu(path)
    pos, cell, sp = H.small_system(40, seed=8)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    eng.compute_node_energies_forces(*H.call_args(ea))
    e_ref, f_ref = eng.node_energies.copy(), eng.node_forces.copy()
    dpos = torch.from_numpy(np.ascontiguousarray(pos)).cuda()
    dty = torch.from_numpy(np.asarray(sp, dtype=np.int32)).cuda()
    dnl = neighbors.DeviceNeighborList()
    E = dnl.build(len(pos), dpos.data_ptr(), dty.data_ptr(), cell, model["r_cut"])
    oE = torch.zeros(len(pos), dtype=torch.float64, device="cuda"); oF = torch.zeros(3 * E, dtype=torch.float64, device="cuda")
    p = dnl.ptr
    eng.compute_device(len(pos), dty.data_ptr(), p["num_neigh"], p["neigh_indices"], p["neigh_types"], p["xyz"], p["r"], E,
                       oE.data_ptr(), oF.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert np.array_equal(oE.cpu().numpy(), e_ref) and np.array_equal(oF.cpu().numpy(), f_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_receiver_chunks_of_the_layer1_adjoint_change_nothing(gpu, tmp_models, dtype):
    """A staging limit far below the message volume (many chunks, down to a few receivers each) gives the same bits."""
    model = H.tiny_model(K=16, L_max=1, n_pts=48, seed=9)
    path = H.write_model(model, tmp_models / "chunks.json")
    pos, cell, sp = H.small_system(60, seed=4)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    eng = gpu(path, dtype)
    eng.compute_node_energies_forces(*H.call_args(ea))
    e_ref, f_ref, h_ref = eng.node_energies.copy(), eng.node_forces.copy(), np.array(eng.H1_adj)
    row_bytes = 4 * 16 * (8 if dtype == "float64" else 4)
    for limit in (len(ea["r"]) * row_bytes // 3, 200 * row_bytes, int(ea["num_neigh"].max()) * row_bytes):
        eng.set_staging_limit(limit)
        print(f"staging limit {limit} bytes", flush=True)
        eng.compute_node_energies_forces(*H.call_args(ea))
        assert np.array_equal(eng.node_energies, e_ref)
        assert np.array_equal(eng.node_forces, f_ref)
        assert np.array_equal(np.array(eng.H1_adj), h_ref)
    eng.set_staging_limit(row_bytes)          # below one receiver's messages
    with pytest.raises(RuntimeError):
        eng.compute_node_energies_forces(*H.call_args(ea))


# (L_max, dtype, one radial table for all pairs, ZBL, density normalisation).  With ghost nodes, ZBL or the density
# normalisation the force array has other contributions before, between and beside those of the two adjoints.
MODE_CASES = [(0, "float64", False, False, False), (1, "float64", False, True, True), (0, "float32", False, True, False),
              (1, "float32", False, True, True), (2, "float64", False, True, True)]
MODE_CASES += [(0, dt, True, zbl, dens) for dt in ("float64", "float32")
               for zbl, dens in ((False, False), (True, False), (False, True), (True, True))]


@pytest.mark.gpu
@pytest.mark.parametrize("L_max,dtype,one_table,zbl,density", MODE_CASES)
def test_pair_style_modes_agree(gpu, tmp_models, L_max, dtype, one_table, zbl, density):
    """The three ways the pair style feeds the engine on one rank give one answer (the reference's
    tests/test_pair_symmetrix_mace.py:28-39): owners as senders (no_domain_decomposition), ghost nodes that go
    through layer 0 (no_mpi_message_passing, one call), and ghost rows of H1 filled by a forward copy with the
    adjoint summed back (mpi_message_passing, stage calls as pair_symmetrix_mace.cpp:372-550 issues them).  The
    first is compared with the oracle, the others with the first."""
    from symmetrix_amd import neighbors
    model = H.tiny_model(K=16, L_max=L_max, n_pts=48, seed=12, pair=not one_table, zbl=zbl, density=density)
    path = H.write_model(model, tmp_models / f"modes{L_max}{dtype}{int(one_table)}{int(zbl)}{int(density)}.json")
    pos, cell, sp = H.small_system(36, seed=21)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N = len(sp)
    eng = gpu(path, dtype)
    assert eng._int("num_radial_tables_0") == (1 if one_table else 6)
    eng.compute_node_energies_forces(*H.call_args(ea))
    orc = _oracle()(model)
    orc.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype, names=[])
    e_ref = eng.node_energies.copy()
    f_ref = eng.reduce_forces(N, ea["neigh_indices"])
    ga = neighbors.ghost_edge_arrays(nl, sp)
    Nl, Ng = ga["num_local_nodes"], ga["num_ghost_nodes"]
    assert Ng > 0
    print(f"ghost mode: {Nl} local + {Ng} ghost nodes, {len(ga['r'])} edges", flush=True)
    eng.compute_ghosted(Nl, Ng, ga["node_types"], ga["num_neigh"], ga["neigh_indices"], ga["neigh_types"], ga["xyz"], ga["r"])
    e_g = eng.node_energies.copy()
    f_g = eng.reduce_forces(N, ga["sender_atom"], ga["receiver_atom"])
    assert e_g.shape == (Nl,)
    ftol = 1e-11 if dtype == "float64" else 2e-5
    assert np.array_equal(e_g, e_ref)      # same edges in the same order for every local receiver
    assert np.abs(f_g - f_ref).max() <= ftol * max(1.0, np.abs(f_ref).max())
    assert np.abs(f_g - H.atom_forces(nl, orc.node_forces, N)).max() <= TOL[dtype]["F"]
    # the same call again, and after an evaluation of the owner layout in between: bit for bit
    eng.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_ghosted(Nl, Ng, ga["node_types"], ga["num_neigh"], ga["neigh_indices"], ga["neigh_types"], ga["xyz"], ga["r"])
    assert np.array_equal(eng.node_energies, e_g)
    assert np.array_equal(eng.reduce_forces(N, ga["sender_atom"], ga["receiver_atom"]), f_g)

    # message-passing mode: local nodes only; H1 of the ghosts copied from their owners, H1_adj summed back
    El = int(ga["num_neigh"][:Nl].sum())
    nt, nn = ga["node_types"][:Nl], ga["num_neigh"][:Nl]
    ni, nty, x, r = ga["neigh_indices"][:El], ga["neigh_types"][:El], ga["xyz"][:3 * El], ga["r"][:El]
    eng2 = gpu(path, dtype)
    eng2.fill("node_energies", Nl); eng2.fill("node_forces", 3 * El)
    if eng2.has_zbl:
        eng2.zbl.compute_ZBL(Nl, nt, nn, nty, eng2.atomic_numbers, r, x)         # pair_symmetrix_mace.cpp:449-452
    eng2.compute_Y(x)
    eng2.compute_R0(Nl, nt, nn, nty, r); eng2.compute_A0(Nl, nt, nn, nty); eng2.compute_A0_scaled(Nl, nt, nn, nty, r)
    eng2.compute_M0(Nl, nt); eng2.compute_H1(Nl)
    nlm_k = eng2.H1.size // Nl
    H1 = np.array(eng2.H1).reshape(Nl, nlm_k)
    eng2.H1 = np.concatenate([H1, H1[ga["ghost_owner"]]]).reshape(-1)          # forward_comm
    eng2.compute_R1(Nl, nt, nn, nty, r); eng2.compute_Phi1(Nl, nn, ni); eng2.compute_A1(Nl)
    eng2.compute_A1_scaled(Nl, nt, nn, nty, r); eng2.compute_M1(Nl, nt); eng2.compute_H2(Nl, nt)
    eng2.compute_readouts(Nl, nt)
    eng2.reverse_H2(Nl, nt, False); eng2.reverse_M1(Nl, nt)
    eng2.reverse_A1_scaled(Nl, nt, nn, nty, x, r, False); eng2.reverse_A1(Nl)
    eng2.reverse_Phi1(Nl, nn, ni, x, r, False, False)
    Hadj = np.array(eng2.H1_adj).reshape(Nl + Ng, nlm_k)
    np.add.at(Hadj, ga["ghost_owner"], Hadj[Nl:])                                # reverse_comm
    eng2.H1_adj = Hadj[:Nl].reshape(-1).copy()
    eng2.reverse_H1(Nl); eng2.reverse_M0(Nl, nt); eng2.reverse_A0_scaled(Nl, nt, nn, nty, x, r)
    eng2.reverse_A0(Nl, nt, nn, nty, x, r)
    etol = 1e-12 if dtype == "float64" else 1e-6
    assert np.abs(eng2.node_energies - e_ref).max() <= etol * max(1.0, np.abs(e_ref).max())
    f_m = eng2.reduce_forces(N, ga["sender_atom"][:El])
    assert np.abs(f_m - f_ref).max() <= ftol * 10 * max(1.0, np.abs(f_ref).max())


@pytest.mark.gpu
def test_rotation_and_replication_through_the_calculator(tmp_models):
    """A rigid rotation of positions and cell leaves the energy alone and rotates the forces; a cell repeated along
    an axis repeats energies and forces.  Both go through the device neighbour list with general triclinic cells."""
    from symmetrix_amd.calc import SymmetrixCalculator
    model = H.tiny_model(K=16, L_max=1, n_pts=64, seed=31, zbl=True, density=True)
    path = H.write_model(model, tmp_models / "rot.json")
    calc = SymmetrixCalculator(path)
    pos, cell, sp = H.small_system(24, density=0.08, seed=13)
    Z = np.array(model["atomic_numbers"])[sp]
    cell = np.diag(cell)
    res = calc.compute(pos, cell, Z)
    e0, f0, en0 = res["energy"], res["forces"].copy(), res["energies"].copy()
    rng = np.random.default_rng(5)
    Q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    if np.linalg.det(Q) < 0:
        Q[:, 0] = -Q[:, 0]
    rot = calc.compute(pos @ Q.T, cell @ Q.T, Z)
    assert abs(rot["energy"] - e0) <= 1e-10 * abs(e0)
    assert np.abs(rot["forces"] - f0 @ Q.T).max() <= 1e-8 * max(1.0, np.abs(f0).max())
    pos2 = np.concatenate([pos, pos + cell[0]])
    cell2 = cell.copy(); cell2[0] *= 2
    rep = calc.compute(pos2, cell2, np.concatenate([Z, Z]))
    assert np.abs(rep["energies"][:len(pos)] - en0).max() <= 1e-10 * max(1.0, np.abs(en0).max())
    assert np.abs(rep["energies"][len(pos):] - en0).max() <= 1e-10 * max(1.0, np.abs(en0).max())
    assert np.abs(rep["forces"][:len(pos)] - f0).max() <= 1e-8 * max(1.0, np.abs(f0).max())
    assert np.abs(rep["stress"] - res["stress"]).max() <= 1e-9 * max(1.0, np.abs(res["stress"]).max())


@pytest.mark.gpu
@pytest.mark.parametrize("L_max", [0, 1])
def test_a_step_captured_in_a_hip_graph_replays_bitwise(gpu, tmp_models, L_max):
    """Callers that cannot launch from the host each step capture the device-resident call once (after a call at the
    same sizes, which allocates) and replay it.  Replays are interleaved with eager calls on other inputs and each
    one is compared with the eager result."""
    import torch
    model = H.tiny_model(K=32, L_max=L_max, n_pts=48, seed=17, zbl=True, density=(L_max == 1))
    path = H.write_model(model, tmp_models / f"graph{L_max}.json")
    eng = gpu(path, "float64")
    pos, cell, sp = H.small_system(50, seed=2)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, E = len(sp), len(ea["r"])
    dev = torch.device("cuda:0")
    t = lambda a, dt: torch.from_numpy(np.ascontiguousarray(a)).to(dev, dtype=dt)
    d = [t(ea["node_types"], torch.int32), t(ea["num_neigh"], torch.int32), t(ea["neigh_indices"], torch.int32),
         t(ea["neigh_types"], torch.int32), t(ea["xyz"], torch.float64), t(ea["r"], torch.float64)]
    xyz0, r0 = d[4].clone(), d[5].clone()
    oE = torch.zeros(N, dtype=torch.float64, device=dev); oF = torch.zeros(3 * E, dtype=torch.float64, device=dev)
    s = torch.cuda.Stream()

    def step():
        eng.compute_device(N, *[x.data_ptr() for x in d], E, oE.data_ptr(), oF.data_ptr(), s.cuda_stream)

    with torch.cuda.stream(s):
        step()
    torch.cuda.synchronize()
    refE, refF = oE.clone(), oF.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step()
    torch.cuda.synchronize()
    rng = np.random.default_rng(0)
    for rep in range(3):
        # eager work on other inputs in between: the same geometry scaled, which changes every intermediate
        scale = 1.0 - 0.01 * (rep + 1)
        d[4].copy_(xyz0 * scale); d[5].copy_(r0 * scale)
        with torch.cuda.stream(s):
            step()
        torch.cuda.synchronize()
        assert not torch.equal(oF, refF)
        d[4].copy_(xyz0); d[5].copy_(r0)
        oE.zero_(); oF.zero_()
        torch.cuda.synchronize()
        print(f"replay {rep}", flush=True)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(oE, refE) and torch.equal(oF, refF)


@pytest.mark.gpu
@pytest.mark.parametrize("L_max,big,one_table", [(0, False, False), (1, False, False), (0, True, False), (0, False, True)])
def test_device_resident_call_checks_its_inputs_on_the_device(gpu, tmp_models, L_max, big, one_table):
    """Arrays handed over as device addresses are checked inside the list preparation; when a check fails, the
    evaluation runs on emptied lists (no unchecked integer is used as an address), node energies and edge forces come
    back as NaN and the next synchronising call (synchronize, get_array, reduce_forces) raises.  Every kernel exits
    normally; the call after is unaffected, also when both are replays of one captured graph.
    `big`: more than 65 536 atoms, where the preparation is made of separate launches; `one_table`: one radial table for
    all species pairs."""
    import torch
    from symmetrix_amd import neighbors, systems
    model = H.tiny_model(K=16 if big else 32, L_max=L_max, n_pts=48, seed=40 + L_max, r_cut=3.0 if big else 4.0,
                         pair=not one_table)
    path = H.write_model(model, tmp_models / f"guard{L_max}{int(big)}{int(one_table)}.json")
    if big:
        pos, cell, sp = systems.fcc_alloy((26, 26, 25), n_species=3, seed=1)     # 67 600 atoms
    else:
        pos, cell, sp = H.small_system(40, seed=5)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, E = len(sp), len(ea["r"])
    dev = torch.device("cuda:0")
    t = lambda a, dt: torch.from_numpy(np.ascontiguousarray(a)).to(dev, dtype=dt)
    names = ["node_types", "num_neigh", "neigh_indices", "neigh_types", "xyz", "r"]
    good = {k: t(ea[k], torch.float64 if k in ("xyz", "r") else torch.int32) for k in names}
    oE = torch.zeros(N, dtype=torch.float64, device=dev); oF = torch.zeros(3 * E, dtype=torch.float64, device=dev)
    eng = gpu(path, "float64")
    stream = torch.cuda.current_stream().cuda_stream

    def run(d):
        eng.compute_device(N, *[d[k].data_ptr() for k in names], E, oE.data_ptr(), oF.data_ptr(), stream)
        torch.cuda.synchronize()

    run(good)
    eng.synchronize()
    e_ref, f_ref = oE.clone(), oF.clone()
    F_ref = eng.reduce_forces(N, ea["neigh_indices"])
    assert torch.isfinite(e_ref).all() and torch.isfinite(f_ref).all()
    bad_cases = {"sender row": ("neigh_indices", 5, N + 3), "edge species": ("neigh_types", 0, 3),
                 "node species": ("node_types", 1, -1), "counts": ("num_neigh", 0, int(ea["num_neigh"][0]) + 1),
                 "edge length": ("r", 3, 2.0 * model["r_cut"])}
    for n_case, (what, (key, pos_, value)) in enumerate(bad_cases.items()):
        d = dict(good); d[key] = good[key].clone(); d[key][pos_] = value
        print(f"bad {what} (L_max {L_max}, {N} atoms)", flush=True)
        oF.zero_()
        run(d)
        assert torch.isnan(oE).all(), what
        assert torch.isnan(oF).all(), what
        with pytest.raises(ValueError):
            if n_case % 2 == 0:
                eng.synchronize()
            else:
                eng.reduce_forces(N, ea["neigh_indices"])     # the per-atom sums of NaN forces are not handed out silently
        eng.synchronize()                       # reported once
        run(good)
        eng.synchronize()
        assert torch.equal(oE, e_ref) and torch.equal(oF, f_ref), what
        assert np.array_equal(eng.reduce_forces(N, ea["neigh_indices"]), F_ref)
    if big:
        return
    # one captured graph, replayed on bad and then on good inputs: a skipped replay leaves nothing behind
    live = {k: good[k].clone() for k in names}
    s = torch.cuda.Stream()

    def step():
        eng.compute_device(N, *[live[k].data_ptr() for k in names], E, oE.data_ptr(), oF.data_ptr(), s.cuda_stream)

    with torch.cuda.stream(s):
        step()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step()
    torch.cuda.synchronize()
    for rep in range(2):
        live["neigh_indices"][5] = N + 3
        torch.cuda.synchronize()
        print(f"graph replay {rep}: bad, then good", flush=True)
        g.replay()
        torch.cuda.synchronize()
        assert torch.isnan(oE).all() and torch.isnan(oF).all()
        live["neigh_indices"].copy_(good["neigh_indices"])
        oE.zero_(); oF.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(oE, e_ref) and torch.equal(oF, f_ref)
        with pytest.raises(ValueError):
            eng.synchronize()                   # the skipped replay is still reported, once
        eng.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_layer0_gradients_on_request_follow_the_calls(gpu, tmp_models, dtype):
    """With several polynomials per channel the whole-pipeline call keeps no M0_grad (its adjoint recomputes it); the
    array is formed when it is asked for, from the evaluation that ran last, and stage-level calls made afterwards
    (which do store gradients, as the reference's methods do) see consistent arrays.  Sequence: evaluation A, ask;
    evaluation B on fewer atoms, reverse_M0 as a stage call (needs the gradients of B), ask; evaluation A again:
    bit-identical to the first."""
    model = H.tiny_model(K=24, L_max=1, n_pts=64, seed=31, pair=False)
    path = H.write_model(model, tmp_models / "lazy_grad.json")
    eng = gpu(path, dtype)
    assert eng._int("contraction_tables") == 3
    tol = 1e-10 if dtype == "float64" else 2e-4
    runs = {}
    for tag, n in (("A", 60), ("B", 23)):
        pos, cell, sp = H.small_system(n, seed=n)
        nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
        orc = _oracle()(model)
        orc.compute_node_energies_forces(*H.call_args(ea))
        runs[tag] = (ea, orc)
    ea, orc = runs["A"]
    eng.compute_node_energies_forces(*H.call_args(ea))
    fA, eA = eng.node_forces.copy(), eng.node_energies.copy()
    assert np.abs(eng.M0_grad - orc.M0_grad).max() <= tol * max(1.0, np.abs(orc.M0_grad).max())
    ea, orc = runs["B"]
    eng.compute_node_energies_forces(*H.call_args(ea))
    a0_adj = eng.A0_adj.copy()
    assert np.abs(a0_adj - orc.A0_adj).max() <= tol * max(1.0, np.abs(orc.A0_adj).max())
    eng.reverse_M0(ea["num_nodes"], ea["node_types"])          # stage call: streams over stored gradients
    assert np.abs(eng.A0_adj - a0_adj).max() <= tol * max(1.0, np.abs(a0_adj).max())
    assert eng.M0_grad.shape == orc.M0_grad.shape
    assert np.abs(eng.M0_grad - orc.M0_grad).max() <= tol * max(1.0, np.abs(orc.M0_grad).max())
    ea, orc = runs["A"]
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(eng.node_forces, fA) and np.array_equal(eng.node_energies, eA)
    assert np.abs(eng.M0_grad - orc.M0_grad).max() <= tol * max(1.0, np.abs(orc.M0_grad).max())


@pytest.mark.gpu
@pytest.mark.parametrize("atoms", [1, 4, 5, 107, 513, 1100])
def test_list_blocks_that_stop_waiting_count_for_themselves(atoms):
    """A block of a list kernel looks for the counts of the blocks before it a bounded number of times, then counts their
    entries itself.  With no look at all every block goes that way: the same list, with and without bins, with and without a
    skin, in an update, and where the first room is outgrown (513 atoms)."""
    import torch
    from symmetrix_amd import _lib, neighbors
    assert torch.cuda.is_available()
    rng = np.random.default_rng(atoms)
    rc = 5.5 if atoms == 513 else 3.3
    cell = np.full(3, (atoms * 8.0) ** (1.0 / 3.0))
    pos = rng.uniform(0, 1, size=(atoms, 3)) * cell
    if atoms == 513:
        pos[:300] *= 0.5        # more pairs than a homogeneous system has
    types = rng.integers(0, 3, size=atoms).astype(np.int32)
    nl = neighbors.DeviceNeighborList()
    for rounds, wait, skin in ((0, True, 0.0), (0, True, 0.4), (0, False, 0.0), (1, True, 0.4), (4096, True, 0.4)):
        _lib.check(_lib.lib().smx_nlist_set_chain_rounds(nl._C.c_void_p(nl._h), rounds))
        nl.set_wait(wait)
        print(f"{atoms} atoms, {rounds} rounds, wait {wait}, skin {skin}", flush=True)
        E = nl.build_host(pos, types, cell, rc, skin=skin)
        got, ref = nl.to_host(), neighbors.neighbor_list(pos, cell, rc)
        assert E == len(ref["r"])
        for k in ("i", "j", "S", "xyz", "r", "first_neigh"):
            assert np.array_equal(got[k], ref[k].reshape(got[k].shape)), k
        if skin:
            moved = pos + rng.uniform(-0.1, 0.1, size=pos.shape)
            E = nl.update_host(moved, rc)
            got, ref = nl.to_host(), neighbors.neighbor_list(moved, cell, rc, offsets=np.zeros((atoms, 3), dtype=int))
            assert E == len(ref["r"])
            for k in ("i", "j", "S", "xyz", "r", "first_neigh"):
                assert np.array_equal(got[k], ref[k].reshape(got[k].shape)), k


@pytest.mark.gpu
@pytest.mark.parametrize("natoms,density,rc,skin", [(1, 0.2, 6.0, 0.0), (512, 0.1, 4.5, 0.0), (513, 0.1, 4.5, 0.0), (700, 0.9, 4.5, 0.0),
                                                    (200, 0.9, 4.5, 0.3), (600, 0.1, 3.0, 1.5)])
def test_list_search_at_the_edges_of_its_ways(natoms, density, rc, skin):
    """All atoms tried (up to 512) or bins, candidates of a receiver ordered in LDS (up to 256) or in memory, lists that
    outgrow the room first taken, with and without a skin: bit for bit the host builder's, twice on the same object."""
    from symmetrix_amd import neighbors
    rng = np.random.default_rng(natoms)
    cell = np.full(3, (natoms / density) ** (1 / 3)) * np.array([1.0, 1.1, 1 / 1.1])
    types = rng.integers(0, 3, size=natoms).astype(np.int32)
    dnl = neighbors.DeviceNeighborList()
    for rep in range(2):
        pos = rng.uniform(-0.2, 1.2, size=(natoms, 3)) * cell
        ref = neighbors.neighbor_list(pos, cell, rc)
        print(f"{natoms} atoms, {len(ref['r'])} edges", flush=True)
        E = dnl.build_host(pos, types, cell, rc, skin=skin)
        got = dnl.to_host()
        assert E == len(ref["r"])
        for k in ("i", "j", "S", "xyz", "r", "first_neigh"):
            assert np.array_equal(got[k], ref[k].reshape(got[k].shape)), k
        assert np.array_equal(got["neigh_types"], types[ref["j"]])


@pytest.mark.gpu
@pytest.mark.parametrize("L_max,K,edge", [(0, 32, 2.6), (0, 32, 1.9), (0, 32, 1.35), (1, 8, 1.9), (1, 8, 1.35)])
def test_senders_with_many_edges(gpu, tmp_models, L_max, K, edge):
    """One atom in a small cell is the sender of all edges: buckets that are ordered in LDS, and longer ones."""
    model = H.tiny_model(K=K, L_max=L_max, n_pts=64, seed=50, r_cut=9.0, pair=False)
    path = H.write_model(model, tmp_models / f"many{L_max}{K}.json")
    nl, ea = H.edges_of(np.array([[0.1, 0.2, 0.3]]), np.full(3, edge), np.array([1], dtype=np.int32), 9.0)
    print(f"{len(ea['r'])} edges", flush=True)
    orc = _oracle()(model)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng = gpu(path, "float64")
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.abs(eng.node_energies - orc.node_energies).max() <= 1e-10 * np.abs(orc.node_energies).max()
    scale = max(1.0, np.abs(orc.node_forces).max())
    assert np.abs(eng.node_forces - orc.node_forces).max() <= 1e-9 * scale
    F, V = eng.reduce_forces(1, nl["j"], receiver_atom=np.zeros(1, dtype=np.int32), virial=True)
    assert np.abs(F).max() <= 1e-9 * scale * len(ea["r"])
    f, d = orc.node_forces.reshape(-1, 3), ea["xyz"].reshape(-1, 3)
    W = 0.5 * (d.T @ f + f.T @ d)
    assert np.abs(V - W[[0, 1, 2, 0, 0, 1], [0, 1, 2, 1, 2, 2]]).max() <= 1e-9 * max(1.0, np.abs(W).max())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,receivers,max_degree", [(20, 40, 50), (64, 12, 40), (65, 24, 35), (130, 24, 35), (16, 515, 9), (16, 3100, 4)])
def test_scalar_features_with_a_coupling_that_mixes_harmonics(gpu, tmp_models, K, receivers, max_degree, dtype):
    """Scalar hidden features whose layer-1 coupling is not diagonal (an output lm is fed by a second harmonic of its l): the
    general edge kernels for scalar features, with one and two channels per lane and several channel groups, one, two and four
    wavefronts per receiver.  The same messages where the adjoint takes the receivers in chunks."""
    model = H.tiny_model(K=K, L_max=0, n_pts=24, seed=K, pair=K != 64)
    q = dict(zip(model["Phi1_lme"], model["Phi1_lelm1lm2"]))
    assert len(q) == len(model["Phi1_lme"]) == 16            # diagonal so far
    for lm, other, c in ((1, 3, 0.4), (4, 8, -0.7), (8, 5, 0.2), (9, 15, 0.9), (12, 11, -0.3)):
        model["Phi1_lme"].append(lm); model["Phi1_lelm1lm2"].append(q[other]); model["Phi1_clebsch_gordan"].append(c)
    rng = np.random.default_rng(receivers)
    degree = np.linspace(0, max_degree, receivers).astype(int) if max_degree > receivers else np.arange(receivers) % (max_degree + 1)
    E = int(degree.sum())
    species = rng.integers(0, 3, size=receivers).astype(np.int32)
    senders = rng.integers(0, receivers, size=E).astype(np.int32)
    x = rng.normal(size=(E, 3))
    x *= (rng.uniform(0.8, 3.9, size=E) / np.linalg.norm(x, axis=1))[:, None]
    args = (receivers, species, degree.astype(np.int32), senders, species[senders], x.ravel(), np.linalg.norm(x, axis=1))
    orc = _oracle()(model)
    eng = gpu(H.write_model(model, tmp_models / f"mixed_{K}.json"), dtype)
    print(f"case K={K} receivers={receivers} edges={E} {dtype}", flush=True)
    orc.compute_node_energies_forces(*args)
    eng.compute_node_energies_forces(*args)
    for name in ("Phi1", "A1", "M1", "H2", "Phi1_adj", "H1_adj", "A0_adj"):
        a, b = np.asarray(getattr(orc, name)), np.asarray(getattr(eng, name))
        assert np.abs(a - b).max(initial=0.0) <= TOL[dtype]["inter"] * 10 * max(1.0, np.abs(a).max()), name
    scale = max(1.0, np.abs(orc.node_forces).max())
    assert np.abs(orc.node_energies - eng.node_energies).max() <= TOL[dtype]["E"] * 10 * max(1.0, np.abs(orc.node_energies).max())
    assert np.abs(orc.node_forces - eng.node_forces).max() <= TOL[dtype]["F"] * scale
    # in chunks: the same sums of messages bit for bit.  (The forces go on from the linear behind them, which is a launch of its
    # own then; for some channel counts the other one forms it in double, in one launch with the sums: the oracle's tolerance.)
    h = eng.H1_adj
    eng.set_staging_limit(max(int(degree.max()), E // 3) * K * (8 if dtype == "float64" else 4))
    eng.compute_node_energies_forces(*args)
    assert np.array_equal(eng.H1_adj, h)
    assert np.abs(orc.node_forces - eng.node_forces).max() <= TOL[dtype]["F"] * scale


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("L_max,K,most,terms", [
    # 160 channels have no chains: from 1 024 atoms linears with the contraction in them, 600 the linears alone, 100 neither
    (0, 160, 1100, False), (1, 160, 1100, False),
    # 32 channels: chains up to 3 072 (l = 0) and 2 048 atoms (l <= 1), linears with the contraction above
    (0, 32, 3100, False), (1, 32, 2100, False),
    # pair repulsion and density normalisation: the linears alone
    (0, 32, 1100, True)])
def test_arrays_that_an_evaluation_does_not_form(gpu, tmp_models, L_max, K, most, terms, dtype):
    """The A-basis and its adjoint stay in registers where the contraction is evaluated behind the linear (in its launch, or in
    a chain) and are formed when somebody asks: alone, in either order, after a stage call, with ghost nodes, and after an
    evaluation of fewer atoms that takes other kernels."""
    from symmetrix_amd import neighbors
    model = H.tiny_model(K=K, L_max=L_max, n_pts=32, seed=60 + L_max, r_cut=3.0, pair=False, zbl=terms, density=terms)
    path = H.write_model(model, tmp_models / f"asked_{L_max}{K}{int(terms)}.json")
    runs = {}
    for n in (most, 600, 100):
        pos, cell, sp = H.small_system(n, density=0.06, seed=n)
        nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
        orc = _oracle()(model)
        orc.compute_node_energies_forces(*H.call_args(ea))
        runs[n] = (nl, ea, sp, orc)
    eng = gpu(path, dtype)

    def same(names, orc, rows=None):
        for name in names:
            a, b = np.asarray(getattr(orc, name)), np.asarray(getattr(eng, name))
            if rows is not None:
                a, b = a.reshape(rows, -1), b.reshape(-1, a.size // rows)[:rows]
            assert a.shape == b.shape, name
            assert np.abs(a - b).max() <= TOL[dtype]["inter"] * 10 * max(1.0, np.abs(a).max()), name

    for n, names in ((most, ("A0", "A1", "A0_adj", "A1_adj")), (most, ("A1_adj", "A0_adj", "A1", "A0", "M0_grad", "M1_grad")),
                     (600, ("A0_adj", "A0", "A1_adj", "A1")), (most, ("A0_adj",)), (100, ("A1", "A0")), (most, ("A1",))):
        print(f"{n} atoms, K {K}, L_max {L_max}, {dtype}: {' '.join(names)}", flush=True)
        nl, ea, sp, orc = runs[n]
        eng.compute_node_energies_forces(*H.call_args(ea))
        same(names, orc)
    # the largest size takes launches per stage (chains differ in the last bits)
    nl, ea, sp, orc = runs[most]
    eng.set_profiling(True)
    eng.compute_node_energies_forces(*H.call_args(ea))
    per_stage = np.array(eng.node_energies)
    assert (eng.stage_times()["M1"] == 0.0) == (not terms)      # (the contraction in the launch of its linear)
    eng.set_profiling(False)
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(per_stage, eng.node_energies)
    # a stage call forms what is left before it does anything else
    eng.compute_node_energies_forces(*H.call_args(ea))
    eng.reverse_M1(ea["num_nodes"], ea["node_types"])
    same(("A1", "A0"), orc)
    # ghost nodes: layer 0 covers them, layer 1 does not
    ga = neighbors.ghost_edge_arrays(nl, sp)
    eng.compute_ghosted(ga["num_local_nodes"], ga["num_ghost_nodes"], ga["node_types"], ga["num_neigh"], ga["neigh_indices"],
                        ga["neigh_types"], ga["xyz"], ga["r"])
    same(("A1", "A1_adj"), orc)
    same(("A0",), orc, rows=len(sp))


@pytest.mark.gpu
@pytest.mark.parametrize("L_max", [0, 1])
def test_stages_without_a_launch_of_their_own_have_no_time(gpu, tmp_models, L_max):
    """Whether a contraction ran inside its linear is told by the engine, not by how short its stage was."""
    model = H.tiny_model(K=32, L_max=L_max, n_pts=32, seed=60 + L_max, r_cut=3.0, pair=False)
    eng = gpu(H.write_model(model, tmp_models / f"stages_{L_max}.json"))
    eng.set_profiling(True)
    for n in (1100, 24, 1100):
        pos, cell, sp = H.small_system(n, density=0.06, seed=n)
        nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
        eng.compute_node_energies_forces(*H.call_args(ea))
        t = eng.stage_times()
        print(f"{n} atoms: {t}", flush=True)
        absent = {"readout", "rev_H2", "rev_M1", "force_sum0", "force_sum1"}
        absent |= {"M1"} if n >= 1024 else set()
        absent |= {"rev_H1", "rev_M0"} | ({"M0"} if n >= 1024 else set()) if L_max == 0 else set()
        assert {k for k, v in t.items() if v == 0.0} == absent
        assert all(v >= 0.0 for v in t.values())


@pytest.mark.gpu
@pytest.mark.parametrize("L_max,K", [(0, 32), (1, 8)])
@pytest.mark.parametrize("n", [255, 256, 257, 512, 513, 1024, 1025, 2100])
def test_buckets_on_both_sides_of_the_lds(gpu, tmp_models, n, L_max, K):
    """One sender of n edges among others of a few: buckets are ordered in the LDS of a wavefront (256 or 512 edges), of a
    block (1 024), or through it into memory.  Sums against the oracle, and the same bits twice and where the adjoint takes
    the receivers in chunks (which orders the buckets in memory first)."""
    model = H.tiny_model(K=K, L_max=L_max, n_pts=32, seed=51, pair=False)
    rng = np.random.default_rng(n)
    N, extra = 7, 60
    senders = rng.permutation(np.concatenate([np.full(n, 3), rng.choice([0, 1, 2, 4, 5], size=extra)])).astype(np.int32)
    E = len(senders)
    degree = np.bincount(rng.integers(0, N, size=E), minlength=N).astype(np.int32)
    species = rng.integers(0, 3, size=N).astype(np.int32)
    x = rng.normal(size=(E, 3))
    x *= (rng.uniform(1.0, 3.9, size=E) / np.linalg.norm(x, axis=1))[:, None]
    args = (N, species, degree, senders, species[senders], x.ravel(), np.linalg.norm(x, axis=1))
    orc = _oracle()(model)
    orc.compute_node_energies_forces(*args)
    eng = gpu(H.write_model(model, tmp_models / f"buckets_{K}.json"), "float64")
    print(f"{n} of {E} edges from one sender, K={K} L_max={L_max}", flush=True)
    eng.compute_node_energies_forces(*args)
    h, f = eng.H1_adj, eng.node_forces
    assert np.abs(h - orc.H1_adj).max() <= 1e-10 * np.abs(orc.H1_adj).max()
    assert np.abs(f - orc.node_forces).max() <= 1e-10 * np.abs(orc.node_forces).max()
    receivers = np.repeat(np.arange(N), degree)
    want = np.zeros((N, 3))
    np.add.at(want, senders, f.reshape(-1, 3)); np.add.at(want, receivers, -f.reshape(-1, 3))
    bound = 1e-13 * np.abs(f).max() * n
    F = eng.reduce_forces(N, senders)
    assert np.abs(F - want).max() <= bound
    shifted = np.where(senders == 3, 6, senders)       # senders that are not the evaluation's: lists of their own
    want = np.zeros((N, 3))
    np.add.at(want, shifted, f.reshape(-1, 3)); np.add.at(want, receivers, -f.reshape(-1, 3))
    assert np.abs(eng.reduce_forces(N, shifted) - want).max() <= bound
    eng.compute_node_energies_forces(*args)
    assert np.array_equal(eng.H1_adj, h) and np.array_equal(eng.node_forces, f) and np.array_equal(eng.reduce_forces(N, senders), F)
    eng.set_staging_limit(int(degree.max()) * K * (1 if L_max == 0 else 4) * 8)
    eng.compute_node_energies_forces(*args)
    assert np.array_equal(eng.H1_adj, h) and np.array_equal(eng.node_forces, f)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max,receivers,max_degree,terms", [
    # degrees on both sides of the chunks of 16 and 17 edges and of the two and four parts a receiver is split into
    (70, 1, 40, 37, 1), (130, 1, 24, 35, 1), (33, 2, 24, 34, 1), (70, 0, 40, 50, 1),
    # two wavefronts per receiver, then one, in either direction
    (16, 1, 515, 9, 1), (16, 1, 2051, 5, 1), (16, 1, 3075, 3, 1), (16, 1, 6147, 3, 1),
    # scalar sender features: two edges at a time in chunks of 44 and 62, one to four channels per lane and an edge alone,
    # channel groups that do not fill their lanes; at 48 channels tables beyond an L2 (four groups)
    (20, 0, 40, 67, 1), (33, 0, 40, 60, 1), (65, 0, 12, 270, 1), (97, 0, 12, 270, 1), (130, 0, 24, 90, 1), (48, 0, 24, 40, 1),
    # a wavefront per receiver, two channels per lane: two wavefronts per SIMD in double, chunks of 44 edges, two at a time and one
    (64, 0, 6145, 47, 1), (128, 0, 6145, 47, 1),
    # coupling entries of three terms
    (32, 1, 20, 20, 3), (32, 2, 20, 20, 3),
])
def test_general_edge_kernels_at_the_edges_of_their_split(gpu, tmp_models, K, L_max, receivers, max_degree, terms, dtype):
    model = H.tiny_model(K=K, L_max=L_max, n_pts=180 if K == 48 else 24, seed=K + L_max, pair=True)
    if terms > 1:   # every coefficient as a sum of three
        for key in ("Phi1_lme", "Phi1_lelm1lm2"):
            model[key] = [v for v in model[key] for _ in range(terms)]
        model["Phi1_clebsch_gordan"] = [v * w for v in model["Phi1_clebsch_gordan"] for w in (0.5, 0.75, -0.25)]
    rng = np.random.default_rng(receivers)
    degree = np.linspace(0, max_degree, receivers).astype(int) if max_degree > receivers else np.arange(receivers) % (max_degree + 1)
    E = int(degree.sum())
    species = rng.integers(0, 3, size=receivers).astype(np.int32)
    senders = rng.integers(0, receivers, size=E).astype(np.int32)
    x = rng.normal(size=(E, 3))
    x *= (rng.uniform(0.8, 3.9, size=E) / np.linalg.norm(x, axis=1))[:, None]
    args = (receivers, species, degree.astype(np.int32), senders, species[senders], x.ravel(), np.linalg.norm(x, axis=1))
    orc = _oracle()(model)
    eng = gpu(H.write_model(model, tmp_models / f"split_{K}_{L_max}_{receivers}_{terms}.json"), dtype)
    print(f"case K={K} L_max={L_max} receivers={receivers} edges={E} terms={terms} {dtype}", flush=True)
    orc.compute_node_energies_forces(*args)
    eng.compute_node_energies_forces(*args)
    names = ["A0", "Phi1", "H1_adj", "A0_adj"]
    for name in names:
        a, b = np.asarray(getattr(orc, name)), np.asarray(getattr(eng, name))
        assert np.abs(a - b).max(initial=0.0) <= TOL[dtype]["inter"] * 10 * max(1.0, np.abs(a).max()), name
    scale = max(1.0, np.abs(orc.node_forces).max())
    assert np.abs(orc.node_energies - eng.node_energies).max() <= TOL[dtype]["E"] * 10 * max(1.0, np.abs(orc.node_energies).max())
    assert np.abs(orc.node_forces - eng.node_forces).max() <= TOL[dtype]["F"] * scale
