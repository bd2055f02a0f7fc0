"""Workloads of the engine as its users call it: which sizes, models, precisions and entry points, how their inputs are
made, and what a pass through each cannot do without.

Five ways in, all public:

  calculator  SymmetrixCalculator.compute(positions, cell, atomic_numbers): host positions in; energies, per-atom forces
              and stress out (structure relaxation, single points, scripts driving a small cell)
  host        MACE.compute_node_energies_forces with numpy edge arrays, node_energies and reduce_forces read back (a caller
              that brings its own neighbour list)
  lammps      MACE.compute_ghosted with numpy edge arrays that hold periodic images as ghost nodes, then reduce_forces (the
              pair style's mode without communication between the layers)
  device      MACE.compute_device with edge arrays that already are on the GPU, outputs into the caller's tensors
  md          one molecular-dynamics force call: DeviceNeighborList.update at moved positions, MACE.compute_device,
              reduce_forces_device with the virial

Models are the benchmark's configurations (random weights of a fixed seed, written once per machine): scalar hidden features
(off_small), hidden features up to l = 1 (off_medium, mp_medium) and up to l = 2 (off_medium_l2), with one radial table for
all species pairs or one per pair, with or without pair repulsion and density normalisation.  Double precision is the
default of every entry point; float32 features are what long runs use."""
from __future__ import annotations

import json
import math
import os
import tempfile

import numpy as np
import torch

from symmetrix_amd import modelgen, neighbors
from symmetrix_amd.calc import SymmetrixCalculator
from symmetrix_amd.mace import MACE


def _case(name, path, model, atoms, dtype, channels=None, tables="one", pair_terms=False):
    case = {"path": path, "model": model, "atoms": atoms, "dtype": dtype, "tables": tables, "pair_terms": pair_terms,
            "channels": channels or modelgen.CONFIGS[model]["num_channels"]}
    return dict(case, name=name) if name else case


def listed():
    return [
        # a handful of molecules from a script: nothing but latency
        _case("calculator_water_24", "calculator", "off_small", 24, "float64"),
        # a metallic cell with a vacancy under relaxation
        _case("calculator_alloy_107", "calculator", "mp_medium", 107, "float64"),
        # molecular dynamics of a small box in the precision that long runs use
        _case("md_organic_501_f32", "md", "off_small", 501, "float32"),
        # the benchmark's headline: energies and edge forces of a 3 000-atom box, arrays on the GPU
        _case("device_organic_3000", "device", "off_small", 3000, "float64"),
        # the same kind of box with a radial table of its own for every species pair (models with a distance transform)
        _case("device_organic_2989_pairs", "device", "off_small", 2989, "float64", tables="pair"),
        # a larger box of the small model
        _case("device_organic_20011_f32", "device", "off_small", 20011, "float32"),
        # a caller with its own neighbour list; a model with pair repulsion and density normalisation
        _case("host_alloy_1999_terms", "host", "mp_medium", 1999, "float64", pair_terms=True),
        # one rank of a domain-decomposed run: ghost atoms as explicit nodes, host arrays
        _case("lammps_water_3000", "lammps", "off_medium", 3000, "float64"),
        # molecular dynamics of bulk water
        _case("md_water_9999_f32", "md", "off_medium", 9999, "float32"),
        # a large water box in double precision
        _case("device_water_24999", "device", "off_medium", 24999, "float64"),
        # hidden features up to l = 2
        _case("device_water_l2_3000_f32", "device", "off_medium_l2", 3000, "float32"),
        # the benchmark's second configuration: 50 000-atom alloy
        _case("device_alloy_50000_f32", "device", "mp_medium", 50000, "float32"),
    ]


# atoms per path: a calculator is used on anything from a molecule to a box, files and host arrays on ordinary sizes, the
# device-resident calls up to the largest
_ATOMS = {"calculator": (12, 6000), "host": (24, 6000), "lammps": (48, 3000), "device": (96, 50000), "md": (96, 30000)}
_SPREAD = [("calculator", 4), ("host", 2), ("lammps", 2), ("device", 6), ("md", 4)]


def draw(rng):
    path = rng.choices([p for p, _ in _SPREAD], [w for _, w in _SPREAD])[0]
    model = rng.choices(["off_small", "off_medium", "mp_medium", "off_medium_l2"], [4, 3, 3, 1])[0]
    channels = rng.choice([32, 64, 96, 128] if model == "off_small" else [64, 128] if model == "off_medium_l2" else [64, 96, 128])
    dtype = rng.choice(["float64", "float32"])
    tables = rng.choices(["one", "pair"], [3, 1])[0]
    pair_terms = rng.random() < 0.25
    lo, hi = _ATOMS[path]
    atoms = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    case = _case(None, path, model, atoms, dtype, channels, tables, pair_terms)
    # not beyond the largest listed case: arithmetic weighted by the width of a value
    most = 0.8 * work(listed()[-1])["flops"]
    cost = work(case)["flops"] * (2.0 if dtype == "float64" else 1.0)
    if cost > most:
        case["atoms"] = max(96, int(atoms * most / cost * rng.uniform(0.6, 1.0)))
    return case


# ---- models -------------------------------------------------------------------------------------------------------------

_model_files, _evaluators, _calculators = {}, {}, {}


def _config(case):
    cfg = dict(modelgen.CONFIGS[case["model"]], num_channels=case["channels"], pair_dependent_radial=case["tables"] == "pair",
               zbl=case["pair_terms"], density_normalisation=case["pair_terms"])
    return cfg


def _model_key(case):
    return (case["model"], case["channels"], case["tables"], case["pair_terms"])


def _model_file(case):
    key = _model_key(case)
    if key not in _model_files:
        path = os.path.join(tempfile.gettempdir(), "smx_case_%s_%d_%s_%d.json" % key)
        if not os.path.exists(path):
            model = modelgen.generate_model(**_config(case))
            with tempfile.NamedTemporaryFile("w", dir=tempfile.gettempdir(), suffix=".json", delete=False) as f:
                f.write("{")
                for n, (k, v) in enumerate(model.items()):
                    f.write((", " if n else "") + json.dumps(k) + ": ")
                    if k.startswith("radial_spline_") and isinstance(v, list) and case["tables"] == "one":
                        text = json.dumps(v[0])     # the same table for every species pair
                        f.write("[" + ", ".join([text] * len(v)) + "]")
                    else:
                        f.write(json.dumps(v))
                f.write("}")
            os.chmod(f.name, 0o644)
            os.replace(f.name, path)
        _model_files[key] = path
    return _model_files[key]


def _evaluator(case):
    """The evaluator a program keeps for a model: one per model and precision."""
    key = _model_key(case) + (case["dtype"],)
    if key not in _evaluators:
        _evaluators[key] = MACE(_model_file(case), case["dtype"])
    return _evaluators[key]


def _calculator(case):
    key = _model_key(case) + (case["dtype"],)
    if key not in _calculators:
        _calculators[key] = SymmetrixCalculator(_model_file(case), dtype=case["dtype"])
    return _calculators[key]


# ---- structures ---------------------------------------------------------------------------------------------------------

def _sites(n, volume, rng, jitter):
    """n of the sites of a cubic lattice that fills a cubic cell of this volume, displaced at random."""
    m = math.ceil(n ** (1.0 / 3.0) - 1e-9)
    length = volume ** (1.0 / 3.0)
    pick = np.sort(rng.permutation(m ** 3)[:n])
    grid = np.stack([pick // (m * m), pick // m % m, pick % m], axis=1) + 0.5
    return (grid + rng.uniform(-jitter, jitter, size=(n, 3))) * (length / m), length


def _structure(case, seed):
    """Positions, cell lengths and species indices, at the densities of the benchmark's systems."""
    rng = np.random.default_rng(seed)
    n = case["atoms"]
    if case["model"] == "off_small":            # organic matter, 0.10 atoms per cubic Angstrom
        pos, length = _sites(n, n / 0.10, rng, 0.22)
        species = rng.choice(4, size=n, p=[0.5, 0.3, 0.1, 0.1])
        cell = np.full(3, length)
    elif case["model"] == "mp_medium":          # perturbed fcc alloy with vacancies
        a = 3.6
        cells = max(8, math.ceil(n / 4))
        m = max(2, int(cells ** (1.0 / 3.0)))
        reps = np.array([m, m, m])
        while 4 * reps.prod() < n:
            reps[np.argmin(reps)] += 1
        basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
        origin = np.stack(np.meshgrid(*[np.arange(r) for r in reps], indexing="ij"), axis=-1).reshape(-1, 1, 3)
        pos = ((origin + basis) * a).reshape(-1, 3)
        pos = pos[np.sort(rng.permutation(len(pos))[:n])] + rng.normal(scale=0.1, size=(n, 3))
        cell = reps * a
        species = rng.integers(0, 5, size=n)
    else:                                       # water, 0.033 molecules per cubic Angstrom (the last one may lack a hydrogen or two)
        mol = math.ceil(n / 3)
        oxygen, length = _sites(mol, mol / 0.033, rng, 0.1)
        axis = rng.integers(0, 3, size=mol)     # two bonds along different axes of the box, either way: no two atoms coincide
        axes = np.stack([axis, (axis + rng.integers(1, 3, size=mol)) % 3])
        d = 0.96 * np.eye(3)[axes] * rng.choice([-1.0, 1.0], size=(2, mol, 1))
        pos = np.stack([oxygen, oxygen + d[0], oxygen + d[1]], axis=1).reshape(-1, 3)[:n] + rng.normal(scale=0.03, size=(n, 3))
        species = np.tile([3, 0, 0], mol)[:n]
        cell = np.full(3, length)
    return np.ascontiguousarray(np.mod(pos, cell)), cell, species.astype(np.int32)


def prepare(case, seed):
    positions, cell, species = _structure(case, seed)
    r_cut = modelgen.CONFIGS[case["model"]]["r_cut"]
    n = case["atoms"]
    state = {"path": case["path"], "n": n}
    if case["path"] == "calculator":
        numbers = np.array(sorted(modelgen.CONFIGS[case["model"]]["atomic_numbers"]))
        return dict(state, calc=_calculator(case), positions=positions, cell=np.diag(cell), numbers=numbers[species])
    state["eval"] = _evaluator(case)
    nl = neighbors.DeviceNeighborList()
    if case["path"] in ("host", "lammps"):
        nl.build_host(positions, species, cell, r_cut)
        found = nl.to_host()
        arrays = neighbors.edge_arrays(found, species) if case["path"] == "host" else neighbors.ghost_edge_arrays(found, species)
        return dict(state, arrays=arrays)
    dev = torch.device("cuda:0")
    state["list"] = nl
    state["energies"] = torch.zeros(n, dtype=torch.float64, device=dev)
    if case["path"] == "device":
        state["edges"] = nl.build_host(positions, species, cell, r_cut)
        # room for the edge forces of any configuration of this size, as a program that keeps its arrays has it
        room = int(1.3 * _edges(case)) + 4096
        if state["edges"] > room:
            raise RuntimeError("more edges than there is room for")
        state["forces"] = torch.zeros((room, 3), dtype=torch.float64, device=dev)
        return state
    # md: a list with a skin, found some steps ago, and the positions of now
    skin = 0.6
    nl.build_host(positions, species, cell, r_cut, skin=skin)
    move = np.random.default_rng([seed, 1]).normal(scale=0.05, size=positions.shape)
    state["positions"] = torch.from_numpy(positions + np.clip(move, -skin / 4, skin / 4)).to(dev)
    state["types"] = torch.from_numpy(species).to(dev)
    state["r_cut"] = r_cut
    return state


def run(state):
    n = state["n"]
    if state["path"] == "calculator":
        got = state["calc"].compute(state["positions"], state["cell"], state["numbers"])
        return {k: got[k] for k in ("energy", "energies", "forces", "stress")}
    ev = state["eval"]
    if state["path"] == "host":
        a = state["arrays"]
        ev.compute_node_energies_forces(a["num_nodes"], a["node_types"], a["num_neigh"], a["neigh_indices"], a["neigh_types"],
                                        a["xyz"], a["r"])
        forces, virial = ev.reduce_forces(n, a["neigh_indices"], virial=True)
        return {"energies": ev.node_energies, "forces": forces, "virial": virial}
    if state["path"] == "lammps":
        a = state["arrays"]
        ev.compute_ghosted(a["num_local_nodes"], a["num_ghost_nodes"], a["node_types"], a["num_neigh"], a["neigh_indices"],
                           a["neigh_types"], a["xyz"], a["r"])
        forces, virial = ev.reduce_forces(n, a["sender_atom"], a["receiver_atom"], virial=True)
        return {"energies": ev.node_energies, "forces": forces, "virial": virial}
    nl, stream = state["list"], torch.cuda.current_stream().cuda_stream
    if state["path"] == "device":
        p, edges = nl.ptr, state["edges"]
        ev.compute_device(n, p["node_types"], p["num_neigh"], p["neigh_indices"], p["neigh_types"], p["xyz"], p["r"], edges,
                          state["energies"].data_ptr(), state["forces"].data_ptr(), stream)
        return {"energies": state["energies"], "forces": state["forces"]}
    types = state["types"].data_ptr()
    edges = nl.update(state["positions"].data_ptr(), types, state["r_cut"], stream)
    p = nl.ptr
    ev.compute_device(n, types, p["num_neigh"], p["neigh_indices"], p["neigh_types"], p["xyz"], p["r"], edges,
                      state["energies"].data_ptr(), 0, stream)
    forces, virial = ev.reduce_forces_device(n, p["neigh_indices"], virial=True)
    return {"energies": state["energies"], "forces": forces, "virial": virial}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------

_DENSITY = {"off_small": 0.10, "mp_medium": 4 / 3.6 ** 3, "off_medium": 0.099, "off_medium_l2": 0.099}


def _edges(case):
    """Edges of a configuration, from its density."""
    return case["atoms"] * _DENSITY[case["model"]] * 4.0 / 3.0 * math.pi * modelgen.CONFIGS[case["model"]]["r_cut"] ** 3


# per hidden degree: paths of layer 1, entries of their coupling block, contracted outputs, monomials of layer 0's polynomials
_PATHS = {0: (4, 16, 16, 94), 1: (10, 88, 40, 410), 2: (17, 243, 71, 882)}


def work(case):
    """Bytes: the edge and node arrays (or the positions, where the list is formed inside), the model's tables and weights read
    once, the outputs written once.  Flops: per edge and channel the radial splines with derivatives, the coupling forward
    and as often again for the adjoint (message and three force components); per atom the channel-mixing products and the
    contractions, forward and adjoint."""
    cfg = modelgen.CONFIGS[case["model"]]
    n, k, s = case["atoms"], case["channels"], 8 if case["dtype"] == "float64" else 4
    e = _edges(case)
    paths, coupling, outputs, monomials = _PATHS[cfg["L_max"]]
    n_lm, t = (cfg["L_max"] + 1) ** 2, len(cfg["atomic_numbers"])
    flops = e * k * (10 * (4 + paths) + 2 * 16 + 2 * coupling + 2 * 32 + 4 * coupling)
    flops += n * k * k * 4 * (16 + n_lm + outputs + 2) + n * k * 12 * (monomials + 94)
    tables = (1 if case["tables"] == "one" else t * (t + 1) // 2) * 255 * 4 * (4 + paths) * k
    weights = k * k * (4 * t + 1 + cfg["L_max"] + outputs / 3 + t + 1) + (monomials + 94) * t * k
    model_bytes = s * (tables + weights)
    # positions 24 and species 4 in; per edge xyz 24, r 8, sender 4, species 4
    arrays = {"calculator": 28 * n, "md": 28 * n}.get(case["path"], 8 * n + 40 * e)
    outs = 8 * n + (24 * e if case["path"] == "device" else 24 * n)
    return {"bytes": arrays + outs + model_bytes, "flops": flops}


def tolerance(case):
    # all outputs are double; with float32 features they carry sums of single-precision products
    return {"rel": 1e-11, "max": 1e-9} if case["dtype"] == "float64" else {"rel": 1e-5, "max": 1e-3}
