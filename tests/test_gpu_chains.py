"""The node-local stages of small systems: chains of them in one launch, an atom per thread block, against the launches per
stage that an evaluation takes which is asked for the times of its stages."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

ARRAYS = ["A0", "M0", "H1", "Phi1", "A1", "M1", "H2", "H2_adj", "M1_adj", "A1_adj", "Phi1_adj", "H1_adj", "M0_adj", "A0_adj", "M1_grad",
          "M0_grad", "node_energies", "node_forces"]


def _both(tmp_models, K, L_max, n, dtype, density=0.1):
    """Whatever an evaluation leaves, by either way."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=3 * K + L_max, r_cut=3.5, pair=False)
    eng = MACE(H.write_model(model, tmp_models / f"chains_{K}_{L_max}.json"), dtype)
    pos, cell, sp = H.small_system(n, density=density, seed=n + K)
    sp = np.where(sp == 1, 2, sp).astype(np.int32)      # a species of the model that the system does not have
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    print(f"K={K} L_max={L_max} atoms={n} edges={len(ea['r'])} {dtype}", flush=True)
    out = []
    for per_stage in (False, True):
        eng.set_profiling(per_stage)
        eng.compute_node_energies_forces(*H.call_args(ea))
        out.append({name: np.array(getattr(eng, name)) for name in ARRAYS})
    return out


def _compare(got, ref, dtype):
    """Both ways form the same sums, of at most 640 products (five blocks of 128 channels), in different orders, and a dozen of
    them follow one another.  A sum of n numbers differs by n/2 roundings of its terms at most, by about sqrt(n) in fact: 30 of
    them each time, against the largest entry, gives 12 * 30 * 2^-53 = 4e-14 and 12 * 30 * 2^-24 = 2e-5; gradients multiply
    three variables (and their errors)."""
    tol = 1e-12 if dtype == "float64" else 1e-4
    for name in ARRAYS:
        a, b = got[name], ref[name]
        assert a.shape == b.shape, name
        assert np.isfinite(a).all(), name
        assert np.abs(a - b).max(initial=0.0) <= tol * max(np.abs(b).max(initial=0.0), 1e-30), name


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("L_max", [0, 1, 2])
@pytest.mark.parametrize("K", [32, 64, 96, 128])
def test_chains_match_launches_per_stage(tmp_models, K, L_max, dtype):
    for n in (2, 23):
        _compare(*_both(tmp_models, K, L_max, n, dtype), dtype)


@pytest.mark.parametrize("n", [768, 769])
def test_chains_end_where_the_rule_says(tmp_models, n):
    """98 304 channels of all atoms at scalar hidden features: the last size with chains (which differ from launches per stage in
    the last bits), and the first without (which does not)."""
    got, ref = _both(tmp_models, 128, 0, n, "float32", density=0.06)
    _compare(got, ref, "float32")
    assert np.array_equal(got["node_energies"], ref["node_energies"]) == (n == 769)


def _ghosted(tmp_models, K, L_max, n, dtype, all_nodes=None):
    """The same for n local atoms whose neighbours across the box are ghost nodes; ghosts without an edge make up all_nodes."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd import neighbors
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=3 * K + L_max, r_cut=3.5, pair=False)
    eng = MACE(H.write_model(model, tmp_models / f"chains_{K}_{L_max}.json"), dtype)
    pos, cell, sp = H.small_system(n, density=0.1, seed=n + K)
    nl, _ = H.edges_of(pos, cell, sp, model["r_cut"])
    g = neighbors.ghost_edge_arrays(nl, sp)
    more = 0 if all_nodes is None else all_nodes - n - g["num_ghost_nodes"]
    assert more >= 0 and g["num_ghost_nodes"] > 0
    none = np.zeros(more, np.int32)
    args = (n, g["num_ghost_nodes"] + more, np.concatenate([g["node_types"], none]), np.concatenate([g["num_neigh"], none]),
            g["neigh_indices"], g["neigh_types"], g["xyz"], g["r"])
    print(f"K={K} L_max={L_max} local={n} ghosts={args[1]} edges={len(g['r'])} {dtype}", flush=True)
    out = []
    for per_stage in (False, True):
        eng.set_profiling(per_stage)
        eng.compute_ghosted(*args)
        out.append({name: np.array(getattr(eng, name)) for name in ARRAYS})
    return out


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max", [(32, 0), (64, 2), (96, 1), (128, 0)])
def test_chains_match_launches_per_stage_with_ghost_nodes(tmp_models, K, L_max, dtype):
    """Layer 0 takes a block per node, ghosts included, layer 1 a block per local one."""
    _compare(*_ghosted(tmp_models, K, L_max, 23, dtype), dtype)


@pytest.mark.parametrize("dtype,nodes", [("float64", 1088), ("float64", 1089), ("float32", 1280), ("float32", 1281)])
def test_chains_end_where_the_rule_for_all_nodes_says(tmp_models, dtype, nodes):
    """139 264 channels of all nodes in double precision, 163 840 in single: the last size with chains and the first without."""
    got, ref = _ghosted(tmp_models, 128, 0, 100, dtype, all_nodes=nodes)
    _compare(got, ref, dtype)
    same = all(np.array_equal(got[name], ref[name]) for name in ("node_energies", "H1", "M1"))
    assert same == (nodes in (1089, 1281))
