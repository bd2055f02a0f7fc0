"""Aggregations and their adjoints inside the chains of small systems: receivers whose edges end on either side of a round of eight, of
the 120 and 80 that a block takes at a time, or that have none; and where the rule ends."""
import numpy as np
import pytest

from tests import helpers as H
from tests.test_gpu_chains import ARRAYS, _compare

pytestmark = pytest.mark.gpu

DEGREES = [0, 1, 7, 8, 9, 79, 80, 81, 119, 120, 121, 248]


def _both(tmp_models, K, L_max, dtype, degree, seed, along, zbl=False):
    """Whatever an evaluation leaves, with chains and by launches per stage; along: layers whose edges the chains took."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=5 * K + L_max, r_cut=3.5, pair=False, zbl=zbl)
    eng = MACE(H.write_model(model, tmp_models / f"chain_edges_{K}_{L_max}_{int(zbl)}.json"), dtype)
    rng = np.random.default_rng(seed)
    N, E = len(degree), int(np.sum(degree))
    species = rng.integers(0, 3, N).astype(np.int32)
    senders = rng.integers(0, N, E).astype(np.int32)
    x = rng.normal(size=(E, 3))
    x *= (rng.uniform(1.0, 3.4, E) / np.linalg.norm(x, axis=1))[:, None]
    print(f"K={K} L_max={L_max} atoms={N} edges={E} {dtype}", flush=True)
    out = []
    for per_stage in (False, True):
        eng.set_profiling(per_stage)
        eng.compute_node_energies_forces(N, species, np.asarray(degree, np.int32), senders, species[senders], x.ravel(), np.linalg.norm(x, axis=1))
        assert eng._int("edges_in_chains") == (0 if per_stage else along)
        out.append({name: np.array(getattr(eng, name)) for name in ARRAYS})
    return out


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("L_max", [0, 1, 2])
@pytest.mark.parametrize("K", [32, 64, 96, 128])
def test_receivers_of_all_lengths(tmp_models, K, L_max, dtype):
    along = 3 if L_max == 0 else 1
    _compare(*_both(tmp_models, K, L_max, dtype, np.random.default_rng(K).permutation(DEGREES), K + L_max, along), dtype)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max", [(64, 0), (96, 0), (128, 1)])
def test_forces_that_are_there_before(tmp_models, K, L_max, dtype):
    """Pair repulsion: every adjoint adds to its forces."""
    _compare(*_both(tmp_models, K, L_max, dtype, DEGREES, K, 3 if L_max == 0 else 1, zbl=True), dtype)


# beyond: atoms more than CUs that hold a block each; n: atoms where they hold several
@pytest.mark.parametrize("K,beyond,n,dtype,along", [(96, 0, 0, "float64", 3), (96, 1, 0, "float64", 0), (128, 0, 0, "float32", 3), (128, 1, 0, "float32", 0),
                                                    (96, 44, 0, "float32", 3), (64, 44, 0, "float64", 3), (32, 0, 2048, "float64", 3), (32, 0, 2049, "float64", 0)])
def test_sizes_at_the_rule(tmp_models, K, beyond, n, dtype, along):
    """With the edges and without, where a CU holds one block and there are as many atoms as CUs, or one more, and elsewhere."""
    import torch
    n = n or torch.cuda.get_device_properties(0).multi_processor_count + beyond
    degree = np.random.default_rng(n).integers(0, 12, n)
    _compare(*_both(tmp_models, K, 0, dtype, degree, n, along), dtype)


def _with_ghosts(tmp_models, K, L_max, n, dtype, all_nodes):
    """n atoms by their owners, and with the neighbours across the box as ghost nodes; ghosts without an edge make up all_nodes."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd import neighbors
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=3 * K + L_max, r_cut=3.5, pair=False)
    eng = MACE(H.write_model(model, tmp_models / f"chain_ghosts_{K}_{L_max}.json"), dtype)
    pos, cell, sp = H.small_system(n, density=0.1, seed=n + K)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    g = neighbors.ghost_edge_arrays(nl, sp)
    more = all_nodes - n - g["num_ghost_nodes"]
    assert more >= 0 and g["num_ghost_nodes"] > 0
    none = np.zeros(more, np.int32)
    print(f"K={K} L_max={L_max} local={n} all={all_nodes} edges={len(g['r'])} {dtype}", flush=True)
    eng.compute_node_energies_forces(*H.call_args(ea))
    own = {name: np.array(getattr(eng, name)) for name in ("node_energies", "M0", "H1", "Phi1")}
    own["forces"] = eng.reduce_forces(n, ea["neigh_indices"])
    own["route"] = eng._int("edges_in_chains")
    eng.compute_ghosted(n, all_nodes - n, np.concatenate([g["node_types"], none]), np.concatenate([g["num_neigh"], none]),
                        g["neigh_indices"], g["neigh_types"], g["xyz"], g["r"])
    got = {name: np.array(getattr(eng, name))[:len(own[name])] for name in ("node_energies", "M0", "H1", "Phi1")}
    receivers = np.concatenate([g["receiver_atom"], np.zeros(more, np.int32)])
    got["forces"] = eng.reduce_forces(n, g["sender_atom"], receivers)
    got["route"] = eng._int("edges_in_chains")
    return own, got


# rounds: of blocks that the CUs hold one of each; nodes where they hold several.  (64 channels reach the line that the chains have for
# all nodes before.)
@pytest.mark.parametrize("K,L_max,dtype,n,rounds,nodes", [(96, 0, "float64", 100, 3, 0), (128, 0, "float64", 100, 2, 0), (128, 0, "float32", 100, 3, 0),
                                                          (128, 1, "float64", 100, 2, 0), (96, 1, "float32", 100, 6, 0),
                                                          (128, 2, "float32", 100, 3, 0), (32, 0, "float64", 1000, 0, 3840)])
def test_ghost_nodes_decide_layer_0(tmp_models, K, L_max, dtype, n, rounds, nodes):
    """Ghost nodes have blocks of their own in the chains of layer 0: beyond a number of them the edges of layer 0 are a launch of their
    own, with the bits of the chains."""
    import torch
    line = nodes + rounds * torch.cuda.get_device_properties(0).multi_processor_count
    for nodes in (line, line + 1):
        own, got = _with_ghosts(tmp_models, K, L_max, n, dtype, nodes)
        assert own["route"] == (3 if L_max == 0 else 1)
        assert got["route"] == own["route"] - (nodes > line)
        for name in ("node_energies", "M0", "H1", "Phi1"):
            assert np.array_equal(got[name], own[name]), name
        # (sums over the images of an atom in another order)
        tol = 1e-12 if dtype == "float64" else 1e-4
        assert np.abs(got["forces"] - own["forces"]).max() <= tol * np.abs(own["forces"]).max()
