"""Aggregations over the edges and their adjoints, over the channels and receivers at which the sums are formed in other ways: four,
two and one wavefront per receiver, one to three channels per lane, with messages and without, l <= 1 and 2 on rows of three that
end in the ninth, l <= 2 with the paths of a receiver in two sets.  Copies of one small system that do not see each other: each must
give what the oracle gives for one of them."""
import numpy as np
import pytest

from tests import helpers as H
from tests.test_gpu_parity import TOL

pytestmark = pytest.mark.gpu

ARRAYS = ["Phi1", "Phi1_adj", "H1_adj", "A0_adj"]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max", [(40, 0), (64, 0), (96, 0), (128, 0), (64, 1), (96, 1), (128, 1), (64, 2), (128, 2), (160, 2)])
def test_copies_of_one_system(tmp_models, K, L_max, dtype):
    import torch
    assert torch.cuda.is_available()
    from oracle.oracle import OracleMACE
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=32, seed=K + L_max, r_cut=3.5, pair=False)
    rng = np.random.default_rng(K + L_max)
    degree = np.array([0, 1, 5, 15, 31, 46, 63, 8], np.int32)
    n, E = len(degree), int(degree.sum())
    species = rng.integers(0, 3, n).astype(np.int32)
    senders = rng.integers(0, n, E).astype(np.int32)
    x = rng.normal(size=(E, 3))
    x *= (rng.uniform(1.0, 3.4, E) / np.linalg.norm(x, axis=1))[:, None]
    r = np.linalg.norm(x, axis=1)
    orc = OracleMACE(model)
    orc.compute_node_energies_forces(n, species, degree, senders, species[senders], x.ravel(), r)
    eng = MACE(H.write_model(model, tmp_models / f"adjoints_{K}_{L_max}.json"), dtype)
    for copies in (75, 325, 790):
        print(f"K={K} L_max={L_max} receivers={n * copies} edges={E * copies} {dtype}", flush=True)
        shifted = (senders[None, :] + n * np.arange(copies, dtype=np.int32)[:, None]).ravel().astype(np.int32)
        eng.compute_node_energies_forces(n * copies, np.tile(species, copies), np.tile(degree, copies), shifted,
                                         np.tile(species[senders], copies), np.tile(x.ravel(), copies), np.tile(r, copies))
        for name in ARRAYS:
            want = np.asarray(getattr(orc, name)).reshape(n, -1)
            got = np.asarray(getattr(eng, name)).reshape(copies, n, -1)
            assert np.abs(got - want).max() <= TOL[dtype]["inter"] * 10 * max(1.0, np.abs(want).max()), name
        want = orc.node_forces.reshape(E, 3)
        got = eng.node_forces.reshape(copies, E, 3)
        assert np.abs(got - want).max() <= TOL[dtype]["F"] * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max", [(32, 1), (72, 2)])
def test_coupling_outside_the_selection_rules(tmp_models, K, L_max, dtype):
    """A file that couples two components which no rotation-equivariant product couples: the way that leaves none out."""
    import torch
    assert torch.cuda.is_available()
    from oracle.oracle import OracleMACE
    from symmetrix_amd import cg
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=32, seed=K, r_cut=3.5, pair=False)
    paths = cg.tensor_product_paths(3, L_max)
    which = paths.index((2, 1, 1))
    num_e = [sum(1 for p in paths if p[0] == l) for l in range(4)]
    e = which - sum(1 for p in paths if p[0] < 2)
    q = sum((2 * a + 1) * (2 * b + 1) for _, a, b in paths[:which])
    model["Phi1_lme"].append(num_e[0] + 3 * num_e[1] + 0 * num_e[2] + e)     # m = 0: m = -2 of l = 2
    model["Phi1_lelm1lm2"].append(q + 2 * 3 + 1)                             # m1 = 1 of l1 = 1, m2 = 0 of l2 = 1
    model["Phi1_clebsch_gordan"].append(0.6)
    pos, cell, sp = H.small_system(30, seed=K)
    _, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    orc, eng = OracleMACE(model), MACE(H.write_model(model, tmp_models / f"rules_{K}_{L_max}.json"), dtype)
    print(f"K={K} L_max={L_max} edges={len(ea['r'])} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    for name in ARRAYS:
        want, got = np.asarray(getattr(orc, name)), np.asarray(getattr(eng, name))
        assert np.abs(got - want).max() <= TOL[dtype]["inter"] * 10 * max(1.0, np.abs(want).max()), name
    assert np.abs(eng.node_forces - orc.node_forces).max() <= TOL[dtype]["F"] * max(1.0, np.abs(orc.node_forces).max())
