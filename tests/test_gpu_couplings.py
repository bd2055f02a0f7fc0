"""Layer-1 couplings of the constant harmonic: like with like (what equivariant models have, a shorter way through the edge
kernels) and any other (the general way)."""
import numpy as np
import pytest

from symmetrix_amd import cg
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _mixed(model, L_max):
    """The same model with a coupling of the constant harmonic between different components of l = l2 = 1."""
    paths = cg.tensor_product_paths(3, L_max)
    num_e = [sum(1 for p in paths if p[0] == l) for l in range(4)]
    which = paths.index((1, 0, 1))
    e = which - sum(1 for p in paths if p[0] < 1)
    q = sum((2 * a + 1) * (2 * b + 1) for _, a, b in paths[:which])
    lme0 = num_e[0]
    extra = [(lme0 + 0 * num_e[1] + e, 0.3, q + 2), (lme0 + 2 * num_e[1] + e, -0.7, q + 1)]     # (m, m2) = (0, 2), (2, 1)
    for lme, c, at in extra:
        model["Phi1_lme"].append(lme)
        model["Phi1_clebsch_gordan"].append(c)
        model["Phi1_lelm1lm2"].append(at)
    return model


@pytest.mark.parametrize("dtype,tol_e,tol_f", [("float64", 1e-10, 1e-8), ("float32", 1e-5, 1e-4)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("K,L_max", [(32, 1), (128, 1), (40, 2)])
def test_couplings_of_the_constant_harmonic(tmp_models, K, L_max, mixed, dtype, tol_e, tol_f):
    """Tolerances of the two precisions as everywhere (parity with the oracle); 40 channels leave lanes without one."""
    import torch
    assert torch.cuda.is_available()
    from oracle.oracle import OracleMACE
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=5 + K, r_cut=3.5, pair=False)
    plain = H.write_model(model, tmp_models / f"coupling_{K}_{L_max}.json")
    path = H.write_model(_mixed(model, L_max), tmp_models / f"coupling_{K}_{L_max}_mixed.json") if mixed else plain
    pos, cell, sp = H.small_system(30, seed=K)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    orc, eng = OracleMACE(model), MACE(path, dtype)
    print(f"K={K} L_max={L_max} mixed={mixed} {dtype} edges={len(ea['r'])}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    for name in ("Phi1", "H1_adj"):
        a, b = getattr(eng, name), getattr(orc, name)
        assert np.abs(a - b).max() <= (1e-11 if dtype == "float64" else 2e-4) * np.abs(b).max(), name
    assert abs(eng.node_energies.sum() - orc.node_energies.sum()) <= tol_e * abs(orc.node_energies.sum())
    assert np.abs(eng.node_forces - orc.node_forces).max() <= tol_f
    if mixed:
        other = MACE(plain, dtype)
        other.compute_node_energies_forces(*H.call_args(ea))
        assert np.abs(eng.Phi1 - other.Phi1).max() > 1e-3 * np.abs(orc.Phi1).max()     # (the couplings do something)
