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
