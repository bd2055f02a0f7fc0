"""The A-basis linears: wavefronts with half of the (l, m) and with all of them, at both sides of the rule that chooses, and column
tiles in pairs only."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

ARRAYS = ["M1", "M1_grad", "M1_adj", "A1_adj", "A0_adj", "H1", "H1_adj", "node_energies"]


def _engine(tmp_models, K, L_max, dtype, density=False):
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, T=(1, 6, 8), n_pts=16 if not density else 48, seed=K + L_max, r_cut=3.0, pair=False, density=density)
    eng = MACE(H.write_model(model, tmp_models / f"linear_{K}_{L_max}_{int(density)}.json"), dtype)
    eng.set_profiling(True)      # small systems would take chains of stages otherwise
    return model, eng


# K, L_max, type, first size whose contraction keeps all (l, m) in a wavefront, and one that the rule leaves with halves
@pytest.mark.parametrize("K,L_max,dtype,n", [(128, 1, "float64", 9217), (128, 0, "float32", 5121), (64, 2, "float32", 10241),
                                             (64, 0, "float64", 18433)])
def test_both_kinds_of_wavefront(tmp_models, K, L_max, dtype, n):
    """The rows of atoms that see each other only are the same bits whatever system they are in: all products form the same sums
    in the same order, polynomials included.  n atoms (all (l, m) in a wavefront) against the first 100 and the last 101 of them."""
    _, eng = _engine(tmp_models, K, L_max, dtype)
    rng = np.random.default_rng(n)
    species = rng.integers(0, 3, n).astype(np.int32)
    i = np.arange(n)
    # one neighbour each, inside groups of ten consecutive atoms that start at multiples of ten; the last 101 begin one early
    cut = n - 101
    start = np.where(i < cut, i // 10 * 10, cut + (i - cut) // 10 * 10)
    size = np.minimum(np.where(i < cut, np.minimum(start + 10, cut), n) - start, 10)
    j = (start + (i - start + 1 + rng.integers(0, 2, n)) % size).astype(np.int32)
    r = rng.uniform(0.8, 2.9, n)
    u = rng.normal(size=(n, 3))
    xyz = u * (r / np.linalg.norm(u, axis=1))[:, None]
    one = np.ones(n, np.int32)
    print(f"K={K} L_max={L_max} atoms={n} {dtype}", flush=True)
    eng.compute_node_energies_forces(n, species, one, j, species[j], xyz, r)
    whole = {name: np.array(getattr(eng, name)).reshape(n, -1) for name in ARRAYS}
    forces = np.array(eng.node_forces).reshape(n, 3)
    for a, b in ((0, 100), (cut, n)):
        s = slice(a, b)
        eng.compute_node_energies_forces(b - a, species[s], one[s], j[s] - a, species[j[s]], xyz[s], r[s])
        for name in ARRAYS:
            got = np.array(getattr(eng, name)).reshape(b - a, -1)
            assert np.isfinite(got).all(), name
            assert np.abs(got - whole[name][s]).max() <= 1e-5 * np.abs(got).max() if dtype == "float32" else \
                np.abs(got - whole[name][s]).max() <= 1e-13 * np.abs(got).max(), name
        got = np.array(eng.node_forces).reshape(-1, 3)
        assert np.abs(got - forces[s]).max() <= (1e-5 if dtype == "float32" else 1e-12) * max(np.abs(got).max(), 1e-3)


# density normalisation: no factors and no contraction in the linears.  The first size is past the lines of all of them (single
# precision), the second past that of the adjoint of A1 only, the third is double and has halves throughout.
@pytest.mark.parametrize("K,L_max,dtype,n", [(128, 1, "float32", 16385), (64, 2, "float32", 6145), (64, 1, "float64", 18433)])
def test_both_kinds_without_a_contraction(tmp_models, K, L_max, dtype, n):
    """As above, bit for bit, against the first 600 and the last 601 atoms (wavefronts with halves)."""
    _, eng = _engine(tmp_models, K, L_max, dtype, density=True)
    rng = np.random.default_rng(n)
    species = rng.integers(0, 3, n).astype(np.int32)
    i, cut = np.arange(n), n - 601
    start = np.where(i < cut, i // 10 * 10, cut + (i - cut) // 10 * 10)
    size = np.minimum(np.where(i < cut, np.minimum(start + 10, cut), n) - start, 10)
    j = (start + (i - start + 1 + rng.integers(0, 2, n)) % size).astype(np.int32)
    r = rng.uniform(0.8, 2.9, n)
    u = rng.normal(size=(n, 3))
    xyz = u * (r / np.linalg.norm(u, axis=1))[:, None]
    one = np.ones(n, np.int32)
    names = ["A0", "A1", "A1_adj", "A0_adj", "Phi1_adj", "node_energies"]
    print(f"K={K} L_max={L_max} atoms={n} {dtype}", flush=True)
    eng.compute_node_energies_forces(n, species, one, j, species[j], xyz, r)
    whole = {name: np.array(getattr(eng, name)).reshape(n, -1) for name in names}
    forces = np.array(eng.node_forces).reshape(n, 3)
    assert np.isfinite(forces).all()
    for a, b in ((0, 600), (cut, n)):
        s = slice(a, b)
        eng.compute_node_energies_forces(b - a, species[s], one[s], j[s] - a, species[j[s]], xyz[s], r[s])
        for name in names:
            assert np.array_equal(np.array(getattr(eng, name)).reshape(b - a, -1), whole[name][s]), name
        assert np.array_equal(np.array(eng.node_forces).reshape(-1, 3), forces[s])


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,n,density", [(160, 17, False), (96, 33, False), (32, 16, False), (160, 9, True), (128, 20, True), (20, 7, True)])
def test_against_the_oracle(tmp_models, K, n, density, dtype):
    """Five pairs of column tiles (in pairs only), three tiles, one pair; rows of a tile left over and none.  With density
    normalisation: rows of more, of exactly and of less than the 2 048 elements that a block takes at a time."""
    from oracle.oracle import OracleMACE
    from tests.test_gpu_parity import _compare
    model, eng = _engine(tmp_models, K, 1, dtype, density=density)
    pos, cell, sp = H.small_system(n, seed=n)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    orc = OracleMACE(model)
    print(f"K={K} atoms={n} edges={len(ea['r'])} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    _compare(orc, eng, dtype)
