"""The A-basis linears: wavefronts with half of the (l, m) and with all of them, at both sides of the rule that chooses, and column
tiles in pairs only."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

ARRAYS = ["M1", "M1_grad", "M1_adj", "A1_adj", "A0_adj", "H1", "H1_adj"]


def _engine(tmp_models, K, L_max, dtype, density=False):
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, T=(1, 6, 8), n_pts=16 if not density else 48, seed=K + L_max, r_cut=3.0, pair=False, density=density)
    eng = MACE(H.write_model(model, tmp_models / f"linear_{K}_{L_max}_{int(density)}.json"), dtype)
    eng.set_profiling(True)      # small systems would take chains of stages otherwise
    return model, eng


def _groups(n, cut, rng):
    """One neighbour each, inside groups of ten consecutive atoms that start at multiples of ten, before `cut` and from there on."""
    species = rng.integers(0, 3, n).astype(np.int32)
    i = np.arange(n)
    start = np.where(i < cut, i // 10 * 10, cut + (i - cut) // 10 * 10)
    size = np.minimum(np.where(i < cut, np.minimum(start + 10, cut), n) - start, 10)
    j = (start + (i - start + 1 + rng.integers(0, 2, n)) % size).astype(np.int32)
    r = rng.uniform(0.8, 2.9, n)
    u = rng.normal(size=(n, 3))
    xyz = u * (r / np.linalg.norm(u, axis=1))[:, None]
    return species, j, xyz, r


def _in_parts(eng, n, part, names, fused, tol=0.0):
    """An evaluation of n atoms against evaluations of the first `part` and the last `part` + 1 of them, which see each other only.
    Whether the linear of layer 1 had the contraction in its launch is seen by the stage times."""
    cut = n - part - 1
    species, j, xyz, r = _groups(n, cut, np.random.default_rng(n))
    one = np.ones(n, np.int32)
    eng.compute_node_energies_forces(n, species, one, j, species[j], xyz, r)
    assert (eng.stage_times()["M1"] == 0.0) == fused
    names = names + ["node_energies", "node_forces"]
    whole = {name: np.array(getattr(eng, name)).reshape(n, -1) for name in names}
    assert all(np.isfinite(a).all() for a in whole.values())
    for a, b in ((0, part), (cut, n)):
        s = slice(a, b)
        eng.compute_node_energies_forces(b - a, species[s], one[s], j[s] - a, species[j[s]], xyz[s], r[s])
        assert (eng.stage_times()["M1"] == 0.0) == fused
        for name in names:
            got = np.array(getattr(eng, name)).reshape(b - a, -1)
            assert np.abs(got - whole[name][s]).max() <= tol * np.abs(got).max(), name


# K, L_max, type, and the first size whose contraction keeps all (l, m) in a wavefront
@pytest.mark.parametrize("K,L_max,dtype,n", [(128, 1, "float64", 9217), (128, 0, "float32", 5121), (64, 2, "float32", 10241),
                                             (64, 0, "float64", 18433)])
def test_both_kinds_of_wavefront(tmp_models, K, L_max, dtype, n):
    """All (l, m) in a wavefront, and the last size with halves of them, each against 1 030 and 1 031 atoms (halves as well, the
    contraction in the launch of the linear).  The products are the same sums in the same order whatever system an atom is in.  The
    polynomials are too, but the compiler may join other multiplications and additions in the two kernels: two sums of at most 112
    monomials, three roundings each, differ by 2 * (112 + 3) of them at most, 230 * 2^-53 = 2.6e-14 and 230 * 2^-24 = 1.4e-5 of the
    sum of magnitudes, and by the root of that in fact (1.7e-15, 9e-7).  What follows is linear in them."""
    _, eng = _engine(tmp_models, K, L_max, dtype)
    print(f"K={K} L_max={L_max} atoms={n} {dtype}", flush=True)
    for atoms in (n, n - 1):
        _in_parts(eng, atoms, 1030, ARRAYS, fused=True, tol=1e-13 if dtype == "float64" else 1e-5)


# density normalisation: no factors and no contraction in the linears.  The first size is past the lines of all of them (single
# precision), the second past that of the adjoint of A1 only, the third is double and has halves throughout.
@pytest.mark.parametrize("K,L_max,dtype,n", [(128, 1, "float32", 16385), (64, 2, "float32", 6145), (64, 1, "float64", 18433)])
def test_both_kinds_without_a_contraction(tmp_models, K, L_max, dtype, n):
    """As above against the first 600 and the last 601 atoms (wavefronts with halves), bit for bit: the
    polynomials have a launch of their own."""
    _, eng = _engine(tmp_models, K, L_max, dtype, density=True)
    print(f"K={K} L_max={L_max} atoms={n} {dtype}", flush=True)
    _in_parts(eng, n, 600, ["A0", "A1", "A1_adj", "A0_adj", "Phi1_adj"], fused=False)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max,n,terms", [
    # from 512 atoms the linears alone, from 1 024 with the contraction of layer 1 (and of layer 0 at scalar features); halves of
    # the (l, m).  Five pairs of column tiles, three tiles (pairs, with a contraction), one pair
    (160, 1, 1031, False), (96, 0, 1024, False), (96, 1, 1050, False), (32, 2, 1025, False), (160, 0, 512, False), (96, 1, 527, False),
    # density normalisation (the linears alone, without factors)
    (64, 1, 1040, True),
    # density normalisation of rows of more, of exactly and of less than the 2 048 elements that a block takes at a time
    (160, 1, 9, True), (128, 1, 20, True), (20, 1, 7, True)])
def test_against_the_oracle(tmp_models, K, L_max, n, terms, dtype):
    """Row tiles of 16 atoms of one species, remainders among them."""
    from oracle.oracle import OracleMACE
    from tests.test_gpu_parity import _compare
    model, eng = _engine(tmp_models, K, L_max, dtype, density=terms)
    pos, cell, sp = H.small_system(n, density=0.06 if n > 100 else 0.08, seed=n)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    orc = OracleMACE(model)
    print(f"K={K} L_max={L_max} atoms={n} edges={len(ea['r'])} {dtype}", flush=True)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert (eng.stage_times()["M1"] == 0.0) == (n >= 1024 and not terms)
    _compare(orc, eng, dtype)
