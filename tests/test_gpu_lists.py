"""The list preparation of an evaluation: one block's scan and one block per species, at the edges of a thread's 16 elements, of
a block's round, and of the number of blocks that count with a ticket; and lists of nothing."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 1025, 16383, 16385, 33000])
def test_lists_of_any_length(tmp_models, n):
    """Energies and forces of an atom depend on its own edges only: a system of n atoms in random order of species, with 0 to 3
    edges each, against the same atoms a few at a time.  A row that the lists lose, repeat or give to another species differs in
    the first digits; what is left is the order of sums (2^-53 of at most 640 terms, a dozen in a row)."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=32, L_max=0, T=(1, 6, 7, 8), n_pts=16, seed=5, r_cut=3.0, pair=False)
    eng = MACE(H.write_model(model, tmp_models / "lists.json"), "float64")
    rng = np.random.default_rng(n)
    species = rng.choice([0, 1, 3], n).astype(np.int32)       # the third species has no atom
    num = rng.integers(0, 4, n).astype(np.int32)
    if n > 1000:
        num[:16 * 7] = 0
        species[-200:] = 3
    i = np.repeat(np.arange(n), num)
    # neighbours inside groups of 8 consecutive atoms, which can be evaluated by themselves
    j = np.minimum(i // 8 * 8 + rng.integers(0, 8, len(i)), n - 1).astype(np.int32)
    r = rng.uniform(0.8, 2.9, len(i))
    u = rng.normal(size=(len(i), 3))
    xyz = u * (r / np.linalg.norm(u, axis=1))[:, None]
    print(f"atoms={n} edges={len(i)}", flush=True)
    eng.compute_node_energies_forces(n, species, num, j, species[j], xyz, r)
    E, F = np.array(eng.node_energies), np.array(eng.node_forces).reshape(-1, 3)
    assert np.isfinite(E).all() and np.isfinite(F).all()
    first = np.concatenate([[0], np.cumsum(num)])
    groups = np.unique(np.concatenate([[0, (n - 1) // 8], rng.integers(0, (n + 7) // 8, 12), np.arange(16384 // 8 - 1, 16384 // 8 + 1)]))
    for g in groups[groups * 8 < n]:
        a, b = g * 8, min(g * 8 + 8, n)
        e = slice(first[a], first[b])
        eng.compute_node_energies_forces(b - a, species[a:b], num[a:b], j[e] - a, species[j[e]], xyz[e], r[e])
        assert np.abs(np.array(eng.node_energies) - E[a:b]).max() <= 1e-12 * np.abs(E).max()
        f = np.array(eng.node_forces).reshape(-1, 3)
        if len(f):
            assert np.abs(f - F[e]).max() <= 1e-12 * max(np.abs(F).max(), 1.0)


def test_lists_refuse_what_they_refused(tmp_models):
    """A species or a sender out of range, a negative count: found by whichever block looks at it."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=32, L_max=0, T=(1, 6, 8), n_pts=16, seed=5, r_cut=3.0, pair=False)
    eng = MACE(H.write_model(model, tmp_models / "lists_bad.json"), "float64")
    n = 20000
    species, num = np.zeros(n, np.int32), np.ones(n, np.int32)
    j = np.roll(np.arange(n), 1).astype(np.int32)
    xyz, r = np.tile([0.0, 0.0, 1.0], (n, 1)), np.ones(n)
    eng.compute_node_energies_forces(n, species, num, j, species, xyz, r)
    good = np.array(eng.node_energies)
    for at in (0, 17000, n - 1):
        for which, value in ((0, 3), (0, -1), (2, n), (2, -1), (3, 3)):
            args = [species.copy(), num, j.copy(), species.copy()]
            args[which][at] = value
            with pytest.raises(Exception):
                eng.compute_node_energies_forces(n, *args, xyz, r)
    eng.compute_node_energies_forces(n, species, num, j, species, xyz, r)
    assert np.array_equal(np.array(eng.node_energies), good)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K,L_max,terms", [(32, 0, False), (32, 1, True), (20, 0, True)])
def test_no_nodes(tmp_models, K, L_max, terms, dtype):
    """A rank without atoms: every stage call for no nodes, before and after other calls, and an evaluation whose nodes are all
    ghosts.  Species groups of no nodes are empty, nothing is written for a node that is not there, and what follows is as before.
    (32 and 20 channels: the readout tail in one launch and in three.)"""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=7, pair=False, zbl=terms, density=terms)
    path = H.write_model(model, tmp_models / f"none_{K}_{L_max}.json")
    pos, cell, sp = H.small_system(40, seed=8)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    n, width = len(sp), (L_max + 1) ** 2 * K
    i0, d0, rows = np.zeros(0, np.int32), np.zeros(0), 5

    def stages(eng):
        """One rank's share of the mode with message passing, `rows` rows of H1 from other ranks."""
        eng.fill("node_energies", 0); eng.fill("node_forces", 0)
        if eng.has_zbl:
            eng.zbl.compute_ZBL(0, i0, i0, i0, eng.atomic_numbers, d0, d0)
        eng.compute_Y(d0); eng.compute_R0(0, i0, i0, i0, d0); eng.compute_A0(0, i0, i0, i0)
        eng.compute_A0_scaled(0, i0, i0, i0, d0); eng.compute_M0(0, i0); eng.compute_H1(0)
        assert len(eng.A0) == len(eng.M0) == len(eng.H1) == 0
        eng.H1 = np.arange(rows * width) * 1e-3
        eng.compute_R1(0, i0, i0, i0, d0); eng.compute_Phi1(0, i0, i0); eng.compute_A1(0)
        eng.compute_A1_scaled(0, i0, i0, i0, d0); eng.compute_M1(0, i0); eng.compute_H2(0, i0); eng.compute_readouts(0, i0)
        assert len(eng.H2) == len(eng.node_energies) == len(eng.M1) == 0
        eng.reverse_H2(0, i0, False); eng.reverse_M1(0, i0); eng.reverse_A1_scaled(0, i0, i0, i0, d0, d0, False); eng.reverse_A1(0)
        eng.reverse_Phi1(0, i0, i0, d0, d0, False, False)
        assert np.array_equal(eng.H1_adj, np.zeros(rows * width)) and len(eng.M1_adj) == 0
        eng.H1_adj = d0
        eng.reverse_H1(0); eng.reverse_M0(0, i0); eng.reverse_A0_scaled(0, i0, i0, i0, d0, d0); eng.reverse_A0(0, i0, i0, i0, d0, d0)
        F, V = eng.reduce_forces(rows, i0, virial=True)
        assert not F.any() and not V.any() and len(eng.node_forces) == 0

    print(f"K={K} L_max={L_max} {dtype}", flush=True)
    eng = MACE(path, dtype)
    stages(eng)
    eng.compute_node_energies_forces(*H.call_args(ea))
    E, F, H1 = np.array(eng.node_energies), np.array(eng.node_forces), np.array(eng.H1)
    fresh = MACE(path, dtype)
    fresh.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(E, fresh.node_energies) and np.array_equal(F, fresh.node_forces)
    # ghosts only: layer 0 for all of them, layer 1 for none
    eng.compute_ghosted(0, n, *H.call_args(ea)[1:])
    assert len(eng.node_energies) == 0 and len(eng.H2) == 0
    assert not np.array(eng.node_forces).any() and len(eng.node_forces) == 3 * len(ea["r"])
    assert np.abs(np.array(eng.H1) - H1).max() <= (1e-12 if dtype == "float64" else 1e-4) * np.abs(H1).max()
    assert not np.array(eng.H1_adj).any()
    stages(eng)
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert np.array_equal(E, eng.node_energies) and np.array_equal(F, eng.node_forces)
