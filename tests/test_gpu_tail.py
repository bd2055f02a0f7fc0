"""H2, the readouts and reverse_H2 in one launch: blocks with one row tile and with several, species with no atom, one atom and
remainders of a tile, every number of channels that the launch takes."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

# one tile; more than one tile per block (256 blocks at 128 channels, 1 024 at 32, 512 else)
SIZES = {32: 16 * 1024 + 40, 48: 16 * 512 + 40, 64: 16 * 512 + 40, 96: 16 * 512 + 40, 128: 16 * 256 + 40}


def _evaluated(tmp_models, K, n, dtype, T, L_max):
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, T=T, n_pts=16, seed=K + n, r_cut=3.0, pair=False)
    eng = MACE(H.write_model(model, tmp_models / f"tail_{K}_{n}_{len(T)}.json"), dtype)
    rng = np.random.default_rng(n + K)
    species = rng.integers(0, len(T), n)
    species[species == 1] = 0                 # the second species: one atom, the last one: none
    species[species == len(T) - 1] = 2 % (len(T) - 1)
    species[n // 2] = 1
    # three neighbours each, all from the first quarter: no message reaches the other atoms
    j = rng.integers(0, max(n // 4, 1), 3 * n)
    r = rng.uniform(0.8, 2.9, 3 * n)
    u = rng.normal(size=(3 * n, 3))
    xyz = u * (r / np.linalg.norm(u, axis=1))[:, None]
    print(f"K={K} atoms={n} species={len(T)} {dtype}", flush=True)
    eng.set_profiling(True)                   # small systems would take chains of stages otherwise
    eng.compute_node_energies_forces(n, species.astype(np.int32), np.full(n, 3, np.int32), j.astype(np.int32),
                                     species[j].astype(np.int32), xyz, r)
    return model, eng, species


def _check(model, eng, species, dtype):
    """Against the same formulas in double precision on the H1 and M1 that the evaluation left.  What the launch does in double
    (all of it, from these arrays) differs by the order of sums of at most 256 products, three in a row: 3 * 256 * 2^-53 = 9e-14 of
    the sum of magnitudes; results kept in single precision are rounded to it, 2^-24 of each (H1_adj twice)."""
    n, K = len(species), model["num_channels"]
    H1 = np.asarray(eng.H1, float).reshape(n, -1, K)
    M1 = np.asarray(eng.M1, float).reshape(n, K)
    WH = np.asarray(model["H2_weights_for_H1"]).reshape(-1, K, K)
    WM = np.asarray(model["H2_weights_for_M1"]).reshape(K, K)
    w1 = np.asarray(model["readout_1_weights"])
    W1 = np.asarray(model["readout_2_weights_1"]).reshape(16, K)
    w2, c = np.asarray(model["readout_2_weights_2"]), model["readout_2_scale_factor"]
    H2, back = np.empty((n, K)), np.empty((n, K))
    for t in np.unique(species):
        H2[species == t] = H1[species == t, 0] @ WH[t] + M1[species == t] @ WM
    hid = H2 @ W1.T
    sig = 1.0 / (1.0 + np.exp(-hid))
    E = np.asarray(model["atomic_energies"])[species] + H1[:, 0] @ w1 + (c * hid * sig) @ w2
    H2_adj = (w2 * c * (sig + hid * sig * (1 - sig))) @ W1
    for t in np.unique(species):
        back[species == t] = H2_adj[species == t] @ WH[t].T
    single = 0.0 if dtype == "float64" else 2.0 ** -24
    seed = w1 if dtype == "float64" else w1.astype(np.float32).astype(float)

    def close(got, want, scale, rounding, name):
        assert np.isfinite(got).all(), name
        assert np.abs(got - want).max() <= (1e-13 + rounding) * scale, name

    def size(*products):
        return max(np.abs(a).max() * np.abs(b).sum(axis=-2).max() for a, b in products)

    s_H2 = size((H1[:, 0], WH), (M1, WM))
    close(np.asarray(eng.H2).reshape(n, K), H2, s_H2, 0.0, "H2")
    # the hidden units pass the error of H2 on through W1 (and c, w2), the adjoints through W1 and the weights once more
    s_hid = s_H2 * np.abs(W1).sum(axis=1).max() * 1.1 * c * np.abs(w2).sum()
    close(np.asarray(eng.node_energies), E, s_hid + np.abs(E).max(), 0.0, "node_energies")
    s_adj = (s_hid + c * np.abs(w2).sum()) * np.abs(W1).max()
    close(np.asarray(eng.H2_adj).reshape(n, K), H2_adj, s_adj, 0.0, "H2_adj")
    M1_adj = H2_adj @ WM.T
    close(np.asarray(eng.M1_adj, float).reshape(n, K), M1_adj, s_adj * np.abs(WM).sum(axis=1).max(), single, "M1_adj")
    H1_adj = np.asarray(eng.H1_adj, float).reshape(n, -1, K)[max(n // 4, 1):]
    close(H1_adj[:, 0], seed + back[max(n // 4, 1):], s_adj * np.abs(WH).sum(axis=2).max() + np.abs(w1).max(), 2 * single, "H1_adj")
    assert not H1_adj[:, 1:].any()


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("K", sorted(SIZES))
def test_tail_against_the_formulas(tmp_models, K, dtype):
    for n, L_max in ((17, 1), (SIZES[K], 0)):
        _check(*_evaluated(tmp_models, K, n, dtype, (1, 6, 7, 8), L_max), dtype)


def test_tail_with_more_species_than_lanes(tmp_models):
    """The tile of a block is looked up 64 species at a time."""
    _check(*_evaluated(tmp_models, 32, 300, "float64", tuple(range(1, 71)), 0), "float64")
