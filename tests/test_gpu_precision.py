"""Precision of sums on the GPU where a comparison of whole evaluations would not show it."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layer", [0, 1])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160])
def test_force_sums_over_channels_are_in_double(tmp_models, K, layer):
    """The force of an edge is a sum over all channels.  With the same radial table and sender features in every channel, two
    channels of opposite adjoints give forces that cancel exactly, and a third of 2^-20 of their size has to be left: a sum in
    single precision keeps 2^-4 of it, one in double all of it (24 + 20 bits).  The three are in different sixteens and
    eights of channels, so no two of them are among those that one lane or its partner adds."""
    import torch
    from symmetrix_amd.mace import MACE
    assert torch.cuda.is_available()
    model = H.tiny_model(K=K, L_max=0, n_pts=48, seed=7, pair=False)
    for key in (f"radial_spline_values_{layer}", f"radial_spline_derivs_{layer}"):
        model[key] = [[row[n // K * K] for n in range(len(row))] for row in model[key]]
    model["H0_weights"] = [1.0] * len(model["H0_weights"])
    model["A0_weights"] = [[np.eye(K).ravel().tolist() for _ in range(4)] for _ in range(len(model["A0_weights"]))]
    eng = MACE(H.write_model(model, tmp_models / f"cancel_{K}_{layer}.json"), "float32")
    pos, cell, sp = H.small_system(50, seed=3)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, nt, nn, ni, nty, xyz, r = H.call_args(ea)
    eng.compute_node_energies_forces(N, nt, nn, ni, nty, xyz, r)
    a = np.random.default_rng(1).normal(size=(N, 16)).astype(np.float32).astype(np.float64)
    got = []
    for large in (1.0, 0.0):
        adj = np.zeros((N, 16, K))
        adj[:, :, 0], adj[:, :, 9], adj[:, :, K - 6] = large * a, 2.0 ** -20 * a, -large * a
        eng.node_forces = np.zeros(3 * len(r))
        if layer == 0:
            eng.A0_adj = adj
            eng.reverse_A0(N, nt, nn, nty, xyz, r)
        else:
            eng.H1 = np.ones(N * K)
            eng.Phi1_adj = adj
            eng.reverse_Phi1(N, nn, ni, xyz, r, True, True)
        got.append(eng.node_forces)
    print(f"K={K} layer {layer}: {len(r)} edges, largest force {np.abs(got[1]).max():.3e}", flush=True)
    assert np.abs(got[1]).max() > 0.0
    assert np.abs(got[0] - got[1]).max() <= 2.0 ** -30 * np.abs(got[1]).max()
