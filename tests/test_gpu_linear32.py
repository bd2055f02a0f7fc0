"""The A-basis linears in single precision on bf16 parts: products against 64 bits, element by element, and a contraction behind them."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _system(model, n):
    pos, cell, sp = H.small_system(n, density=0.05, seed=n)
    return H.edges_of(pos, cell, sp, model["r_cut"])[1], sp


def _engine(tmp_models, K, L_max):
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, T=(1, 6, 8), n_pts=16, seed=K + L_max, r_cut=3.0, pair=False, density=False)
    eng = MACE(H.write_model(model, tmp_models / f"linear32_{K}_{L_max}.json"), "float32")
    eng.set_profiling(True)      # small systems would take chains of stages otherwise
    return model, eng


# 16 columns per wavefront (few atoms) and 32 at 128 channels, two blocks of columns at 256; 96 channels; remainders of a row tile
@pytest.mark.parametrize("K,L_max,n", [(128, 0, 513), (128, 0, 2049), (128, 1, 527), (128, 1, 2065), (128, 2, 1025), (256, 0, 640), (96, 0, 1025), (96, 2, 1039)])
def test_products(tmp_models, K, L_max, n):
    """What is left out of a product is below 2^-25 of it, its factors are exact, and a sum of `inner` terms is rounded 6 / 32 times a
    term and once more: (6 inner / 32 + 2) 2^-24 of the sum of magnitudes at most."""
    model, eng = _engine(tmp_models, K, L_max)
    ea, sp = _system(model, n)
    print(f"K={K} L_max={L_max} atoms={n} edges={len(ea['r'])}", flush=True)
    eng.compute_node_energies_forces(*H.call_args(ea))
    get = lambda name: np.array(getattr(eng, name)).reshape(n, -1, K)
    w32 = lambda w: np.array(w, dtype=np.float32).astype(np.float64)

    def check(got, x, w, what):
        ref, size = x @ w, np.abs(x) @ np.abs(w)
        assert (np.abs(got - ref) <= (6 * w.shape[0] / 32 + 2) * 2.0 ** -24 * size).all(), what

    if L_max == 0 and n >= 1024:      # (else the adjoint has been written over Phi0)
        Phi0, A0 = get("Phi0"), get("A0")
        for t in range(3):
            for l in range(4):
                check(A0[sp == t, l * l:(l + 1) ** 2], Phi0[sp == t, l * l:(l + 1) ** 2], w32(model["A0_weights"][t][l]).reshape(K, K), "A0")
    Phi1, A1, A1_adj, Phi1_adj = get("Phi1"), get("A1"), get("A1_adj"), get("Phi1_adj")
    off = 0
    for l in range(4):
        w = w32(model["A1_weights"][l]).reshape(-1, K)
        ne = len(w) // K
        for m in range(2 * l + 1):
            check(A1[:, l * l + m], Phi1[:, off:off + ne].reshape(n, -1), w, "A1")
            # (the operand is M1_grad . M1_adj, rounded as A1_adj is)
            for e in range(ne):
                check(Phi1_adj[:, off + e], A1_adj[:, l * l + m], w[e * K:(e + 1) * K].T, "Phi1_adj")
            off += ne


@pytest.mark.parametrize("K,L_max,n", [(128, 0, 2049), (128, 1, 1040), (128, 2, 1024)])
def test_contraction(tmp_models, K, L_max, n):
    from oracle.oracle import OracleMACE
    from tests.test_gpu_parity import _compare
    model, eng = _engine(tmp_models, K, L_max)
    ea, _ = _system(model, n)
    print(f"K={K} L_max={L_max} atoms={n} edges={len(ea['r'])}", flush=True)
    orc = OracleMACE(model)
    orc.compute_node_energies_forces(*H.call_args(ea))
    eng.compute_node_energies_forces(*H.call_args(ea))
    assert eng.stage_times()["M1"] == 0.0      # in the launch of the linear
    _compare(orc, eng, "float32")
