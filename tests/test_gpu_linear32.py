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


# 16 columns per wavefront (few atoms) and 32 at 128 channels, two and three blocks of columns at 192 to 288; 96 channels; remainders of a row tile
@pytest.mark.parametrize("K,L_max,n", [(128, 0, 513), (128, 0, 2049), (128, 1, 527), (128, 1, 2065), (128, 2, 1025), (256, 0, 640), (96, 0, 1025), (96, 2, 1039), (192, 0, 1025), (288, 1, 1030)])
def test_products(tmp_models, K, L_max, n):
    """What is left out of a product is at most 1.002 2^-24 of it, its factors are exact, and a sum of `inner` terms is rounded 6 / 32
    times a term: (6 inner / 32 + 2) 2^-24 of the sum of magnitudes at most."""
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


@pytest.mark.parametrize("K,L_max,n", [(128, 0, 2049), (128, 1, 1040), (128, 2, 1024), (256, 0, 2049)])
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


def _check_range(got, x, w, what):
    """As in test_products where the parts form a sum; numbers above 2^103 and sums above 2^80 are sums in single precision, of a rounding
    a term.  A rounding is half of the smallest number of single precision, 2^-149, at least: one of them at the end of a sum of parts, one a
    term else."""
    K = w.shape[0]
    with np.errstate(invalid="ignore", over="ignore"):
        ref, size = x @ w, np.abs(x) @ np.abs(w)
        plain = (np.abs(x) >= 2.0 ** 103).any(-1)[..., None] | (np.abs(w) >= 2.0 ** 103).any(0) | (size >= 2.0 ** 79)
        assert np.array_equal(np.isnan(got), np.isnan(ref)), what
        assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)]), what
        ok = np.isfinite(ref) & (size <= 3.4e38)      # (single precision may not hold a larger sum on the way)
        err = np.abs(got - ref) - np.where(plain, K, 6 * K / 32 + 2) * 2.0 ** -24 * size
    assert (err <= np.where(plain, K, 1) * 2.0 ** -150)[ok].all(), what


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("K", [96, 128])
def test_range(tmp_models, K, weights):
    """Rows of all sizes that single precision holds, infinities and NaN; columns of weights of all sizes; the numbers whose products lose most."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    n = 1030
    model = H.tiny_model(K=K, L_max=0, T=(1, 6, 8), n_pts=16, seed=K, r_cut=3.0, pair=False, density=False)
    W = [np.array(w).reshape(K, K) for w in model["A1_weights"]]
    if weights:
        for c, power in enumerate([-140, -122, -112, -100, 76, 100, 110, 120]):
            for w in W:
                w[:, c] *= 2.0 ** power
    worst = 1.0038986206      # of its square 2^-24.01 is left out
    for w in W:
        w[:, 9] = worst
    model["A1_weights"] = [w.ravel().tolist() for w in W]
    W = [w.astype(np.float32).astype(np.float64) for w in W]
    eng = MACE(H.write_model(model, tmp_models / f"linear32_range_{K}_{weights}.json"), "float32")
    rng = np.random.default_rng(K)
    x = rng.normal(size=(n, 16, K))
    for i, power in ((0, -140), (1, -126), (17, -112), (18, -100), (33, 76), (34, 100), (50, 120)):
        x[i] *= 2.0 ** power
    x[51] = 0.0
    x[52] = worst
    x[66, :, 7] = np.inf
    x[67, :, 8] = -np.inf
    x[82, :, 9] = np.nan
    x[98, :, 10] = np.finfo(np.float32).max
    x[114, :, ::2] *= 2.0 ** 110
    x[114, :, 1::2] *= 2.0 ** -130
    x = x.astype(np.float32).astype(np.float64)
    print(f"K={K} atoms={n} weights={weights}", flush=True)
    eng.Phi1 = x.ravel()
    eng.compute_A1(n)
    A1 = np.array(eng.A1).reshape(n, 16, K)
    eng.A1_adj = x.ravel()
    eng.reverse_A1(n)
    Phi1_adj = np.array(eng.Phi1_adj).reshape(n, 16, K)
    for l in range(4):
        m = slice(l * l, (l + 1) ** 2)
        _check_range(A1[:, m], x[:, m], W[l], "A1")
        _check_range(Phi1_adj[:, m], x[:, m], W[l].T, "Phi1_adj")


def test_small_factors(tmp_models):
    """Energies so small that the factors of the adjoint rows are next to the smallest numbers."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    K, n = 128, 528
    model = H.tiny_model(K=K, L_max=0, T=(1, 6, 8), n_pts=16, seed=7, r_cut=3.0, pair=False, density=False)
    for name in ("readout_1_weights", "readout_2_weights_2"):
        model[name] = (np.array(model[name]) * 2.0 ** -118).tolist()
    eng = MACE(H.write_model(model, tmp_models / "linear32_small.json"), "float32")
    eng.set_profiling(True)
    ea, _ = _system(model, n)
    eng.compute_node_energies_forces(*H.call_args(ea))
    get = lambda name: np.array(getattr(eng, name)).reshape(n, -1, K)
    A1_adj, Phi1_adj = get("A1_adj"), get("Phi1_adj")
    print(f"largest factor {np.abs(A1_adj).max():.2e}, edges {len(ea['r'])}", flush=True)
    assert 0.0 < np.abs(A1_adj).max() < 2.0 ** -100
    for l in range(4):
        w = np.array(model["A1_weights"][l], dtype=np.float32).astype(np.float64).reshape(K, K)
        m = slice(l * l, (l + 1) ** 2)
        # (A1_adj is rounded to the smallest number, and the operand is a product like it)
        err = np.abs(Phi1_adj[:, m] - A1_adj[:, m] @ w.T) - (6 * K / 32 + 3) * 2.0 ** -24 * (np.abs(A1_adj[:, m]) @ np.abs(w.T))
        assert (err <= 2.0 ** -149 * (2 + np.abs(w.T).sum(0))).all()
