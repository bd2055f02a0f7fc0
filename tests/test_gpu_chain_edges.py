"""Aggregations and their adjoints inside the chains of small systems: receivers whose edges end on either side of a round of eight, of
the 120 and 80 that a block takes at a time, or that have none; and where the rule ends."""
import numpy as np
import pytest

from tests import helpers as H
from tests.test_gpu_chains import ARRAYS, _compare

pytestmark = pytest.mark.gpu

DEGREES = [0, 1, 7, 8, 9, 79, 80, 81, 119, 120, 121, 248]


def _both(tmp_models, K, L_max, dtype, degree, seed):
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=K, L_max=L_max, n_pts=48, seed=5 * K + L_max, r_cut=3.5, pair=False)
    eng = MACE(H.write_model(model, tmp_models / f"chain_edges_{K}_{L_max}.json"), dtype)
    rng = np.random.default_rng(seed)
    N, E = len(degree), int(np.sum(degree))
    species = rng.integers(0, 3, N).astype(np.int32)
    senders = rng.integers(0, N, E).astype(np.int32)
    x = rng.normal(size=(E, 3))
    x *= (rng.uniform(1.0, 3.4, E) / np.linalg.norm(x, axis=1))[:, None]
    print(f"K={K} L_max={L_max} atoms={N} edges={E} {dtype}", flush=True)
    out = []
    for per_stage in (False, True):
        eng.set_profiling(per_stage)
        eng.compute_node_energies_forces(N, species, np.asarray(degree, np.int32), senders, species[senders], x.ravel(), np.linalg.norm(x, axis=1))
        out.append({name: np.array(getattr(eng, name)) for name in ARRAYS})
    return out


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("L_max", [0, 1, 2])
@pytest.mark.parametrize("K", [32, 64, 96, 128])
def test_receivers_of_all_lengths(tmp_models, K, L_max, dtype):
    _compare(*_both(tmp_models, K, L_max, dtype, np.random.default_rng(K).permutation(DEGREES), K + L_max), dtype)


@pytest.mark.parametrize("K,n,dtype", [(96, 256, "float64"), (96, 257, "float64"), (128, 257, "float32"), (96, 300, "float32"), (64, 300, "float64")])
def test_sizes_at_the_rule(tmp_models, K, n, dtype):
    """With the edges and without, where a CU holds one block and there are as many atoms as CUs, or one more."""
    degree = np.random.default_rng(n).integers(0, 12, n)
    _compare(*_both(tmp_models, K, 0, dtype, degree, n), dtype)
