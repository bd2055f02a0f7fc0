"""The virial, whose partial sums the last block of the reduction adds up: one block, remainders of the four atoms of a block, more blocks
than a wavefront has lanes, and more atoms than there are blocks for."""
import numpy as np
import pytest

from tests import helpers as H
from tests.test_gpu_reductions import _virial

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 5, 255, 257, 2049, 8193])
def test_virial_of_any_number_of_blocks(tmp_models, n):
    """Against a sum in another order (of magnitudes, 1e-13 is a bound for n terms in double), and the same bits every time."""
    import torch
    assert torch.cuda.is_available()
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=16, L_max=0, n_pts=16, seed=7, r_cut=3.0, pair=False)
    eng = MACE(H.write_model(model, tmp_models / "virial.json"))
    rng = np.random.default_rng(n)
    species = rng.integers(0, 3, n).astype(np.int32)
    j = rng.permutation(n).astype(np.int32)
    r = rng.uniform(0.8, 2.9, n)
    u = rng.normal(size=(n, 3))
    xyz = u * (r / np.linalg.norm(u, axis=1))[:, None]
    print(f"{n} atoms", flush=True)
    eng.compute_node_energies_forces(n, species, np.ones(n, np.int32), j, species[j], xyz.ravel(), r)
    f = eng.node_forces
    first = None
    for _ in range(3):
        F, V = eng.reduce_forces(n, j, virial=True)
        assert np.abs(V - _virial(xyz, f)).max() <= 1e-13 * np.abs(_virial(np.abs(xyz), np.abs(f))).max()
        assert first is None or np.array_equal(V, first)
        first = V
        assert np.array_equal(eng.reduce_forces(n, j), F)      # (without a virial: no ticket is taken)
