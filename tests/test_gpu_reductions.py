"""Caller-side reductions on the GPU: which edges they cover after the calls that may come before them."""
import ctypes as C

import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _virial(xyz, forces):
    d, f = np.asarray(xyz).reshape(-1, 3), np.asarray(forces).reshape(-1, 3)
    W = 0.5 * (d.T @ f + f.T @ d)
    return W[[0, 1, 2, 0, 0, 1], [0, 1, 2, 1, 2, 2]]


def _no_alloc(eng, atoms, senders, forces, virial):
    import torch
    from symmetrix_amd import _lib
    p = lambda t: C.c_void_p(t.data_ptr()) if t is not None else None
    rc = _lib.lib().smx_reduce_forces_device_noalloc(eng._h, atoms, p(senders), p(forces), p(virial), None)
    assert rc == 0, _lib.lib().smx_last_error().decode()
    torch.cuda.synchronize()


def test_virial_covers_every_edge_after_a_stage_call_over_leading_nodes(tmp_models):
    """A stage may cover the leading nodes of a longer edge list.  The forces of all edges are there, and all of them belong
    to the virial (a sum of E terms in double, in another order: 1e-13 of the sum of magnitudes is a bound for any E here)."""
    import torch
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=16, L_max=1, n_pts=48, seed=23, zbl=True)
    eng = MACE(H.write_model(model, tmp_models / "leading.json"))
    pos, cell, sp = H.small_system(60, seed=5)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, nt, nn, ni, nty, xyz, r = H.call_args(ea)
    senders = torch.from_numpy(ni).cuda()
    eng.compute_node_energies_forces(N, nt, nn, ni, nty, xyz, r)
    for leading in (N, 23, 1, 0):
        print(f"{leading} of {N} nodes, {len(r)} edges", flush=True)
        eng.compute_ZBL(leading, nt[:leading], nn[:leading], nty, r, xyz)
        f = eng.node_forces
        want, bound = _virial(xyz, f), 1e-13 * np.abs(_virial(np.abs(xyz), np.abs(f))).max()
        F, V = eng.reduce_forces(N, ni, virial=True)
        assert np.abs(V - want).max() <= bound
        dF = torch.zeros((N, 3), dtype=torch.float64, device="cuda:0"); dV = torch.zeros(6, dtype=torch.float64, device="cuda:0")
        _no_alloc(eng, N, senders, dF, dV)
        assert np.abs(dV.cpu().numpy() - want).max() <= bound
        assert np.array_equal(dF.cpu().numpy(), F)
        dV.zero_()
        _no_alloc(eng, N, senders, None, dV)
        assert np.abs(dV.cpu().numpy() - want).max() <= bound


def test_no_alloc_virial_of_a_skipped_evaluation_is_nan(tmp_models):
    """Device arrays that fail their checks leave empty lists: the virial says so as the forces do."""
    import torch
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=16, L_max=1, n_pts=48, seed=23)
    eng = MACE(H.write_model(model, tmp_models / "skipped.json"))
    pos, cell, sp = H.small_system(40, seed=5)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d = [t(ea[k]) for k in ("node_types", "num_neigh", "neigh_indices", "neigh_types", "xyz", "r")]
    senders = d[2].clone()
    d[3][0] = 3                      # a species the model does not have
    eng.compute_device(len(sp), *[x.data_ptr() for x in d], len(ea["r"]))
    dF = torch.zeros((len(sp), 3), dtype=torch.float64, device="cuda:0"); dV = torch.zeros(6, dtype=torch.float64, device="cuda:0")
    _no_alloc(eng, len(sp), senders, dF, dV)
    assert torch.isnan(dV).all() and torch.isnan(dF).any()
    dV.zero_()
    _no_alloc(eng, len(sp), senders, None, dV)
    assert torch.isnan(dV).all()
    with pytest.raises(ValueError):
        eng.synchronize()
