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
    assert torch.isnan(dV).all() and torch.isnan(dF).all()
    dV.zero_()
    _no_alloc(eng, len(sp), senders, None, dV)
    assert torch.isnan(dV).all()
    with pytest.raises(ValueError):
        eng.synchronize()
    # the reason is reported once; the sums stay NaN, whichever sender lists they are formed from
    owners = np.arange(len(sp), dtype=np.int32)
    for kw in (dict(), dict(receiver_atom=owners)):
        F, V = eng.reduce_forces(len(sp), ea["neigh_indices"], virial=True, **kw)
        assert np.isnan(F).all() and np.isnan(V).all()
    # stage calls do not take up the unchecked arrays
    with pytest.raises(ValueError, match="before its inputs exist"):
        eng.compute_Phi1(len(sp), ea["num_neigh"], ea["neigh_indices"])


def test_nothing_is_reduced_after_a_refused_evaluation(tmp_models):
    """Host arrays that fail their checks: the call raises, and so does every use of what it would have computed, until an
    evaluation or a sequence of stage calls has made new forces."""
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=16, L_max=0, n_pts=48, seed=23, zbl=True)
    eng = MACE(H.write_model(model, tmp_models / "refused.json"))
    pos, cell, sp = H.small_system(30, seed=5)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, nt, nn, ni, nty, xyz, r = H.call_args(ea)
    owners = np.arange(N, dtype=np.int32)
    good = (N, nt, nn, ni, nty, xyz, r)
    eng.compute_node_energies_forces(*good)
    f_ref, (F_ref, V_ref) = eng.node_forces, eng.reduce_forces(N, ni, virial=True)
    assert np.abs(F_ref).max() > 0.0
    for key, at, value in (("species of an edge", 4, 3), ("species of a node", 1, -1), ("sender", 3, N), ("length", 6, 2.0 * model["r_cut"])):
        bad = list(good)
        bad[at] = good[at].copy(); bad[at][7] = value
        print(key, flush=True)
        with pytest.raises(ValueError):
            eng.compute_node_energies_forces(*bad)
        for kw in (dict(), dict(virial=True), dict(receiver_atom=owners)):
            with pytest.raises(ValueError, match="refused"):
                eng.reduce_forces(N, ni, **kw)
        with pytest.raises(ValueError, match="before its inputs exist"):
            eng.reverse_Phi1(N, nn, ni, xyz, r)      # (species are those of the refused call)
        # forces made by stage calls alone
        eng.compute_ZBL(N, nt, nn, nty, r, xyz)
        f = eng.node_forces
        assert np.isfinite(f).all() and np.abs(f).max() > 0.0
        assert np.allclose(eng.reduce_forces(N, ni), H.atom_forces(nl, f, N), rtol=0, atol=1e-12 * max(1.0, np.abs(f).max()))
        eng.compute_node_energies_forces(*good)
        assert np.array_equal(eng.node_forces, f_ref)
        F, V = eng.reduce_forces(N, ni, virial=True)
        assert np.array_equal(F, F_ref) and np.array_equal(V, V_ref)


def test_stage_inputs_that_were_refused_are_not_used_later(tmp_models):
    """A stage call that refuses its arrays leaves none of them behind: later stages ask for them, and go on once they have
    been given."""
    from symmetrix_amd.mace import MACE
    model = H.tiny_model(K=16, L_max=1, n_pts=48, seed=23)
    eng = MACE(H.write_model(model, tmp_models / "stage_refused.json"))
    pos, cell, sp = H.small_system(30, seed=5)
    nl, ea = H.edges_of(pos, cell, sp, model["r_cut"])
    N, nt, nn, ni, nty, xyz, r = H.call_args(ea)

    def through_phi1():
        eng.compute_Y(xyz); eng.compute_R0(N, nt, nn, nty, r); eng.compute_A0(N, nt, nn, nty)
        eng.compute_M0(N, nt); eng.compute_H1(N); eng.compute_R1(N, nt, nn, nty, r); eng.compute_Phi1(N, nn, ni)
        return eng.Phi1

    ref = through_phi1()
    for what, bad in (("species of the nodes", (nt + 3, nn, nty, r)), ("species of the edges", (nt, nn, nty - 1, r)),
                      ("lengths", (nt, nn, nty, r + model["r_cut"]))):
        print(what, flush=True)
        with pytest.raises(ValueError):
            eng.compute_R1(N, *bad)
        with pytest.raises(ValueError, match="before its inputs exist"):
            eng.compute_Phi1(N, nn, ni)
        eng.compute_R1(N, nt, nn, nty, r)
        eng.compute_Phi1(N, nn, ni)
        assert np.array_equal(eng.Phi1, ref)
    with pytest.raises(ValueError):
        eng.compute_Phi1(N, nn, ni + N)
    assert np.array_equal(through_phi1(), ref)
