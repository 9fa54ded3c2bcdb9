"""Empty and degenerate inputs on the GPU path, against the CPU oracle: a structure without atoms inside a batch, atoms
without neighbours, a cell with one atom, rows of length zero in the force / virial operators.  The reference handles
them through the same loops as everything else (a row of numneigh = 0 contributes its bias energy and no force,
nep.h:379-529, linearMtp.h:228-352; a structure with binum = 0 keeps the zeros its outputs start from)."""
import numpy as np
import pytest

from ai2pot_amd import mtp_param, synth
from test_gpu_mtp import close, gpu_efv
from test_gpu_nep import check, run_gpu

pytestmark = pytest.mark.gpu


def _gas(oracle, n, box, nt, seed, rcut, dmin, umax=120):
    lat, pos = synth.random_packed(n, [box, box, box], dmin, seed)
    return oracle.nblist(lat, synth.rng_randint(seed + 1, n, nt), pos, rcut, umax)


def _batch_with_an_empty_structure(oracle, nt, rcut):
    """structure 0: dense; structure 1: no atoms at all; structure 2: a thin gas in which most atoms have no neighbour"""
    dense = _gas(oracle, 48, 9.5, nt, 71, rcut, 2.1)
    gas = _gas(oracle, 12, 40.0, nt, 73, rcut, 5.0)
    assert (gas[2] == 0).sum() >= 6                  # atoms without neighbours
    nb = synth.pack_batch([dense, dense, gas])
    nb["binum"][1] = 0                               # every row of structure 1 is padding
    nb["bnumneigh"][1] = 0
    return nb


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_nep_empty_structure_and_isolated_atoms(oracle, np_dtype):
    m = synth.nep_model()
    nb = _batch_with_an_empty_structure(oracle, 3, 7.0)
    nb = dict(nb, brcs=nb["brcs"].astype(np_dtype))
    out = run_gpu(m, nb, np_dtype)
    ref = oracle.nep_efv(m, nb, np_dtype)
    check(out, ref, np_dtype)
    e, f, v = out
    assert e[1] == 0 and not f[1].any() and not v[1].any()
    # an atom without neighbours: its energy is the network at q = 0 plus the bias, its force is zero
    lone = np.flatnonzero(nb["bnumneigh"][2, :nb["binum"][2]] == 0)
    assert not f[2, nb["bilist"][2, lone]].any()


@pytest.mark.parametrize("level", [10, 16, 20])
def test_mtp_empty_structure_and_isolated_atoms(oracle, level):
    nt = 2
    m = synth.mtp_model(mtp_param.mtp_param(level), nt, 8, 5.0, 1.0, 3100 + level, lo=-0.05, hi=0.05)
    nb = _batch_with_an_empty_structure(oracle, nt, 5.0)
    e, f, v = gpu_efv(m, nb)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)
    assert e[1] == 0 and not f[1].any() and not v[1].any()
    # all atoms of a species isolated: the energy is the sum of their biases
    gas = _gas(oracle, 6, 60.0, nt, 75, 5.0, 12.0)
    assert not gas[2].any()
    nb1 = synth.pack_batch([gas])
    e1, f1, v1 = gpu_efv(m, nb1)
    assert abs(e1[0] - m["type_bias"][gas[5]].sum()) <= 1e-12 * max(1.0, abs(e1[0]))
    assert not f1.any() and not v1.any()


def test_mtp_loss_with_isolated_atoms(oracle):
    """Training step on a batch that holds a structure of isolated atoms: its coefficient gradient is zero, the
    gradients of the linear coefficients and the bias follow the energy error alone."""
    from test_gpu_mtp import gpu_loss
    nt = 2
    m = synth.mtp_model(mtp_param.mtp_param(10), nt, 8, 5.0, 1.0, 3110, lo=-0.05, hi=0.05)
    dense = _gas(oracle, 40, 9.0, nt, 77, 5.0, 2.1)
    gas = _gas(oracle, 9, 60.0, nt, 79, 5.0, 12.0)
    assert not gas[2].any()
    nb = synth.pack_batch([dense, gas])
    B, P = nb["bilist"].shape
    rng = np.random.default_rng(3)
    labels = dict(energy=rng.normal(size=B), force=rng.normal(size=(B, P, 3)), virial=rng.normal(size=(B, 9)))
    w = (1.0, 0.7, 0.3)
    ref = oracle.mtp_loss_step(m, nb, w, labels)
    got = gpu_loss(m, nb, labels, w)
    for k in ("bloss", "rmse", "energy", "force", "virial", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], ref[k]), k
    assert not got["dcoeffs"][1].any()


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_list_of_one_atom_and_of_a_thin_gas(oracle, np_dtype):
    """One atom in a cell wider than the cutoff has no neighbour; in a cell narrower than the cutoff its own images are
    its neighbours.  Compared with the oracle entry by entry."""
    import torch
    from ai2pot_amd import nblist
    dev = torch.device("cuda:0")
    cases = [(np.eye(3) * 30.0, np.array([[1.0, 2.0, 3.0]]), 5.0),
             (np.diag([3.1, 30.0, 2.9]), np.array([[0.5, 0.5, 0.5]]), 5.0),
             (np.eye(3) * 25.0, np.array([[1.0, 1.0, 1.0], [2.5, 1.0, 1.0], [20.0, 20.0, 20.0]]), 4.0)]
    for lat, pos, rcut in cases:
        ty = np.zeros(len(pos), np.int32)
        for sort in (False, True):
            ref = oracle.nblist(lat.astype(np_dtype), ty, pos.astype(np_dtype), rcut, 40, sort=sort)
            out = nblist.find_info4mlff_device(lat.astype(np_dtype), torch.from_numpy(ty).to(dev),
                                               torch.from_numpy(pos.astype(np_dtype)).to(dev), rcut, 40, sort=sort)
            got = [o.cpu().numpy() if hasattr(o, "cpu") else o for o in out]
            assert got[0] == ref[0] and got[6] == ref[6]
            for g, r in zip(got[1:6], ref[1:6]):
                assert g.dtype == r.dtype and np.array_equal(g, r)


def test_force_and_virial_operators_with_rows_of_length_zero(oracle):
    import torch
    from ai2pot_amd import ops
    rng = np.random.default_rng(11)
    B, P, U = 2, 7, 5
    numneigh = rng.integers(0, U + 1, size=(B, P)).astype(np.int32)
    numneigh[0, :3] = 0
    numneigh[1] = 0                                   # a structure whose rows are all empty
    first = rng.integers(0, P, size=(B, P, U)).astype(np.int32)
    dei = rng.normal(size=(B, P, U, 3))
    rcs = rng.normal(size=(B, P, U, 3))
    binum = np.full(B, P, np.int32)
    ilist = np.tile(np.arange(P, dtype=np.int32), (B, 1))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    f = ops.ForceSrOp(t(binum), t(ilist), t(numneigh), t(first), 0, U, t(dei))[0].cpu().numpy()
    v = ops.VirialSrOp(t(numneigh), t(rcs), U, t(dei))[0].cpu().numpy()
    for b in range(B):
        fr, _ = oracle.fvt_force(ilist[b], numneigh[b], first[b], 0, dei[b])
        vr, _, _ = oracle.fvt_virial(numneigh[b], rcs[b], dei[b])
        assert np.abs(f[b] - fr).max() <= 1e-13 * max(1.0, np.abs(fr).max())
        assert np.abs(v[b].reshape(9) - vr).max() <= 1e-13 * max(1.0, np.abs(vr).max())
    assert not f[1].any() and not v[1].any()


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_device_resident_step_on_a_thin_gas(oracle, np_dtype):
    """Compact lists + NEP on them where most rows are empty and no atom has a neighbour inside the angular cutoff;
    then one atom alone in its cell."""
    from test_gpu_nep_gather import _calc, _check, _step
    m = synth.nep_model(seed=3301)
    n = 40
    lat, pos = synth.random_packed(n, [60.0, 61.0, 62.0], 4.5, 331)
    ty = synth.rng_randint(332, n, 3)
    calc = _calc(m, lat, ty, n, np_dtype, path="gather")
    out = _step(calc, pos, np_dtype)
    ref = oracle.nblist(lat.astype(np_dtype), ty, pos.astype(np_dtype), 7.0, 200)
    assert (ref[2] == 0).sum() >= n // 2 and ref[2].any()
    assert np.array_equal(calc.numneigh.cpu().numpy(), ref[2])
    assert np.array_equal(calc.firstneigh.cpu().numpy(), ref[3])
    _check(out, oracle.nep_efv(m, synth.pack_batch([ref]), np_dtype), np_dtype)
    lat1, pos1, ty1 = np.eye(3) * 30.0, np.array([[3.0, 4.0, 5.0]]), np.array([1], np.int32)
    calc1 = _calc(m, lat1, ty1, 1, np_dtype, path="gather")
    e, f, v = _step(calc1, pos1, np_dtype)
    ref1 = oracle.nblist(lat1.astype(np_dtype), ty1, pos1.astype(np_dtype), 7.0, 200)
    er, fr, vr = oracle.nep_efv(m, synth.pack_batch([ref1]), np_dtype)
    assert np.allclose(e.ravel(), np.ravel(er), rtol=1e-10 if np_dtype == np.float64 else 1e-5, atol=0)
    assert not f.any() and not v.any()


def test_nep_loss_with_isolated_atoms(oracle):
    """NEP training step on a batch that holds a structure of isolated atoms: against the loss restated in the oracle
    and its central differences."""
    from test_gpu_nep_loss import GRADS, PARAMS, close as lclose, gpu_loss
    nt = 2
    dense = _gas(oracle, 40, 10.0, nt, 81, 5.5, 2.1)
    gas = _gas(oracle, 9, 60.0, nt, 83, 5.5, 12.0)
    assert not gas[2].any()
    nb = synth.pack_batch([dense, gas])
    B, P = nb["bilist"].shape
    m = synth.nep_model(ntypes=nt, seed=741, rmax_radial=5.5, rmax_angular=4.0, num_neurons=11, type_map=(14, 8))
    labels = dict(energy=synth.rng_normal(91, B, -5.0, 2.0), force=synth.rng_normal(92, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(93, B * 9, 0.0, 0.5).reshape(B, 9))
    w = (0.9, 1.3, 0.4)
    got = gpu_loss(m, nb, labels, w)
    bloss, rmse, e, f, v = oracle.nep_loss(m, nb, w, labels)
    assert lclose(got["bloss"], bloss) and lclose(got["rmse"], rmse)
    d = {k: synth.rng_normal(410 + i, np.size(m[k])).reshape(np.shape(m[k])) for i, k in enumerate(PARAMS)}
    fd = oracle.nep_loss_dirderiv(m, nb, w, labels, d, h=1e-6)
    an = sum(got[gk] @ np.ravel(d[pk]) for gk, pk in zip(GRADS, PARAMS))
    assert np.allclose(an, fd, rtol=2e-6, atol=1e-9), (an, fd)
    assert not got[GRADS[0]][1].any()                 # no pair: no coefficient gradient from the second structure


# A structure that is said to have more rows than the lists hold: those of the lists are evaluated, and nothing behind them is read
# (the operators refuse such a count unless they are told not to look at the lists).
@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,n_r,beyond", [(70, 5, 1), (70, 5, 200), (49153, 6, 1), (49153, 6, 300)])
def test_nep_rows_beyond_the_lists(monkeypatch, np_dtype, n, n_r, beyond):
    """n_r = 5 takes the kernel for any shape, 49,153 atoms in fp64 the staged one (fp32: four atoms to a wavefront); the last
    workgroup of both has rows to spare."""
    from ai2pot_amd import ops
    monkeypatch.setattr(ops, "_validate_batch", lambda *a: None)
    B, U = 2, 8
    m = synth.nep_model(n_radial_basis=n_r, seed=77)
    first = np.full((B, n, U), -1, np.int32)
    near = np.array([-3, -2, -1, 1, 2, 3])
    first[:, :, :6] = (np.arange(n)[:, None] + near) % n
    rcs = np.zeros((B, n, U, 3), np_dtype)
    rcs[:, :, :6, 0] = 1.9 * near
    rcs[:, :, :6, 1:] = 0.3 * synth.rng_normal(5, B * n * 6 * 2).reshape(B, n, 6, 2)
    nb = dict(binum=np.full(B, n, np.int32), bilist=np.tile(np.arange(n, dtype=np.int32), (B, 1)),
              bnumneigh=np.full((B, n), 6, np.int32), bfirstneigh=first, brcs=rcs,
              btypes=synth.rng_randint(6, B * n, 3).reshape(B, n).astype(np.int32), nghost=0, umax=U)
    want = run_gpu(m, nb, np_dtype)
    got = run_gpu(m, dict(nb, binum=nb["binum"] + beyond), np_dtype)
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0 and np.array_equal(a, b)


@pytest.mark.parametrize("model", ["nep", "mtp", "nnmtp"])
def test_loss_rows_beyond_the_lists(oracle, monkeypatch, model):
    """The errors are divided by the number of rows: twice as many halve the loss and its gradients, to the last bit."""
    import test_gpu_mtp
    import test_gpu_nep_loss
    import test_gpu_nnmtp
    from ai2pot_amd import ops
    monkeypatch.setattr(ops, "_validate_batch", lambda *a: None)
    w = (1.0, 0.7, 0.3)
    if model == "nep":                                # (three angular functions: the kernel for any shape)
        m, nb, labels = test_gpu_nep_loss.larger_case(oracle, 2, (41, 41), l_max=2, n_a=3)
        run = lambda lists: test_gpu_nep_loss.gpu_loss(m, lists, labels, w)
    elif model == "mtp":
        m, nb, labels = test_gpu_mtp.loss_inputs(oracle, 10, 2, sizes=(37, 37))
        run = lambda lists: test_gpu_mtp.gpu_loss(m, lists, labels, w)
    else:
        m, nb, labels = test_gpu_nnmtp.loss_inputs(oracle, 8, 2, 7, sizes=(37, 37))
        run = lambda lists: test_gpu_nnmtp.gpu_loss(m, lists, labels, w, True)
    assert (nb["binum"] == nb["bilist"].shape[1]).all()
    want, got = run(nb), run(dict(nb, binum=2 * nb["binum"]))
    for k in want:
        if k in ("energy", "force", "virial"):
            assert np.array_equal(got[k], want[k]), k
        elif k != "rmse":
            assert np.abs(want[k]).max() > 0 and np.array_equal(got[k], want[k] / 2), k
