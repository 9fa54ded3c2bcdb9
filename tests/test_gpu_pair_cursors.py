"""Cursors of the pair reduction that are zero between calls (csrc/pair_reduce.hip): calls of other kinds and sizes in turn,
calls that were refused, lists that run over, atoms without a row and atoms that no pair names give the bits of a call with
a workspace of its own, and every output is written."""
import numpy as np
import pytest

from ai2pot_amd import mtp_param, synth
from conftest import to_device
from test_gpu_mtp import gpu_efv
from test_gpu_nep import run_gpu as run_nep

pytestmark = pytest.mark.gpu


def _lists(np_dtype, P, U, nghost, named, seed):
    """Rows for the even centres only; pairs name the first `named` atoms; the rest of the atoms gather nothing."""
    rng = np.random.default_rng(seed)
    nn = rng.integers(0, U + 1, (2, P)).astype(np.int32)
    u = rng.normal(size=(2, P, U, 3))
    rcs = u / np.linalg.norm(u, axis=3, keepdims=True) * rng.uniform(2.0, 6.5, (2, P, U, 1))
    rows = (P + 1) // 2
    il = np.zeros((2, P), np.int32)
    il[:, :rows] = np.arange(0, P, 2)
    return dict(binum=np.array([rows, max(rows - 2, 0)], np.int32), bilist=il, bnumneigh=nn, nghost=nghost,
                bfirstneigh=rng.integers(0, named, (2, P, U)).astype(np.int32), brcs=rcs.astype(np_dtype),
                btypes=rng.integers(0, 2, (2, P + nghost)).astype(np.int32))


def _force(nb, np_dtype, dei):
    import torch
    from ai2pot_amd import ops
    dtype = torch.float32 if np_dtype == np.float32 else torch.float64
    d = to_device(nb, dtype)
    return [ops.ForceSrOp(d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"], nb["nghost"], dei.shape[2],
                          torch.from_numpy(dei).to("cuda:0"))[0].cpu().numpy()]


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_calls_in_turn(np_dtype, monkeypatch):
    from ai2pot_amd import _lib
    monkeypatch.setenv("AI2POT_POISON_OUTPUTS", "1")
    nep = synth.nep_model(ntypes=2, type_map=(1, 2), sigma=0.12)
    mtp = synth.mtp_model(mtp_param.mtp_param(10), 2, 8, 6.0, 1.0, 7)
    calls = []
    for P, U, nghost, named, seed in ((23, 40, 5, 23, 1), (1, 3, 0, 1, 2), (90, 70, 30, 100, 3)):
        nb = _lists(np_dtype, P, U, nghost, named, seed)
        dei = np.random.default_rng(seed).normal(size=nb["brcs"].shape).astype(np_dtype)
        over = dict(nb, bfirstneigh=nb["bfirstneigh"] % max(1, named // 8))    # most pairs beyond their targets' segments
        calls += [lambda nb=nb: run_nep(nep, nb, np_dtype), lambda nb=nb: gpu_efv(mtp, nb, np_dtype),
                  lambda nb=over, dei=dei: _force(nb, np_dtype, dei), lambda nb=over: run_nep(nep, nb, np_dtype)]
    bad = _lists(np_dtype, 23, 40, 0, 23, 4)
    bad["bfirstneigh"][0, :3, :5] = 1000
    bad["bnumneigh"][0, :3] = 5

    def alone(call):
        _lib.check(_lib.lib().a2p_workspace_release())
        return call()
    want = [alone(c) for c in calls]
    for w in want:
        assert all(np.isfinite(x).all() for x in w)
    order = np.random.default_rng(9).permutation(np.repeat(np.arange(len(calls)), 3))
    for k, i in enumerate(order):
        if k % 5 == 0:
            with pytest.raises(RuntimeError, match="neighbour index"):
                run_nep(nep, bad, np_dtype)
        got = calls[i]()
        assert all(np.array_equal(g, w) for g, w in zip(got, want[i])), (k, i)
