"""The CPython module's lists: ordinary arrays, filled through pinned blocks that the library reuses (csrc/common.hip,
pinned_take).  Lists that are kept stay what they were while others are built and dropped, also past the size of the
pinned blocks; each array is memory of its own."""
import os
import sys

import numpy as np
import pytest

from ai2pot_amd import synth
from test_gpu_nblist import assert_same

pytestmark = pytest.mark.gpu
LIBDIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ai2pot_amd", "_lib")


def test_kept_lists_stay(oracle):
    if LIBDIR not in sys.path:
        sys.path.append(LIBDIR)
    import nblist
    n, umax = 60, 20000                               # 19 MB and 34 MB a list
    kept = []
    for k in range(12):
        dt = (np.float32, np.float64)[k % 2]
        lat, pos = synth.random_packed(n, [11.0, 10.0, 10.5], 2.0, 70 + k)
        ty = synth.rng_randint(k, n, 3)
        args = (lat.astype(dt), ty, pos.astype(dt), 4.0, umax, True, [True, True, True], k % 3 == 0)
        for _ in range(2):                            # a dropped list between the kept ones: its block is taken again
            dropped = nblist.find_info4mlff(*args)
        out = nblist.find_info4mlff(*args)
        assert all(np.array_equal(a, b) for a, b in zip(dropped[1:6], out[1:6]))
        del dropped
        kept.append((out if k % 4 else out[4], args))
    for out, args in kept:
        want = oracle.nblist(args[0], args[1], args[2], 4.0, umax, sort=args[7])
        if isinstance(out, tuple):
            assert_same(out, want)
        else:                                         # one array kept alone
            assert np.array_equal(out.view(np.uint8), want[4].view(np.uint8))
    with pytest.raises(RuntimeError):
        nblist.find_info4mlff(*args[:4], 3, *args[5:])
    assert_same(nblist.find_info4mlff(*args), want)   # nothing is left behind by the failed call


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_arrays_are_ordinary_memory(oracle, dt):
    """A non-blocking copy of an array to the device has read it when it returns, as of any array that is not pinned: what
    the caller writes into the array afterwards is not what arrives, however long the queue ahead of the copy.  No array
    keeps another's memory."""
    import torch
    if LIBDIR not in sys.path:
        sys.path.append(LIBDIR)
    import nblist
    lat, pos = synth.random_packed(300, [19.0, 18.0, 17.5], 2.0, 11)
    ty = synth.rng_randint(5, 300, 3)
    args = (lat.astype(dt), ty, pos.astype(dt), 5.0, 200, True, [True, True, True], False)
    out = nblist.find_info4mlff(*args)
    want = oracle.nblist(args[0], ty, args[2], 5.0, 200)
    assert_same(out, want)
    queue = torch.zeros(1 << 26, device="cuda:0")
    for a in out[1:6]:
        assert a.flags.owndata and not torch.from_numpy(a).is_pinned()
    for _ in range(200):                              # about 20 ms
        queue.add_(1.0)
    up = [torch.from_numpy(a).to("cuda:0", non_blocking=True) for a in out[1:6]]
    for a in out[1:6]:
        a[...] = 77
    for g, w in zip(up, want[1:6]):
        assert np.array_equal(g.cpu().numpy(), w)


def test_a_large_list_is_not_kept_on_the_device(oracle):
    """Lists beyond the size of a pinned block (64 MiB) take no part of the workspace, which would hold the largest of them
    for good."""
    from ai2pot_amd import _lib
    import ctypes
    if LIBDIR not in sys.path:
        sys.path.append(LIBDIR)
    import nblist
    L = _lib.lib()
    L.a2p_workspace_bytes.restype = ctypes.c_size_t
    lat, pos = synth.random_packed(300, [19.0, 18.0, 17.5], 2.0, 11)
    ty = synth.rng_randint(5, 300, 3)
    args = lambda umax: (lat, ty, pos, 5.0, umax, True, [True, True, True], False)
    small = nblist.find_info4mlff(*args(200))
    before = L.a2p_workspace_bytes()
    out = nblist.find_info4mlff(*args(9000))          # 76 MB
    assert L.a2p_workspace_bytes() - before < 16 << 20
    assert_same(out, oracle.nblist(lat, ty, pos, 5.0, 9000))
    assert all(np.array_equal(a, b) for a, b in zip(small[1:6], nblist.find_info4mlff(*args(200))[1:6]))
