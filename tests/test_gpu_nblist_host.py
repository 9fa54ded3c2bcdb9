"""The CPython module's lists: five arrays over one host block that the library pins and reuses (csrc/common.hip,
host_alloc).  Lists that are kept stay what they were while others are built and dropped, also past the library's share
of pinned memory."""
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
    n, umax = 60, 20000                               # 19 MB and 34 MB a list: more than 256 MiB are alive at the end
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
        else:                                         # one array holds the block on its own
            assert np.array_equal(out.view(np.uint8), want[4].view(np.uint8))
    with pytest.raises(RuntimeError):
        nblist.find_info4mlff(*args[:4], 3, *args[5:])
    assert_same(nblist.find_info4mlff(*args), want)   # nothing is left behind by the failed call
