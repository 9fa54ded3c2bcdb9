"""Neighbour lists over boxes of few and of many bins: the offsets of the bins' records come from one launch, two or three."""
import numpy as np
import pytest
import torch
from scipy.spatial import cKDTree

from ai2pot_amd.nblist import find_info4mlff_device

pytestmark = pytest.mark.gpu
RCUT, UMAX, N = 6.0, 200, 4999                       # (more atoms than are binned in one launch)


# bins of half the cutoff; one more than their number is summed up: in tiles of 4096 by one launch up to 16 of them, in tiles of
# 2048 by two up to 2048 of them, by three beyond
# Their counters are cleared ahead for the bins of a cell's size (none for the largest boxes): half a cell has fewer than there are.
@pytest.mark.parametrize("dims,cell", [((63, 65, 1), 1.0), ((64, 64, 1), 1.0), ((64, 64, 15), 1.0), ((64, 64, 15), 0.5), ((64, 16, 64), 1.0), ((41, 40, 41), 1.0),
                                       ((255, 128, 128), 1.0), ((256, 128, 128), 1.0)])
def test_every_pair_once(dims, cell):
    rng = np.random.default_rng(sum(dims))
    top = (np.array(dims) - 0.5) * RCUT / 2           # the corners fix the box
    # places 1.5 apart, moved by up to 0.5: none closer than 0.5; a third of the atoms in a part of the box, so that the largest
    # boxes have pairs as well
    cells = np.maximum((top / 1.5).astype(int), 1)
    part = np.minimum(cells, np.maximum(20, 3600 // (cells.min() + 1) ** 2))
    places = {tuple(c) for c in rng.integers(0, part, (N // 3, 3))}
    while len(places) < N - 2:
        places.add(tuple(rng.integers(0, cells)))
    x = np.array(sorted(places), dtype=np.float64)[rng.permutation(len(places))]
    x = np.concatenate([[[0.0] * 3, top], np.minimum((x + 0.5) * 1.5 + rng.uniform(-0.5, 0.5, x.shape), top - 0.01)])
    x = x[np.linalg.norm(x - top, axis=1) + (np.arange(len(x)) == 1) > 0.6]
    n = len(x)
    lattice = np.diag((top + 40.0) * cell)
    out = find_info4mlff_device(lattice, torch.zeros(n, dtype=torch.int32, device="cuda:0"), torch.from_numpy(x).to("cuda:0"), RCUT, UMAX,
                                True, (False, False, False))
    count, first = out[2].cpu().numpy().reshape(n), out[3].cpu().numpy().reshape(n, UMAX)
    pairs = cKDTree(x).query_pairs(RCUT, output_type="ndarray")
    d = np.linalg.norm(x[pairs[:, 0]] - x[pairs[:, 1]], axis=1)
    assert d.min() > 0.1 and np.abs(d - RCUT).min() > 1e-9              # (none whose side of the cutoff is a matter of rounding)
    want = np.sort(np.concatenate([pairs[:, 0] * n + pairs[:, 1], pairs[:, 1] * n + pairs[:, 0]]))
    assert count.max() <= UMAX
    got = np.sort(np.concatenate([i * n + first[i, :count[i]] for i in range(n)]).astype(np.int64))
    assert np.array_equal(got, want)
