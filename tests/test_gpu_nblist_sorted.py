"""Sorted rows put in order by the wavefront that builds them (csrc/nblist.hip): rows with all distances distinct, rows
with equal ones (the reference's std::sort decides, so the order is compared bit for bit), row lengths around the
wavefront's width and up to the longest row it takes, and the lengths beyond that."""
import numpy as np
import pytest

from ai2pot_amd import synth
from test_gpu_nblist import assert_same, gpu_list

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
# neighbours in the perfect crystal: 0, 12, 54, 78, 140, 248; a row buffer of 16-byte stores needs umax % 4 == 0
@pytest.mark.parametrize("umax,rcut", [(200, 2.0), (200, 4.0), (200, 6.0), (200, 6.6), (200, 8.4), (256, 10.0), (260, 10.0),
                                       (202, 8.4)])
@pytest.mark.parametrize("moved", ["none", "few", "all"])
def test_rows_of_a_crystal(oracle, dt, umax, rcut, moved):
    lat, pos = synth.fcc_cell(4, 4.05, 0.0, 1)
    n = pos.shape[0]
    if moved == "few":                                           # tied and untied rows side by side
        pos[::37] += 0.07 * synth.rng_normal(3, pos[::37].size).reshape(-1, 3)
    elif moved == "all":
        pos += 0.05 * synth.rng_normal(4, pos.size).reshape(-1, 3)
    pos = np.mod(pos, lat[0, 0])
    types = synth.rng_randint(5, n, 2)
    want = oracle.nblist(lat.astype(dt), types, pos.astype(dt), rcut, umax, sort=True)
    assert_same(gpu_list(lat.astype(dt), types, pos.astype(dt), rcut, umax, sort=True), want)
