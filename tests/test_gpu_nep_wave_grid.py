"""The NEP kernel with four atoms per wavefront over the sizes of its launches: wavefronts of a workgroup, workgroups of a
compute unit and rows of a wavefront change with the number of rows."""
import numpy as np
import pytest

from ai2pot_amd import synth
from test_gpu_nep import check, run_gpu
from test_gpu_nep_wave import _lists

pytestmark = pytest.mark.gpu
ROWS, U = 71, 72


def _block(np_dtype, ntypes):
    rng = np.random.default_rng(11)
    n = rng.integers(0, U + 1, ROWS).astype(np.int32)
    u = rng.normal(size=(ROWS, U, 3))
    u /= np.linalg.norm(u, axis=2, keepdims=True)
    r = np.where(rng.random((ROWS, U)) < 0.35, rng.uniform(2.0, 3.99, (ROWS, U)), rng.uniform(4.01, 7.5, (ROWS, U)))
    return dict(n=n, first=rng.integers(0, ROWS, (ROWS, U)).astype(np.int32), rcs=(u * r[..., None]).astype(np_dtype),
                types=rng.integers(0, ntypes, ROWS).astype(np.int32))


def _copies(blk, copies, batch):
    """`copies` of the block as one structure, the last without its last row; `batch` such structures."""
    first = (blk["first"][None] + ROWS * np.arange(copies, dtype=np.int32)[:, None, None]).reshape(-1, U)
    one = dict(bilist=np.arange(ROWS * copies, dtype=np.int32), bnumneigh=np.tile(blk["n"], copies), bfirstneigh=first,
               brcs=np.tile(blk["rcs"], (copies, 1, 1)), btypes=np.tile(blk["types"], copies))
    nb = {k: np.array(np.broadcast_to(v, (batch,) + v.shape)) for k, v in one.items()}
    return dict(nb, binum=np.full(batch, ROWS * copies - 1, np.int32), nghost=0)


# fp32 at three species: up to 2560 rows a wavefront each; then four rows each, up to 4096 four wavefronts to a workgroup, up to
# 8192 two such workgroups, beyond it twelve wavefronts, beyond 12288 several times four rows each; fp64 from 1024 rows on four
# wavefronts throughout.  One species: several workgroups of any size.
@pytest.mark.parametrize("np_dtype", [np.float32, np.float64])
@pytest.mark.parametrize("ntypes,copies,batch", [(3, 1, 1), (3, 14, 1), (3, 36, 1), (3, 37, 1), (3, 57, 1), (3, 58, 1), (3, 115, 1), (3, 116, 1), (3, 180, 1), (3, 600, 1),
                                                 (3, 1, 61), (3, 3, 61), (1, 180, 1), (5, 60, 3)])
def test_every_launch_gives_the_same(np_dtype, ntypes, copies, batch):
    blk = _block(np_dtype, ntypes)
    m = synth.nep_model(ntypes=ntypes, num_neurons=30, type_map=(1, 2, 3, 4, 5), sigma=0.12)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    e2, f2, _ = run_gpu(m, _copies(blk, 2, 1), np_dtype)               # (a launch of nine workgroups' worth at most)
    e3, _, v3 = run_gpu(m, _copies(blk, 3, 1), np_dtype)
    _, _, v2 = run_gpu(m, _copies(blk, 2, 1), np_dtype)
    e, f, v = run_gpu(m, _copies(blk, copies, batch), np_dtype)
    # An atom's sums run over up to 72 pairs in another order when its lane or chunk is another; a pair's force is a sum over the
    # 24 x 4 moments: 100 roundings of the largest term, with room for the cancellation of pairs of a dozen times the sum.
    eps = np.finfo(np_dtype).eps
    inner = f2.reshape(2, ROWS, 3)[0]
    tol = 1200 * eps * np.abs(inner).max()
    f = f.reshape(batch, copies, ROWS, 3)
    if copies > 1:
        assert np.abs(f[:, :-1] - inner).max() <= tol
    assert np.abs(f[:, -1] - f2.reshape(2, ROWS, 3)[1]).max() <= tol
    # energies and virials: those of two blocks and so many times those of one more
    per_e, per_v = e3 - e2, v3 - v2
    scale = max(copies, 3) * eps * 1200
    assert np.abs(e - (e2 + (copies - 2) * per_e)).max() <= scale * np.abs(e3).max()
    assert np.abs(v - (v2 + (copies - 2) * per_v)).max() <= scale * np.abs(v3).max()


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n_r,l_max,ntypes,H,nghost,skin", [(6, 4, 3, 50, 0, 0.0), (4, 3, 1, 30, 7, 1.0),
                                                            (6, 3, 5, 65, 0, 1.0), (4, 4, 2, 7, 3, 0.0)])
def test_tile_edges_of_four_atoms(oracle, np_dtype, n_r, l_max, ntypes, H, nghost, skin):
    """Rows of 0 to 200 slots with 0 to 200 of them inside the angular cutoff (several tiles and several rounds of 64 pairs
    beside rows of one), 39 structures of them: four rows to a wavefront in either precision."""
    nb = _lists(np_dtype, ntypes, nghost, skin)
    m = synth.nep_model(ntypes=ntypes, n_radial_basis=n_r, l_max=l_max, num_neurons=H, type_map=(1, 2, 3, 4, 5), sigma=0.12)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    ref = oracle.nep_efv(m, nb, np_dtype)
    many = {k: np.concatenate([v] * 13) if isinstance(v, np.ndarray) else v for k, v in nb.items()}
    e, f, v = run_gpu(m, many, np_dtype)
    for k in range(0, 39, 3):
        check((e[k:k + 3], f[k:k + 3], v[k:k + 3]), ref, np_dtype)


@pytest.mark.parametrize("np_dtype", [np.float32, np.float64])
@pytest.mark.parametrize("copies,batch", [(29, 4), (2, 61), (1, 130)])
def test_rows_in_runs_and_in_turn(np_dtype, copies, batch):
    """Above 2048 sets of four rows a workgroup takes a run of rows: every structure as it comes out alone, with from none to
    all of its rows in use."""
    m = synth.nep_model(ntypes=3, num_neurons=30, type_map=(1, 2, 3, 4, 5), sigma=0.12)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    nb = _copies(_block(np_dtype, 3), copies, batch)
    P = nb["bilist"].shape[1]
    nb["binum"] = (np.arange(batch) * 37 % (P + 1)).astype(np.int32)
    nb["binum"][-1] = P
    assert batch * -(-P // 4) > 2048
    e, f, v = run_gpu(m, nb, np_dtype)
    eps = np.finfo(np_dtype).eps
    for b in (0, 1, batch // 2, batch - 1):
        one = {k: a[b:b + 1] if isinstance(a, np.ndarray) else a for k, a in nb.items()}
        e1, f1, v1 = run_gpu(m, one, np_dtype)
        # (the roundings of test_every_launch_gives_the_same; the sums of a structure grow with its rows)
        assert np.abs(f[b] - f1[0]).max() <= 1200 * eps * np.abs(f1).max()
        assert np.abs(e[b] - e1[0]).max() <= 1200 * eps * copies * max(np.abs(e1).max(), 1.0)
        assert np.abs(v[b] - v1[0]).max() <= 1200 * eps * copies * max(np.abs(v1).max(), 1.0)


@pytest.mark.parametrize("np_dtype", [np.float32, np.float64])
@pytest.mark.parametrize("copies,batch,most", [(29, 8, 0), (29, 8, 1), (1, 130, 0)])
def test_runs_of_structures_with_places_to_spare(np_dtype, copies, batch, most):
    """Runs of rows by the places of the lists, and by the rows in use where all structures leave a quarter of the places empty (up to
    64 of them are looked at: the second of 130 is not, and uses all of its places)."""
    m = synth.nep_model(ntypes=3, num_neurons=30, type_map=(1, 2, 3, 4, 5), sigma=0.12)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    nb = _copies(_block(np_dtype, 3), copies, batch)
    P = nb["bilist"].shape[1]
    top = P - P // 4 + most
    assert batch * -(-P // 4) > 2048
    nb["binum"] = np.resize(np.array([0, 1, 5, top // 3, top - 1, top - 2, top - 4, top], np.int32), batch)
    if batch > 64:
        nb["binum"][1] = P
    e, f, v = run_gpu(m, nb, np_dtype)
    eps = np.finfo(np_dtype).eps
    for b in range(8):
        one = {k: a[b:b + 1] if isinstance(a, np.ndarray) else a for k, a in nb.items()}
        e1, f1, v1 = run_gpu(m, one, np_dtype)
        # (the roundings of test_every_launch_gives_the_same; the sums of a structure grow with its rows)
        assert np.abs(f[b] - f1[0]).max() <= 1200 * eps * np.abs(f1).max()
        assert np.abs(e[b] - e1[0]).max() <= 1200 * eps * copies * max(np.abs(e1).max(), 1.0)
        assert np.abs(v[b] - v1[0]).max() <= 1200 * eps * copies * max(np.abs(v1).max(), 1.0)
    for b in range(8, batch):
        if b % 8 != 1:
            assert abs(e[b] - e[b % 8]) <= 1200 * eps * copies * max(abs(e[b % 8]), 1.0)
