"""The wavefront-per-atom gradient kernel of the NEP loss at the edges of its tiles (64 slots of a row, 32 pairs inside the
angular cutoff, 16 columns of a matrix instruction), against the kernel for any shape: the same model with one more basis
function, whose coefficients are zero, takes that kernel and has the same gradients in its other entries; and against
central differences of the oracle's loss."""
import numpy as np
import pytest

from ai2pot_amd import synth
from test_gpu_nep_loss import GRADS, PARAMS, close, gpu_loss

pytestmark = pytest.mark.gpu
ROWS = [0, 1, 16, 17, 63, 64, 65, 129, 200]
INNER = [0, 1, 15, 16, 17, 32, 33, 64, 65]


def edges(np_dtype, n_r, l_max, ntypes, H):
    """Model, batch and labels whose rows and angular neighbours lie at the tiles' edges."""
    rng = np.random.default_rng(7)
    P, U = len(ROWS) * len(INNER), 200
    rows = np.repeat(ROWS, len(INNER))
    nb = dict(binum=np.array([P, P - 5, 1], np.int32), bilist=np.tile(rng.permutation(P), (3, 1)).astype(np.int32),
              bnumneigh=np.tile(rows, (3, 1)).astype(np.int32),
              bfirstneigh=rng.integers(0, P, (3, P, U)).astype(np.int32), brcs=np.zeros((3, P, U, 3), np_dtype),
              btypes=rng.integers(0, ntypes, (3, P)).astype(np.int32), nghost=0)
    u = rng.normal(size=(3, P, U, 3))
    # the first slots of a row, in random order, are inside the angular cutoff of 4, as many as its quota; the last of the
    # others lie beyond the radial one
    place = np.stack([[np.concatenate([rng.permutation(n), np.arange(n, U)]) for n in rows] for _ in range(3)])
    inner = place < np.tile(INNER, len(ROWS))[None, :, None]
    r = np.where(inner, rng.uniform(2.0, 3.99, inner.shape), rng.uniform(4.01, 7.4, inner.shape))
    nb["brcs"][:] = u * (r / np.linalg.norm(u, axis=3))[..., None]

    m = synth.nep_model(ntypes=ntypes, n_radial_basis=n_r, l_max=l_max, num_neurons=H, sigma=0.12)
    m["type_map"] = np.arange(1, ntypes + 1, dtype=np.int32)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    labels = dict(energy=rng.normal(-5.0, 2.0, 3), force=rng.normal(size=(3, P, 3)), virial=rng.normal(size=(3, 9)))
    return m, nb, labels


@pytest.mark.parametrize("np_dtype,n_r,l_max,ntypes,H", [(np.float64, 6, 4, 3, 50), (np.float64, 4, 3, 1, 30),
                                                         (np.float64, 6, 3, 5, 65), (np.float32, 6, 4, 3, 50),
                                                         (np.float32, 4, 3, 2, 30), (np.float32, 4, 4, 17, 4)])
def test_tile_edges(np_dtype, n_r, l_max, ntypes, H):
    m, nb, labels = edges(np_dtype, n_r, l_max, ntypes, H)
    wide = dict(m, chebyshev_size=9)
    c = m["coeffs"].reshape(-1, 8)
    wide["coeffs"] = np.concatenate([c, np.zeros((len(c), 1))], axis=1).ravel()
    got = gpu_loss(m, nb, labels, (0.9, 1.3, 0.4), np_dtype)
    want = gpu_loss(wide, nb, labels, (0.9, 1.3, 0.4), np_dtype)
    want["dcoeffs"] = want["dcoeffs"].reshape(3, -1, 9)[..., :8].reshape(3, -1)
    # both kernels add some 80 rows of up to 200 terms, in different orders: at most 300 roundings of the largest partial
    # sum, itself a few times the result
    tol = 1e-12 if np_dtype == np.float64 else 300 * 2.0**-24 * 4
    for k in GRADS:
        assert close(got[k], want[k], tol), (k, np.abs(got[k] - want[k]).max() / np.abs(want[k]).max())


@pytest.mark.parametrize("n_r,l_max,ntypes,H", [(6, 4, 3, 50), (4, 3, 1, 30), (6, 3, 2, 65), (4, 4, 3, 4)])
def test_tile_edges_against_the_oracle(oracle, n_r, l_max, ntypes, H):
    """Loss, and its derivative along a direction in one group of parameters at a time, by central differences of the
    oracle's own loss."""
    m, nb, labels = edges(np.float64, n_r, l_max, ntypes, H)
    w, h = (0.9, 1.3, 0.4), 1e-6
    got = gpu_loss(m, nb, labels, w)
    bloss = oracle.nep_loss(m, nb, w, labels)[0]
    assert close(got["bloss"], bloss)
    for i, (gk, pk) in enumerate(zip(GRADS, PARAMS)):
        d = synth.rng_normal(500 + i, np.size(m[pk])).reshape(np.shape(m[pk]))
        an, fd = got[gk] @ np.ravel(d), oracle.nep_loss_dirderiv(m, nb, w, labels, {pk: d}, h=h)
        # the difference's own errors: two losses with some hundred roundings of their terms over 2 h, and the third
        # derivative over 6 h**-2
        size = np.abs(got[gk]) @ np.abs(np.ravel(d))
        assert np.all(np.abs(an - fd) <= 100 * 2.3e-16 * bloss / h + 1e-7 * size), (pk, an, fd)


@pytest.mark.parametrize("np_dtype,bar", [(np.float64, 1e-11), (np.float32, 300 * 2.0**-24 * 4)])
@pytest.mark.parametrize("copies", [15, 44, 100])
def test_rows_without_neighbours_among_many(np_dtype, bar, copies):
    """A wavefront with several rows (batches of more than 2048 rows in fp32, 1024 in fp64) has the right ones behind a row
    without neighbours: each copy of the batch has the gradients of the batch alone, where a wavefront has one row.  The
    residual forces may come from another kernel there, so the bars are those of sums in another order, in fp64 with three
    orders for cancellation."""
    m, nb, labels = edges(np_dtype, 6, 4, 3, 50)
    nb = dict(nb, binum=np.array([81, 76, 40], np.int32))
    one = gpu_loss(m, nb, labels, (0.9, 1.3, 0.4), np_dtype)
    many = lambda d: {k: np.concatenate([v] * copies) if np.ndim(v) else v for k, v in d.items()}
    got = gpu_loss(m, many(nb), many(labels), (0.9, 1.3, 0.4), np_dtype)
    for k in GRADS:
        assert got[k].shape[0] == 3 * copies
        for c in range(copies):
            assert close(got[k][3 * c:3 * c + 3], one[k], bar), (k, c)


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
@pytest.mark.parametrize("lone", [(0,), (4699,), (3, 2050, 4100), tuple(range(0, 4700, 7)), tuple(range(4, 4700))])
def test_lone_atoms_of_a_large_structure(np_dtype, lone):
    """4700 rows, so that a wavefront has two or three (fp64 five), of which `lone` have no neighbours: against the kernel for
    any shape, as above."""
    rng = np.random.default_rng(len(lone))
    P, U, H, ntypes = 4700, 24, 20, 3
    rows = rng.integers(1, U + 1, P)
    rows[list(lone)] = 0
    u = rng.normal(size=(1, P, U, 3))
    r = rng.uniform(2.0, 7.4, (1, P, U))
    nb = dict(binum=np.array([P], np.int32), bilist=np.arange(P, dtype=np.int32)[None], bnumneigh=rows[None].astype(np.int32),
              bfirstneigh=rng.integers(0, P, (1, P, U)).astype(np.int32),
              brcs=(u * (r / np.linalg.norm(u, axis=3))[..., None]).astype(np_dtype),
              btypes=rng.integers(0, ntypes, (1, P)).astype(np.int32), nghost=0)
    beyond = np.arange(U) >= rows[:, None]                  # padded entries hold anything
    nb["bfirstneigh"][0, beyond] = rng.choice([-1, 1 << 30, P], beyond.sum())
    nb["brcs"][0, beyond] = np.nan
    m = synth.nep_model(ntypes=ntypes, n_radial_basis=4, l_max=3, num_neurons=H, sigma=0.12)
    m["type_map"] = np.arange(1, ntypes + 1, dtype=np.int32)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    labels = dict(energy=rng.normal(-5.0, 2.0, 1), force=rng.normal(size=(1, P, 3)), virial=rng.normal(size=(1, 9)))
    wide = dict(m, chebyshev_size=9)
    c = m["coeffs"].reshape(-1, 8)
    wide["coeffs"] = np.concatenate([c, np.zeros((len(c), 1))], axis=1).ravel()
    got = gpu_loss(m, nb, labels, (0.9, 1.3, 0.4), np_dtype)
    want = gpu_loss(wide, nb, labels, (0.9, 1.3, 0.4), np_dtype)
    want["dcoeffs"] = want["dcoeffs"].reshape(1, -1, 9)[..., :8].reshape(1, -1)
    # sums over 4700 rows, whose roundings are of random sign: 3 sqrt(4700) of the largest partial sum, itself a few times the
    # result; fp64 as above
    tol = 1e-11 if np_dtype == np.float64 else 3 * 69 * 2.0**-24 * 10
    for k in GRADS:
        assert close(got[k], want[k], tol), (k, np.abs(got[k] - want[k]).max() / np.abs(want[k]).max())
