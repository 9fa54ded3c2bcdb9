"""The passes over the neighbours of the moment tensor potentials where their layouts can go wrong: basic moments whose
powers of z have gaps, occur twice or are high, or that make many polynomials, and linear-solver components for one to four groups of columns and for rows with
few neighbours (pairs of neighbours that have no second one)."""
import numpy as np
import pytest

from ai2pot_amd import mtp_param, synth
from test_gpu_mtp import close, gpu_efv, gpu_loss, loss_inputs, model_to_device, structure
from conftest import to_device

pytestmark = pytest.mark.gpu

# (mu, a, b, c): z^0 and z^2 of a row without z^1, a row without its constant, and the same moment twice
GAPS = [(0, 0, 0, 0), (0, 0, 0, 2), (0, 1, 0, 1), (0, 1, 1, 3), (1, 0, 0, 1), (1, 0, 2, 0)]
TWICE = GAPS[:4] + [(0, 0, 0, 2)] + GAPS[4:] + [(1, 0, 2, 0)]
# a polynomial in z longer than a thread's sums, and more polynomials than a wavefront has lanes
LONG = GAPS + [(1, 0, 0, 11)]
MANY = [(mu, a, b, 0) for mu in (0, 1) for a in range(8) for b in range(8 - a)]


def tables(basic):
    nb = len(basic)
    times = [(0, 1, 2, nb), (2, 3, 1, nb), (4, 5, 1, nb + 1), (nb, nb + 1, 3, nb + 2), (nb - 1, nb - 1, 1, nb + 2)]
    mapping = [0, 1, nb - 1, nb, nb + 2]
    return dict(alpha_moments_count=nb + 3, alpha_index_basic=np.array(basic, np.int32),
                alpha_index_times=np.array(times, np.int32), alpha_moment_mapping=np.array(mapping, np.int32),
                nmus=2)


@pytest.mark.parametrize("basic", [GAPS, TWICE, LONG, MANY], ids=["gaps", "twice", "long", "many"])
def test_irregular_basic_moments(oracle, basic):
    """Energies, forces, virials and loss gradients against the oracle: fp64, 1e-10 as for the shipped tables."""
    nt = 2
    nb = synth.pack_batch([structure(oracle, n, (8.5, 9.0, 9.5), nt, 21 + n, 5.0) for n in (40, 23)])
    m = synth.mtp_model(tables(basic), nt, 6, 5.0, 1.5, 3200)
    m["q_scaler"] = np.linspace(0.8, 1.3, m["q_scaler"].size)
    for got, ref in zip(gpu_efv(m, nb), oracle.mtp_efv(m, nb)):
        assert close(got, ref)
    B, P = nb["bilist"].shape
    labels = dict(energy=synth.rng_normal(1, B, -4 * 40, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w), oracle.mtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], ref[k]), k


ROWS = [0, 1, 2, 3, 4, 5, 15, 16, 17, 23, 24, 25, 31, 32, 33, 40, 41, 47, 48, 49, 63, 64, 65, 80]


@pytest.mark.parametrize("level", [8, 12, 16, 20, 22])            # 1, 1, 2, 4 and 5 tiles: one or two to a wavefront, or shared by four and two
def test_passes_by_row_length(oracle, level):
    """The sums of the basic moments and the pair derivatives for rows that fill a matrix product, half a wavefront, a wavefront and
    the neighbour table, one neighbour more and one less.  Energies, forces, virials and loss gradients against the oracle: fp64, 1e-10."""
    nt, rc = 2, 7.0
    nb = dict(synth.pack_batch([structure(oracle, len(ROWS), (7.0, 7.2, 7.4), nt, 57, rc, umax=140)]))
    assert nb["bnumneigh"].min() >= max(ROWS)
    nb["bnumneigh"] = np.array([ROWS], np.int32)
    m = synth.mtp_model(mtp_param.mtp_param(level), nt, 8, rc, 1.5, 3300 + level, lo=-0.05, hi=0.05)
    m["q_scaler"] = np.linspace(0.8, 1.3, m["q_scaler"].size)
    for got, ref in zip(gpu_efv(m, nb), oracle.mtp_efv(m, nb)):
        assert close(got, ref)
    n = len(ROWS)
    labels = dict(energy=synth.rng_normal(1, 1, -4 * n, 3), force=synth.rng_normal(2, n * 3).reshape(1, n, 3),
                  virial=synth.rng_normal(3, 9, 0, 0.5).reshape(1, 9))
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w), oracle.mtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], ref[k]), k


@pytest.mark.parametrize("levels", [1, 2, 5, 62, 63, 64, 65, 129, 130])
def test_products_by_number_of_levels_and_multiplicity(oracle, levels):
    """Products that depend on the one before, so that a wavefront makes as many steps as there are levels, odd and even, less and
    more than the 64 whose control words it holds at a time; lists with one, two and three products of a multiplicity, among them
    negative ones and one beyond 21 bits.  Energies, forces, virials and loss gradients against the oracle: fp64, 1e-10."""
    nt, nbasic = 2, len(GAPS)
    times = []
    for k in range(levels):                                       # sums that stay of the order of a product of two
        at = nbasic + k
        times += [(at - 1 if k else 1, 0, 1, at), (2, 3, -3, at), (4, 5, 1, at), (1, 3, 2, at)]
    last = nbasic + levels
    times += [(0, 0, (1 << 21) + 1, last), (1, 1, -(1 << 21), last), (last - 1, 2, 1, last)]
    t = dict(alpha_moments_count=last + 1, alpha_index_basic=np.array(GAPS, np.int32),
             alpha_index_times=np.array(times, np.int32), alpha_moment_mapping=np.array(sorted({0, 2, nbasic, last - 1, last}), np.int32), nmus=2)
    nb = synth.pack_batch([structure(oracle, n, (8.5, 9.0, 9.5), nt, 21 + n, 5.0) for n in (12, 7)])
    m = synth.mtp_model(t, nt, 6, 5.0, 1.5, 3200)
    m["q_scaler"] = np.linspace(0.8, 1.3, m["q_scaler"].size)
    m["linear_coeffs"][-1] *= 1e-6                                # of the order of the others
    for got, ref in zip(gpu_efv(m, nb), oracle.mtp_efv(m, nb)):
        assert np.isfinite(ref).all() and close(got, ref)
    B, P = nb["bilist"].shape
    labels = dict(energy=synth.rng_normal(1, B, -4 * 12, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w), oracle.mtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], ref[k]), k


@pytest.mark.parametrize("level", [8, 14, 16, 18])                # 1, 1, 2 and 4 groups of 64 pieces
@pytest.mark.parametrize("U", [1, 2, 3, 9, None])
def test_components_by_group_and_row_length(oracle, level, U):
    """All columns from one pass against a pass per column, fp64 1e-10."""
    from ai2pot_amd import _lib, ops
    import torch
    m, nb, _ = loss_inputs(oracle, level, 2, sizes=(20, 13))
    if U is not None:
        nb = dict(nb)
        nb["bnumneigh"] = np.minimum(nb["bnumneigh"], U)
        nb["bnumneigh"][0, 3] = 0
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    args = (m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
            d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])
    L = _lib.lib()
    before = L.a2p_mtp_components_route(1)
    try:
        one = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        L.a2p_mtp_components_route(0)
        per_column = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
    finally:
        L.a2p_mtp_components_route(before)
    for a, b in zip(one, per_column):
        assert np.abs(b).max() > 0
        assert close(a, b)


@pytest.mark.parametrize("lists", ["whole", "rows left out", "one atom named by all"])
@pytest.mark.parametrize("basic", [GAPS, TWICE, LONG, MANY, MANY + [(1, 0, 0, 8)]], ids=["gaps", "twice", "long", "many", "many, gap"])
def test_components_of_irregular_tables(oracle, basic, lists):
    """The vectors of the basic moments by polynomials and one by one, columns cut into pieces of any length, and the virial summed
    over the atoms that the pairs name: atoms without a row of their own, and one with more pairs than are ranked in LDS.  All
    columns from one pass against a pass per column, fp64 1e-10."""
    from ai2pot_amd import _lib, ops
    import torch
    nt = 2
    nb = synth.pack_batch([structure(oracle, n, (8.5, 9.0, 9.5), nt, 21 + n, 5.0) for n in (40, 23)])
    if lists == "rows left out":
        nb["binum"] = nb["binum"] - 17
    if lists == "one atom named by all":
        nb["bfirstneigh"] = np.where(nb["bfirstneigh"] >= 0, 5, nb["bfirstneigh"]).astype(np.int32)
        assert nb["bnumneigh"][0].sum() > 256
    m = synth.mtp_model(tables(basic), nt, 6, 5.0, 1.5, 3200)
    m["q_scaler"] = np.linspace(0.8, 1.3, m["q_scaler"].size)
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    args = (m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
            d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])
    L = _lib.lib()
    before = L.a2p_mtp_components_route(1)
    try:
        one = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        L.a2p_mtp_components_route(0)
        per_column = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
    finally:
        L.a2p_mtp_components_route(before)
    for a, b in zip(one, per_column):
        assert np.abs(b).max() > 0
        assert close(a, b)


def components_by_both_routes(m, nb):
    """Energy, force and virial columns from one pass over the atoms, and from a pass per column."""
    from ai2pot_amd import _lib, ops
    import torch
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    args = (m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
            d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])
    L = _lib.lib()
    before = L.a2p_mtp_components_route(1)
    try:
        one = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        L.a2p_mtp_components_route(0)
        per_column = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
    finally:
        L.a2p_mtp_components_route(before)
    return one, per_column


@pytest.mark.parametrize("level", [8, 16])                        # 11 columns and 94: one of them to a lane, and two
@pytest.mark.parametrize("pairs", [63, 64, 65, 127, 128, 129, 130, 255, 256, 257])
def test_components_by_pairs_that_name_an_atom(oracle, level, pairs):
    """An atom named by as many pairs as a wavefront ranks at a time, as have their displacements in LDS, and as are ranked at
    all, one more and one less: all columns from one pass against a pass per column, fp64 1e-10."""
    m, nb, _ = loss_inputs(oracle, level, 2, sizes=(40, 23))
    first = nb["bfirstneigh"].copy()
    first[0][first[0] == 5] = 6
    used = np.argwhere(np.arange(first.shape[2]) < nb["bnumneigh"][0][:, None])
    for ii, u in used[::len(used) // pairs][:pairs]:              # (over all rows, at places of any order)
        first[0, ii, u] = 5
    nb = dict(nb, bfirstneigh=first)
    assert sum((first[0, i, :n] == 5).sum() for i, n in enumerate(nb["bnumneigh"][0])) == pairs
    for a, b in zip(*components_by_both_routes(m, nb)):
        assert np.abs(b).max() > 0
        assert close(a, b)


# a power of z left out and a moment given twice: as many coefficients as basic moments, though not one for each
ONE_OF_EACH = [(0, 0, 0, 0), (0, 0, 0, 2), (0, 1, 0, 0), (0, 1, 0, 0), (1, 0, 0, 0), (1, 0, 0, 1)]


def test_as_many_coefficients_as_basic_moments(oracle):
    test_irregular_basic_moments(oracle, ONE_OF_EACH)
    nt = 2
    nb = synth.pack_batch([structure(oracle, n, (8.5, 9.0, 9.5), nt, 21 + n, 5.0) for n in (40, 23)])
    m = synth.mtp_model(tables(ONE_OF_EACH), nt, 6, 5.0, 1.5, 3200)
    for a, b in zip(*components_by_both_routes(m, nb)):
        assert np.abs(b).max() > 0
        assert close(a, b)


def test_components_in_chunks_of_structures(oracle):
    """Enough pair derivatives (level 16: 92 columns, more than 200 MB) that the structures are taken in chunks, the last
    one shorter: every structure equal to the call with that structure alone, bit for bit, in force columns too."""
    from ai2pot_amd import ops
    import torch
    m, nb, _ = loss_inputs(oracle, 16, 2, sizes=(48,))
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    n, B = int(nb["binum"][0]), 91
    keys = ("binum", "bilist", "bnumneigh", "bfirstneigh", "brcs", "btypes")
    assert nb["bnumneigh"].sum() * B * 3 * m["q_scaler"].size * 8 > (200 << 20) and n * B >= 4096

    def components(t):
        return ops.mtp_lin_components(
            m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], t["binum"], t["bilist"], t["bnumneigh"],
            t["bfirstneigh"], t["brcs"], t["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])

    batch = {k: d[k].expand(B, *d[k].shape[1:]).contiguous() for k in keys}
    alone = components(d)
    for whole, one in zip(components(batch), alone):
        assert torch.equal(whole, one.expand_as(whole))


# A million neighbours and more in one row: lengths at which a single-precision quotient makes chunks of 33 for a table of
# 32, or of 49 for 48 (with the reciprocal rounded to nearest or one place above), and one that it gets right.
@pytest.mark.parametrize("level,n", [(10, 1 << 20), (10, 2618352), (10, 5449248), (8, 2625408), (20, 2074272), (20, 4154976)])
def test_rows_of_millions(level, n):
    """A row whose neighbours all lie beyond the cutoff but a few, the last one of every 1000th chunk: energies, forces and
    virials of the row of those few."""
    from ai2pot_amd import mtp_param
    m = synth.mtp_model(mtp_param.mtp_param(level), 1, 6, 5.0, 1.5, 3210)
    cap = 48 if level < 20 else 32
    size = -(-n // -(-n // cap))
    at = np.arange(size - 1, n, 1000 * size)
    rng = np.random.default_rng(level)
    few = rng.normal(size=(len(at), 3))
    few *= (rng.uniform(2.0, 4.9, len(at)) / np.linalg.norm(few, axis=1))[:, None]
    common = dict(binum=np.array([1], np.int32), bilist=np.zeros((1, 2), np.int32), btypes=np.zeros((1, 2), np.int32), nghost=0)
    row = lambda r: dict(common, bnumneigh=np.array([[len(r), 0]], np.int32), bfirstneigh=np.ones((1, 2, len(r)), np.int32),
                         brcs=np.stack([r, r])[None])
    far = np.full((n, 3), 4.0)
    far[at] = few
    # sums of the same few hundred terms in another order
    for got, want in zip(gpu_efv(m, row(far)), gpu_efv(m, row(few))):
        assert np.abs(want).max() > 0
        assert close(got, want)
