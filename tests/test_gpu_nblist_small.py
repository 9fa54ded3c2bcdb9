"""Lists of structures whose binning one launch does (csrc/nblist.hip, small_bins_kernel): atom counts around its
threads and its limit, cells told axis by axis and cells whose images are tried one by one, open boundaries, and boxes
that do not fit (atoms far outside the cell), where the build starts over on the general route."""
import numpy as np
import pytest

from ai2pot_amd import synth
from test_gpu_nblist import assert_same, gpu_list

pytestmark = pytest.mark.gpu


def jittered(n, seed, density=0.04, shape=(1.0, 1.2, 0.9)):
    m = int(np.ceil(n ** (1 / 3)))
    L = np.array(shape) * (n / density / np.prod(shape)) ** (1 / 3)
    site = np.argsort(synth.rng_uniform(seed, m ** 3), kind="stable")[:n]       # any order of the atoms
    f = (np.stack([site // (m * m), site // m % m, site % m], 1) + 0.25 * synth.rng_uniform(seed + 1, 3 * n).reshape(n, 3)) / m
    return L, f


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 500, 1023, 1024, 1025, 2049, 4095, 4096, 4097])
def test_atom_counts(oracle, dt, n):
    L, f = jittered(n, n)
    ty = synth.rng_randint(n, n, 3)
    for sort in (False, True):
        args = (np.diag(L).astype(dt), ty, (f * L).astype(dt), 5.0, 120)
        assert_same(gpu_list(*args, sort=sort), oracle.nblist(*args, sort=sort))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("pbc", [(True, True, True), (True, False, True), (False, False, False)])
@pytest.mark.parametrize("n,tilt,rcut", [(7, 0.0, 6.0), (90, 0.3, 6.0), (560, 0.3, 6.0), (600, 0.3, 6.0), (120, 0.0, 7.5), (30, 0.0, 12.0)])
def test_cells(oracle, dt, pbc, n, tilt, rcut):
    """Five and more images along an axis, triclinic cells on both sides of the limit (atoms x images), fractional input."""
    L, f = jittered(n, 7 * n)
    lat = np.diag(L)
    lat[1, 0], lat[2, 1] = tilt * L[0], -tilt * L[1]
    ty = synth.rng_randint(n, n, 2)
    for is_cart in (True, False):
        x = (f @ lat if is_cart else f).astype(dt)
        args = (lat.astype(dt), ty, x, rcut, 400)
        a = gpu_list(*args, is_cart=is_cart, pbc=pbc)
        assert_same(a, oracle.nblist(*args, is_cart=is_cart, pbc=pbc))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_atoms_outside_the_cell(oracle, dt):
    """A few bins beyond the cell (fits), a dozen cells away (does not), and back, into fresh and into kept buffers."""
    import torch
    from ai2pot_amd.calculator import NepCalculator
    n = 800
    L, f = jittered(n, 5)
    ty = synth.rng_randint(3, n, 3)
    lat = np.diag(L).astype(dt)
    m = synth.nep_model(rmax_radial=5.0, rmax_angular=4.0)
    calc = NepCalculator(m, n, lat, ty, umax=120, dtype=torch.float32 if dt == np.float32 else torch.float64, path="segments")
    for far in (0.0, 0.2, 12.0, 0.1, 12.0, 0.0):
        x = f * L
        x[::3, 0] += far * L[0]
        x[1::3, 2] -= 0.5 * far * L[2]
        args = (lat, ty, x.astype(dt), 5.0, 120)
        want = oracle.nblist(*args)
        assert_same(gpu_list(*args), want)
        calc.step(torch.from_numpy(x.astype(dt)).to("cuda:0"))
        calc.check()
        nn = calc.numneigh.cpu().numpy()
        assert np.array_equal(nn, want[2])
        first, rcs = calc.firstneigh.cpu().numpy(), calc.rcs.cpu().numpy()
        for i in range(n):
            assert np.array_equal(first[i, :nn[i]], want[3][i, :nn[i]]) and np.array_equal(rcs[i, :nn[i]], want[4][i, :nn[i]])
    bad = (f * L).astype(dt)
    bad[401] = np.nan
    try:
        gpu_list(lat, ty, bad, 5.0, 120)
    except RuntimeError:
        pass
    args = (lat, ty, (f * L).astype(dt), 5.0, 120)
    assert_same(gpu_list(*args), oracle.nblist(*args))            # still usable


def sync_free_builds(oracle, lat, ty, xs, rcut, umax, pbc=(True, True, True)):
    """A synchronised build of xs[0], then builds of the others that do not read the extents back: each against the
    oracle, with nothing flagged."""
    import torch
    from ai2pot_amd import _lib, nblist
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    lib = _lib.lib()
    for k, x in enumerate(xs):
        before = lib.a2p_nblist_sync_free(1 if k else 0)
        try:
            out = nblist.find_info4mlff_device(lat, d(ty), d(x), rcut, umax, True, pbc, False, check=False)
            _lib.check_status(torch.cuda.current_stream().cuda_stream)
        finally:
            lib.a2p_nblist_sync_free(before)
        got = tuple(o.cpu().numpy() if hasattr(o, "cpu") else o for o in out)
        assert_same(got, oracle.nblist(lat, ty, x, rcut, umax, pbc=pbc))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("beyond", [24, 30])
def test_wire_whose_box_grows_past_a_byte(oracle, dt, beyond):
    """A wire of 220 bins with one atom `beyond` bins outside it in the synchronised build and up to 21 bins further out
    afterwards (within the eighth that the box may grow by): boxes of up to 280 bins along the axis."""
    n, bin_size = 900, 2.5
    lat = np.diag([220 * bin_size, 2.4, 2.4]).astype(dt)
    x = np.stack([np.sort(synth.rng_uniform(5, n)) * lat[0, 0], *(2.4 * synth.rng_uniform(6, 2 * n).reshape(2, n))], 1)
    ty = synth.rng_randint(7, n, 2)
    xs = []
    for more in (0, 2, 12, 21):
        y = x.copy()
        y[n // 2, 0] = (220 + beyond + more) * bin_size
        xs.append(y.astype(dt))
    sync_free_builds(oracle, lat, ty, xs, 2 * bin_size, 60, pbc=(True, False, False))


def growing_boxes(n, outside):
    """Cell, cutoff and positions whose boxes grow within the eighth: 16 bins along an axis, and an atom outside the cell."""
    L, f = jittered(n, n, density=0.045, shape=(1.0, 1.0, 1.0))
    bin_size = L[0] / 15.9
    x = f * L
    far = np.argmax(x.sum(1))
    x[far] = L + outside * bin_size
    spread = x.copy()
    spread[far] += 1.9 * bin_size
    # crowded around the origin, where eight cells meet and every atom has eight images in reach
    corner = np.where(x < 0.5 * L, 0.45 * x, L - 0.45 * (L - x))
    return L, 2.0 * bin_size, [x, 0.999 * x, spread, corner, x]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [2300, 4096])
@pytest.mark.parametrize("outside", [-1.1, 0.9])
def test_sync_free_box_grown_by_an_eighth(oracle, dt, n, outside):
    """Atoms that spread or crowd together within the box of the synchronised build and its eighth: boxes of more bins, and
    more images, than the one launch holds in LDS are binned all the same."""
    L, rcut, xs = growing_boxes(n, outside)
    sync_free_builds(oracle, np.diag(L).astype(dt), synth.rng_randint(n, n, 2), [x.astype(dt) for x in xs], rcut, 1200)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_more_images_than_lds(oracle, dt):
    """The same crowd of 4096 atoms (26,000 images) in synchronised builds: plain, sorted and in compact lists' records."""
    import torch
    from ai2pot_amd.calculator import NepCalculator
    L, rcut, xs = growing_boxes(4096, -1.1)
    lat, ty, x = np.diag(L).astype(dt), synth.rng_randint(9, 4096, 2), xs[3].astype(dt)
    for sort in (False, True):
        assert_same(gpu_list(lat, ty, x, rcut, 600, sort=sort), oracle.nblist(lat, ty, x, rcut, 600, sort=sort))
    m = synth.nep_model(rmax_radial=rcut, rmax_angular=0.7 * rcut)
    kw = dict(umax=400, dtype=torch.float32 if dt == np.float32 else torch.float64)
    if dt == np.float32:
        gather = NepCalculator(m, 4096, lat, ty, path="gather", **kw)
        rows = NepCalculator(m, 4096, lat, ty, path="segments", **kw)
        d = torch.from_numpy(x).to("cuda:0")
        e, f, v = gather.step(d)
        gather.check()
        e0, f0, v0 = rows.step(d)
        rows.check()
        # 400 terms a row, of either sign: two summation orders in single precision
        for a, b in ((e, e0), (f, f0), (v, v0)):
            assert (a - b).abs().max() <= 1e-5 * b.abs().max()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("tilt", [0.0, 0.1])
def test_one_plane_of_bins_with_more_images_than_lds(oracle, dt, tilt):
    """2400 atoms in one plane across x, around the corner of the other two axes: 9600 images for one workgroup; in a tilted
    cell the images are tried one by one (1600 atoms with nine images each stay below the limit of that way)."""
    n = 2400 if tilt == 0.0 else 1600
    u = synth.rng_uniform(11, 3 * n).reshape(n, 3)
    lat = np.diag([6.0, 30.0, 30.0])
    lat[2, 1] = tilt * 30.0
    x = np.stack([2.8 + 0.4 * u[:, 0], (9.0 * u[:, 1] - 4.5) % 30.0, (9.0 * u[:, 2] - 4.5) % 30.0], 1)
    ty = synth.rng_randint(12, n, 2)
    sync_free_builds(oracle, lat.astype(dt), ty, [x.astype(dt)] * 2, 5.0, n, pbc=(False, True, True))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("spacing", [0.005, 0.0059])
def test_more_than_a_thousand_images_along_an_axis(oracle, dt, axis, spacing):
    """One atom in a cell far shorter than the cutoff: 1201 and 1019 images along the axis, ten bits' worth on either side."""
    lat = np.diag([20.0, 18.0, 22.0])
    lat[axis, axis] = spacing
    x = np.array([[0.1, 0.2, 0.3]])
    pbc = [a == axis for a in range(3)]
    args = (lat.astype(dt), np.zeros(1, np.int32), x.astype(dt), 3.0, 1300)
    assert_same(gpu_list(*args, pbc=pbc), oracle.nblist(*args, pbc=pbc))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_workspace_of_a_short_cell(oracle, dt):
    """A slab of the box has room for one image along x to an atom, also where the cell is four bins long: 32 slabs of nine images
    to an atom, 16 bytes (fp64 32) a record and 8 for the images' numbers, and an eighth that a workspace is allocated
    ahead.  Atoms six cells away along x, where a slab would hold
    several of an atom's images, are listed as well."""
    import ctypes
    from ai2pot_amd import _lib
    n, L = 3800, np.array([12.0, 80.0, 80.0])
    f = np.stack([np.arange(n) % 5 / 5, np.arange(n) // 5 % 28 / 28, np.arange(n) // 140 / 28], 1) + 0.02 * synth.rng_uniform(9, 3 * n).reshape(n, 3)
    ty = synth.rng_randint(4, n, 2)
    held = _lib.lib().a2p_workspace_bytes
    held.restype = ctypes.c_size_t
    _lib.check(_lib.lib().a2p_workspace_release())
    x = f * L
    for far in (0.0, 2.0, 6.0, 0.0):
        x[::7, 0] = f[::7, 0] * L[0] + far * L[0]
        args = (np.diag(L).astype(dt), ty, x.astype(dt), 6.0, 120)
        assert_same(gpu_list(*args), oracle.nblist(*args))
        assert held() < 32 * 9 * n * (8 + 4 * np.dtype(dt).itemsize) * 9 // 8 + (4 << 20)


def test_coordinates_whose_rounding_counts_beside_the_cell(oracle):
    """fp32, 2 ** 22 A from the origin: coordinates are half an A apart there, and images of an atom a cell and a half."""
    n = 60
    L, f = jittered(n, 11, density=0.02)
    lat, ty = np.diag(L).astype(np.float32), synth.rng_randint(3, n, 2)
    site = np.stack(np.unravel_index(np.arange(n), (4, 4, 4)), 1)
    import torch
    from ai2pot_amd import _lib
    from ai2pot_amd.nblist import find_info4mlff_device
    for at in (0.0, 2.0 ** 12, 2.0 ** 17, 2.0 ** 22):
        x = (site * np.float32(L.min() / 4) + np.float32(at) * np.array([1, 0, 0])).astype(np.float32)
        args = (lat, ty, x, 5.0, 200)
        want = oracle.nblist(*args)
        for k in range(2):                               # (the second knows the box of the first, and that it goes the general way)
            assert_same(gpu_list(*args), want)
        # without a synchronisation there is no second try: such a structure takes the general route at once
        t, c = torch.from_numpy(ty.astype(np.int32)).to("cuda:0"), torch.from_numpy(x).to("cuda:0")
        before = _lib.lib().a2p_nblist_sync_free(1)
        try:
            for k in range(2):
                got = find_info4mlff_device(lat, t, c, 5.0, 200, check=False)
                _lib.check_status(torch.cuda.current_stream().cuda_stream)
                assert_same(tuple(o.cpu().numpy() if hasattr(o, "cpu") else o for o in got), want)
        finally:
            _lib.lib().a2p_nblist_sync_free(before)
