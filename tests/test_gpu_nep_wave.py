"""The wavefront-per-atom NEP kernel at the edges of its tiles: row lengths around 64 and 128 slots, 0 to 200 neighbours
inside the angular cutoff (which takes them 16 at a time), ghosts, a structure without atoms, places kept between calls."""
import ctypes as c

import numpy as np
import pytest

from ai2pot_amd import synth
from conftest import to_device
from test_gpu_nep import _model_to_device, check, run_gpu

pytestmark = pytest.mark.gpu
ROWS = [0, 1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 200]
INNER = [0, 1, 16, 17, 33, 200]


def _lists(np_dtype, ntypes, nghost, skin):
    rng = np.random.default_rng(5)
    P, U = len(ROWS) * len(INNER), 200
    nb = dict(binum=np.array([P, 0, P - 5], np.int32), bilist=np.tile(rng.permutation(P), (3, 1)).astype(np.int32),
              bnumneigh=np.tile(np.repeat(ROWS, len(INNER)), (3, 1)).astype(np.int32),
              bfirstneigh=rng.integers(0, P + nghost, (3, P, U)).astype(np.int32), brcs=np.zeros((3, P, U, 3), np_dtype),
              btypes=rng.integers(0, ntypes, (3, P + nghost)).astype(np.int32), nghost=nghost)
    u = rng.normal(size=(3, P, U, 3))
    u /= np.linalg.norm(u, axis=3, keepdims=True)
    # slot k of a row is inside the angular cutoff of 4 if its place in a random order comes before the row's quota
    quota = np.tile(INNER, len(ROWS))[None, :, None]
    inner = rng.permuted(np.tile(np.arange(U), (3, P, 1)), axis=2) * nb["bnumneigh"][:, :, None] < quota * U
    r = np.where(inner, rng.uniform(2.0, 3.99, inner.shape), rng.uniform(4.01, 7.0 + skin, inner.shape))
    nb["brcs"][:] = u * r[..., None]
    return nb


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n_r,l_max,ntypes,H,nghost,skin", [(6, 4, 3, 50, 0, 0.0), (4, 3, 1, 30, 7, 1.0),
                                                            (6, 3, 5, 65, 0, 1.0), (4, 4, 2, 7, 3, 0.0)])
def test_tile_edges(oracle, np_dtype, n_r, l_max, ntypes, H, nghost, skin):
    import torch
    from ai2pot_amd import _lib
    nb = _lists(np_dtype, ntypes, nghost, skin)
    m = synth.nep_model(ntypes=ntypes, n_radial_basis=n_r, l_max=l_max, num_neurons=H, type_map=(1, 2, 3, 4, 5), sigma=0.12)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)     # sums over up to 200 neighbours stay off saturation
    ref = oracle.nep_efv(m, nb, np_dtype)
    out = run_gpu(m, nb, np_dtype)
    check(out, ref, np_dtype)

    # the same through places recorded by one call and used by the next: bit-identical where every pair is inside the
    # cutoffs (others have a place here and none in the plain call, and the unit of a target's exact sum is chosen by the
    # number of its places: 2**-52 of the sum's bound either way)
    dtype = torch.float32 if np_dtype == np.float32 else torch.float64
    md, d = _model_to_device(m, dtype), to_device(nb, dtype)
    B, P, U = d["bfirstneigh"].shape
    dev, vp = d["brcs"].device, lambda t: c.c_void_p(t.data_ptr())
    rank = torch.full((B, P, U), -7, dtype=torch.int32, device=dev)
    incoming = torch.full((B, P + nghost), -7, dtype=torch.int32, device=dev)
    e, f, v = (torch.empty(s, dtype=dtype, device=dev) for s in ((B,), (B, P + nghost, 3), (B, 9)))
    fn = getattr(_lib.lib(), "a2p_nep_efv_ranked_" + ("f32" if dtype == torch.float32 else "f64"))
    stream = torch.cuda.current_stream().cuda_stream
    for valid in (0, 1, 1):
        _lib.check(fn(*(c.c_int(i) for i in (8, n_r, 4, l_max, H, ntypes)), vp(md["coeffs"]), vp(md["w0"]), vp(md["b0"]),
                      vp(md["w1"]), vp(md["type_bias"]), vp(md["q_scaler"]), c.c_double(m["rmax_radial"]),
                      c.c_double(m["rmax_angular"]), *(c.c_int(i) for i in (B, P, U, nghost)), vp(d["binum"]),
                      vp(d["bilist"]), vp(d["bnumneigh"]), vp(d["bfirstneigh"]), vp(d["brcs"]), vp(d["btypes"]),
                      vp(rank), vp(incoming), c.c_int(valid), vp(e), vp(f), vp(v), None, c.c_void_p(stream)))
        torch.cuda.synchronize()
        _lib.check_status(stream)
        got = [t.cpu().numpy().reshape(o.shape) for t, o in zip((e, f, v), out)]
        check(got, ref, np_dtype)
        assert skin or all(np.array_equal(g, o) for g, o in zip(got, out))


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_no_row_beyond_the_last(oracle, np_dtype):
    """A row count beyond the padded length counts the rows there are (the operators of the bind library take it unread),
    with a workgroup for every four of them and with fewer."""
    import torch
    from ai2pot_amd import ops
    nb = _lists(np_dtype, 3, 0, 0.0)
    m = synth.nep_model(sigma=0.12)
    m["q_scaler"] = np.linspace(5.0, 10.0, m["q_scaler"].size)
    P = nb["bilist"].shape[1]
    dtype = torch.float32 if np_dtype == np.float32 else torch.float64
    md = _model_to_device(m, dtype)
    for copies in (1, 300):                          # (18 and 3 workgroups of four rows for 72)
        d = to_device({k: np.repeat(v[:1], copies, axis=0) if isinstance(v, np.ndarray) else v for k, v in nb.items()}, dtype)
        out = []
        for rows in (P, P + 100000):
            r = ops.nepToEFVOp(m["chebyshev_size"], m["n_radial_basis"], m["n_angular_basis"], m["l_max"], md["coeffs"],
                               md["w0"], md["b0"], md["w1"], md["type_bias"], torch.full_like(d["binum"], rows), d["bilist"],
                               d["bnumneigh"], d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], 0, m["rmax_radial"],
                               m["rmax_angular"], md["q_scaler"], 0.0, 0.0, None, None, validate=False)
            out.append([t.cpu() for t in r])
        assert all(torch.equal(a, b) for a, b in zip(*out))
