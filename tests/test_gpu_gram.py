"""Normal equations of three weighted matrices (csrc/gram.hip) against the products in numpy, in double, at column counts
around the 16 columns of a tile and the 24 tiles of a workgroup, and at row counts around the 32 rows of a pass.  And the
force components of a list that names an atom by more pairs than a row has room for, and by more than the 256 that are
ranked in LDS (csrc/mtp.hip comp_force_kernel), against one pass per column."""
import ctypes as c
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LIBDIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ai2pot_amd", "_lib")


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,rows", [(1, (1, 3, 0)), (15, (31, 32, 33)), (16, (5, 700, 9)), (95, (64, 24576, 576)),
                                    (111, (2, 97, 18)), (112, (0, 4096, 0)), (290, (8, 3000, 72)), (575, (3, 200, 27))])
def test_normal_equations(dtype, n, rows):
    import torch
    from ai2pot_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(n)
    w = (1.3, 0.4, 2.1)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    X = [rng.normal(size=(r, n)).astype(dtype) for r in rows]
    y = [rng.normal(size=r).astype(dtype) for r in rows]
    Xd, yd = [t(a) for a in X], [t(a) for a in y]
    A = torch.full((n, n), float("nan"), dtype=Xd[0].dtype, device="cuda:0")
    b = torch.full((n,), float("nan"), dtype=Xd[0].dtype, device="cuda:0")
    ptrs = lambda ts: (c.c_void_p * 3)(*[a.data_ptr() if a.numel() else 0 for a in ts])
    fn = L.a2p_normal_equations_f64 if dtype == "float64" else L.a2p_normal_equations_f32
    _lib.check(fn(c.c_int(n), (c.c_longlong * 3)(*rows), (c.c_double * 3)(*w), ptrs(Xd), ptrs(yd),
                  c.c_void_p(A.data_ptr()), c.c_void_p(b.data_ptr()),
                  c.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    A, b = A.cpu().numpy().astype(np.float64), b.cpu().numpy().astype(np.float64)
    X, y = [a.astype(np.float64) for a in X], [a.astype(np.float64) for a in y]
    Ar, br = sum(k * a.T @ a for k, a in zip(w, X)), sum(k * a.T @ v for k, a, v in zip(w, X, y))
    # every product once rounded, at most max(rows) additions in a row: |error| <= (rows + 2) eps sum |w x x|
    eps = (max(rows) + 2) * np.finfo(dtype).eps
    assert np.all(np.abs(A - Ar) <= eps * sum(k * np.abs(a).T @ np.abs(a) for k, a in zip(w, X)))
    assert np.all(np.abs(b - br) <= eps * sum(k * np.abs(a).T @ np.abs(v) for k, a, v in zip(w, X, y)))
    assert np.array_equal(A, A.T)


# 55 and 66 tiles: the last column count with sixteen threads to an entry of the blocks' sum, and the first ones with four, from
# fewer blocks than those to more
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,rows", [(159, (1, 33, 9)), (159, (9, 24576, 81)), (160, (1, 0, 0)), (160, (1, 33, 9)),
                                    (175, (9, 24576, 81)), (176, (3, 150, 27))])
def test_sum_of_the_blocks(dtype, n, rows):
    test_normal_equations(dtype, n, rows)


@pytest.mark.parametrize("named", [9, 300])
def test_an_atom_named_by_many_pairs(oracle, named):
    import torch
    from ai2pot_amd import _lib, ops
    from conftest import to_device
    from test_gpu_mtp import close, loss_inputs, model_to_device
    m, nb, _ = loss_inputs(oracle, 10, 2, sizes=(60, 41))
    U = 8
    nb = dict(nb, bnumneigh=np.minimum(nb["bnumneigh"], U), bfirstneigh=nb["bfirstneigh"][:, :, :U].copy(),
              brcs=nb["brcs"][:, :, :U].copy())
    left = named                                         # pairs of structure 0 that name atom 3
    for i in range(60):
        k = min(left, int(nb["bnumneigh"][0, i]))
        nb["bfirstneigh"][0, i, :k] = 3
        left -= k
    assert left == 0
    md, d = model_to_device(m, torch.float64), to_device(nb, torch.float64)
    args = (m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
            d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])
    L = _lib.lib()
    before = L.a2p_mtp_components_route(1)
    cap = L.a2p_pair_segment_capacity(512)               # the passes per column have segments of a fixed length
    try:
        one = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        again = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        L.a2p_mtp_components_route(0)
        per_column = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
    finally:
        L.a2p_mtp_components_route(before)
        L.a2p_pair_segment_capacity(cap)
    for a, b, c_ in zip(one, per_column, again):
        assert np.abs(b).max() > 0 and close(a, b) and np.array_equal(a, c_)


def _solver(oracle, dtype):
    import torch
    from conftest import to_device
    from test_gpu_mtp import loss_inputs, model_to_device
    torch.ops.load_library(os.path.join(LIBDIR, "libmtpr_bind.so"))
    m, nb, lab = loss_inputs(oracle, 10, 2, sizes=(17, 12, 23))
    md, d = model_to_device(m, dtype), to_device(nb, dtype)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0", dtype)
    labels = [t(lab[k]) for k in ("energy", "force", "virial")]
    z = torch.zeros(0, dtype=dtype, device="cuda:0")
    args = (m["chebyshev_size"], m["scaling"], md["coeffs"], md["linear_coeffs"], md["type_bias"], m["alpha_moments_count"],
            md["alpha_index_basic"], md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"],
            d["bnumneigh"], d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], 0, m["rmax"], m["rmin"], md["q_scaler"],
            0.0, 0.0, z, z)
    return labels, args


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_one_answer_from_both_entry_points(oracle, dtype):
    """The operator of the bind library and the Python one are the same calls: the same bits."""
    import torch
    from ai2pot_amd import ops
    labels, args = _solver(oracle, getattr(torch, dtype))
    for a, b in zip(torch.ops.mtpr.LinMatrixLinVectorOp(1.0, 0.7, 0.3, *labels, *args),
                    ops.LinMatrixLinVectorOp(1.0, 0.7, 0.3, *labels, *args)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("entry", ["bind", "python"])
def test_labels_that_want_a_gradient(oracle, entry):
    """lin_vector is linear in the labels: u . lin_vector is their product with its gradient, and the numbers are those of
    labels that want none."""
    import torch
    labels, args = _solver(oracle, torch.float64)
    from ai2pot_amd import ops
    op = torch.ops.mtpr.LinMatrixLinVectorOp if entry == "bind" else ops.LinMatrixLinVectorOp
    A0, b0 = op(1.0, 0.7, 0.3, *labels, *args)
    leaves = [l.clone().requires_grad_(True) for l in labels]
    A, b = op(1.0, 0.7, 0.3, *leaves, *args)
    assert torch.allclose(A, A0, rtol=1e-11, atol=1e-13 * float(A0.abs().max()))
    assert torch.allclose(b, b0, rtol=1e-11, atol=1e-13 * float(b0.abs().max()))
    u = torch.linspace(-1.0, 1.3, b.numel(), dtype=torch.float64, device="cuda:0")
    grads = torch.autograd.grad((u * b).sum(), leaves)
    total = sum((g * l).sum() for g, l in zip(grads, labels))
    assert abs(float(total - (u * b0).sum())) <= 1e-11 * float((u * b0).abs().sum())
    if entry == "bind":
        return                                               # (registered operators have no batching rule)
    # and a batch of labels, mapped over
    A2, b2 = torch.func.vmap(lambda *l: tuple(op(1.0, 0.7, 0.3, *l, *args)))(*[torch.stack([l, 2.0 * l]) for l in labels])
    assert torch.allclose(A2[1], A0, rtol=1e-11, atol=1e-13 * float(A0.abs().max()))
    assert torch.allclose(b2, torch.stack([b0, 2.0 * b0]), rtol=1e-11, atol=2e-13 * float(b0.abs().max()))
