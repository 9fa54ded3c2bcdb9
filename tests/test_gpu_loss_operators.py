"""The loss operators' backward through torch.ops (one weighted sum over the per-structure gradients of all parameters,
csrc/common.hip weighted_rows_kernel) against the matrix products it stands for, at batch sizes around its runs and
unrolled loads; the early status word; gradients that are themselves differentiated; outputs written in place."""
import os

import numpy as np
import pytest

from ai2pot_amd import mtp_param, synth
from conftest import to_device

pytestmark = pytest.mark.gpu
LIBDIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ai2pot_amd", "_lib")


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("B", [1, 3, 4, 31, 32, 33, 65])
@pytest.mark.parametrize("sizes", [(1,), (63, 1, 64), (640, 3300, 150, 150, 3), (5, 0, 7, 1, 2, 9, 130, 8)])
def test_weighted_rows(dtype, B, sizes):
    import ctypes
    import torch
    from ai2pot_amd import _lib
    dt = getattr(torch, dtype)
    g = torch.Generator(device="cuda:0").manual_seed(B)
    parts = [torch.randn((B, n), generator=g, device="cuda:0", dtype=dt) for n in sizes]
    w = torch.randn(B, generator=g, device="cuda:0", dtype=dt)
    out = torch.full((sum(sizes) + 1,), 7.0, device="cuda:0", dtype=dt)
    L = _lib.lib()
    fn = L.a2p_weighted_rows_f32 if dtype == "float32" else L.a2p_weighted_rows_f64
    ptr = (ctypes.c_void_p * len(sizes))(*[p.data_ptr() if p.numel() else w.data_ptr() for p in parts])
    num = (ctypes.c_longlong * len(sizes))(*sizes)
    _lib.check(fn(ctypes.c_int(B), ctypes.c_void_p(w.data_ptr()), ctypes.c_int(len(sizes)), ptr, num,
                  ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    want = torch.cat([(w.double()[:, None] * p.double()).sum(0) for p in parts])
    # sums in double, rounded once: half an ulp of the result beside the rounding of B products in double
    eps = np.finfo(dtype).eps
    bound = torch.cat([(w.double().abs()[:, None] * p.double().abs()).sum(0) for p in parts]) * B * 2.3e-16 + want.abs() * eps
    assert bool(((out[:-1].double() - want).abs() <= bound).all()) and float(out[-1]) == 7.0
    # results in places of their own: the same bits, and nothing beside them
    outs = [torch.full((n + 1,), 7.0, device="cuda:0", dtype=dt) for n in sizes]
    fn = L.a2p_weighted_rows_split_f32 if dtype == "float32" else L.a2p_weighted_rows_split_f64
    dst = (ctypes.c_void_p * len(sizes))(*[o.data_ptr() for o in outs])
    _lib.check(fn(ctypes.c_int(B), ctypes.c_void_p(w.data_ptr()), ctypes.c_int(len(sizes)), ptr, num, dst,
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(torch.cat([o[:-1] for o in outs]), out[:-1]) and all(float(o[-1]) == 7.0 for o in outs)


def _loss(oracle, dtype):
    import torch
    torch.ops.load_library(os.path.join(LIBDIR, "libmtpr_bind.so"))
    m = synth.mtp_model(mtp_param.mtp_param(8), 2, 8, 5.0, 0.5, 31)
    lists = []
    for k, n in enumerate((9, 14, 11)):
        lat, pos = synth.random_packed(n, [8.0, 7.5, 8.5], 2.0, 40 + k)
        lists.append(oracle.nblist(lat, synth.rng_randint(50 + k, n, 2), pos, 5.0, 200))
    nb = to_device(synth.pack_batch(lists), dtype)
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0", dtype)
    i = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).to("cuda:0")
    par = [f(m[k]).requires_grad_(True) for k in ("coeffs", "linear_coeffs", "type_bias")]
    B, P = nb["bilist"].shape
    lab = (f(synth.rng_normal(1, B)), f(synth.rng_normal(2, B * P * 3).reshape(B, P, 3)), f(synth.rng_normal(3, B * 9).reshape(B, 9)))
    z = torch.zeros(0, dtype=dtype, device="cuda:0")

    def call(first=None):
        return torch.ops.mtpr.linearMtpToLossOp(
            1.0, 1.0, 1.0, *lab, 8, 1.0, *par, int(m["alpha_moments_count"]), i(m["alpha_index_basic"]),
            i(m["alpha_index_times"]), i(m["alpha_moment_mapping"]), int(m["nmus"]), nb["binum"], nb["bilist"],
            nb["bnumneigh"], nb["bfirstneigh"] if first is None else first, nb["brcs"], nb["btypes"], i(m["type_map"]), 0,
            5.0, 0.5, f(m["q_scaler"]), 0.0, 0.0, z, z)
    return call, par, nb


def test_backward_of_the_backward_and_in_place_outputs(oracle):
    import torch
    call, par, nb = _loss(oracle, torch.float64)
    w = torch.tensor([0.3, -1.1, 0.7], dtype=torch.float64, device="cuda:0", requires_grad=True)
    out = call()
    plain = torch.autograd.grad((out[0] * w.detach()).sum(), par, retain_graph=True)
    graphed = torch.autograd.grad((out[0] * w).sum(), par, create_graph=True)
    for a, b in zip(plain, graphed):
        assert torch.allclose(a, b, rtol=1e-12, atol=1e-14)
    d = torch.autograd.grad(graphed[2].sum(), w)[0]             # linear in the weights
    one = [torch.autograd.grad(call()[0][k], par)[2].sum() for k in range(3)]
    assert torch.allclose(d, torch.stack(one), rtol=1e-12)
    kept = [t.clone() for t in out[1:]]
    out[1].detach().mul_(2.0)                                   # the others are tensors of their own
    assert torch.equal(out[2], kept[1]) and torch.equal(out[3], kept[2])


def test_bad_index_is_raised_by_the_call_itself(oracle):
    import torch
    call, par, nb = _loss(oracle, torch.float64)
    bad = nb["bfirstneigh"].clone()
    bad[1, 2, 0] = 999
    want = call()[0].detach().clone()
    for _ in range(2):
        with pytest.raises(RuntimeError, match="neighbour index"):
            call(bad)
        assert torch.equal(call()[0].detach(), want)            # nothing is left behind for the next call


def test_gradients_of_a_batch_of_weights(oracle):
    """is_grads_batched hands the backward pass one wrapped tensor for all weight vectors: the Jacobian of the
    per-structure losses in one pass, and any other batch of weights."""
    import torch
    call, par, nb = _loss(oracle, torch.float64)
    one = [torch.autograd.grad(call()[0][k], par) for k in range(3)]
    w = torch.tensor([[1.0, 0.0, 0.0], [0.0, 1.0, 0.0], [0.0, 0.0, 1.0], [0.3, -1.1, 0.7]], dtype=torch.float64, device="cuda:0")
    got = torch.autograd.grad(call()[0], par, w, is_grads_batched=True)
    for i, g in enumerate(got):
        assert g.shape == (4,) + tuple(par[i].shape)
        want = torch.einsum("kb,b...->k...", w, torch.stack([o[i] for o in one]))
        # a product of three terms in another order
        assert torch.allclose(g, want, rtol=1e-13, atol=1e-15 * float(want.abs().max()))


def test_forward_derivative_of_the_gradient(oracle):
    """A weight vector with a tangent: the gradients carry the tangent's own gradients (they are linear in the weights)."""
    import torch
    import torch.autograd.forward_ad as fwad
    call, par, nb = _loss(oracle, torch.float64)
    w, t = (torch.tensor(v, dtype=torch.float64, device="cuda:0") for v in ([0.3, -1.1, 0.7], [1.5, 0.2, -0.4]))
    want, want_t = (torch.autograd.grad(call()[0], par, v) for v in (w, t))
    with fwad.dual_level():
        got = [fwad.unpack_dual(g) for g in torch.autograd.grad(call()[0], par, fwad.make_dual(w, t))]
        got = [(g.primal.clone(), None if g.tangent is None else g.tangent.clone()) for g in got]
    for (p, d), a, b in zip(got, want, want_t):
        assert d is not None
        assert torch.allclose(p, a, rtol=1e-13, atol=1e-15 * float(a.abs().max()))
        assert torch.allclose(d, b, rtol=1e-13, atol=1e-15 * float(b.abs().max()))


def test_gradients_are_tensors_of_their_own(oracle):
    """Each gradient has its own storage, no larger than it is: kept or saved alone it keeps nothing else."""
    import torch
    call, par, nb = _loss(oracle, torch.float64)
    grads = torch.autograd.grad(call()[0].sum(), par)
    assert len({g.untyped_storage().data_ptr() for g in grads}) == len(grads)
    for g, p in zip(grads, par):
        assert g.shape == p.shape and g.is_contiguous() and g.data_ptr() % 256 == 0
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size()
