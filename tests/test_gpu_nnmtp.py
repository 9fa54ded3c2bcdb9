"""GPU parity of the neural-network MTP operators (energy / force / virial, site energies,
descriptors) against the CPU oracle and the reference's committed outputs.  Bar: fp64 within
1e-10 relative, fp32 within 1e-4 / 1e-3 as for the linear MTP."""
import os

import numpy as np
import pytest

from ai2pot_amd import mtp_param, synth
from conftest import to_device

pytestmark = pytest.mark.gpu


def model_to_device(m, dtype, device="cuda:0"):
    import torch
    out = dict(m)
    for k in ("coeffs", "w0", "w1", "type_bias", "q_shifter", "q_scaler"):
        out[k] = torch.from_numpy(np.ascontiguousarray(m[k], np.float64)).to(dtype).to(device)
    for k in ("alpha_index_basic", "alpha_index_times", "alpha_moment_mapping", "type_map"):
        out[k] = torch.from_numpy(np.ascontiguousarray(m[k], np.int32)).to(device)
    return out


def op_args(m, md, d):
    return (m["chebyshev_size"], md["coeffs"], md["w0"], md["w1"], md["type_bias"], m["alpha_moments_count"],
            md["alpha_index_basic"], md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"],
            d["bilist"], d["bnumneigh"], d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], d["nghost"],
            m["rmax"], m["rmin"], md["q_shifter"], md["q_scaler"])


def run(m, nb, np_dtype=np.float64):
    import torch
    from ai2pot_amd import ops
    dtype = torch.float64 if np_dtype == np.float64 else torch.float32
    md = model_to_device(m, dtype)
    args = op_args(m, md, to_device(nb, dtype))
    e, f, v = ops.nnMtpToEFVOp(*args, 0.0, 0.0, None, None)
    e2, f2 = ops.nnMtpToEFOp(*args, 0.0, 0.0, None, None)
    es = ops.nnMtpToEsitesOp(*args, 0.0, 0.0, None, None)[0]
    desc = ops.nnMtpToDescriptorsOp(*(args[:2] + args[5:20]))[0]
    torch.cuda.synchronize()
    assert torch.equal(e, e2) and torch.equal(f, f2)
    return [t.cpu().numpy() for t in (e, f, v, es, desc)]


def close(a, b, tol=1e-10):
    return np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-300)


def structure(oracle, n, box, nt, seed, rcut, umax=120):
    lat, pos = synth.random_packed(n, list(box), 2.0, seed)
    return oracle.nblist(lat, synth.rng_randint(seed + 1, n, nt), pos, rcut, umax)


@pytest.mark.parametrize("level,nt,H", [(6, 1, 3), (8, 2, 7), (12, 2, 64), (16, 3, 20), (20, 4, 50), (22, 2, 100)])
def test_levels(oracle, level, nt, H):
    nb = synth.pack_batch([structure(oracle, 40, (8.5, 9.0, 9.5), nt, 21, 5.0),
                           structure(oracle, 25, (8.0, 7.5, 9.0), nt, 31, 5.0)])
    m = synth.nnmtp_model(mtp_param.mtp_param(level), nt, 8, H, 5.0, 1.8, 3200 + level, lo=-0.05, hi=0.05)
    e, f, v, es, desc = run(m, nb)
    er, fr, vr, esr = oracle.nnmtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr) and close(es, esr)
    assert np.all(es[1, 25:] == 0)
    lin = dict(m); lin["scaling"] = 1.0; lin["linear_coeffs"] = np.zeros(m["q_scaler"].size)
    assert close(desc, oracle.mtp_esites(lin, nb)[1])


@pytest.mark.parametrize("level,nt,H", [(8, 2, 7), (16, 3, 20)])
def test_against_reference_outputs(oracle, level, nt, H):
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "nnmtp.npz")) as z:
        g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L%02d/" % level)}
    lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
    ty = synth.rng_randint(22, 48, nt)
    m = synth.nnmtp_model(mtp_param.mtp_param(level), nt, 8, H, 5.0, 1.8, 3200 + level)
    o = oracle.nblist(lat, ty, pos, 5.0, 100)
    nb = synth.pack_batch([o, o])
    nb["brcs"][1] *= 1.01
    e, f, v, es, _ = run(m, nb)
    assert close(e, g["E"]) and close(f, g["F"]) and close(v, g["V"]) and close(es, g["esites"])


def test_ghosts_and_fp32(oracle):
    inum, ilist, numneigh, first, rcs, types, _ = structure(oracle, 64, (9.0, 9.5, 10.0), 2, 1004, 5.0, umax=150)
    nl = 40
    first = first.copy()
    first[first < 0] = 0
    nb = dict(binum=np.array([nl], np.int32), bilist=ilist[None, :nl].copy(), bnumneigh=numneigh[None, :nl].copy(),
              bfirstneigh=first[None, :nl].copy(), brcs=rcs[None, :nl].copy(), btypes=types[None, :].copy(),
              nghost=inum - nl)
    m = synth.nnmtp_model(mtp_param.mtp_param(10), 2, 8, 16, 5.0, 1.5, 3004)
    e, f, v, es, _ = run(m, nb)
    er, fr, vr, esr = oracle.nnmtp_efv(m, nb)
    assert f.shape == (1, inum, 3)
    assert close(e, er) and close(f, fr) and close(v, vr) and close(es, esr)
    e32, f32, v32, es32, _ = run(m, nb, np.float32)
    assert close(e32, er, 1e-4) and close(f32, fr, 1e-3) and close(v32, vr, 1e-3) and close(es32, esr, 1e-4)


def test_errors(oracle):
    import torch
    from ai2pot_amd import ops
    nb = synth.pack_batch([structure(oracle, 30, (8.5, 9.0, 9.5), 2, 21, 5.0)])
    m = synth.nnmtp_model(mtp_param.mtp_param(8), 2, 8, 5, 5.0, 1.8, 5)
    md = model_to_device(m, torch.float64)
    args = list(op_args(m, md, to_device(nb, torch.float64)))
    with pytest.raises(RuntimeError):                       # w0 of the wrong size
        ops.nnMtpToEFVOp(*(args[:2] + [md["w0"][:-1].contiguous()] + args[3:]))
    with pytest.raises(RuntimeError):                       # ZBL switched on without its parameter tensors
        ops.nnMtpToEFVOp(*args, 2.0, 1.0, None, None)


def loss_inputs(oracle, level, nt, H, sizes=(48, 30, 37)):
    lists = [structure(oracle, n, (8.5 + 0.1 * i, 9.0, 9.5), nt, 21 + 5 * i, 5.0) for i, n in enumerate(sizes)]
    nb = synth.pack_batch(lists)
    B, P = nb["bilist"].shape
    m = synth.nnmtp_model(mtp_param.mtp_param(level), nt, 8, H, 5.0, 1.5, 3300 + level)
    labels = dict(energy=synth.rng_normal(1, B, -4 * 40, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    return m, nb, labels


def gpu_loss(m, nb, labels, w, exact, want_grad=True):
    import torch
    from ai2pot_amd import ops
    md = model_to_device(m, torch.float64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    args = op_args(m, md, to_device(nb, torch.float64))
    r = ops.nnmtp_loss_step(w[0], w[1], w[2], t(labels["energy"]), t(labels["force"]), t(labels["virial"]), *args,
                            want_grad=want_grad, exact_gradient=exact)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in r.items()}


@pytest.mark.parametrize("level,nt,H", [(8, 2, 7), (10, 1, 12), (12, 3, 5)])
def test_loss_step_complete_derivative(oracle, level, nt, H):
    """exact_gradient=True against the oracle's forward-mode derivative of the loss (which agrees
    with finite differences)."""
    m, nb, labels = loss_inputs(oracle, level, nt, H)
    w = (1.0, 0.7, 0.3)
    got = gpu_loss(m, nb, labels, w, True)
    ref = oracle.nnmtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "energy", "force", "virial", "dcoeffs", "dw0", "dw1", "dbias"):
        assert close(got[k], ref[k]), k
    fwd = gpu_loss(m, nb, labels, w, True, want_grad=False)
    assert np.array_equal(fwd["bloss"], got["bloss"]) and "dcoeffs" not in fwd


@pytest.mark.parametrize("sizes", [(1, 2, 3), (4, 5, 16), (63, 68), (256, 257), (275, 15)], ids=str)
def test_gradients_by_number_of_rows(oracle, sizes):
    """The rows' gradients are summed in four runs, 64 rows and then sixteen of a species at a time, as those of the linear potentials."""
    boxes = [max(4.0, (n / 0.05) ** (1 / 3)) for n in sizes]
    nb = synth.pack_batch([structure(oracle, n, (a, a, a), 3, 41 + n, 4.0) for n, a in zip(sizes, boxes)])
    B, P = nb["bilist"].shape
    m = synth.nnmtp_model(mtp_param.mtp_param(8), 3, 8, 5, 4.0, 1.0, 3408, lo=-0.05, hi=0.05)
    labels = dict(energy=synth.rng_normal(1, B, -4 * 40, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w, True), oracle.nnmtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dw0", "dw1", "dbias"):
        assert close(got[k], ref[k]), k


@pytest.mark.parametrize("level", [8, 12, 16])              # 9, 29 and 92 inputs; 64 threads, and 256 for the loss gradient
@pytest.mark.parametrize("H", [1, 4, 5, 16, 33, 65, 257])
def test_readout_by_neighbouring_lanes(oracle, level, H):
    """Neurons and inputs summed by sixteen lanes each down to one, and more of them than the workgroup has threads: energies,
    forces, virials and the loss gradient against the oracle, fp64 1e-10."""
    m, nb, labels = loss_inputs(oracle, level, 2, H, sizes=(13, 9))
    e, f, v, _, _ = run(m, nb)
    er, fr, vr, _ = oracle.nnmtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w, True), oracle.nnmtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dw0", "dw1", "dbias"):
        assert close(got[k], ref[k]), k


@pytest.mark.parametrize("level", [14, 18, 20])            # 52, 163 and 288 inputs: 64 threads, 256, and more inputs than those
@pytest.mark.parametrize("H", [1, 15, 16, 17, 64, 65, 200])
def test_readout_in_rounds(oracle, level, H):
    """Neurons in more rounds than one, with wavefronts that have none in the last, and a second round of inputs, in both precisions:
    energies, forces and virials against the oracle, fp64 1e-10, fp32 1e-4 and 1e-3 as above."""
    m, nb, _ = loss_inputs(oracle, level, 2, H, sizes=(13, 9))
    er, fr, vr, esr = oracle.nnmtp_efv(m, nb)
    for dt, te, tf in ((np.float64, 1e-10, 1e-10), (np.float32, 1e-4, 1e-3)):
        e, f, v, es, _ = run(m, nb, dt)
        assert close(e, er, te) and close(es, esr, te) and close(f, fr, tf) and close(v, vr, tf)


def many_inputs(oracle, S, H):
    """A table of one radial function whose first S basic moments are the scalar ones: more than 96 inputs leave no room for the
    tangents of the inputs where they wait otherwise."""
    basic = [(0, a, b, c) for a in range(9) for b in range(9 - a) for c in range(9 - a - b)]
    tables = dict(alpha_moments_count=len(basic), alpha_index_basic=np.array(basic, np.int32),
                  alpha_index_times=np.zeros((0, 4), np.int32), alpha_moment_mapping=np.arange(S, dtype=np.int32), nmus=1)
    _, nb, labels = loss_inputs(oracle, 8, 2, H, sizes=(11, 7))
    return synth.nnmtp_model(tables, 2, 6, H, 5.0, 1.5, 3400), nb, labels


@pytest.mark.parametrize("S", [96, 97, 130])
@pytest.mark.parametrize("H", [1, 5])
def test_loss_step_of_many_inputs(oracle, S, H):
    """The complete derivative against the oracle, fp64 1e-10; and, with both formulas, the gradient with and without inputs
    whose weights are zero."""
    m, nb, labels = many_inputs(oracle, S, H)
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w, True), oracle.nnmtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dw0", "dw1", "dbias"):
        assert close(got[k], ref[k]), k
    few = many_inputs(oracle, 90, H)[0]
    w0 = np.zeros((2, H, S))
    w0[:, :, :90] = np.reshape(few["w0"], (2, H, 90))
    m = dict(m, coeffs=few["coeffs"], w0=w0.reshape(np.shape(m["w0"])), w1=few["w1"], type_bias=few["type_bias"])
    for k in ("q_shifter", "q_scaler"):
        m[k] = np.concatenate([few[k], m[k][90:]])
    for exact in (False, True):
        a, b = gpu_loss(m, nb, labels, w, exact), gpu_loss(few, nb, labels, w, exact)
        B = len(nb["binum"])
        assert close(a["dw0"].reshape(B, 2, H, S)[..., :90], b["dw0"].reshape(B, 2, H, 90), 1e-12)
        for k in ("bloss", "dcoeffs", "dw1", "dbias"):
            assert close(a[k], b[k], 1e-12), k


@pytest.mark.parametrize("level", [8, 12, 16, 20])
@pytest.mark.parametrize("H", [3, 20, 65])
def test_readout_of_an_infinite_input(oracle, level, H):
    """An input that overflows (the last one: lanes with no input of their own must not count it) saturates every neuron at
    plus or minus one: energies are sums of the second layer's weights and the forces vanish.  fp64 1e-13: H additions."""
    m, nb, _ = loss_inputs(oracle, level, 2, H, sizes=(13, 9))
    m["q_scaler"] = m["q_scaler"].copy()
    m["q_scaler"][-1] = 5e-324
    lin = dict(m); lin["scaling"] = 1.0; lin["linear_coeffs"] = np.zeros(m["q_scaler"].size)
    last = oracle.mtp_esites(lin, nb)[1][..., -1] - m["q_shifter"][-1]
    w0, w1 = np.reshape(m["w0"], (2, H, -1)), np.reshape(m["w1"], (2, H))
    ref = np.zeros(last.shape)
    for b, n in enumerate(nb["binum"]):
        for ii in range(n):
            t = nb["btypes"][b, nb["bilist"][b, ii]]
            ref[b, ii] = m["type_bias"][t] + np.sum(w1[t] * np.sign(w0[t, :, -1] * last[b, ii]))
    e, f, v, es, _ = run(m, nb)
    assert close(es, ref, 1e-13) and close(e, ref.sum(1), 1e-13) and not f.any() and not v.any()


@pytest.mark.parametrize("level,nt,H", [(8, 2, 7), (16, 3, 20)])
def test_loss_step_reference_formulas(oracle, level, nt, H):
    """exact_gradient=False (the operators' default) against the committed output of the reference's
    NNMtpLoss::find_loss_backward; and the two modes agree where the reference's formulas are
    complete: on w1 and type_bias always, on everything for an energy-only loss."""
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "nnmtp.npz")) as z:
        g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L%02d/" % level)}
    lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
    ty = synth.rng_randint(22, 48, nt)
    m = synth.nnmtp_model(mtp_param.mtp_param(level), nt, 8, H, 5.0, 1.8, 3200 + level)
    o = oracle.nblist(lat, ty, pos, 5.0, 100)
    nb = synth.pack_batch([o, o])
    nb["brcs"][1] *= 1.01
    B, P = nb["bilist"].shape
    labels = dict(energy=synth.rng_normal(1, B, -4 * 48, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    got = gpu_loss(m, nb, labels, (1.0, 0.7, 0.3), False)
    for k in ("bloss", "energy", "force", "virial", "dcoeffs", "dw0", "dw1", "dbias"):
        assert close(got[k], g["loss_" + k]), k
    full = gpu_loss(m, nb, labels, (1.0, 0.7, 0.3), True)
    assert close(full["dw1"], got["dw1"]) and close(full["dbias"], got["dbias"])
    assert not close(full["dcoeffs"], got["dcoeffs"], 1e-4)          # the omitted terms are not small
    e_only_ref, e_only_full = (gpu_loss(m, nb, labels, (1.0, 0.0, 0.0), x) for x in (False, True))
    for k in ("dcoeffs", "dw0", "dw1", "dbias"):
        assert close(e_only_ref[k], e_only_full[k]), k


def test_loss_autograd_contract(oracle):
    """One output, bloss[B]; backward = grad_output @ per-structure gradients to coeffs, w0, w1, type_bias."""
    import torch
    from ai2pot_amd import ops
    m, nb, labels = loss_inputs(oracle, 8, 2, 7)
    md = model_to_device(m, torch.float64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    for k in ("coeffs", "w0", "w1", "type_bias"):
        md[k].requires_grad_(True)
    args = op_args(m, md, to_device(nb, torch.float64))
    out = ops.nnMtpToLossOp(1.0, 0.7, 0.3, t(labels["energy"]), t(labels["force"]), t(labels["virial"]), *args,
                            0.0, 0.0, None, None, exact_gradient=True)
    assert len(out) == 1 and out[0].shape == (3,)
    out[0].mean().backward()
    ref = oracle.nnmtp_loss_step(m, nb, (1.0, 0.7, 0.3), labels)
    for k, g in (("coeffs", "dcoeffs"), ("w0", "dw0"), ("w1", "dw1"), ("type_bias", "dbias")):
        assert close(md[k].grad.cpu().numpy(), ref[g].mean(0)), k
    # energy + force variant = zero virial weight
    for k in ("coeffs", "w0", "w1", "type_bias"):
        md[k].grad = None
    out2 = ops.nnMtpToEFLossOp(1.0, 0.7, t(labels["energy"]), t(labels["force"]), *args, 0.0, 0.0, None, None,
                               exact_gradient=True)
    out2[0].sum().backward()
    ref2 = oracle.nnmtp_loss_step(m, nb, (1.0, 0.7, 0.0), labels)
    assert close(out2[0].detach().cpu().numpy(), ref2["bloss"])
    assert close(md["w0"].grad.cpu().numpy(), ref2["dw0"].sum(0))


@pytest.mark.parametrize("level,nt,H", [(8, 2, 7), (10, 1, 6)])
def test_site_energy_backward(oracle, level, nt, H):
    """Autograd of nnMtpToEsitesOp against the oracle's forward-mode derivative (two species, a padded
    structure) and, for one species, against the committed output of the reference's
    find_e_sites_backward (for several species the reference mis-assigns its w0 / w1 rows)."""
    import torch
    from ai2pot_amd import ops
    lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
    ty = synth.rng_randint(22, 48, nt)
    m = synth.nnmtp_model(mtp_param.mtp_param(level), nt, 8, H, 5.0, 1.8, 3200 + level)
    o = oracle.nblist(lat, ty, pos, 5.0, 100)
    nb = synth.pack_batch([o, o])
    nb["brcs"][1] *= 1.01
    B, P = nb["bilist"].shape
    gout = synth.rng_normal(4, B * P).reshape(B, P)
    md = model_to_device(m, torch.float64)
    for k in ("coeffs", "w0", "w1", "type_bias"):
        md[k].requires_grad_(True)
    args = op_args(m, md, to_device(nb, torch.float64))
    es = ops.nnMtpToEsitesOp(*args, 0.0, 0.0, None, None)[0]
    (es * torch.from_numpy(gout).to("cuda:0")).sum().backward()
    ref = oracle.nnmtp_esites_bwd(m, nb, gout)
    for k, r in zip(("coeffs", "w0", "w1", "type_bias"), ref):
        assert close(md[k].grad.cpu().numpy(), r.sum(0)), k
    if nt == 1:
        with np.load(os.path.join(os.path.dirname(__file__), "golden", "nnmtp.npz")) as z:
            g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L%02d/" % level)}
        for k, gk in (("coeffs", "es_dcoeffs"), ("w0", "es_dw0"), ("w1", "es_dw1"), ("type_bias", "es_dbias")):
            assert close(md[k].grad.cpu().numpy(), g[gk].sum(0)), k
