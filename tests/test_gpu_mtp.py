"""GPU parity of the linear-MTP energy / force / virial path and of the training-loss step
against the CPU oracle.  Bar: fp64 within 1e-10 relative (the tolerance the task states for
MTP energies, forces and virials; gradients are held to the same bar against the oracle's
independent forward-mode derivative)."""
import numpy as np
import pytest

from ai2pot_amd import mtp_param, synth
from conftest import to_device

pytestmark = pytest.mark.gpu


def model_to_device(m, dtype, device="cuda:0"):
    import torch
    out = dict(m)
    for k in ("coeffs", "linear_coeffs", "type_bias", "q_scaler"):
        out[k] = torch.from_numpy(np.ascontiguousarray(m[k], np.float64)).to(dtype).to(device)
    for k in ("alpha_index_basic", "alpha_index_times", "alpha_moment_mapping", "type_map"):
        out[k] = torch.from_numpy(np.ascontiguousarray(m[k], np.int32)).to(device)
    return out


def gpu_efv(m, nb, np_dtype=np.float64, virial=True):
    import torch
    from ai2pot_amd import ops
    dtype = torch.float64 if np_dtype == np.float64 else torch.float32
    md = model_to_device(m, dtype)
    d = to_device(nb, dtype)
    fn = ops.linearMtpToEFVOp if virial else ops.linearMtpToEFOp
    out = fn(m["chebyshev_size"], m["scaling"], md["coeffs"], md["linear_coeffs"], md["type_bias"],
             m["alpha_moments_count"], md["alpha_index_basic"], md["alpha_index_times"],
             md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"],
             d["brcs"], d["btypes"], md["type_map"], d["nghost"], m["rmax"], m["rmin"], md["q_scaler"],
             0.0, 0.0, None, None)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in out]


def close(a, b, tol=1e-10):
    return np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-300)


def structure(oracle, n, box, nt, seed, rcut, umax=120, dmin=2.0):
    lat, pos = synth.random_packed(n, list(box), dmin, seed)
    ty = synth.rng_randint(seed + 1, n, nt)
    return oracle.nblist(lat, ty, pos, rcut, umax)


def test_mos2_known_answer(oracle):
    """Set-up of the reference's unit test (mtpr/tests/test_linearMtp.cc, level 16):
    E = -0.938157350795572, F[1][z] = -0.520135157048249."""
    lat, types, frac = synth.mos2_fixture()
    nb = synth.pack_batch([oracle.nblist(lat, types, frac, 5.0, 20, is_cart=False, sort=True)])
    m = synth.mtp_model_closed_form(mtp_param.mtp_param(16))
    e, f, v = gpu_efv(m, nb)
    assert abs(e[0] - (-0.938157350795572)) < 1e-11
    assert abs(f[0, 1, 2] - (-0.520135157048249)) < 1e-11
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)


@pytest.mark.parametrize("level,nt,K", [(6, 1, 8), (8, 2, 8), (10, 1, 8), (12, 2, 6), (16, 3, 8), (20, 4, 10),
                                        (22, 2, 12)])
def test_levels(oracle, level, nt, K):
    o = structure(oracle, 40, (8.5, 9.0, 9.5), nt, 21, 5.0)
    o2 = structure(oracle, 25, (8.0, 7.5, 9.0), nt, 31, 5.0)
    nb = synth.pack_batch([o, o2])
    m = synth.mtp_model(mtp_param.mtp_param(level), nt, K, 5.0, 1.8, 3000 + level, lo=-0.05, hi=0.05)
    m["q_scaler"] = np.linspace(0.7, 1.4, m["q_scaler"].size)
    e, f, v = gpu_efv(m, nb)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)
    e2, f2 = gpu_efv(m, nb, virial=False)
    assert close(e2, er) and close(f2, fr)


def test_config1_full_size(oracle):
    """Benchmark configuration 1: 216-atom diamond cell, level 10, one species, rcut 5, rmin 0.5."""
    lat, pos = synth.diamond_cell()
    ty = np.zeros(216, np.int32)
    nb = synth.pack_batch([oracle.nblist(lat, ty, pos, 5.0, 200)])
    m = synth.mtp_model(mtp_param.mtp_param(10), 1, 8, 5.0, 0.5, 3001, type_map=[14])
    e, f, v = gpu_efv(m, nb)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)


def test_config3_reduced_and_ghosts(oracle):
    """Configuration 3's model (level 20, 4 species, K = 10, rmax 5.5, rmin 1.8) on 512 atoms at
    its density, plus the same list seen as 400 local atoms + 112 ghosts."""
    o = structure(oracle, 512, (21.72, 21.72, 21.72), 4, 1004, 5.5, umax=200)
    m = synth.mtp_model(mtp_param.mtp_param(20), 4, 10, 5.5, 1.8, 3004, lo=-0.05, hi=0.05,
                        type_map=[75, 41, 16, 34])
    nb = synth.pack_batch([o])
    e, f, v = gpu_efv(m, nb)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)
    assert np.abs(f.sum(1)).max() < 1e-9 * np.abs(f).max()
    inum, ilist, numneigh, first, rcs, types, _ = o
    nl = 400
    first = first.copy()
    first[first < 0] = 0
    nbg = dict(binum=np.array([nl], np.int32), bilist=ilist[None, :nl].copy(), bnumneigh=numneigh[None, :nl].copy(),
               bfirstneigh=first[None, :nl].copy(), brcs=rcs[None, :nl].copy(), btypes=types[None, :].copy(),
               nghost=inum - nl)
    eg, fg, vg = gpu_efv(m, nbg)
    er, fr, vr = oracle.mtp_efv(m, nbg)
    assert fg.shape == (1, inum, 3)
    assert close(eg, er) and close(fg, fr) and close(vg, vr)


def test_config3_full_size(oracle):
    """Benchmark configuration 3 at full size: 8192 atoms in one cell, level 20, 4 species, K = 10,
    rmax 5.5, rmin 1.8, against the oracle; the net force vanishes."""
    lat, pos = synth.random_packed(8192, [64.0, 51.2, 50.0], 2.0, 1004)
    ty = synth.rng_randint(2004, 8192, 4)
    nb = synth.pack_batch([oracle.nblist(lat, ty, pos, 5.5, 200)])
    m = synth.mtp_model(mtp_param.mtp_param(20), 4, 10, 5.5, 1.8, 3004, lo=-0.05, hi=0.05,
                        type_map=[75, 41, 16, 34])
    e, f, v = gpu_efv(m, nb)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr) and close(v, vr)
    assert np.abs(f.sum(1)).max() < 1e-9 * np.abs(f).max()


def test_config4_full_size(oracle):
    """Benchmark configuration 4 at full size: one training step over 64 structures of 128 atoms,
    level 16, 3 species.  Every per-structure result of the batch (loss, energy, forces, virial,
    gradient rows) equals the one-structure call's bit for bit; six of the structures are checked
    against the oracle (the whole batch takes it 20 s)."""
    rho = synth.rng_uniform(1005, 64, 0.03, 0.05)
    lists = []
    for b in range(64):
        Lb = (128.0 / rho[b]) ** (1.0 / 3.0)
        lat, pos = synth.random_packed(128, [Lb, Lb, Lb], 2.0, 11005 + b)
        lists.append(oracle.nblist(lat, synth.rng_randint(21005 + b, 128, 3), pos, 5.0, 200))
    nb = synth.pack_batch(lists)
    m = synth.mtp_model(mtp_param.mtp_param(16), 3, 8, 5.0, 0.0, 3005)
    B, P = nb["bilist"].shape
    labels = dict(energy=synth.rng_normal(4005, B * P, -4.0, 0.2).reshape(B, P).sum(1),
                  force=synth.rng_normal(4006, B * P * 3, 0.0, 1.0).reshape(B, P, 3),
                  virial=synth.rng_normal(4007, B * 9, 0.0, 0.5).reshape(B, 9))
    w = (1.0, 1.0, 1.0)
    got = gpu_loss(m, nb, labels, w)
    keys = ("bloss", "energy", "force", "virial", "dcoeffs", "dlinear", "dbias")
    pick = [0, 7, 21, 38, 50, 63]
    sub = {k: (v[pick].copy() if hasattr(v, "shape") else v) for k, v in nb.items()}
    sub_labels = {k: v[pick] for k, v in labels.items()}
    ref = oracle.mtp_loss_step(m, sub, w, sub_labels)
    for k in keys:
        assert close(got[k][pick], ref[k]), k
    for b in (0, 38, 63):
        one = {k: (v[b:b + 1].copy() if hasattr(v, "shape") else v) for k, v in nb.items()}
        r1 = gpu_loss(m, one, {k: v[b:b + 1] for k, v in labels.items()}, w)
        for k in keys:
            assert np.array_equal(r1[k][0], got[k][b]), k


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_reproducible(oracle, np_dtype):
    """Two runs give bit-identical results: the pairs claim their segment entries in an order that
    changes from run to run, the sums over a segment do not depend on it."""
    nb = synth.pack_batch([structure(oracle, 400, (20.0, 21.0, 19.0), 2, 31, 5.0)])
    m = synth.mtp_model(mtp_param.mtp_param(10), 2, 8, 5.0, 0.5, 3032, lo=-0.05, hi=0.05)
    a = gpu_efv(m, nb, np_dtype)
    b = gpu_efv(m, nb, np_dtype)
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


def test_fp32_runs_close_to_fp64(oracle):
    o = structure(oracle, 40, (8.5, 9.0, 9.5), 2, 21, 5.0)
    nb = synth.pack_batch([o])
    m = synth.mtp_model(mtp_param.mtp_param(12), 2, 8, 5.0, 1.8, 3012)
    e, f, v = gpu_efv(m, nb, np.float32)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er, 1e-4) and close(f, fr, 1e-3) and close(v, vr, 1e-3)


def loss_inputs(oracle, level, nt, sizes=(48, 30, 37), P=None):
    lists = [structure(oracle, n, (8.5 + 0.1 * i, 9.0, 9.5), nt, 21 + 5 * i, 5.0) for i, n in enumerate(sizes)]
    nb = synth.pack_batch(lists, natoms_pad=P)
    B, P = nb["bilist"].shape
    m = synth.mtp_model(mtp_param.mtp_param(level), nt, 8, 5.0, 0.0 if level == 16 else 1.5, 3100 + level)
    m["q_scaler"] = np.linspace(0.8, 1.3, m["q_scaler"].size)
    labels = dict(energy=synth.rng_normal(1, B, -4 * 40, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    return m, nb, labels


def gpu_loss(m, nb, labels, w, want_grad=True):
    import torch
    from ai2pot_amd import ops
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    r = ops.mtp_loss_step(w[0], w[1], w[2], t(labels["energy"]), t(labels["force"]), t(labels["virial"]),
                          m["chebyshev_size"], m["scaling"], md["coeffs"], md["linear_coeffs"], md["type_bias"],
                          m["alpha_moments_count"], md["alpha_index_basic"], md["alpha_index_times"],
                          md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
                          d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], 0, m["rmax"], m["rmin"],
                          md["q_scaler"], want_grad=want_grad)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in r.items()}


@pytest.mark.parametrize("level,nt", [(8, 2), (10, 1), (12, 3)])
def test_loss_step(oracle, level, nt):
    m, nb, labels = loss_inputs(oracle, level, nt)
    w = (1.0, 0.7, 0.3)
    got = gpu_loss(m, nb, labels, w)
    ref = oracle.mtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "rmse", "energy", "force", "virial", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], ref[k]), k
    fwd = gpu_loss(m, nb, labels, w, want_grad=False)
    assert np.array_equal(fwd["bloss"], got["bloss"]) and "dcoeffs" not in fwd


@pytest.mark.parametrize("sizes", [(1, 2, 3), (4, 5, 16), (63, 68), (256, 257), (275, 15)], ids=str)
def test_gradients_by_number_of_rows(oracle, sizes):
    """The rows' gradients are summed in four runs, 64 rows and then sixteen of a species at a time: structures that leave runs empty, fill
    them, or have one row more.  fp64 against the oracle, 1e-10."""
    boxes = [max(4.0, (n / 0.05) ** (1 / 3)) for n in sizes]
    nb = synth.pack_batch([structure(oracle, n, (a, a, a), 3, 41 + n, 4.0) for n, a in zip(sizes, boxes)])
    B, P = nb["bilist"].shape
    m = synth.mtp_model(mtp_param.mtp_param(8), 3, 8, 4.0, 1.0, 3108)
    m["q_scaler"] = np.linspace(0.8, 1.3, m["q_scaler"].size)
    labels = dict(energy=synth.rng_normal(1, B, -4 * 40, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    w = (1.0, 0.7, 0.3)
    got, ref = gpu_loss(m, nb, labels, w), oracle.mtp_loss_step(m, nb, w, labels)
    for k in ("bloss", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], ref[k]), k


def test_loss_level16_against_golden(oracle):
    """Level 16 (configuration 4's level) against the committed output of the reference's own
    find_loss_backward (tests/golden/mtp.npz), where the oracle's forward-mode derivative is slow."""
    import os
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "mtp.npz")) as z:
        g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L16/")}
    lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
    ty = synth.rng_randint(22, 48, 3)
    m = synth.mtp_model(mtp_param.mtp_param(16), 3, 8, 5.0, 1.8, 3016)
    o = oracle.nblist(lat, ty, pos, 5.0, 100)
    nb = synth.pack_batch([o, o])
    nb["brcs"][1] *= 1.01
    B, P = nb["bilist"].shape
    labels = dict(energy=synth.rng_normal(1, B, -4 * 48, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    got = gpu_loss(m, nb, labels, (1.0, 0.7, 0.3))
    for k in ("bloss", "rmse", "energy", "force", "virial", "dcoeffs", "dlinear", "dbias"):
        assert close(got[k], g["loss_" + k]), k


def test_loss_autograd_contract(oracle):
    """The operator returns [bloss, e_rmse, f_rmse, v_rmse] and back-propagates
    grad_output @ dloss/dtheta to coeffs, linear_coeffs and type_bias only."""
    import torch
    from ai2pot_amd import ops
    m, nb, labels = loss_inputs(oracle, 8, 2)
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    for k in ("coeffs", "linear_coeffs", "type_bias"):
        md[k].requires_grad_(True)
    out = ops.linearMtpToLossOp(1.0, 0.7, 0.3, t(labels["energy"]), t(labels["force"]), t(labels["virial"]),
                                m["chebyshev_size"], m["scaling"], md["coeffs"], md["linear_coeffs"],
                                md["type_bias"], m["alpha_moments_count"], md["alpha_index_basic"],
                                md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"],
                                d["bilist"], d["bnumneigh"], d["bfirstneigh"], d["brcs"], d["btypes"],
                                md["type_map"], 0, m["rmax"], m["rmin"], md["q_scaler"], 0.0, 0.0, None, None)
    assert len(out) == 4 and out[0].shape == (3,) and all(o.shape == (1,) for o in out[1:])
    out[0].mean().backward()
    ref = oracle.mtp_loss_step(m, nb, (1.0, 0.7, 0.3), labels)
    assert close(md["coeffs"].grad.cpu().numpy(), ref["dcoeffs"].mean(0))
    assert close(md["linear_coeffs"].grad.cpu().numpy(), ref["dlinear"].mean(0))
    assert close(md["type_bias"].grad.cpu().numpy(), ref["dbias"].mean(0))


def esites_args(m, md, d):
    return (m["chebyshev_size"], m["scaling"], md["coeffs"], md["linear_coeffs"], md["type_bias"],
            m["alpha_moments_count"], md["alpha_index_basic"], md["alpha_index_times"],
            md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"],
            d["brcs"], d["btypes"], md["type_map"], d["nghost"], m["rmax"], m["rmin"], md["q_scaler"])


@pytest.mark.parametrize("level,nt", [(8, 2), (10, 1), (16, 3), (20, 2)])
def test_site_energies_and_descriptors(oracle, level, nt):
    """linearMtpToEsitesOp / linearMtpToDescriptorsOp against the oracle (itself pinned to the
    reference's committed outputs), with a padded structure and, at level 20, the wide kernel."""
    import torch
    from ai2pot_amd import ops
    m, nb, _ = loss_inputs(oracle, level, nt, sizes=(48, 30), P=52)
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    args = esites_args(m, md, d)
    es = ops.linearMtpToEsitesOp(*args, 0.0, 0.0, None, None)[0]
    desc = ops.linearMtpToDescriptorsOp(*(args[:3] + args[5:20]))[0]
    es_ref, desc_ref = oracle.mtp_esites(m, nb)
    assert es.shape == es_ref.shape and desc.shape == desc_ref.shape
    assert close(es.cpu().numpy(), es_ref) and close(desc.cpu().numpy(), desc_ref)
    assert np.all(es.cpu().numpy()[1, 30:] == 0) and np.all(desc.cpu().numpy()[1, 30:] == 0)
    e = ops.linearMtpToEFVOp(*args, 0.0, 0.0, None, None)[0]
    assert close(es.sum(1).cpu().numpy(), e.cpu().numpy())
    if level > 10:
        return
    B, P = nb["bilist"].shape
    gout = synth.rng_normal(4, B * P).reshape(B, P)
    dc, dl, db = ops.mtp_esites_backward(torch.from_numpy(gout).to("cuda:0"), *args)
    rc, rl, rb = oracle.mtp_esites_bwd(m, nb, gout)
    assert close(dc.cpu().numpy(), rc) and close(dl.cpu().numpy(), rl) and close(db.cpu().numpy(), rb)


def test_site_energies_against_golden_and_autograd(oracle):
    """Level 16 against the committed outputs of the reference's find_e_sites, find_descriptors and
    find_e_sites_backward; then the operator's autograd contract: gradients reach coeffs,
    linear_coeffs and type_bias, summed over structures and rows (linearMtpOp.cc:4002-4005)."""
    import os
    import torch
    from ai2pot_amd import ops
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "mtp.npz")) as z:
        g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L16/")}
    lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
    ty = synth.rng_randint(22, 48, 3)
    m = synth.mtp_model(mtp_param.mtp_param(16), 3, 8, 5.0, 1.8, 3016)
    o = oracle.nblist(lat, ty, pos, 5.0, 100)
    nb = synth.pack_batch([o, o])
    nb["brcs"][1] *= 1.01
    B, P = nb["bilist"].shape
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    for k in ("coeffs", "linear_coeffs", "type_bias"):
        md[k].requires_grad_(True)
    args = esites_args(m, md, d)
    es = ops.linearMtpToEsitesOp(*args, 0.0, 0.0, None, None)[0]
    desc = ops.linearMtpToDescriptorsOp(*(args[:3] + args[5:20]))[0]
    assert close(es.detach().cpu().numpy(), g["esites"]) and close(desc.cpu().numpy(), g["desc"])
    assert not desc.requires_grad
    gout = synth.rng_normal(4, B * P).reshape(B, P)
    (es * torch.from_numpy(gout).to("cuda:0")).sum().backward()
    assert close(md["coeffs"].grad.cpu().numpy(), g["es_dcoeffs"].sum(0))
    assert close(md["linear_coeffs"].grad.cpu().numpy(), g["es_dlinear"].sum(0))
    assert close(md["type_bias"].grad.cpu().numpy(), g["es_dbias"].sum(0))


def basis_args(m, md, d, coeffs, brcs):
    import torch
    n_moms = m["alpha_moments_count"]
    mus4moms = torch.zeros((n_moms, 1), dtype=torch.int32, device="cuda:0")       # only its first dimension is read
    num_mus4moms = torch.zeros((n_moms,), dtype=torch.int32, device="cuda:0")
    return (md["alpha_index_basic"], md["alpha_index_times"], md["alpha_moment_mapping"], num_mus4moms, mus4moms,
            torch.tensor(m["nmus"], dtype=torch.int32), int(md["type_map"].numel()), m["chebyshev_size"], m["scaling"],
            coeffs, d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"], brcs, d["btypes"], int(brcs.shape[2]),
            m["rmax"], m["rmin"])


@pytest.mark.parametrize("level,nt", [(8, 2), (10, 1), (16, 3), (20, 2)])
def test_legacy_basis_operator(oracle, level, nt):
    """mtpBasisOp: forward = the scalar moments; backward for weights w of the moments against the oracle
    (pinned to the reference's MtpBasis::find_val_der + find_der_backward), with a padded structure and, at
    level 20, the wide kernel; fp32 to its own tolerance."""
    import torch
    from ai2pot_amd import ops
    m, nb, _ = loss_inputs(oracle, level, nt, sizes=(48, 30), P=52)
    B, P = nb["bilist"].shape
    S = m["alpha_moment_mapping"].size
    w = synth.rng_normal(5, B * P * S).reshape(B, P, S)
    want_c = level <= 16
    drcs_ref, dc_ref = oracle.mtp_basis_bwd(m, nb, w, want_dcoeffs=want_c)
    _, desc_ref = oracle.mtp_esites(m, nb)
    for dtype, tol in ((torch.float64, 1e-10), (torch.float32, 2e-4)):
        md = model_to_device(m, dtype)
        d = to_device(nb, dtype)
        coeffs = md["coeffs"].clone().requires_grad_(want_c)
        brcs = d["brcs"].clone().requires_grad_(True)
        val = ops.mtpBasisOp(*basis_args(m, md, d, coeffs, brcs))[0]
        assert val.shape == desc_ref.shape and close(val.detach().cpu().numpy(), desc_ref, tol)
        (val * torch.from_numpy(w).to(dtype).to("cuda:0")).sum().backward()
        got = brcs.grad.cpu().numpy()
        assert got.shape == drcs_ref.shape and close(got, drcs_ref, tol)
        beyond = np.arange(got.shape[2])[None, None, :] >= nb["bnumneigh"][:, :, None]
        assert np.all(got[beyond] == 0) and np.all(got[1, 30:] == 0)
        if want_c:
            assert coeffs.grad.shape == coeffs.shape and close(coeffs.grad.cpu().numpy().ravel(), dc_ref.sum(0), tol)
    # one gradient only: the other pass is skipped
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    wt = torch.from_numpy(w).to("cuda:0")
    only_r, none_c = ops.mtp_basis_backward(wt, m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"],
                                            md["alpha_index_basic"], md["alpha_index_times"], md["alpha_moment_mapping"],
                                            m["nmus"], nt, d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"],
                                            d["brcs"], d["btypes"], m["rmax"], m["rmin"], want_dcoeffs=False)
    assert none_c is None and close(only_r.cpu().numpy(), drcs_ref)


def test_legacy_basis_operator_against_golden(oracle):
    """Levels 8 and 16 against the committed outputs of the reference's MtpBasis::find_val_der and
    find_der_backward (dense derivative arrays contracted with the weights)."""
    import os
    import torch
    from ai2pot_amd import ops
    for level, nt in ((8, 2), (16, 3)):
        with np.load(os.path.join(os.path.dirname(__file__), "golden", "mtp.npz")) as z:
            g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L%02d/" % level)}
        lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
        ty = synth.rng_randint(22, 48, nt)
        m = synth.mtp_model(mtp_param.mtp_param(level), nt, 8, 5.0, 1.8, 3000 + level)
        o = oracle.nblist(lat, ty, pos, 5.0, 100)
        nb = synth.pack_batch([o, o])
        nb["brcs"][1] *= 1.01
        B, P = nb["bilist"].shape
        S = m["alpha_moment_mapping"].size
        w = synth.rng_normal(5, B * P * S).reshape(B, P, S)
        md = model_to_device(m, torch.float64)
        d = to_device(nb, torch.float64)
        coeffs = md["coeffs"].clone().requires_grad_(True)
        brcs = d["brcs"].clone().requires_grad_(True)
        val = ops.mtpBasisOp(*basis_args(m, md, d, coeffs, brcs))[0]
        assert close(val.detach().cpu().numpy(), g["desc"])
        (val * torch.from_numpy(w).to("cuda:0")).sum().backward()
        width = g["basis_drcs"].shape[2]
        got = brcs.grad.cpu().numpy()
        assert close(got[:, :, :width], g["basis_drcs"]) and np.all(got[:, :, width:] == 0)
        assert close(coeffs.grad.cpu().numpy().ravel(), g["basis_dcoeffs"].sum(0))


def test_site_energies_with_ghosts(oracle):
    """Rows are the local atoms; neighbours may be ghosts (index >= natoms_pad)."""
    import torch
    from ai2pot_amd import ops
    o = structure(oracle, 64, (9.0, 9.5, 10.0), 2, 1004, 5.0, umax=150)
    m = synth.mtp_model(mtp_param.mtp_param(10), 2, 8, 5.0, 1.5, 3004)
    inum, ilist, numneigh, first, rcs, types, _ = o
    nl = 40
    first = first.copy()
    first[first < 0] = 0
    nbg = dict(binum=np.array([nl], np.int32), bilist=ilist[None, :nl].copy(), bnumneigh=numneigh[None, :nl].copy(),
               bfirstneigh=first[None, :nl].copy(), brcs=rcs[None, :nl].copy(), btypes=types[None, :].copy(),
               nghost=inum - nl)
    md = model_to_device(m, torch.float64)
    d = to_device(nbg, torch.float64)
    args = esites_args(m, md, d)
    es = ops.linearMtpToEsitesOp(*args, 0.0, 0.0, None, None)[0]
    es_ref, _ = oracle.mtp_esites(m, nbg)
    assert close(es.cpu().numpy(), es_ref)
    gout = synth.rng_normal(5, nl).reshape(1, nl)
    got = ops.mtp_esites_backward(torch.from_numpy(gout).to("cuda:0"), *args)
    ref = oracle.mtp_esites_bwd(m, nbg, gout)
    for a, b in zip(got, ref):
        assert close(a.cpu().numpy(), b)


@pytest.mark.parametrize("level,nt", [(8, 2), (10, 1), (12, 3)])
def test_linear_system(oracle, level, nt):
    """LinMatrixLinVectorOp against the oracle (a padded batch), fp64 1e-10."""
    import torch
    from ai2pot_amd import ops
    m, nb, labels = loss_inputs(oracle, level, nt)
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    A, b = ops.LinMatrixLinVectorOp(1.0, 0.7, 0.3, t(labels["energy"]), t(labels["force"]), t(labels["virial"]),
                                    *esites_args(m, md, d), 0.0, 0.0, None, None)
    Ar, br = oracle.mtp_lin_system(m, nb, (1.0, 0.7, 0.3), labels)
    assert close(A.cpu().numpy(), Ar) and close(b.cpu().numpy(), br)


@pytest.mark.parametrize("level,nt,U", [(10, 1, None), (16, 3, None), (20, 2, None), (22, 2, None), (16, 2, 8)])
def test_components_in_one_pass_equal_a_pass_per_column(oracle, level, nt, U):
    """The components of the linear system, all columns from one pass over the atoms (the adjoints of all scalar
    moments as one gather over their ancestors), against one energy / force / virial pass per column: a padded batch
    with rows in a permuted order (rows of 30-odd neighbours take two chunks of the table at level 16), and (U = 8) lists
    cut short, in which most pairs have no counterpart from the other end."""
    import torch
    from ai2pot_amd import _lib, ops
    m, nb, _ = loss_inputs(oracle, level, nt, sizes=(30, 41) if level >= 20 else (48, 30, 37))
    if U is not None:                                    # keep the first U neighbours of every row
        nb = dict(nb)
        nb["bnumneigh"] = np.minimum(nb["bnumneigh"], U)
    B, P = nb["bilist"].shape
    perm = np.argsort(synth.rng_normal(9, P))            # rows of a structure in another order than its atoms
    for b in range(B):
        n = int(nb["binum"][b])
        order = perm[perm < n]
        for k in ("bilist", "bnumneigh", "bfirstneigh", "brcs"):
            nb[k][b, :n] = nb[k][b, order]
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    args = (m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
            d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])
    L = _lib.lib()
    before = L.a2p_mtp_components_route(1)
    try:
        one = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        again = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
        L.a2p_mtp_components_route(0)
        per_column = [t.cpu().numpy() for t in ops.mtp_lin_components(*args)]
    finally:
        L.a2p_mtp_components_route(before)
    for a, b, c in zip(one, per_column, again):
        assert np.abs(b).max() > 0
        assert close(a, b)
        assert np.array_equal(a, c)                      # bit-reproducible


@pytest.mark.parametrize("level", [10, 16])
@pytest.mark.parametrize("sizes", [(1,), (3, 2), (4,), (5, 1), (8, 6, 3), (9,)])
def test_components_of_few_atoms(oracle, level, sizes):
    """Rows of structures that fill the sets of four which are summed together, begin one or leave one short."""
    from ai2pot_amd import _lib, ops
    import torch
    m, nb, _ = loss_inputs(oracle, level, 2, sizes=sizes)
    md, d = model_to_device(m, torch.float64), to_device(nb, torch.float64)
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
        assert close(a, b)


def test_components_of_a_count_beyond_the_rows(oracle):
    """A structure that is said to have more rows than the lists hold: those of the lists are evaluated, and neither the next
    structure's nor what lies behind the last one's (sizes of which a set of four leaves some over)."""
    import torch
    from ai2pot_amd import ops
    m, nb, _ = loss_inputs(oracle, 10, 2, sizes=(9, 9, 9))
    md, d = model_to_device(m, torch.float64), to_device(nb, torch.float64)
    assert d["bilist"].shape[1] == 9
    run = lambda binum: [t.cpu().numpy() for t in ops.mtp_lin_components(
        m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
        md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], binum, d["bilist"], d["bnumneigh"], d["bfirstneigh"],
        d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"], validate=False)]
    for beyond in (1, 3, 9):
        for a, b in zip(run(d["binum"] + beyond), run(d["binum"])):
            assert np.abs(b).max() > 0 and np.array_equal(a, b)


def test_components_in_single_precision(oracle):
    """The fp32 instance of the one-pass components against the fp64 one (the plan's byte offsets are halved for
    4-byte moments)."""
    import torch
    from ai2pot_amd import ops
    m, nb, _ = loss_inputs(oracle, 12, 2, sizes=(30, 24))
    out = {}
    for dt in (torch.float64, torch.float32):
        md = model_to_device(m, dt)
        d = to_device(nb, dt)
        out[dt] = [t.double().cpu().numpy() for t in ops.mtp_lin_components(
            m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"], md["alpha_index_basic"],
            md["alpha_index_times"], md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
            d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])]
    for a, b in zip(out[torch.float32], out[torch.float64]):
        assert close(a, b, 2e-4)


def test_components_flag_bad_lists(oracle):
    """The one-pass components check their lists like the energy / force / virial kernel: a neighbour index or a type
    outside its range, or a row longer than umax, is skipped on the device and reported; nothing is read or written
    out of bounds, and a good call afterwards is right."""
    import torch
    from ai2pot_amd import _lib, ops
    m, nb, _ = loss_inputs(oracle, 10, 2, sizes=(30, 24))
    md = model_to_device(m, torch.float64)

    def run(lists):
        d = to_device(lists, torch.float64)
        return ops.mtp_lin_components(m["chebyshev_size"], m["scaling"], md["coeffs"], m["alpha_moments_count"],
                                      md["alpha_index_basic"], md["alpha_index_times"], md["alpha_moment_mapping"],
                                      m["nmus"], d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"], d["brcs"],
                                      d["btypes"], md["type_map"], m["rmax"], m["rmin"], md["q_scaler"])
    good = [t.cpu().numpy() for t in run(nb)]
    P = nb["bilist"].shape[1]
    for key, where, value in (("bfirstneigh", (0, 3, 1), P + 5), ("bfirstneigh", (1, 0, 0), -7),
                              ("btypes", (0, 2), 9), ("bilist", (1, 4), P + 1),
                              ("bnumneigh", (0, 1), nb["bfirstneigh"].shape[2] + 3)):
        bad = {k: (v.copy() if hasattr(v, "copy") else v) for k, v in nb.items()}
        bad[key][where] = value
        with pytest.raises((_lib.A2PError, RuntimeError)):      # (the row length is checked on the host first)
            run(bad)
    again = [t.cpu().numpy() for t in run(nb)]
    for a, b in zip(good, again):
        assert np.array_equal(a, b)


def test_linear_system_and_schmidt_against_golden(oracle):
    """Level 16 against the committed outputs of the reference's CPU launcher and of its Gram-Schmidt."""
    import os
    import torch
    from ai2pot_amd import ops
    with np.load(os.path.join(os.path.dirname(__file__), "golden", "mtp.npz")) as z:
        g = {k.split("/")[1]: z[k] for k in z.files if k.startswith("L16/")}
    lat, pos = synth.random_packed(48, [8.5, 9.0, 9.5], 2.0, 21)
    ty = synth.rng_randint(22, 48, 3)
    m = synth.mtp_model(mtp_param.mtp_param(16), 3, 8, 5.0, 1.8, 3016)
    m["q_scaler"] = np.linspace(0.7, 1.4, m["q_scaler"].size)
    o = oracle.nblist(lat, ty, pos, 5.0, 100)
    nb = synth.pack_batch([o, o])
    nb["brcs"][1] *= 1.01
    B, P = nb["bilist"].shape
    labels = dict(energy=synth.rng_normal(1, B, -4 * 48, 3), force=synth.rng_normal(2, B * P * 3).reshape(B, P, 3),
                  virial=synth.rng_normal(3, B * 9, 0, 0.5).reshape(B, 9))
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    A, b = ops.LinMatrixLinVectorOp(1.0, 0.7, 0.3, t(labels["energy"]), t(labels["force"]), t(labels["virial"]),
                                    *esites_args(m, md, d), 0.0, 0.0, None, None)
    assert close(A.cpu().numpy(), g["lin_matrix"]) and close(b.cpu().numpy(), g["lin_vector"])
    oc = ops.CoeffsSchmidtOrthOp(3, m["nmus"], 8, md["coeffs"])[0]
    assert oc.shape == md["coeffs"].shape and close(oc.cpu().numpy(), g["orth_coeffs"], 1e-13)
    oc32 = ops.CoeffsSchmidtOrthOp(3, m["nmus"], 8, md["coeffs"].float())[0]
    assert oc32.dtype == torch.float32 and close(oc32.cpu().numpy(), g["orth_coeffs"], 1e-5)


def test_errors(oracle):
    import torch
    from ai2pot_amd import _lib, ops
    o = structure(oracle, 30, (8.5, 9.0, 9.5), 2, 21, 5.0)
    nb = synth.pack_batch([o])
    m = synth.mtp_model(mtp_param.mtp_param(8), 2, 8, 5.0, 1.8, 5)
    md = model_to_device(m, torch.float64)
    d = to_device(nb, torch.float64)
    bad = md["alpha_index_times"].clone()
    bad[0, 3] = 0                                       # a product may not write a basic moment
    with pytest.raises(_lib.A2PError):
        ops.linearMtpToEFVOp(8, 1.0, md["coeffs"], md["linear_coeffs"], md["type_bias"],
                             m["alpha_moments_count"], md["alpha_index_basic"], bad, md["alpha_moment_mapping"],
                             m["nmus"], d["binum"], d["bilist"], d["bnumneigh"], d["bfirstneigh"], d["brcs"],
                             d["btypes"], md["type_map"], 0, 5.0, 1.8, md["q_scaler"], 0.0, 0.0, None, None)
    with pytest.raises(RuntimeError):                   # coefficient count does not match
        ops.linearMtpToEFVOp(8, 1.0, md["coeffs"][:-1].contiguous(), md["linear_coeffs"], md["type_bias"],
                             m["alpha_moments_count"], md["alpha_index_basic"], md["alpha_index_times"],
                             md["alpha_moment_mapping"], m["nmus"], d["binum"], d["bilist"], d["bnumneigh"],
                             d["bfirstneigh"], d["brcs"], d["btypes"], md["type_map"], 0, 5.0, 1.8,
                             md["q_scaler"], 0.0, 0.0, None, None)
    e, f, v = gpu_efv(m, nb)
    er, fr, vr = oracle.mtp_efv(m, nb)
    assert close(e, er) and close(f, fr)
