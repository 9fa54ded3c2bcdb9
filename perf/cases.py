"""The work this framework is timed on: what its users call, over the range of sizes they call it with.

Seven paths, each through the entry points a user's program goes through:

  ase     one evaluation of a host program (an ASE calculator): nblist.find_info4mlff on NumPy arrays, its results
          copied to the GPU, the energy / force / virial operator, the three results back on the host
  md      one step of a device-resident molecular-dynamics loop: NepCalculator.step (list rebuild + energy, forces, virial)
  efv     one energy / force / virial operator call on lists that are on the GPU already: a periodic batch, or the owned
          atoms and ghosts of a LAMMPS domain (lists longer than the cutoff by the skin)
  train   one training step's share of the operators: loss of a batch of structures and its gradients
  solver  the normal equations of the linear parameters of a moment tensor potential
  list    the neighbour list on device tensors with its padded outputs
  fvt     force and virial reductions of a descriptor network's pair derivatives, forward and backward

Inputs are jittered lattices with vacancies at the densities of the benchmark's configurations.
"""
import math
import os
import sys

import numpy as np
import torch

import ai2pot_amd
from ai2pot_amd import mtp_param, synth
from ai2pot_amd.calculator import NepCalculator
from ai2pot_amd.nblist import find_info4mlff_device

LIB = os.path.join(os.path.dirname(os.path.abspath(ai2pot_amd.__file__)), "_lib")
UMAX = 200          # umax_num_neigh_atoms of the models
SKIN = 2.0          # LAMMPS' default for metal units
JITTER = 0.15       # thermal displacements, per coordinate
PBC = [True, True, True]


def _load():
    if not hasattr(_load, "done"):
        for name in ("nep", "mtpr", "nnmtp", "fvt_sr_op", "nblist"):
            torch.ops.load_library(os.path.join(LIB, "lib%s_bind.so" % name))
        _load.done = True


# ---- cases ---------------------------------------------------------------------------------------------------
def _nep(**kw):
    return dict(dict(model="nep", dtype="f32", species=3, n_radial=6, l_max=4, neurons=50, rcut=7.0, rcut_angular=4.0,
                     density=0.033), **kw)


def _mtp(**kw):
    return dict(dict(model="mtp", dtype="f64", species=3, level=16, cheb=8, rcut=5.0, rmin=0.5, density=0.05), **kw)


def listed():
    return [
        # a molecule-sized cell under an ASE optimiser or a phonon script: all latency
        _nep(name="ase_nep_108", path="ase", atoms=108),
        # small device-resident dynamics with the calculator's defaults
        _nep(name="md_nep_4096", path="md", atoms=4096, sync_free=False),
        # the headline: a large cell, list rebuilt every step, no host synchronisation in the step
        _nep(name="md_nep_1048576", path="md", atoms=1048576, sync_free=True),
        # one MPI rank's domain under LAMMPS: owned atoms, ghosts, lists with a skin
        _nep(name="lammps_nep_20011", path="efv", atoms=20011, batch=1, ghosts=True),
        # the smallest moment tensor potential in use: 216-atom cell, one species
        _mtp(name="efv_mtp10_216", path="efv", atoms=216, batch=1, ghosts=False, species=1, level=10),
        # an accurate moment tensor potential on a production cell
        _mtp(name="efv_mtp20_8192", path="efv", atoms=8192, batch=1, ghosts=False, species=4, level=20, cheb=10, rcut=5.5,
             rmin=1.8),
        # training on a large batch, both model families
        _nep(name="train_nep_64x128", path="train", batch=64, atoms=128, ragged=False, rcut=6.0, density=0.04),
        _mtp(name="train_mtp16_64x128", path="train", batch=64, atoms=128, ragged=False, rmin=0.0, density=0.04),
        # training on a small batch of small structures of different sizes, as a first fit does
        _mtp(name="train_nnmtp12_5x47", path="train", model="nnmtp", batch=5, atoms=47, ragged=True, level=12, species=2,
             neurons=20, rmin=1.5, density=0.04),
        # linear least-squares fit of the moment tensor potential
        _mtp(name="solver_mtp16_64x128", path="solver", batch=64, atoms=128, ragged=False, rmin=0.0, density=0.04),
        # sorted lists of a large cell in double precision
        dict(name="list_sorted_131072", path="list", atoms=131072, dtype="f64", sort=True, rcut=6.0, density=0.04, species=2),
        # a descriptor network's force and virial with their gradients
        dict(name="fvt_4x1000", path="fvt", batch=4, atoms=1000, ragged=False, dtype="f64", rcut=6.0, density=0.04, species=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["ase", "md", "md", "efv", "efv", "efv", "train", "train", "train", "solver", "list", "fvt"])
    if path in ("list", "fvt"):
        c = dict(path=path, dtype=rng.choice(["f32", "f64"]), rcut=round(rng.uniform(4.5, 7.0), 2),
                 density=round(rng.uniform(0.03, 0.05), 4), species=rng.randint(1, 4))
        if path == "list":
            c.update(atoms=_log_int(rng, 300, 131072), sort=rng.random() < 0.5)
        else:
            c.update(batch=rng.randint(1, 8), atoms=_log_int(rng, 50, 2000), ragged=rng.random() < 0.5)
        return c
    if path == "solver":
        return _mtp(path=path, batch=_log_int(rng, 2, 64), atoms=_log_int(rng, 16, 128), ragged=rng.random() < 0.5,
                    species=rng.randint(1, 3), level=rng.choice([8, 10, 12, 14, 16]),
                    density=round(rng.uniform(0.03, 0.05), 4))
    family = "nep" if path == "md" else rng.choice(["nep", "mtp"] if path == "ase" else ["nep", "mtp", "mtp", "nnmtp"])
    density = round(rng.uniform(0.03, 0.05), 4)
    if family == "nep":
        c = _nep(path=path, species=rng.randint(1, 4), n_radial=rng.choice([4, 6]), l_max=rng.choice([3, 4, 4]),
                 neurons=rng.choice([30, 50]), rcut=round(rng.uniform(5.0, 7.0), 2), density=density,
                 dtype=rng.choice(["f32", "f32", "f32", "f64"]))
        top = 32768
    else:
        top = {"mtp": [8, 10, 12, 14, 16, 18, 20], "nnmtp": [8, 10, 12, 14, 16]}[family]
        c = _mtp(path=path, model=family, species=rng.randint(1, 4), level=rng.choice(top), cheb=rng.choice([8, 10]),
                 rcut=round(rng.uniform(4.5, 5.5), 2), rmin=rng.choice([0.0, 0.5, 1.5]), density=density,
                 dtype=rng.choice(["f64", "f64", "f64", "f32"]))
        if family == "nnmtp":
            c["neurons"] = rng.choice([10, 20, 30])
        top = 8192
    if path == "ase":
        c.update(atoms=_log_int(rng, 12, 3000))
    elif path == "md":
        c.update(atoms=_log_int(rng, 200, 600000 if c["dtype"] == "f32" and c["l_max"] == 4 else 60000),
                 sync_free=rng.random() < 0.5)
    elif path == "efv":
        ghosts = rng.random() < 0.4
        c.update(atoms=_log_int(rng, 400 if ghosts else 20, top), batch=1, ghosts=ghosts)
        if not ghosts and c["atoms"] * 8 <= top and rng.random() < 0.5:
            c["batch"] = rng.randint(2, 8)
    else:
        c.update(batch=_log_int(rng, 1, 64), atoms=_log_int(rng, 12, 128), ragged=rng.random() < 0.5)
    return c


# ---- inputs --------------------------------------------------------------------------------------------------
def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _structure(n, case, gen):
    """n atoms of a jittered fcc lattice with vacancies, cell by cell: box length, positions [n, 3], types [n]."""
    dev = gen.device
    m = max(1, math.ceil((n / 4) ** (1 / 3) - 1e-9))
    box = (n / case["density"]) ** (1 / 3)
    sites = torch.randperm(4 * m ** 3, generator=gen, device=dev)[:n].sort().values
    cell, base = sites // 4, sites % 4
    shift = torch.tensor([[0.0, 0.0, 0.0], [0.0, 0.5, 0.5], [0.5, 0.0, 0.5], [0.5, 0.5, 0.0]], dtype=torch.float64, device=dev)
    ijk = torch.stack([cell // (m * m), cell // m % m, cell % m], 1).to(torch.float64)
    x = (ijk + shift[base]) * (box / m) + JITTER * torch.randn((n, 3), generator=gen, device=dev, dtype=torch.float64)
    x = torch.remainder(x, box).to(_dtype(case))
    types = torch.randint(0, case["species"], (n,), generator=gen, device=dev, dtype=torch.int32)
    return box, x.contiguous(), types


def _lattice(box, case):
    return np.eye(3, dtype=np.float32 if case["dtype"] == "f32" else np.float64) * box


def _batch(case, gen):
    """The seven padded tensors of a batch of structures, as a data loader hands them over."""
    dev, dt = gen.device, _dtype(case)
    B, P = case["batch"], case["atoms"]
    sizes = [P] * B
    if case.get("ragged"):
        low = max(2, P // 3)
        sizes = [P] + torch.randint(low, P + 1, (B - 1,), generator=gen, device=dev).tolist()
    nb = dict(binum=torch.tensor(sizes, dtype=torch.int32, device=dev), nghost=0,
              brcs=torch.zeros((B, P, UMAX, 3), dtype=dt, device=dev))
    for k in ("bilist", "bnumneigh", "btypes"):
        nb[k] = torch.zeros((B, P), dtype=torch.int32, device=dev)
    nb["bfirstneigh"] = torch.zeros((B, P, UMAX), dtype=torch.int32, device=dev)
    for b, n in enumerate(sizes):
        box, x, t = _structure(n, case, gen)
        _, il, nn, first, rcs, ty, _ = find_info4mlff_device(_lattice(box, case), t, x, case["rcut"], UMAX)
        for k, v in (("bilist", il), ("bnumneigh", nn), ("bfirstneigh", first), ("brcs", rcs), ("btypes", ty)):
            nb[k][b, :n] = v
    return nb


def _domain(case, gen):
    """One periodic cell as a LAMMPS domain: every atom owned, its images within cutoff + skin of the box as ghosts."""
    dev, n = gen.device, case["atoms"]
    box, x, t = _structure(n, case, gen)
    reach = case["rcut"] + SKIN
    _, il, nn, first, rcs, _, _ = find_info4mlff_device(_lattice(box, case), t, x, reach, UMAX)
    index = torch.full((27, n), -1, dtype=torch.int64, device=dev)
    index[13] = torch.arange(n, device=dev)
    types, count = [t], n
    for s in range(27):
        if s == 13:
            continue
        p = x + box * torch.tensor([s // 9 - 1, s // 3 % 3 - 1, s % 3 - 1], dtype=x.dtype, device=dev)
        keep = ((p > -reach - 1e-3) & (p < box + reach + 1e-3)).all(1).nonzero()[:, 0]
        index[s, keep] = count + torch.arange(keep.numel(), device=dev)
        types.append(t[keep])
        count += keep.numel()
    # the exchange of ghosts is sized beforehand, so that a few of them name no row's neighbour
    total = max(count, n + 100 + int(1.15 * n * ((1.0 + 2.0 * reach / box) ** 3 - 1.0)))
    types.append(torch.zeros(total - count, dtype=torch.int32, device=dev))
    j = first.clamp(min=0).long()
    s = torch.round((x[:, None] + rcs - x[j]) / box).long() + 1
    named = index[s[..., 0] * 9 + s[..., 1] * 3 + s[..., 2], j]
    first = torch.where(first >= 0, named, torch.full_like(named, -1)).to(torch.int32)
    return dict(binum=torch.tensor([n], dtype=torch.int32, device=dev), bilist=il[None].contiguous(),
                bnumneigh=nn[None].contiguous(), bfirstneigh=first[None].contiguous(), brcs=rcs[None].contiguous(),
                btypes=torch.cat(types)[None].contiguous(), nghost=total - n)


def _model(case, seed):
    nt = case["species"]
    tm = tuple(range(1, nt + 1))
    if case["model"] == "nep":
        return synth.nep_model(ntypes=nt, n_radial_basis=case["n_radial"], l_max=case["l_max"], num_neurons=case["neurons"],
                               rmax_radial=case["rcut"], rmax_angular=case["rcut_angular"], seed=seed, type_map=tm)
    tables = mtp_param.mtp_param(case["level"])
    if case["model"] == "nnmtp":
        return synth.nnmtp_model(tables, nt, case["cheb"], case["neurons"], case["rcut"], case["rmin"], seed, type_map=tm)
    return synth.mtp_model(tables, nt, case["cheb"], case["rcut"], case["rmin"], seed, lo=-0.05, hi=0.05, type_map=tm)


def _on_gpu(m, case, dev, grad=False):
    """The model's arrays as tensors; the trained ones as leaves that want a gradient."""
    out = {}
    for k, v in m.items():
        if isinstance(v, np.ndarray):
            whole = v.dtype.kind == "i"
            out[k] = torch.from_numpy(np.ascontiguousarray(v)).to(torch.int32 if whole else _dtype(case)).to(dev)
            if grad and not whole and k not in ("q_scaler", "q_shifter"):
                out[k].requires_grad_(True)
        else:
            out[k] = v
    return out


def _lists(nb):
    return nb["binum"], nb["bilist"], nb["bnumneigh"], nb["bfirstneigh"], nb["brcs"], nb["btypes"]


def _arguments(case, m, nb, zbl):
    """The operators' arguments from the model on; the loss operators take the weights and labels before them."""
    off = (0.0, 0.0, zbl, zbl)                                     # no ZBL correction: the models' default
    if case["model"] == "nep":
        return (m["chebyshev_size"], m["n_radial_basis"], m["n_angular_basis"], m["l_max"], m["coeffs"], m["w0"], m["b0"],
                m["w1"], m["type_bias"], *_lists(nb), m["type_map"], nb["nghost"], m["rmax_radial"], m["rmax_angular"],
                m["q_scaler"], *off)
    tables = (int(m["alpha_moments_count"]), m["alpha_index_basic"], m["alpha_index_times"], m["alpha_moment_mapping"],
              int(m["nmus"]))
    cut = (m["type_map"], nb["nghost"], m["rmax"], m["rmin"])
    if case["model"] == "nnmtp":
        return (m["chebyshev_size"], m["coeffs"], m["w0"], m["w1"], m["type_bias"], *tables, *_lists(nb), *cut,
                m["q_shifter"], m["q_scaler"], *off)
    return (m["chebyshev_size"], 1.0, m["coeffs"], m["linear_coeffs"], m["type_bias"], *tables, *_lists(nb), *cut,
            m["q_scaler"], *off)


def _efv_operator(case):
    return {"nep": lambda: torch.ops.nep.nepToEFVOp, "mtp": lambda: torch.ops.mtpr.linearMtpToEFVOp,
            "nnmtp": lambda: torch.ops.nnmtp.nnMtpToEFVOp}[case["model"]]()


def _labels(case, nb, gen):
    B, P = nb["bilist"].shape
    dt, dev = _dtype(case), gen.device
    normal = lambda *s: torch.randn(s, generator=gen, device=dev, dtype=torch.float64)
    e = -4.0 * nb["binum"].double() + 0.2 * nb["binum"].double().sqrt() * normal(B)
    return e.to(dt), normal(B, P, 3).to(dt), (0.5 * normal(B, 9)).to(dt)


def prepare(case, seed):
    _load()
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    path, dt = case["path"], _dtype(case)
    s = dict(path=path)
    if path == "ase":
        if LIB not in sys.path:
            sys.path.append(LIB)
        import nblist
        box, x, t = _structure(case["atoms"], case, gen)
        m = _on_gpu(_model(case, seed), case, dev)
        s.update(find=nblist.find_info4mlff, lattice=_lattice(box, case), coords=x.cpu().numpy(), types=t.cpu().numpy(),
                 rcut=case["rcut"], model=m, case=dict(case), dev=dev, zbl=torch.zeros(0, dtype=dt, device=dev),
                 op=_efv_operator(case))
    elif path == "md":
        box, x, t = _structure(case["atoms"], case, gen)
        s.update(coords=x, calc=NepCalculator(_model(case, seed), case["atoms"], _lattice(box, case), t.cpu().numpy(),
                                              umax=UMAX, dtype=dt, device=dev, sync_free=case["sync_free"]))
    elif path == "efv":
        nb = _domain(case, gen) if case["ghosts"] else _batch(case, gen)
        m = _on_gpu(_model(case, seed), case, dev)
        s.update(op=_efv_operator(case), args=_arguments(case, m, nb, torch.zeros(0, dtype=dt, device=dev)))
    elif path in ("train", "solver"):
        nb = _batch(case, gen)
        m = _on_gpu(_model(case, seed), case, dev, grad=path == "train")
        args = (1.0, 1.0, 1.0, *_labels(case, nb, gen), *_arguments(case, m, nb, torch.zeros(0, dtype=dt, device=dev)))
        if path == "solver":
            s.update(op=torch.ops.mtpr.LinMatrixLinVectorOp, args=args)
        else:
            op = {"nep": lambda: torch.ops.nep.nepToLossOp, "mtp": lambda: torch.ops.mtpr.linearMtpToLossOp,
                  "nnmtp": lambda: torch.ops.nnmtp.nnMtpToLossOp}[case["model"]]()
            s.update(op=op, args=args, params=[v for v in m.values() if isinstance(v, torch.Tensor) and v.requires_grad])
    elif path == "list":
        box, x, t = _structure(case["atoms"], case, gen)
        s.update(args=(torch.from_numpy(_lattice(box, case)), t, x, case["rcut"], UMAX, True, PBC, case["sort"]))
    else:
        nb = _batch(case, gen)
        valid = torch.arange(UMAX, device=dev) < nb["bnumneigh"][..., None]
        dei = torch.randn(nb["brcs"].shape, generator=gen, device=dev, dtype=dt) * valid[..., None]
        B, P = nb["bilist"].shape
        s.update(lists=(nb["binum"], nb["bilist"], nb["bnumneigh"], nb["bfirstneigh"]), brcs=nb["brcs"].requires_grad_(True),
                 dei=dei.requires_grad_(True), gf=torch.randn((B, P, 3), generator=gen, device=dev, dtype=dt),
                 gv=torch.randn((B, 3, 3), generator=gen, device=dev, dtype=dt))
    return s


# ---- one pass ------------------------------------------------------------------------------------------------
def run(s):
    path = s["path"]
    if path == "md":
        return s["calc"].step(s["coords"])
    if path in ("efv", "solver"):
        return s["op"](*s["args"])
    if path == "train":
        out = s["op"](*s["args"])
        return [t.detach() for t in out], torch.autograd.grad(out[0].mean(), s["params"])
    if path == "list":
        return torch.ops.nblist.find_info4mlff(*s["args"])
    if path == "fvt":
        binum, bilist, bnumneigh, bfirstneigh = s["lists"]
        f = torch.ops.fvt.ForceSrOp(binum, bilist, bnumneigh, bfirstneigh, 0, UMAX, s["dei"])[0]
        v = torch.ops.fvt.VirialSrOp(bnumneigh, s["brcs"], UMAX, s["dei"])[0]
        return (f.detach(), v.detach()) + torch.autograd.grad([f, v], [s["brcs"], s["dei"]], [s["gf"], s["gv"]])
    n, il, nn, first, rcs, ty, nghost = s["find"](s["lattice"], s["types"], s["coords"], s["rcut"], UMAX, True, PBC, False)
    up = lambda a: torch.from_numpy(a).to(s["dev"])[None]
    nb = dict(binum=torch.tensor([n], dtype=torch.int32, device=s["dev"]), bilist=up(il), bnumneigh=up(nn),
              bfirstneigh=up(first), brcs=up(rcs), btypes=up(ty), nghost=nghost)
    e, f, v = s["op"](*_arguments(s["case"], s["model"], nb, s["zbl"]))
    return e.cpu(), f.cpu(), v.cpu()


# ---- what a pass cannot do without -----------------------------------------------------------------------------
def _neighbours(case, r):
    return case["density"] * 4.0 / 3.0 * math.pi * r ** 3


def _flops(case, nn, backward):
    """Per atom (an FMA counts two): descriptors, read-out, forces and virial; with backward also the gradient of the
    loss with respect to the parameters."""
    if case["model"] == "nep":
        K, n_r, n_a, H = 8, case["n_radial"], 4, case["neurons"]
        D, cK, na = n_r + n_a * case["l_max"], 14 * 8 + 24, _neighbours(case, case["rcut_angular"])
        f = (nn * (14 + cK + 4 * K * n_r + 3 * n_r) + na * (cK + 4 * K * n_a + 210 + 480 * n_a) + 144 * n_a + 4 * D * H +
             15 * H)
        return 3.5 * f if backward else f
    t = mtp_param.mtp_param(case["level"])
    K, nmus, nb, S = case["cheb"], int(t["nmus"]), len(t["alpha_index_basic"]), len(t["alpha_moment_mapping"])
    kmax, nt = int(t["alpha_index_basic"][:, 1:].sum(1).max()), len(t["alpha_index_times"])
    f = nn * (8 + 8 * K + 30 + 4 * K * nmus + 4 * kmax + 29 * nb) + 9 * nt + 4 * S
    if backward:
        f += nn * (2 * (8 * K + 30 + 4 * kmax + 4 * K * nmus) + 70 * nb) + 24 * nt + 6 * S
    if case["model"] == "nnmtp":
        f += (3 if backward else 1) * case["neurons"] * (4 * S + 15)
    return f


def work(case):
    path, s = case["path"], 4 if case["dtype"] == "f32" else 8
    nn = _neighbours(case, case["rcut"])
    atoms = case["atoms"] * case.get("batch", 1) * (2.0 / 3.0 if case.get("ragged") else 1.0)
    row, padded = nn * (4 + 3 * s), UMAX * (4 + 3 * s)            # a row's valid entries; a row as it is stored
    if path == "ase":
        return dict(bytes=atoms * (3 * s + 4 + 12 + padded + 3 * s), flops=atoms * _flops(case, nn, False))
    if path == "md":
        return dict(bytes=atoms * (3 * s + 4 + 12 + row + 3 * s), flops=atoms * _flops(case, nn, False))
    if path == "efv":
        if case["ghosts"]:
            row *= ((case["rcut"] + SKIN) / case["rcut"]) ** 3
        return dict(bytes=atoms * (12 + row + 3 * s), flops=atoms * _flops(case, nn, False))
    if path == "train":
        return dict(bytes=atoms * (12 + row + 3 * s), flops=atoms * _flops(case, nn, True))
    if path == "solver":
        t = mtp_param.mtp_param(case["level"])
        n = len(t["alpha_moment_mapping"]) + case["species"]
        # a derivative per column, coordinate and neighbour, and the products of the columns
        return dict(bytes=atoms * (12 + row + 3 * s) + n * n * s,
                    flops=atoms * (_flops(case, nn, False) + nn * 3 * 2 * n + 3 * n * (n + 1)))
    if path == "list":
        return dict(bytes=atoms * (3 * s + 4 + 12 + padded), flops=atoms * nn * 30)
    return dict(bytes=atoms * (2 * nn * 3 * s + nn * 4 + 2 * UMAX * 3 * s + 6 * s), flops=atoms * nn * 60)


def tolerance(case):
    if case["path"] == "list":
        return "exact"
    if case["dtype"] == "f64":
        return {"rel": 1e-10}
    return {"rel": 1e-5, "max": 1e-3}
