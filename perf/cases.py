"""What a user of this framework has it do, as measurable cases.

Every case goes through the public entry points of ``edus_amd.native``: the time
loop of one problem (steps, with the observables every ``res`` steps), a batch of
problems, the mean-field time loop, the whole drop-in program on an input file,
and the two setup computations that run on the GPU (the Wannier contraction and
the Coulomb coefficients).  Sizes are those of the benchmark workloads, of the
reference's example run and of the test-suite, or lie between them.

The tables of a problem (H, D, U, rho0, the stencil) are made here from the seed:
smooth periodic matrices on a hexagonal lattice, with a gap between the filled
and the empty bands, so that ``exact`` can restate a pass in plain torch.
"""
import ctypes as C
import math
import os
import tempfile

import numpy as np
import torch

from edus_amd import native as N

A_LAT = 2.5 / 0.529177249  # bohr
EV = 1.0 / 27.211396
STEPPERS = {"rk4": N.STEPPER_RK4, "ab": N.STEPPER_AB, "taylor": N.STEPPER_TAYLOR}
PRECISIONS = {"fp64": N.PRECISION_FP64, "mixed": N.PRECISION_MIXED, "mixed32": N.PRECISION_MIXED32,
              "bf16x3": N.PRECISION_BF16X3}
# offsets of the two-shell hexagonal stencil, in grid steps
OFFSETS = [(-1, -1), (-1, 0), (0, -1), (0, 1), (1, 0), (1, 1), (-2, -1), (-1, -2), (-1, 1), (1, -1), (1, 2), (2, 1)]


def listed():
    return [
        # the smallest production run: 3-band boron nitride with dephasing on 60 x 60 k
        _steps("hbn3_60x60_rk4", 3, 60, 60, "rk4", 4, steps=20, res=10, nch=1, diss=True),
        # the reference's published example: 70 x 70, Adams-Bashforth 5, observables every
        # 5 steps, input file in, output files out
        {"name": "example_70x70_ab5_files", "kind": "run", "n": 70, "order": 5, "steps": 1000, "res": 5},
        # a fine grid of a small tight-binding model, odd sizes, in-plane field
        _steps("bands4_251x307_rk4", 4, 251, 307, "rk4", 4, steps=20, res=10, pol=2),
        # Wannier models of three sizes, linear polarisation
        _steps("bands8_200x200_rk4", 8, 200, 200, "rk4", 4, steps=20, res=10),
        _steps("bands16_200x200_rk4", 16, 200, 200, "rk4", 4, steps=20, res=10),
        _steps("bands32_128x128_rk4", 32, 128, 128, "rk4", 4, steps=20, res=10),
        # an odd band count on an odd grid, multistep stepper, dephasing
        _steps("bands13_61x85_ab4_dephasing", 13, 61, 85, "ab", 4, steps=20, res=10, diss=True),
        # the mixed-precision form with the Taylor stepper
        _steps("bands24_96x100_taylor4_mixed", 24, 96, 100, "taylor", 4, steps=20, res=10, precision="mixed"),
        # the Hartree-Fock mean field on the excitonic workload's grid
        {"name": "coulomb3_300x300_ab4", "kind": "coulomb", "n1": 300, "n2": 300, "stepper": "ab", "order": 4, "steps": 20,
         "res": 10, "ncut": 20},
        # a scan over materials and pulses: small problems of 2, 4 and 8 bands stepped together
        {"name": "scan_12_instances", "kind": "batch", "count": 12, "lo": 48, "hi": 144, "steps": 10},
        # setup: H(k) and r(k) of a Wannier model from its lattice sums
        {"name": "wannier16_R441_96x96", "kind": "wannier", "nw": 16, "rmax": 10, "n1": 96, "n2": 96, "form": "fp64"},
        # setup: the mean-field coefficients from the lattice sum of the screened interaction
        {"name": "coulomb_coefficients", "kind": "coefficients", "nb": 3, "ncut": 20, "n_sum": 999, "shell": 28.0,
         "n_peak": 9999},
    ]


def _steps(name, nb, n1, n2, stepper, order, steps, res, nch=0, diss=False, pol=1, precision="fp64"):
    """pol: number of field components that are not zero (1: along z, 2: in the plane)."""
    return {"name": name, "kind": "steps", "nb": nb, "n1": n1, "n2": n2, "stepper": stepper, "order": order, "steps": steps,
            "res": res, "nch": nch, "diss": diss, "pol": pol, "precision": precision}


def draw(rng):
    def grid(most):
        """Two grid lengths, their product spread over its logarithm, up to `most` k points."""
        nk = math.exp(rng.uniform(math.log(900), math.log(most)))
        r = rng.uniform(0.8, 1.25)
        return max(24, int(math.sqrt(nk * r))), max(24, int(math.sqrt(nk / r)))

    kind = rng.choice(["steps"] * 6 + ["coulomb", "batch", "wannier", "coefficients", "run"])
    if kind == "steps":
        nb = rng.choice([2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 14, 16, 18, 20, 24, 27, 28, 32])
        n1, n2 = grid(min(110000, 16384 * 1024 // (nb * nb)))
        stepper = rng.choice(["rk4", "rk4", "ab", "taylor"])
        order = {"rk4": 4, "ab": rng.randint(2, 5), "taylor": rng.choice([4, 6])}[stepper]
        forms = ["fp64"] * 3 + (["mixed", "mixed32"] if nb > 4 else []) + (["bf16x3"] if nb > 8 else [])
        c = _steps("", nb, n1, n2, stepper, order, steps=20, res=rng.choice([5, 10, 20]), nch=rng.choice([0, 0, 1]) if nb > 2 else 0,
                   diss=rng.random() < 0.3, pol=rng.choice([1, 1, 2]), precision=rng.choice(forms))
    elif kind == "coulomb":
        n1, n2 = grid(90000)
        stepper = rng.choice(["rk4", "ab"])
        c = {"kind": kind, "n1": n1, "n2": n2, "stepper": stepper, "order": 4, "steps": 20, "res": rng.choice([5, 10]),
             "ncut": rng.randint(8, 20)}
    elif kind == "batch":
        c = {"kind": kind, "count": rng.randint(4, 12), "lo": rng.randint(31, 48), "hi": rng.randint(64, 144), "steps": 10}
    elif kind == "wannier":
        nw = rng.choice([4, 8, 11, 16, 20])
        n1, n2 = grid(9216 * 256 // (nw * nw))
        c = {"kind": kind, "nw": nw, "rmax": rng.randint(5, 10), "n1": n1, "n2": n2,
             "form": rng.choice(["fp64", "fp64", "fp32", "bf16x3"])}
    elif kind == "coefficients":
        c = {"kind": kind, "nb": rng.choice([2, 3, 4]), "ncut": rng.randint(8, 20), "n_sum": 2 * rng.randint(150, 450) + 1,
             "shell": rng.uniform(12.0, 28.0), "n_peak": 2 * rng.randint(2000, 4500) + 1}
    else:  # the input reader takes even grids only
        c = {"kind": kind, "n": 2 * rng.randint(16, 35), "order": rng.randint(2, 5), "steps": 100 * rng.randint(4, 10),
             "res": rng.choice([5, 10])}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _lattice():
    """Rows b1, b2 of the reciprocal lattice of the hexagonal cell (sample in the yz plane)."""
    c30, s30 = math.cos(math.pi / 6), math.sin(math.pi / 6)
    a = A_LAT * np.array([[c30, s30], [c30, -s30]])
    b = np.zeros((2, 3))
    b[:, 1:] = 2 * math.pi * np.linalg.inv(a).T
    return b


def _stencil(n1, n2):
    """nbr [nk][12] and w_b b [12][3] of the gradient on an n1 x n2 grid: equal weights on +b and -b with
    sum_b w_b b b^T = 1 in the plane (minimum-norm solution)."""
    b = _lattice() / np.array([[n1], [n2]])
    vec = np.array([m1 * b[0] + m2 * b[1] for m1, m2 in OFFSETS])
    half = [i for i, (m1, m2) in enumerate(OFFSETS) if (m1, m2) > (0, 0)]
    eq = np.array([[2 * vec[i][p] * vec[i][q] for i in half] for p, q in ((1, 1), (1, 2), (2, 2))])
    w = np.linalg.lstsq(eq, np.array([1.0, 0.0, 1.0]), rcond=None)[0]
    wb = np.zeros((len(OFFSETS), 3))
    for i, wi in zip(half, w):
        wb[i] = wi * vec[i]
        wb[OFFSETS.index((-OFFSETS[i][0], -OFFSETS[i][1]))] = -wi * vec[i]
    i1, i2 = np.divmod(np.arange(n1 * n2), n2)
    nbr = np.stack([((i1 + m1) % n1) * n2 + (i2 + m2) % n2 for m1, m2 in OFFSETS], axis=1).astype(np.int32)
    return nbr, wb


def _kgrid(n1, n2, dev):
    k1 = -0.5 + torch.arange(n1, dtype=torch.float64, device=dev) / n1
    k2 = -0.5 + torch.arange(n2, dtype=torch.float64, device=dev) / n2
    return torch.stack(torch.meshgrid(k1, k2, indexing="ij"), -1).reshape(-1, 2)


def _hermitian(rng, k, nb, scale, count=1):
    """`count` smooth periodic Hermitian matrices S(k) = A_0 + sum_R (A_R e^{2 pi i k.R} + h.c.), |R| <= 2."""
    R = [(0, 1), (1, 0), (1, 1), (1, -1), (0, 2), (2, 0)]
    coef = rng.normal(size=(1 + len(R), count * nb * nb, 2)) @ np.array([1.0, 1j])
    coef *= scale / np.array([1.0] + [1.0 + 2.0 * (p * p + q * q) for p, q in R])[:, None]
    ph = torch.exp(2j * math.pi * (k @ torch.tensor([[0.0, 0.0]] + [list(map(float, r)) for r in R], dtype=torch.float64, device=k.device).T))
    S = (ph @ torch.tensor(coef, device=k.device)).reshape(-1, count, nb, nb)
    return S + S.mH


def _model(case, seed, dev):
    """Tables of one problem on `dev`, in the reference's layouts (complex128)."""
    nb, n1, n2, nch = case["nb"], case["n1"], case["n2"], case.get("nch", 0)
    nv = max(nch + 1, nb // 2) if nb > 1 else 1
    rng = np.random.default_rng(seed)
    k = _kgrid(n1, n2, dev)
    S = _hermitian(rng, k, nb, 0.6 / math.sqrt(nb))[:, 0]
    U = torch.linalg.matrix_exp(1j * S)
    e = np.concatenate([np.full(nch, -0.7), -0.08 - 0.25 * np.sort(rng.uniform(size=nv - nch))[::-1], 0.12 + 0.4 * np.sort(rng.uniform(size=nb - nv))])
    amp, phi = 0.03 * rng.uniform(size=(nb, 2)), 2 * math.pi * rng.uniform(size=(nb, 2))
    ang = 2 * math.pi * k[:, None, :] + torch.tensor(phi, device=dev)
    ek = torch.tensor(e, device=dev) + (torch.tensor(amp, device=dev) * torch.cos(ang)).sum(-1)
    H = (U.mH * ek[:, None, :]) @ U
    H = 0.5 * (H + H.mH)
    D = _hermitian(rng, k, nb, 0.25 / math.sqrt(nb), 3).real.to(torch.complex128).permute(0, 2, 3, 1).contiguous()
    occ = torch.zeros(nb, dtype=torch.float64, device=dev)
    occ[:nv] = 1.0
    rho0 = (U.mT * occ) @ U.conj()  # transposed storage: rho0_ij = sum_v U_vi conj(U_vj)
    T = np.zeros((nb, nb))
    if case.get("diss"):
        T[:] = 0.0024
        np.fill_diagonal(T, 0.0)
        for c in range(nch):
            T[c, :] = T[:, c] = 0.004
            T[c, c] = 0.004
    nbr, wb = _stencil(n1, n2)
    return {"nk": n1 * n2, "nb": nb, "nch": nch, "ncc": nv, "H": H, "D": D, "U": U, "rho0": rho0, "T": T, "nbr": nbr, "wb": wb,
            "wx2": 0.55 if nch else 0.0, "dims": (1, n1, n2)}


def _gradient(H, nbr, wb):
    """Stencil gradient of H, [k][i][j][x]."""
    G = torch.zeros((*H.shape, 3), dtype=H.dtype, device=H.device)
    t = torch.tensor(nbr, dtype=torch.int64, device=H.device)
    for n in range(nbr.shape[1]):
        d = H[t[:, n]] - H
        for x in range(3):
            if wb[n, x]:
                G[..., x] += wb[n, x] * d
    return G


def _dt(case):
    return {"rk4": 0.05, "ab": 0.03, "taylor": 0.03}[case["stepper"]]


def _fields(case, seed):
    """Field evaluations of the pass's steps, [steps][evals][6], around the peak of a
    gaussian pump in the plane, and half the probe on the core transitions."""
    rng = np.random.default_rng([seed, 1])
    e0, w, ph, ang = rng.uniform(0.2, 0.5) * 0.01944, rng.uniform(0.4, 1.0) * EV, rng.uniform(0, 2 * math.pi), rng.uniform(0.1, 1.0)
    pol = np.array([0.0, math.cos(ang), math.sin(ang)]) if case.get("pol", 1) == 2 else np.array([0.0, 0.0, 1.0])
    dt, n = _dt(case), case["steps"]
    at = [0.0, 0.5, 1.0] if case["stepper"] == "rk4" else [0.0]
    t = (np.arange(n)[:, None] + np.array(at)) * dt
    env = e0 * np.exp(-((t - 0.5 * n * dt) / 400.0) ** 2) * np.cos(w * t + ph)
    f = np.zeros((n, len(at), 6))
    f[..., :3] = env[..., None] * pol
    if case.get("nch", 0):
        f[..., 3] = 1e-4 * np.exp(-((t - 0.5 * n * dt) / 3.0) ** 2)
    return f, np.ones(n, dtype=np.uint8)


def _tau_inverse(order, dt):
    t = dt * np.arange(1, order)
    return np.linalg.inv(t[:, None] ** np.arange(1, order))


def _coulomb_tables(nb, ncut, seed):
    """Decaying mean-field coefficients with the structure of the generator's: A, D real, B, C imaginary."""
    rng = np.random.default_rng([seed, 2])
    m = np.arange(ncut)
    decay = (0.05 / (1.0 + m[:, None] ** 2 + m[None, :] ** 2)).reshape(-1, 1)
    q = [decay * (1.0 + 0.3 * rng.uniform(size=(ncut * ncut, nb * nb))) * f for f in (1.0, 0.3j, 0.3j, 0.5)]
    screen = (0.02 * (1.0 + 0.3 * rng.uniform(size=nb * nb))).astype(complex)
    vh = 0.3 * rng.uniform(size=(nb, nb))
    return {"ncut": ncut, "A": q[0].astype(complex), "B": q[1], "C": q[2], "D": q[3].astype(complex), "screen": screen,
            "vh": (0.5 * (vh + vh.T)).astype(complex)}


class _Coulomb(C.Structure):
    """edus_coulomb of include/edus.h."""
    _fields_ = [("ncut", C.c_int32), ("diag_basis", C.c_int32)] + [(n, C.POINTER(C.c_double)) for n in ("A", "B", "C", "D", "screen", "vh")]


def _problem(m, case, coul=None):
    """native.Problem of a model, and the host arrays behind it (alive until the engine is made)."""
    p, keep = N.Problem(), []

    def host(a):
        a = np.ascontiguousarray(a.cpu().numpy() if torch.is_tensor(a) else a)
        keep.append(a)
        return a.ctypes.data_as(C.POINTER(C.c_int32 if a.dtype == np.int32 else C.c_double))

    p.nk, p.nb, p.nch, p.ncc, p.n_nbr = m["nk"], m["nb"], m["nch"], m["ncc"], m["nbr"].shape[1]
    p.stepper, p.order, p.precision = STEPPERS[case["stepper"]], case["order"], PRECISIONS[case.get("precision", "fp64")]
    p.nbr, p.nbr_wb, p.T = host(m["nbr"]), host(m["wb"]), host(m["T"])
    p.H, p.D, p.U, p.rho0 = host(m["H"]), host(m["D"]), host(m["U"]), host(m["rho0"])
    p.gradH = host(_gradient(m["H"], m["nbr"], m["wb"]))
    p.wx2, p.dt, p.nktot = m["wx2"], _dt(case), float(m["nk"])
    p.j_norm, p.tabs_norm = 0.05 / m["nk"], 1.4 / m["nk"]
    if case["stepper"] == "taylor":
        p.taylor_tau_inv = host(_tau_inverse(case["order"], _dt(case)))
    for i in range(3):
        p.nk_dims[i] = m["dims"][i]
    if coul:
        q = _Coulomb()
        q.ncut, q.diag_basis = coul["ncut"], 0
        for n in ("A", "B", "C", "D", "screen", "vh"):
            setattr(q, n, host(coul[n]))
        keep.append(q)
        p.coulomb = C.cast(C.pointer(q), C.c_void_p)
    return p, keep


def _members(case, seed):
    """The problems of a scan: grid, band count and pulse of each."""
    rng = np.random.default_rng([case["count"], case["lo"], case["hi"]])  # sizes belong to the case, values to the seed
    out = []
    for i in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        out.append({"nb": (8, 4, 2)[i % 3], "n1": n, "n2": n, "stepper": "rk4", "order": 4, "steps": case["steps"], "pol": 2})
    return [(c, seed * 1000 + i) for i, c in enumerate(out)]


def _coulomb_case(case):
    return {**case, "nb": 3, "nch": 1}


def _wannier_model(case, seed):
    rng = np.random.default_rng(seed)
    r, nw = case["rmax"], case["nw"]
    R = np.array([(0, i, j) for i in range(-r, r + 1) for j in range(-r, r + 1)], dtype=np.int32)
    n = len(R)
    decay = np.exp(-np.linalg.norm(R, axis=1) * 2.5 / 2.0)
    X = rng.normal(size=(n, nw, nw, 4, 2)) @ np.array([1.0, 1j]) * decay[:, None, None, None]
    X = 0.5 * (X + X[::-1].conj().transpose(0, 2, 1, 3))  # R runs to -R in reverse order: H(-R) = H(R)^+
    return R, np.ascontiguousarray(0.05 * X[..., 0]), np.ascontiguousarray(0.5 * X[..., 1:])


def _coefficient_params(case, seed):
    rng = np.random.default_rng(seed)
    b = _lattice()
    m = np.arange(-80, 81)
    g = np.stack(np.meshgrid(m, m, indexing="ij"), -1).reshape(-1, 2)
    g = g[np.linalg.norm(g @ b, axis=1) < case["shell"] * np.linalg.norm(b[0])]
    disp = np.zeros((case["nb"], 3))
    disp[:, 1:] = rng.uniform(-1.5, 1.5, size=(case["nb"], 2))
    return {"nb": case["nb"], "ncut": case["ncut"], "n_sum": case["n_sum"], "n_peak": case["n_peak"], "rytova": 1,
            "g": g.astype(np.int32), "b1": b[0], "b2": b[1], "eps_area": A_LAT ** 2 * math.sqrt(3) / 2, "qtf": 0.01,
            "r0": 18.89726, "q_peak": 0.02, "disp": disp}


def _input_text(case, seed):
    """The reference's example input (Haldane model of boron nitride, circular pump), its pulse from the seed."""
    rng = np.random.default_rng(seed)
    return ("NEWINPUT\n\ntdse{\ntightbinding Haldane_CoreBN_Nedge gap=  7.25 t1=  -2.3 t2= 0 phi0= 0.0\n"
            f"dt 0.1 au\nt_fin 1650.0 au\nAdams_Bashforth {case['order']}\nnum_pump_pulses 1\n}}\n\n"
            f"nkPT{{\n1 {case['n']} {case['n']}\n}}\n\ndecoherence{{\ncorehole 0.00396892 au\n}}\n\n"
            f"laserpump sin2 {{\ncycles 1\nwavelength {rng.uniform(150.0, 200.0)!r} nm\nintensity {rng.uniform(0.5, 2.0) * 1e12!r} wcm2\n"
            "polarization circular 0 1 0 0 0 1\n}\n\n"
            "laserprobe gaussian {\nsigma 0.08 fs\ndelay 0 fs\nintensity 10.e+06\nfrequency 15.06\npolarization 1 0 0\n}\n\n"
            f"observables{{\nit_resolution {case['res']}\nTAbs\nCurrent\n}}\n")


def prepare(case, seed):
    kind, dev = case["kind"], _device()
    if kind == "run":
        tmp = tempfile.TemporaryDirectory()
        path = os.path.join(tmp.name, "input.txt")
        with open(path, "w") as f:
            f.write(_input_text(case, seed))
        return {"case": case, "tmp": tmp, "setup": N.Setup(path), "out": tmp.name}
    if kind == "wannier":
        return {"case": case, "model": _wannier_model(case, seed)}
    if kind == "coefficients":
        return {"case": case, "params": _coefficient_params(case, seed)}
    if kind == "batch":
        members, keep = _members(case, seed), []
        for c, s in members:
            keep.append(_problem(_model(c, s, dev), c))
        fields = [_fields(c, s) for c, s in members]
        return {"case": case, "batch": N.Batch([p for p, _ in keep]), "fields": [f for f, _ in fields], "on": [g for _, g in fields]}
    coul = None
    if kind == "coulomb":
        case = _coulomb_case(case)
        coul = _coulomb_tables(case["nb"], case["ncut"], seed)
    m = _model(case, seed, dev)
    p, keep = _problem(m, case, coul)
    eng = N.Engine(p)
    f, on = _fields(case, seed)
    return {"case": case, "engine": eng, "fields": f, "on": on, "ncc": m["ncc"]}


# ---------------------------------------------------------------- passes

def _elements(case, ncc):
    """k-resolved elements that a run prints: the last filled band, the first empty one, the coherence between them."""
    return [] if ncc >= case["nb"] else [(ncc - 1, ncc - 1), (ncc, ncc), (ncc - 1, ncc)]


def _whole_state(case):
    return case["n1"] * case["n2"] * case["nb"] ** 2 <= 100_000


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        s, n = state["setup"], case["steps"]
        s.run(state["out"], max_steps=n)
        return {f: np.fromfile(os.path.join(state["out"], "Output", f + ".txt"), sep=" ") for f in ("J1", "J2", "Losses")}
    if kind == "wannier":
        R, HR, rR = state["model"]
        form = case["form"]
        H, D = N.wannier_hk([1, case["n1"], case["n2"]], R, HR, rR, case["nw"], fp32=form == "fp32", bf16x3=form == "bf16x3")
        return {"H": H, "D": D}
    if kind == "coefficients":
        return N.coulomb_coefficients(state["params"])
    if kind == "batch":
        state["batch"].step(state["fields"], state["on"])
        return [m.observables() for m in state["batch"].members]
    eng, f, on, res = state["engine"], state["fields"], state["on"], case["res"]
    out = {"obs": []}
    for s in range(0, case["steps"], res):
        eng.step(f[s:s + res], on[s:s + res])
        out["obs"].append(eng.observables())
    if _whole_state(case):
        out["state"] = eng.get_state()
    else:
        out["elements"] = [eng.eigen_element(i, j) for i, j in _elements(case, state["ncc"])]
    return out


# ---------------------------------------------------------------- what a pass cannot do without

def _step_work(case):
    """Bytes and flops of the case's steps: packed Hermitian matrices (8 nb^2 bytes), per right-hand side the state in,
    H, the dipole components of the field, U with dephasing, and the stepper's own state arrays."""
    nb, nk = case["nb"], case["n1"] * case["n2"]
    pk = 8.0 * nb * nb
    op = pk if case.get("precision", "fp64") == "fp64" else pk / 2
    rhs = op * (1 + case.get("pol", 1) + (1 if case.get("nch", 0) else 0)) + (2 * op if case.get("diss") else 0)
    per = {"rk4": 4 * rhs + 16 * pk, "ab": rhs + (2 + case["order"]) * pk, "taylor": rhs + (2 + case["order"]) * pk}[case["stepper"]]
    evals = 4 if case["stepper"] == "rk4" else 1
    flops = evals * (8.0 * nb ** 3 * (5 if case.get("diss") else 1) + 24.0 * nb * nb)
    return {"bytes": case["steps"] * nk * per, "flops": case["steps"] * nk * flops}


def _observe_work(case):
    """One evaluation of the observables: state, U, H, three components of D and of the gradient of H."""
    nb, nk = case["nb"], case["n1"] * case["n2"]
    return {"bytes": nk * 8.0 * nb * nb * 10, "flops": nk * (8.0 * nb ** 3 * 2 + 60.0 * nb * nb)}


def work(case):
    kind = case["kind"]
    if kind == "run":
        n = {"nb": 3, "n1": case["n"], "n2": case["n"], "stepper": "ab", "order": case["order"], "steps": case["steps"], "nch": 1,
             "diss": True, "pol": 2}
        s, o = _step_work(n), _observe_work(n)
        m = case["steps"] / case["res"]
        return {"bytes": s["bytes"] + m * o["bytes"], "flops": s["flops"] + m * o["flops"]}
    if kind == "wannier":
        nk, nw2, nr = case["n1"] * case["n2"], case["nw"] ** 2, (2 * case["rmax"] + 1) ** 2
        return {"bytes": 64.0 * nw2 * (nk + nr), "flops": 32.0 * nk * nr * nw2}
    if kind == "coefficients":
        ng = 3.63 * case["shell"] ** 2
        pair = case["nb"] * (case["nb"] - 1) // 2
        q = case["n_sum"] ** 2 + 0.56 * (0.0133 * case["n_peak"]) ** 2 * 4
        return {"bytes": 8.0 * (case["n_sum"] ** 2 * (1 + 2 * pair)), "flops": q * ng * (20 + 10.0 * pair)}
    if kind == "batch":
        w = [f(c) for c, _ in _members(case, 0) for f in (_step_work, _observe_work)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    case = _coulomb_case(case) if kind == "coulomb" else case
    nb, nk = case["nb"], case["n1"] * case["n2"]
    s, o, m = _step_work(case), _observe_work(case), math.ceil(case["steps"] / case["res"])
    w = {k: s[k] + m * o[k] for k in s}
    if kind == "coulomb":
        evals = case["steps"] * (4 if case["stepper"] == "rk4" else 1)
        w["bytes"] += evals * nk * 8.0 * nb * nb
        # the two transforms, separable: rows, then columns
        w["flops"] += evals * 2 * nb * nb * 4.0 * case["ncut"] * (nk + 2 * case["ncut"] * (case["n1"] + case["n2"]) / 2) * 2
    w["bytes"] += nk * 16.0 * nb * nb if _whole_state(case) else 3 * nk * (24.0 * nb * nb + 16)
    return w


# ---------------------------------------------------------------- the same passes in plain torch, 64 bits

class _Plain:
    """One problem's time loop, restated."""

    def __init__(self, case, seed, dev, coul=None):
        self.case, self.m = case, _model(case, seed, dev)
        m = self.m
        nb, nch = m["nb"], m["nch"]
        self.P = m["rho0"].clone()
        self.dt, self.hist = _dt(case), []
        self.nbr = torch.tensor(m["nbr"], dtype=torch.int64, device=dev)
        core = torch.zeros((nb, nb), dtype=torch.bool, device=dev)
        core[:nch, nch:] = True
        self.rwa = core.to(torch.complex128) * (1j * m["wx2"])
        self.core = core | core.T
        self.T = torch.tensor(m["T"], device=dev, dtype=torch.complex128)
        self.diss = bool((m["T"] != 0).any())
        U = m["U"]
        tv = torch.tensor(np.diag(m["T"])[:m["ncc"]].copy(), device=dev, dtype=torch.complex128)
        self.hole = (U[:, :m["ncc"]].mT * tv) @ U[:, :m["ncc"]].conj()
        self.up = torch.triu(torch.ones(nb, nb, device=dev, dtype=torch.complex128), 1)
        self.coul, self.n_cond, self.Hr = None, 0.0, m["H"]
        if coul:
            self.coul = {k: torch.tensor(v, device=dev) if isinstance(v, np.ndarray) else v for k, v in coul.items()}
            nc, (_, n1, n2) = coul["ncut"], m["dims"]
            mm = torch.arange(nc, dtype=torch.float64, device=dev)
            a1 = 2 * math.pi * mm[:, None] * (-0.5 + torch.arange(n1, dtype=torch.float64, device=dev) / n1)
            a2 = 2 * math.pi * mm[:, None] * (-0.5 + torch.arange(n2, dtype=torch.float64, device=dev) / n2)
            self.trig = [torch.cos(a1), torch.sin(a1), torch.cos(a2), torch.sin(a2)]
            self.corr = (1 - 4 * math.pi ** 2 * (mm[:, None] ** 2 + mm[None, :] ** 2) / (m["nk"] * 27)) / m["nk"]
            self.X0, self.EH0 = 0.0, 0.0
            self.X0, self.EH0 = self._modes(self.P)

    def _hermitise(self, V):
        """From the upper triangle and the real part of the diagonal."""
        u = V * self.up
        return u + u.mH + torch.diag_embed(torch.diagonal(V, dim1=1, dim2=2).real).to(V.dtype)

    def _modes(self, P):
        """(X_mn of the four trig products [4][mn][i][j], Hartree shift), minus their equilibrium values."""
        c, nb = self.coul, self.m["nb"]
        n1, n2 = self.m["dims"][1:]
        nc = c["ncut"]
        G = P.reshape(n1, n2, nb * nb)
        t = [x.to(torch.complex128) for x in self.trig]
        F = [torch.einsum("ma,ane->mne", t[a], torch.einsum("nb,abe->ane", t[2 + b], G)) * self.corr[..., None] for a in (0, 1) for b in (0, 1)]
        F = [f.reshape(nc * nc, nb, nb) for f in F]
        A, B, Cc, D = (c[k].reshape(nc * nc, nb, nb).clone() for k in "ABCD")
        i = torch.arange(nb, device=P.device)
        A[:, i, i], D[:, i, i] = A[:, :1, 0].expand(-1, nb), D[:, :1, 0].expand(-1, nb)
        B[:, i, i] = Cc[:, i, i] = 0
        cc, cs, sc, ss = F
        X = torch.stack([A * cc + D * ss + B * cs + Cc * sc, A * cs - D * sc + Cc * ss - B * cc,
                         A * sc - D * cs + B * ss - Cc * cc, A * ss + D * cc - B * sc - Cc * cs])
        u = X * self.up
        X = u + u.mH + torch.diag_embed(torch.diagonal(X, dim1=2, dim2=3))
        EH = c["vh"].real @ torch.diagonal(cc[0]).real
        return X - self.X0, EH - self.EH0

    def _mean_field(self, P):
        c, m = self.coul, self.m
        nb, nc = m["nb"], c["ncut"]
        n1, n2 = m["dims"][1:]
        X, EH = self._modes(P)
        X = X.mT.reshape(4, nc, nc, nb * nb)  # the reconstruction reads X_ji
        t = [x.to(torch.complex128) for x in self.trig]
        Tc = torch.einsum("mne,nb->mbe", X[0], t[2]) + torch.einsum("mne,nb->mbe", X[1], t[3])
        Ts = torch.einsum("mne,nb->mbe", X[2], t[2]) + torch.einsum("mne,nb->mbe", X[3], t[3])
        xk = -(torch.einsum("ma,mbe->abe", t[0], Tc) + torch.einsum("ma,mbe->abe", t[1], Ts)).reshape(-1, nb, nb)
        if self.n_cond > 1e-20:
            s = c["screen"].reshape(nb, nb).conj().clone()
            i = torch.arange(nb, device=P.device)
            s[i, i] = c["screen"][0].conj()
            xk = xk - s * (P - m["rho0"]).mT
        return self._hermitise(m["H"] + xk + torch.diag(EH).to(torch.complex128))

    def rhs(self, P, E):
        m = self.m
        Ep, Eq = ([float(v) for v in E[:3]], [float(v) for v in E[3:]])
        Hm = self.Hr = self._mean_field(P) if self.coul else m["H"]
        Dp = sum(Ep[x] * m["D"][..., x] for x in range(3))
        Dq = sum(Eq[x] * m["D"][..., x] for x in range(3))
        X = P @ (Hm + torch.where(self.core, Dq, Dp)).mT
        V = -1j * (X - X.mH) + self.rwa * P
        if self.diss:
            Uc = m["U"].conj()
            V = V - Uc @ (self.T * (Uc @ P @ m["U"].mT)) @ Uc + self.hole
        V = self._hermitise(V)
        for n in range(len(OFFSETS)):
            cn = float(sum(Ep[x] * m["wb"][n, x] for x in range(3)))
            V = V + cn * P[self.nbr[:, n]]
        return V

    def step(self, E):
        dt, P, how = self.dt, self.P, self.case["stepper"]
        if how == "rk4":
            k1 = self.rhs(P, E[0])
            k2 = self.rhs(P + 0.5 * dt * k1, E[1])
            k3 = self.rhs(P + 0.5 * dt * k2, E[1])
            k4 = self.rhs(P + dt * k3, E[2])
            self.P = P + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
            return
        o = self.case["order"]
        f = self.rhs(P, E[0])
        while len(self.hist) < o - 1:
            self.hist.append(torch.zeros_like(f))
        if how == "ab":
            co = {1: [1], 2: [3 / 2, -1 / 2], 3: [23 / 12, -16 / 12, 5 / 12], 4: [55 / 24, -59 / 24, 37 / 24, -9 / 24],
                  5: [1901 / 720, -2774 / 720, 2616 / 720, -1274 / 720, 251 / 720]}[o]
            d = dt * sum(c * h for c, h in zip(co, [f] + self.hist))
        else:
            ti = _tau_inverse(o, dt)
            d = dt * f
            for i in range(1, o):
                d = d + dt ** (i + 1) / (i + 1) * sum(float(ti[i - 1, p]) * (f - self.hist[p]) for p in range(o - 1))
        self.P = P + d
        self.hist = ([f] + self.hist)[:o - 1]

    def observables(self):
        m, P = self.m, self.P
        nb, nch, nk = m["nb"], m["nch"], m["nk"]
        U = m["U"]
        if self.coul:
            U = torch.linalg.eigh(self.Hr.cpu())[1].mH.to(P.device)
        pk = torch.diagonal(U.conj() @ P @ U.mT, dim1=1, dim2=2).real
        pop = pk.sum(0) / nk
        filled = torch.arange(nb, device=P.device) < m["ncc"]
        hole = torch.where(filled, 1 - pk, pk)
        G = _gradient(self.Hr, m["nbr"], m["wb"])
        j1 = torch.einsum("kij,kijx->x", P, G).real * (0.05 / nk)
        j2 = torch.einsum("kij,kijx->x", P, torch.stack([self.Hr @ m["D"][..., x].mH for x in range(3)], -1)) * (0.05 / nk)
        ta = -2 * torch.einsum("kij,kijx->x", P[:, :nch, nch:], m["D"][:, :nch, nch:]) * (1.4 / nk)
        if self.coul:
            self.n_cond = float(torch.where(filled, 1 - pop, pop).max())
        two = lambda v: torch.view_as_real(v.to(torch.complex128)).reshape(-1).cpu().numpy()  # noqa: E731
        return {"pop": pop.cpu().numpy(), "j1": two(j1), "j2": two(j2), "tabs": two(ta),
                "pminmax": np.array([float(hole.min().clamp(max=1.0)), float(hole.abs().max())])}

    def element(self, i, j):
        U = self.m["U"]
        v = torch.einsum("ki,kij,kj->k", U[:, i].conj(), self.P, U[:, j])
        return (v.real + 0j if i == j else v).to(torch.complex128).cpu().numpy()


def exact(case, seed):
    kind, dev = case["kind"], _device()
    if kind == "run":
        return None  # its tables are the framework's own; the text files are compared with the start's
    if kind == "wannier":
        return _exact_wannier(case, seed, dev)
    if kind == "coefficients":
        return _exact_coefficients(_coefficient_params(case, seed), dev)
    if kind == "batch":
        out = []
        for c, s in _members(case, seed):
            p = _Plain(c, s, dev)
            for E in _fields(c, s)[0]:
                p.step(E)
            out.append(p.observables())
        return out
    coul = None
    if kind == "coulomb":
        case = _coulomb_case(case)
        coul = _coulomb_tables(case["nb"], case["ncut"], seed)
    p = _Plain(case, seed, dev, coul)
    f, out = _fields(case, seed)[0], {"obs": []}
    for s in range(0, case["steps"], case["res"]):
        for E in f[s:s + case["res"]]:
            p.step(E)
        out["obs"].append(p.observables())
    if _whole_state(case):
        out["state"] = p.P.cpu().numpy()
    else:
        out["elements"] = [p.element(i, j) for i, j in _elements(case, p.m["ncc"])]
    return out


def _exact_wannier(case, seed, dev):
    R, HR, rR = _wannier_model(case, seed)
    n1, n2, nw = case["n1"], case["n2"], case["nw"]
    k = _kgrid(n1, n2, dev)
    ph = torch.exp(2j * math.pi * (k @ torch.tensor(R[:, 1:].astype(float), device=dev).T))
    H = (ph @ torch.tensor(HR, device=dev).reshape(len(R), -1)).reshape(-1, nw, nw)
    D = (ph @ torch.tensor(rR, device=dev).reshape(len(R), -1)).reshape(-1, nw, nw, 3)
    i = torch.arange(nw, device=dev)
    H[:, i, i] = H[:, i, i].real + 0j
    D[:, i, i] = D[:, i, i].real + 0j
    return {"H": H.cpu().numpy(), "D": (0.5 * (D + D.transpose(1, 2))).cpu().numpy()}


def _screened(q, p, qtf2, dev):
    """W(q) = sum_G V(|q + G|) e^{i (q + G).(d_i - d_j)}: the diagonal value and one complex value per pair i < j."""
    b = torch.tensor(np.stack([p["b1"], p["b2"]]), device=dev)
    nb, disp = p["nb"], torch.tensor(p["disp"], device=dev)
    beta = torch.stack([b @ (disp[i] - disp[j]) for i in range(nb) for j in range(i + 1, nb)], 1)
    g = torch.tensor(p["g"].astype(float), device=dev)
    eg, w0, wp = torch.exp(1j * (g @ beta)), [], []
    for part in q.split(4096):
        v = (part[:, None, :] + g) @ b
        r = torch.linalg.norm(v, dim=-1)
        V = 2 * math.pi / (p["eps_area"] * torch.sqrt(r * r + qtf2) * (r * p["r0"] + 1))
        w0.append(V.sum(1))
        wp.append((V.to(torch.complex128) @ eg) * torch.exp(1j * (part @ beta)))
    return torch.cat(w0), torch.cat(wp)


def _exact_coefficients(p, dev):
    nb, nc, n = p["nb"], p["ncut"], p["n_sum"]
    pairs = [(i, j) for i in range(nb) for j in range(i + 1, nb)]
    x = -0.5 + torch.arange(n, dtype=torch.float64, device=dev) / (n - 1)
    w0, wp = _screened(torch.stack(torch.meshgrid(x, x, indexing="ij"), -1).reshape(-1, 2), p, p["qtf"] ** 2, dev)
    simpson = torch.full((n,), 2.0, dtype=torch.float64, device=dev)
    simpson[1::2] = 4.0
    simpson[0] = simpson[-1] = 1.0
    simpson /= 3 * (n - 1)
    m = torch.arange(nc, dtype=torch.float64, device=dev)
    arg = 2 * math.pi * m[:, None] * x
    c, s = torch.cos(arg) * simpson, torch.sin(arg) * simpson
    sc = 4.0 * torch.where(m > 0, 1.0, 0.5).outer(torch.where(m > 0, 1.0, 0.5)).to(torch.float64)
    both = lambda u, v, f: (sc * (u @ f.reshape(n, n) @ v.T)).reshape(-1)  # noqa: E731
    A, B, Cc, D = (torch.zeros((nc * nc, nb * nb), dtype=torch.complex128, device=dev) for _ in range(4))
    A[:, 0], D[:, 0] = both(c, c, w0) + 0j, both(s, s, w0) + 0j
    for k, (i, j) in enumerate(pairs):
        re, im = wp[:, k].real.contiguous(), wp[:, k].imag.contiguous()
        A[:, i * nb + j], D[:, i * nb + j] = both(c, c, re) + 0j, both(s, s, re) + 0j
        B[:, i * nb + j], Cc[:, i * nb + j] = 1j * both(c, s, im), 1j * both(s, c, im)
    # Hartree term at q = 0, V = 0 where the offsets sum to zero or less
    b = np.stack([p["b1"], p["b2"]])
    cart = p["g"] @ b
    r = np.linalg.norm(cart, axis=1)
    V = np.where(p["g"].sum(1) <= 0, 0.0, 2 * math.pi / (p["eps_area"] * np.sqrt(r * r + p["qtf"] ** 2) * (r * p["r0"] + 1)))
    vh = np.zeros((nb, nb), dtype=complex)
    np.fill_diagonal(vh, V.sum())
    for i, j in pairs:
        vh[i, j] = vh[j, i] = (V * np.cos(cart @ (p["disp"][i] - p["disp"][j]))).sum()
    # the correction around q = 0 on the finer grid
    npk = p["n_peak"]
    lo = int(npk * 0.45)
    f = -0.5 + np.arange(lo, npk - lo) * (1.0 / (npk - 1))
    q = np.stack(np.meshgrid(f, f, indexing="ij"), -1).reshape(-1, 2)
    q2 = ((q @ b) ** 2).sum(1)
    q = torch.tensor(q[(q2 < p["q_peak"] ** 2) & (q2 > 1e-17)], device=dev)
    screen = np.zeros(nb * nb, dtype=complex)
    if len(q):
        w0, wp = _screened(q, p, 0.0, dev)
        a1, a2 = 2 * math.pi * q[:, :1] * m, 2 * math.pi * q[:, 1:] * m
        tr = [torch.cos(a1), torch.sin(a1), torch.cos(a2), torch.sin(a2)]
        for i in range(nb):
            for j in range(i, nb):
                at = i * nb + j
                series = sum(((u.to(torch.complex128) @ K[:, at].reshape(nc, nc)) * v).sum(1)
                             for K, u, v in ((A, tr[0], tr[2]), (B, tr[0], tr[3]), (Cc, tr[1], tr[2]), (D, tr[1], tr[3])))
                w = w0 + 0j if i == j else wp[:, pairs.index((i, j))]
                screen[at] = complex((w - series).sum().item()) / npk ** 2
    h = [t.cpu().numpy() for t in (A, B, Cc, D)]
    return {"A": h[0], "B": h[1], "C": h[2], "D": h[3], "screen": screen, "vh": vh}
