"""The work this framework is measured on: the calls a GW run makes, through
the public entry points, over the range of their sizes.

A GW run builds W by batched Sternheimer solves (one operator per set of k+q
points, systems = bands x perturbations, shifts = frequencies), takes it to a
dielectric matrix, continues it to the frequencies Sigma needs, builds G the
same way, and forms Sigma from both.  Each kind below is one of those calls:

  apply    the shifted Hamiltonian on a block of vectors
  solve    a lock-step batch of multishift systems
  stream   a queue of systems through a fixed number of solver slots
  adjoint  the backward solve and dL/dV_loc of a stored forward solve
  response columns of the dielectric matrix (solve, density, Hartree kernel)
  green    G(G, G'; omega) of one k-point, taken to real space
  sigma    Sigma_c from W's continuation and G(r, r') (real-space products)
  robust   continuation of W by the robust Pade approximant, and one evaluation
  aaa      continuation of W by AAA, and one evaluation
  conv     the frequency convolution as a GEMM

Cells are the fcc cell of sternheimergw_amd.cell (a = 10.26 bohr, seeded
V_loc); 24^3 at 6 Ha and 48^3 at 25 Ha are its two configurations.  All data
are complex128, the type the framework computes in.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from sternheimergw_amd import _lib, batch, cell, green, operators, scf, sigma, sigma_real

HA2RY = 2.0
ALAT = 10.26
THRESHOLD = 1e-10         # default of green_function and solve_linter
ECUT_MAX = {24: 8.0, 32: 12.0, 36: 16.0, 48: 25.0}   # Ha; the sphere each box holds


def listed():
    return [
        # one band of a few: what a single-system solve applies per product
        {"name": "apply-24-4", "kind": "apply", "box": 24, "ecut": 6.0, "lmax": 1, "nbnd": 4,
         "nq": 1, "nvec": 4},
        # one q-batch of the 25 Ha cell, ragged spheres of four k+q points
        {"name": "apply-48-256", "kind": "apply", "box": 48, "ecut": 25.0, "lmax": 3, "nbnd": 16,
         "nq": 4, "nvec": 256},
        # the small cell's whole W solve: 4 bands x 8 frequencies
        {"name": "solve-24-4x8", "kind": "solve", "box": 24, "ecut": 6.0, "lmax": 1, "nbnd": 4,
         "nq": 1, "npert": 1, "nshift": 8},
        # an ordinary cell: 8 bands x 2 q x 2 perturbations, odd shift count
        {"name": "solve-36-32x15", "kind": "solve", "box": 36, "ecut": 13.0, "lmax": 2, "nbnd": 8,
         "nq": 2, "npert": 2, "nshift": 15},
        # the 25 Ha cell in production form: 16 bands x 4 q x 12 G streamed
        {"name": "stream-48-768x32", "kind": "stream", "box": 48, "ecut": 25.0, "lmax": 3,
         "nbnd": 16, "nq": 4, "npert": 12, "nshift": 32, "slots": 512},
        # gradient with respect to V_loc: 6 Ha sphere on a 48^3 box
        {"name": "adjoint-48-128x16", "kind": "adjoint", "box": 48, "ecut": 6.0, "lmax": 1,
         "nbnd": 8, "nq": 2, "npert": 8, "nshift": 16},
        # 16 columns of the dielectric matrix of the 25 Ha cell, 16 frequencies
        {"name": "response-48-16", "kind": "response", "box": 48, "ecut": 25.0, "lmax": 3,
         "nbnd": 16, "npert": 16, "nfreq": 16, "num_g": 100},
        # G of one k-point on a 16^3 correlation grid, all G' columns at once
        {"name": "green-24-113", "kind": "green", "box": 24, "ecut": 6.0, "lmax": 1, "nbnd": 4,
         "n": 16, "n_p": 16, "num_g": 113, "num_g_p": 113, "nfreq": 4},
        # Sigma_c on the 24^3 correlation grid: 2 Sigma x 4 Green's frequencies
        {"name": "sigma-24-1500", "kind": "sigma", "n": 24, "n_p": 24, "num_g": 1500,
         "num_g_p": 1500, "ncoul": 2, "nsigma": 2},
        # W of 400 x 400 elements continued from 32 points of a circle
        {"name": "robust-400-32", "kind": "robust", "num_g": 400, "nfreq": 32},
        # the same from 35 points of the imaginary axis by AAA
        {"name": "aaa-400-35", "kind": "aaa", "num_g": 400, "nfreq": 35},
        # four output frequencies of the convolution at N_G = 1500
        {"name": "conv-1500-4x8", "kind": "conv", "n": 1500, "nout": 4, "nin": 8},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: any kind, sizes over the range the listed ones span."""
    kind = rng.choice(["apply", "solve", "stream", "adjoint", "response", "green", "sigma",
                       "robust", "aaa", "conv"])
    c = {"kind": kind}
    if kind in ("apply", "solve", "stream", "adjoint", "response", "green"):
        box = rng.choice([24, 32, 36, 48])
        if kind == "green":
            box = rng.choice([24, 32])
        ecut = round(rng.uniform(6.0, ECUT_MAX[box]), 2)
        if kind == "adjoint":
            ecut = round(rng.uniform(6.0, 8.0), 2)
        c.update(box=box, ecut=ecut, lmax=rng.randint(1, 3), nbnd=rng.randint(1, 16))
    if kind == "apply":
        c.update(nq=rng.randint(1, 4), nvec=round(_log(rng, 1, 512)))
    elif kind == "solve":
        c.update(nq=rng.randint(1, 2), npert=rng.randint(1, 4), nshift=rng.randint(1, 32))
    elif kind == "stream":
        c.update(nq=rng.randint(1, 2), npert=rng.randint(4, 12), nshift=rng.randint(1, 32),
                 slots=rng.choice([64, 128, 256, 512]))
    elif kind == "adjoint":
        c.update(nq=rng.randint(1, 2), npert=rng.randint(1, 8), nshift=rng.randint(1, 16))
    elif kind == "response":
        c.update(npert=rng.randint(1, 8), nfreq=rng.randint(2, 12), num_g=rng.randint(20, 100))
    elif kind == "green":
        c.update(n=rng.choice([16, 18]), n_p=rng.choice([16, 18]), num_g=rng.randint(27, 137),
                 num_g_p=rng.randint(27, 137), nfreq=rng.randint(1, 6))
    elif kind == "sigma":
        n, n_p = rng.choice([16, 18, 24]), rng.choice([16, 18, 24])
        c.update(n=n, n_p=n_p, num_g=rng.randint(n ** 3 // 40, n ** 3 // 9),
                 num_g_p=rng.randint(n_p ** 3 // 40, n_p ** 3 // 9), ncoul=rng.randint(1, 2),
                 nsigma=rng.randint(1, 2))
    elif kind == "robust":
        c.update(num_g=round(_log(rng, 40, 400)), nfreq=rng.randint(12, 40))
    elif kind == "aaa":
        c.update(num_g=round(_log(rng, 40, 400)), nfreq=rng.randint(12, 40))
    else:
        c.update(n=round(_log(rng, 150, 1500)), nout=rng.randint(1, 4), nin=rng.randint(1, 8))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)
    return g


def _randn(shape, gen):
    return torch.randn(shape, dtype=torch.complex128, device=_dev(), generator=gen)


def _shortest(num, nonzero=False):
    g = cell.shortest_millers(num + 1)
    return g[1:num + 1] if nonzero else g[:num]


def _workload(case, seed):
    """The cell with its k+q spheres, projectors, occupied states and
    right-hand sides; imaginary shifts on [0, 4 Ha].  The spheres are the
    case's, V_loc and with it every state is the seed's."""
    q, scale = cell.c2_qpoints(case.get("nq", 1))
    nshift = case.get("nshift", 1)
    omega, _ = cell.gauss_legendre(0.0, 4.0, nshift)
    npert = case["npert"] if case["kind"] in ("solve", "stream", "adjoint") else 1
    return cell.build_workload("case", box=(case["box"],) * 3, ecut_ha=case["ecut"],
                               nbnd=case["nbnd"], lchan=list(range(case["lmax"] + 1)),
                               qpoints=q, ecut_scale=scale, omega_ha=1j * omega, alat=ALAT,
                               seed=seed, pert_mill=_shortest(npert))


def _dense(w, group, with_valence=True):
    """H (+ alpha_pv P_v) of one k+q group from V(G - G'), on the GPU."""
    s = w.spheres[group]
    vg = torch.from_numpy(np.fft.fftn(w.vloc) / w.vloc.size).to(_dev())
    m = torch.from_numpy(s.mill.astype(np.int64)).to(_dev())
    d = m[:, None, :] - m[None, :, :]
    n1, n2, n3 = w.box
    h = vg[d[..., 2] % n3, d[..., 1] % n2, d[..., 0] % n1]
    h = h + torch.diag(torch.from_numpy(s.kin).to(_dev())).to(h.dtype)
    np_ = w.nproj if with_valence else w.nproj_beta
    p = torch.from_numpy(w.proj[group, :np_, : s.npw]).to(_dev())
    dc = torch.from_numpy(w.dcoef[group, :np_]).to(_dev())
    return h + (p.T * dc[None, :]) @ p.conj()


def _spectral(h, rhs, sigma_):
    """x[s, k] = (h + sigma[s, k])^-1 rhs[s] from the eigenvectors of h."""
    lam, u = torch.linalg.eigh(h)
    c = rhs @ u.conj()
    return (c[:, None, :] / (lam[None, None, :] + sigma_[:, :, None])) @ u.T


def _solutions(w, sigma_, rhs=None):
    """Solutions (nsys, nshift, ld) of the workload's systems at sigma_."""
    out = torch.zeros((w.nsys, sigma_.shape[1], w.ld), dtype=torch.complex128, device=_dev())
    rhs = torch.from_numpy(w.rhs).to(_dev()) if rhs is None else rhs
    sig = torch.from_numpy(np.ascontiguousarray(sigma_)).to(_dev())
    for g in range(len(w.spheres)):
        at = torch.from_numpy(np.nonzero(w.group == g)[0]).to(_dev())
        n = w.spheres[g].npw
        out[at, :, :n] = _spectral(_dense(w, g), rhs[at, :n], sig[at])
    return out


def _vectors(w, nvec, seed):
    """Vectors as a Krylov space has them: random, falling off with the
    kinetic energy; groups in order, shifts of the workload's bands."""
    rng = np.random.default_rng(seed)
    group = np.sort(np.arange(nvec) % len(w.spheres)).astype(np.int32)
    x = np.zeros((nvec, w.ld), dtype=np.complex128)
    for v in range(nvec):
        s = w.spheres[group[v]]
        x[v, : s.npw] = (rng.standard_normal(s.npw) + 1j * rng.standard_normal(s.npw)) / (1.0 + s.kin)
    sig = -(w.eps_v[rng.integers(0, w.nbnd, nvec)] + 1j * rng.uniform(0.0, 8.0, nvec))
    return x, group, sig


def _w_poles(case, seed):
    """Pole strengths and positions of every element: pairs (p, p*) so that W
    is real where its argument is, outside radius 1.5."""
    ne = case["num_g"] ** 2
    gen = _gen(seed)
    npole = 3
    r = 1.5 + 2.5 * torch.rand((npole, ne), dtype=torch.float64, device=_dev(), generator=gen)
    phi = math.pi * torch.rand((npole, ne), dtype=torch.float64, device=_dev(), generator=gen)
    a = torch.randn((npole, ne), dtype=torch.float64, device=_dev(), generator=gen)
    if case["kind"] == "aaa":      # off the imaginary axis the samples lie on
        phi = 0.4 * phi
    return a, torch.polar(r, phi)


def _w_at(poles, z):
    a, p = poles
    return (a / (z - p) + a / (z - p.conj())).sum(0)


def _mesh(case):
    n = case["nfreq"]
    if case["kind"] == "robust":
        return np.exp(2j * np.pi * np.arange(n) / n)
    x, _ = cell.gauss_legendre(0.0, 8.0, n)
    return 1j * x


def _eval_freq(case):
    return 0.3 + 0.4j if case["kind"] == "robust" else 0.25 + 1.1j


def _corr_n(num_g):
    return next(n for n in (16, 18, 24) if n ** 3 >= num_g)


# plasmon-pole W on the imaginary axis, sampled at the solver's frequencies
SOLVER = 1j * np.array([0.0, 0.5, 1.5, 4.0])
MU = 0.05
SIGMA_FREQ = np.array([-0.2, 0.3])
COUL = 1j * np.array([0.1, 0.6])
WEIGHT = np.array([0.4, 0.6])


def _sigma_w(case, seed):
    gen = _gen(seed)
    ng = max(case["num_g"], case["num_g_p"])
    fall = 1.0 / (1.0 + 0.01 * torch.arange(ng, dtype=torch.float64, device=_dev()))
    amp = _randn((ng, ng), gen) * fall[:, None] * fall[None, :]
    om = 0.8 + 2.0 * torch.rand((ng, ng), dtype=torch.float64, device=_dev(), generator=gen)
    gam = 3.0 + torch.rand((ng, ng), dtype=torch.float64, device=_dev(), generator=gen)
    return torch.stack([amp / (z * z - om * om) + 0.3 * amp.conj() / (z * z - gam * gam)
                        for z in SOLVER.tolist()])


def _green_r(case, seed):
    nr, nr_p = case["n"] ** 3, case["n_p"] ** 3
    gen = _gen(seed + 1)
    return _randn((2 * case["ncoul"], nr_p, nr), gen) * 1e-3


def _omega_cell():
    return cell.fcc_lattice(ALAT)[2]


def _green_omega(case):
    return np.linspace(-0.4, 0.6, case["nfreq"]) + 1j * np.linspace(0.3, 1.2, case["nfreq"])


def _freqs(nf):
    x, _ = cell.gauss_legendre(0.0, 4.0, nf - 1)
    return np.concatenate([[0.0], 1j * x * HA2RY])


def prepare(case, seed):
    dev, kind = _dev(), case["kind"]
    st = {"case": case, "kind": kind}
    if kind in ("apply", "solve", "stream", "adjoint", "response", "green"):
        w = _workload(case, seed)
        op = operators.PwOperator.from_workload(w, with_valence=kind != "green")
        st.update(w=w, op=op)
    if kind == "apply":
        x, group, sig = _vectors(w, case["nvec"], seed)
        st.update(x=torch.from_numpy(x).to(dev), group=torch.from_numpy(group).to(dev),
                  sigma=torch.from_numpy(sig).to(dev),
                  ax=torch.zeros(x.shape, dtype=torch.complex128, device=dev))
    elif kind in ("solve", "stream", "adjoint"):
        slots = min(case["slots"], w.nsys) if kind == "stream" else w.nsys
        st.update(
            solver=batch.BatchSolver(op, slots, w.nshift, w.ld, lmax=4, threshold=THRESHOLD,
                                     shift_test=True),
            rhs=torch.from_numpy(w.rhs).to(dev), h_sigma=np.ascontiguousarray(w.sigma),
            sigma=torch.from_numpy(np.ascontiguousarray(w.sigma)).to(dev), h_group=w.group,
            group=torch.from_numpy(w.group).to(dev),
            x=torch.zeros((w.nsys, w.nshift, w.ld), dtype=torch.complex128, device=dev))
        if kind == "adjoint":
            st["c"] = -st["rhs"]
            st["weight"] = _adjoint_weight(w)
            st["y"] = st["x"]
            st["x"] = _solutions(w, w.sigma)
            st["grad"] = torch.zeros(tuple(reversed(w.box)), dtype=torch.float64, device=dev)
    elif kind == "response":
        _a, bg, vol = cell.fcc_lattice(ALAT)
        st.update(setup=scf.LinterSetup(op, w, 0), bg=bg, vol=vol,
                  pert=_shortest(case["npert"], nonzero=True), g=_shortest(case["num_g"]),
                  freq=_freqs(case["nfreq"]), gcut2=8.0 * case["ecut"])
    elif kind == "green":
        st.update(omega=_green_omega(case),
                  grid=green.CorrGrid(case["n"], _shortest(case["num_g"])),
                  grid_p=green.CorrGrid(case["n_p"], _shortest(case["num_g_p"])))
    elif kind == "sigma":
        st.update(grid=green.CorrGrid(case["n"], _shortest(case["num_g"])),
                  grid_p=green.CorrGrid(case["n_p"], _shortest(case["num_g_p"])),
                  green=_green_r(case, seed),
                  w=sigma_real.ScreenedCoulomb(_sigma_w(case, seed), SOLVER, _lib.PADE_APPROX,
                                               sigma_real.NO_SYMMETRY))
    elif kind in ("robust", "aaa"):
        ng = case["num_g"]
        poles = _w_poles(case, seed)
        n = _corr_n(ng)
        grid = green.CorrGrid(n, _shortest(ng))
        st.update(w=torch.stack([_w_at(poles, z).reshape(ng, ng) for z in _mesh(case).tolist()]),
                  grid=grid, gmap=torch.arange(ng, dtype=torch.int32, device=dev),
                  out=torch.empty((grid.nr, grid.nr), dtype=torch.complex128, device=dev))
    else:
        n, nout, nin = case["n"], case["nout"], case["nin"]
        gen = _gen(seed)
        fall = 1.0 / (1.0 + 0.01 * torch.arange(n, dtype=torch.float64, device=dev))
        st.update(g=_randn((nout, nin, n, n), gen) / math.sqrt(n),
                  w=_randn((nin, n, n), gen) * fall[:, None] * fall[None, :],
                  weight=torch.from_numpy(cell.gauss_legendre(0.0, 4.0, nin)[1]).to(dev),
                  s=torch.empty((nout, n, n), dtype=torch.complex128, device=dev))
    return st


def _adjoint_weight(w):
    wt = cell.gauss_legendre(0.0, 4.0, w.nshift)[1]
    return torch.from_numpy((1.0 / (1.0 + w.pert_q2))[:, None] * wt[None, :]).to(_dev())


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case, kind = st["case"], st["kind"]
    if kind == "apply":
        _lib.check(_lib.lib().sgw_operator_apply_device(
            st["op"].handle, case["nvec"], _ptr(st["group"]), _ptr(st["sigma"]), _ptr(st["x"]),
            st["w"].ld, _ptr(st["ax"]), _stream()))
        return st["ax"]
    if kind == "solve":
        ierr, _it = st["solver"].solve(st["group"], st["rhs"], st["sigma"], st["h_sigma"], st["x"])
        return {"x": st["x"], "ierr": ierr}
    if kind == "stream":
        ierr, _it = st["solver"].solve_stream(st["h_group"], st["rhs"], st["sigma"],
                                              st["h_sigma"], st["x"])
        return {"x": st["x"], "ierr": ierr}
    if kind == "adjoint":
        loss, ierr = st["solver"].adjoint(st["group"], st["c"], st["sigma"], st["h_sigma"],
                                          st["weight"], st["x"], st["y"], st["grad"])
        return {"loss": loss, "y": st["y"], "grad": st["grad"], "ierr": ierr}
    if kind == "response":
        return scf.coulomb_columns_direct(st["setup"], st["pert"], st["freq"], st["g"],
                                          bg=st["bg"], gcut2=st["gcut2"], threshold=THRESHOLD,
                                          volume=st["vol"])
    if kind == "green":
        g = green.green_function(st["op"], 0, st["w"].spheres[0].mill, st["omega"], st["grid"],
                                 st["grid_p"], threshold=THRESHOLD)
        return green.invfft6(g, st["grid"], _omega_cell(), st["grid_p"])
    if kind == "sigma":
        nc, ns = case["ncoul"], case["nsigma"]
        return sigma_real.sigma_correlation(st["grid"], st["grid_p"], _omega_cell(), 0.5, MU,
                                            COUL[:nc], WEIGHT[:nc], SIGMA_FREQ[:ns], st["green"],
                                            st["w"])
    if kind in ("robust", "aaa"):
        model = _lib.PADE_ROBUST if kind == "robust" else _lib.AAA_APPROX
        scr = sigma_real.ScreenedCoulomb(st["w"].clone(), _mesh(case), model,
                                         sigma_real.NO_SYMMETRY, thres=1e-10)
        scr.eval_into(_eval_freq(case), st["grid"], st["grid"], st["gmap"], st["gmap"], st["out"])
        return {"coeff": scr.coeff, "w": st["out"]}
    n = case["n"]
    sigma.conv_device(st["g"], st["w"], st["weight"], st["s"], n, n, case["nout"], case["nin"],
                      -1.0 / (2.0 * math.pi))
    return st["s"]


# ---------------------------------------------------------------------------
# the same in plain torch
# ---------------------------------------------------------------------------
def _box(mill, n):
    m = np.asarray(mill, dtype=np.int64)
    return torch.from_numpy((m[:, 0] % n) + n * ((m[:, 1] % n) + n * (m[:, 2] % n))).to(_dev())


def _to_box(coef, at, n):
    """sum_G c(G) e^{iGr} of rows of coefficients, on (rows, n, n, n)."""
    b = torch.zeros((coef.shape[0], n ** 3), dtype=torch.complex128, device=_dev())
    b[:, at] = coef
    return torch.fft.ifftn(b.view(-1, n, n, n), dim=(1, 2, 3), norm="forward")


def _fft6_inv(block, at, at_p, n, n_p, volume):
    """f(r, r') = 1/V sum e^{-iGr} f(G, G') e^{iG'r'}; block[c][r], f[r'][r]."""
    rows = torch.zeros((block.shape[1], n_p ** 3), dtype=torch.complex128, device=_dev())
    rows[:, at_p] = block.T
    rows = torch.fft.ifftn(rows.view(-1, n_p, n_p, n_p), dim=(1, 2, 3), norm="forward")
    rows = rows.reshape(block.shape[1], -1)
    f = torch.zeros((n_p ** 3, n ** 3), dtype=torch.complex128, device=_dev())
    f[:, at] = rows.T
    return torch.fft.fftn(f.view(-1, n, n, n), dim=(1, 2, 3)).reshape(n_p ** 3, n ** 3) / volume


def _fft6_fwd(f, at, at_p, n, n_p, volume):
    b = torch.fft.ifftn(f.view(-1, n, n, n), dim=(1, 2, 3)).reshape(f.shape)[:, at]
    b = torch.fft.fftn(b.T.reshape(-1, n_p, n_p, n_p), dim=(1, 2, 3), norm="forward")
    return b.reshape(at.numel(), -1)[:, at_p].T * volume


def _thiele(w):
    """Coefficients of the continued fraction through W at SOLVER."""
    z = SOLVER.tolist()
    g, a = [x for x in w], [w[0]]
    for p in range(1, len(z)):
        g = g[:p] + [(g[p - 1] / g[i] - 1.0) / (z[i] - z[p - 1]) for i in range(p, len(z))]
        a.append(g[p])
    return a


def _thiele_at(a, x):
    z, v = SOLVER.tolist(), 0.0
    for p in range(len(z) - 1, 0, -1):
        v = a[p] * (x - z[p - 1]) / (1.0 + v)
    return a[0] / (1.0 + v)


def exact(case, seed):
    kind, dev = case["kind"], _dev()
    if kind in ("apply", "solve", "stream", "adjoint", "response", "green"):
        w = _workload(case, seed)
    if kind == "apply":
        x, group, sig = _vectors(w, case["nvec"], seed)
        x, out = torch.from_numpy(x).to(dev), torch.zeros(x.shape, dtype=torch.complex128, device=dev)
        sig = torch.from_numpy(sig).to(dev)
        for g in range(len(w.spheres)):
            at = torch.from_numpy(np.nonzero(group == g)[0]).to(dev)
            n = w.spheres[g].npw
            out[at, :n] = x[at, :n] @ _dense(w, g).T + sig[at, None] * x[at, :n]
        return out
    if kind in ("solve", "stream"):
        return {"x": _solutions(w, w.sigma), "ierr": None}
    if kind == "adjoint":
        c = -torch.from_numpy(w.rhs).to(dev)
        x, y = _solutions(w, w.sigma), _solutions(w, w.sigma.conj(), c)
        wt, n = _adjoint_weight(w), case["box"]
        grad = torch.zeros((n, n, n), dtype=torch.float64, device=dev)
        for s in range(w.nsys):
            sp = w.spheres[w.group[s]]
            at = _box(sp.mill, n)
            xr, yr = (_to_box(t[s, :, : sp.npw], at, n) for t in (x, y))
            grad -= (wt[s, :, None, None, None] * (yr.conj() * xr).real).sum(0) / n ** 3
        loss = float((wt * (c[:, None, :].conj() * x).sum(2).real).sum())
        return {"loss": loss, "y": y, "grad": grad, "ierr": None}
    if kind == "response":
        return _response(case, w)
    if kind == "green":
        sq = w.spheres[0]
        h = _dense(w, 0, with_valence=False)
        lam, u = torch.linalg.eigh(h)
        key = {tuple(m): i for i, m in enumerate(sq.mill.tolist())}
        row = [key.get(tuple(m), -1) for m in _shortest(case["num_g"]).tolist()]
        col = [key.get(tuple(m), -1) for m in _shortest(case["num_g_p"]).tolist()]
        row = [-1 if r + 1 >= sq.npw else r for r in row]     # the reference's row mask
        mask = torch.tensor([r >= 0 for r in row], device=dev)[None, :] \
            & torch.tensor([c >= 0 for c in col], device=dev)[:, None]
        at, at_p = _box(_shortest(case["num_g"]), case["n"]), _box(_shortest(case["num_g_p"]), case["n_p"])
        out = []
        for om in _green_omega(case).tolist():
            gf = -(u / (lam - om)[None, :]) @ u.conj().T
            out.append(_fft6_inv(torch.where(mask, gf[row][:, col].T, 0.0), at, at_p, case["n"],
                                 case["n_p"], _omega_cell()))
        return torch.stack(out)
    if kind == "sigma":
        a, gr = _thiele(_sigma_w(case, seed)), _green_r(case, seed)
        ng, ngp, n, n_p = case["num_g"], case["num_g_p"], case["n"], case["n_p"]
        at, at_p = _box(_shortest(ng), n), _box(_shortest(ngp), n_p)
        coul, vol = COUL[:case["ncoul"]], _omega_cell()
        out = torch.zeros((case["nsigma"], ngp, ng), dtype=torch.complex128, device=dev)
        for i, fs in enumerate((MU + SIGMA_FREQ[:case["nsigma"]]).tolist()):
            for j, fg in enumerate(np.concatenate([MU + coul, MU - coul]).tolist()):
                fc = complex(fs - fg)
                fc = fc.conjugate() if fc.real * fc.imag < 0 else fc
                f = _fft6_inv(_thiele_at(a, fc)[:ngp, :ng], at, at_p, n, n_p, vol)
                f *= gr[j]
                out[i] += 0.5 * WEIGHT[j % case["ncoul"]] * _fft6_fwd(f, at, at_p, n, n_p, vol)
        return out
    if kind in ("robust", "aaa"):
        ng, nr = case["num_g"], _corr_n(case["num_g"]) ** 3
        out = torch.zeros((nr, nr), dtype=torch.complex128, device=dev)
        out[:ng, :ng] = _w_at(_w_poles(case, seed), _eval_freq(case)).reshape(ng, ng)
        return {"coeff": None, "w": out}
    st = prepare(case, seed)
    out = torch.zeros_like(st["s"])
    for j in range(case["nin"]):       # column-major matrices: S^T = W^T G^T
        out += st["weight"][j] * (st["w"][j] @ st["g"][:, j])
    return out * (-1.0 / (2.0 * math.pi))


def _response(case, w):
    n, nf, nb, dev = case["box"], case["nfreq"], w.nbnd, _dev()
    _a, bg, vol = cell.fcc_lattice(ALAT)
    sq, freq = w.spheres[0], _freqs(nf)
    omegas = torch.from_numpy(np.concatenate([freq, -freq[1:]])).to(dev)
    at, gat = _box(sq.mill, n), _box(_shortest(case["num_g"]), n)
    psi = _to_box(torch.from_numpy(w.psi_k).to(dev), _box(w.sphere_k.mill, n), n)
    ev = torch.from_numpy(w.evq[0]).to(dev)
    lam, u = torch.linalg.eigh(_dense(w, 0))
    eps = torch.from_numpy(w.eps_v).to(dev)
    den = lam[None, None, :] - (eps[:, None, None] + omegas[None, :, None])
    m = np.arange(n)
    m = np.where(m <= n // 2, m, m - n)
    m3, m2, m1 = np.meshgrid(m, m, m, indexing="ij")
    g = np.stack([m1, m2, m3], -1) @ bg
    q = sq.kvec - w.sphere_k.kvec
    q2 = ((g + q) ** 2).sum(-1)
    kern = np.where(((g ** 2).sum(-1) <= 8.0 * case["ecut"]) & (q2 > 1e-16),
                    2.0 * 4.0 * np.pi / np.maximum(q2, 1e-300), 0.0)
    kern = torch.from_numpy(kern).to(dev)
    pert = _shortest(case["npert"], nonzero=True)
    out = torch.zeros((len(pert), nf, gat.numel()), dtype=torch.complex128, device=dev)
    for ip, pm in enumerate(pert):
        one = torch.ones((1, 1), dtype=torch.complex128, device=dev)
        dv = torch.fft.fftn(psi * _to_box(one, _box(pm[None, :], n), n), dim=(1, 2, 3),
                            norm="forward").reshape(nb, -1)[:, at]
        rhs = -(dv - (dv @ ev.conj().T) @ ev)
        x = ((rhs @ u.conj())[:, None, :] / den) @ u.T
        dpsi = torch.cat([x[:, :1], 0.5 * (x[:, 1:nf] + x[:, nf:])], 1)
        for f in range(nf):
            drho = -(4.0 / vol) * (psi.conj() * _to_box(dpsi[:, f], at, n)).sum(0)
            dvh = torch.fft.fftn(drho, norm="forward") * kern
            out[ip, f] = dvh.reshape(-1)[gat]
        hit = np.all(_shortest(case["num_g"]) == pm[None, :], axis=1)
        out[ip, :, torch.from_numpy(hit).to(dev)] += 1.0
    return out.cpu().numpy()


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _fft(n):
    return 5.0 * n * math.log2(n)


def _apply_work(case):
    """Bytes and flops of one vector, and the bytes all vectors share."""
    _a, b, _v = cell.fcc_lattice(ALAT)
    s = cell.make_sphere(b, np.zeros(3), case["ecut"])
    n, npw = case["box"], s.npw
    ncol = len({(m[0], m[1]) for m in s.mill.tolist()})
    row = 2 * int(np.abs(s.mill[:, 0]).max()) + 1
    nproj = 2 * (case["lmax"] + 1) ** 2 + case["nbnd"]
    flops = 2.0 * (ncol + n * row + n * n) * _fft(n) + 2.0 * n ** 3 + 16.0 * nproj * npw + 10.0 * npw
    shared = 8.0 * n ** 3 + case.get("nq", 1) * npw * (16.0 * nproj + 20.0)
    return npw, 32.0 * npw, flops, shared


SOLVE_ITER = 10   # BiCGStab(4) iterations of a typical system at the threshold


def work(case):
    kind = case["kind"]
    if kind == "apply":
        _npw, per, flops, shared = _apply_work(case)
        return {"bytes": case["nvec"] * per + shared, "flops": case["nvec"] * flops}
    if kind in ("solve", "stream", "adjoint", "response", "green"):
        npw, _per, flops, shared = _apply_work(case)
        nq, nsh = case.get("nq", 1), case.get("nshift", 1)
        nsys = case["nbnd"] * nq * case.get("npert", 1)
        if kind == "response":
            nsh = 2 * case["nfreq"] - 1
        if kind == "green":
            nsys, nsh = case["num_g_p"], case["nfreq"]
        # 8 products, 2 x 26 axpy's of the seed and 2 x 14 of every shift an iteration
        f = nsys * SOLVE_ITER * (8.0 * flops + 8.0 * npw * (52 + 28 * nsh))
        by = shared + 16.0 * nsys * npw * (1 + nsh)
        if kind == "adjoint":
            by += 16.0 * nsys * npw * nsh
            f += nsys * nsh * flops
        if kind == "response":
            by = shared + 16.0 * case["npert"] * case["nfreq"] * case["num_g"] \
                + 16.0 * case["nbnd"] * case["box"] ** 3
            f += nsys * case["nfreq"] * (0.5 * flops + 8.0 * case["box"] ** 3)
        if kind == "green":
            nr, nr_p = case["n"] ** 3, case["n_p"] ** 3
            by = shared + 16.0 * nsh * nr * nr_p
            f += nsh * 3.0 * (nr_p * case["n"] ** 2 * _fft(case["n"])
                              + case["num_g"] * case["n_p"] ** 2 * _fft(case["n_p"]))
        return {"bytes": by, "flops": f}
    if kind == "sigma":
        n, n_p, ng, ngp = (case[k] for k in ("n", "n_p", "num_g", "num_g_p"))
        prods = 2 * case["ncoul"] * case["nsigma"]
        nr, nr_p = n ** 3, n_p ** 3
        by = prods * 16.0 * (nr * nr_p + 4.0 * ng * ngp) + 16.0 * case["nsigma"] * ng * ngp
        f = prods * (2 * 3.0 * (nr_p * n * n * _fft(n) + ng * n_p * n_p * _fft(n_p))
                     + 6.0 * nr * nr_p)
        return {"bytes": by, "flops": f}
    if kind in ("robust", "aaa"):
        ne, n = case["num_g"] ** 2, case["nfreq"]
        nr = _corr_n(case["num_g"]) ** 3
        m = n // 2 - 2 if kind == "robust" else 7
        # one factorisation of an (m + 1) x m matrix per element, a sample sum
        return {"bytes": 16.0 * (2 * n * ne + nr * nr), "flops": ne * 8.0 * (n * n + 2.0 * m ** 3)}
    n, nout, nin = case["n"], case["nout"], case["nin"]
    return {"bytes": 16.0 * n * n * (nout * nin + nin + nout), "flops": 8.0 * n ** 3 * nout * nin}
