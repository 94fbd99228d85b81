"""The work that programs have this library do, as cases that can be timed
and compared: whole evaluations of a system (density, potential, energy, H psi,
forces, stress), SCF iterations, the class-level FourierTransform calls and
SlaterDet::gram, at Gamma, with two spins and over k-points, in every precision.

A case is a dict of plain values:
  op      evaluate    ef.evaluate (one BOSampleStepper evaluation)
          graph       the same, captured once and replayed
          scf         density, charge mixing, potential, H psi, PSDA step
          transforms  compute_density and rs_mul_add on a grid of the caller's maps
          gram        SlaterDet::gram of bands that are not yet orthonormal
  na, nb  atoms of the two species;  proj "sp" or "spd" projectors on the first
  a0 a1 a2, ecut (Ry), bands (per spin set and k-point: all bands), nspin, nkp
  prec    fp64, fp32, bf16x3, bf16x2;  stress: the stress tensor too

Bands are torch tensors, handed to the library by their address.  exact()
evaluates the same model in plain 64-bit torch with analytic Fourier transforms of the
species' Gaussians (the library splines tabulated ones, as Qbox does, which
agrees to about 1e-7), energies as explicit sums, forces and stress by
autograd.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "qbox-public_amd"))
import qbg  # noqa: E402
from qbg import configs as cf  # noqa: E402

PI = math.pi
TERMS = ("ekin", "eps", "enl", "ehart", "exc", "esr", "eself", "etotal", "total_charge")


def _case(name, op, na, nb, cell, ecut, bands, prec, proj="sp", nspin=1, nkp=1, stress=False):
    return dict(name=name, op=op, na=na, nb=nb, proj=proj, a0=float(cell[0]), a1=float(cell[1]),
                a2=float(cell[2]), ecut=float(ecut), bands=bands, nspin=nspin, nkp=nkp, prec=prec,
                stress=stress)


def listed():
    c16, c24, c36 = (16.0,) * 3, (24.0,) * 3, (36.0,) * 3
    return [
        # a molecule-sized system, one evaluation per geometry: latency and launches
        _case("small-fp64", "evaluate", 8, 0, c16, 30, 16, "fp64"),
        # the same inside a captured loop, as serving many small systems does
        _case("small-graph", "graph", 8, 0, c16, 30, 16, "bf16x2"),
        # a small magnetic cell of unequal edges, an odd number of bands
        _case("spin-fp32", "evaluate", 9, 7, (15.0, 17.5, 21.0), 45, 47, "fp32", nspin=2),
        # the ordinary size of a condensed-phase run
        _case("medium-bf16x2", "evaluate", 64, 0, c24, 60, 128, "bf16x2"),
        # an ordinary slab-like cell with d projectors, in full precision
        _case("slab-fp64", "evaluate", 38, 23, (19.0, 22.0, 34.0), 50, 131, "fp64", proj="spd"),
        # the large workload of the benchmark, mixed and FP64
        _case("large-bf16x2", "evaluate", 128, 128, c36, 70, 512, "bf16x2"),
        _case("large-fp64", "evaluate", 128, 128, c36, 70, 512, "fp64"),
        # variable-cell steps: forces and the stress tensor
        _case("stress-bf16x3", "evaluate", 64, 64, (28.0, 30.0, 32.0), 60, 256, "bf16x3",
              stress=True),
        # Brillouin-zone sampling of a small cell: the complex basis, three k-points
        _case("kpoints-bf16x2", "evaluate", 16, 16, (15.0, 15.5, 16.0), 55, 64, "bf16x2", nkp=3),
        # one iteration of the self-consistent loop, small in FP64, large mixed
        _case("scf-fp64", "scf", 30, 10, (20.0, 20.0, 20.0), 45, 90, "fp64"),
        _case("scf-large-bf16x2", "scf", 128, 128, c36, 70, 512, "bf16x2"),
        # the class-level calls of a host program that keeps its own functional
        _case("transforms-fp32", "transforms", 8, 0, (21.0, 23.0, 26.0), 52, 75, "fp32"),
    ]


def draw(rng):
    op = rng.choice(["evaluate"] * 5 + ["graph", "scf", "scf", "transforms", "gram"])
    nat = int(round(math.exp(rng.uniform(math.log(2), math.log(160)))))
    na = max(1, int(round(nat * rng.uniform(0.3, 1.0))))
    nb = max(0, nat - na)
    nkp = rng.choice([1, 1, 1, 2, 4]) if op == "evaluate" and nat <= 48 else 1
    # bohr^3 per atom from a dense solid to a dilute liquid; unequal edges
    vol = (na + nb) * math.exp(rng.uniform(math.log(130), math.log(500))) + 300.0
    r = [math.exp(rng.uniform(-0.2, 0.2)) for _ in range(3)]
    s = (vol / (r[0] * r[1] * r[2])) ** (1.0 / 3.0)
    ecut = rng.uniform(25, 85)
    bands = max(2, int(round((na + nb) * rng.uniform(1.6, 2.6))))
    # no dearer than the largest listed case
    while bands * nkp * vol * ecut ** 1.5 > 0.25 * 512 * 36.0 ** 3 * 70.0 ** 1.5:
        ecut *= 0.9
    nspin = 2 if op in ("evaluate", "graph") and nkp == 1 and rng.random() < 0.25 else 1
    prec = rng.choice(["fp64", "fp64", "fp32", "bf16x3", "bf16x2", "bf16x2"])
    if op == "transforms":
        prec = rng.choice(["fp64", "fp32"])
    if op == "gram":
        prec = "fp64"
    c = _case("", op, na, nb, [round(s * x, 2) for x in r], round(ecut, 1), bands, prec,
              proj=rng.choice(["sp", "sp", "spd"]), nspin=nspin, nkp=nkp,
              stress=op == "evaluate" and rng.random() < 0.25)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
def _system(case, seed):
    """The SystemDef: atoms on randomly chosen sites of a lattice, displaced."""
    rng = np.random.default_rng([seed, 1])
    cell = np.diag([case["a0"], case["a1"], case["a2"]])
    L = np.diag(cell)
    nat = case["na"] + case["nb"]
    h = (L.prod() / nat) ** (1.0 / 3.0)
    n = np.maximum(1, np.ceil(L / h).astype(int))
    sites = np.stack(np.meshgrid(*[np.arange(m) for m in n], indexing="ij"), -1).reshape(-1, 3)
    f = rng.permutation(sites)[:nat] + rng.uniform(-0.12, 0.12, (nat, 3))
    first = cf.SPECIES_D if case["proj"] == "spd" else cf.SPECIES_A
    species, na = [first], [case["na"]]
    if case["nb"]:
        species.append(cf.SPECIES_B)
        na.append(case["nb"])
    nst, two = case["bands"], case["nspin"] == 2
    occ = np.full(nst, 1.0 if two else 2.0)
    return cf.SystemDef("perf", cell, case["ecut"], species, na, nst, seed, 0.0, tau=f / n * L,
                        nspin=case["nspin"], nst_up=(nst + 1) // 2 if two else 0, occ_bands=occ)


def _kpoints(case):
    """A list of k-points and weights, or (None, None) at Gamma."""
    if case["nkp"] == 1:
        return None, None
    k = [[0.0, 0.0, 0.0], [0.5, 0.0, 0.0], [0.25, 0.25, 0.0], [0.25, -0.25, 0.5]][:case["nkp"]]
    w = np.array([1.0, 2.0, 3.0, 2.0][:case["nkp"]])
    return np.array(k), w / w.sum()


def _bands(g2, nst, gamma, gen, orthonormal=True):
    """Smooth random bands (nst x ngw), orthonormal where a program has them so."""
    c = torch.randn(nst, g2.numel(), dtype=torch.complex128, device="cuda", generator=gen)
    c /= 1.0 + g2
    if gamma:
        c[:, 0] = c[:, 0].real.to(c.dtype)
    if not orthonormal:
        return c
    if gamma:
        p = torch.view_as_real(c).reshape(nst, -1)
        s = 2.0 * (p @ p.t()) - torch.outer(p[:, 0], p[:, 0])
        p = torch.linalg.inv(torch.linalg.cholesky(s)) @ p
        return torch.view_as_complex(p.reshape(nst, -1, 2).contiguous())
    return torch.linalg.inv(torch.linalg.cholesky(c @ c.conj().t())) @ c


class Buffer:
    """A tensor as the library's device array."""

    def __init__(self, t):
        self.t = t
        self.p = ctypes.c_void_p(t.data_ptr())


class State:
    def __del__(self):
        for k in ("graph", "grid", "stepper", "mixer", "ef"):
            if hasattr(self, k):
                getattr(self, k).release()


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = qbg.Context(0)
    return _ctx


def prepare(case, seed):
    st = State()
    st.case, st.ctx = case, _context()
    sd = st.sysdef = _system(case, seed)
    kp, wt = _kpoints(case)
    st.ef = qbg.EnergyFunctional(st.ctx, sd, kpoints=kp, weights=wt)
    gen = torch.Generator("cuda").manual_seed(seed)
    op, nst = case["op"], case["bands"]
    c = torch.zeros(case["nkp"] * nst, st.ef.ngw, dtype=torch.complex128, device="cuda")
    for ik in range(case["nkp"]):
        g2 = torch.from_numpy(st.ef.kset_basis(ik)["kpg2"]).cuda()
        rows = slice(ik * nst, (ik + 1) * nst)
        sets = [(0, nst)]
        if case["nspin"] == 2:
            sets = [(0, sd.nst_up), (sd.nst_up, nst)]
        for b0, b1 in sets:
            c[rows][b0:b1, :g2.numel()] = _bands(g2, b1 - b0, kp is None, gen, op != "gram")
    st.c = Buffer(c)
    st.h = Buffer(torch.zeros_like(c)) if op != "gram" else None
    torch.cuda.synchronize()
    if op == "transforms":
        b = st.ef.basis(0)
        st.grid = qbg.Grid(st.ctx, st.ef.np0, st.ef.np1, st.ef.np2, b["ip"], b["im"],
                           b["zvec_to_val"])
        n = st.ef.N
        st.v = Buffer(torch.randn(n, dtype=torch.float64, device="cuda", generator=gen))
        st.rho = Buffer(torch.zeros(n, dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
    if op == "scf":
        st.stepper = qbg.WfStepper(st.ef, "psda")
        st.mixer = qbg.Mixer(st.ef)
        st.mixer.restart()
    if op == "graph":
        st.ef.evaluate(st.c, st.h, forces=True, prec=case["prec"])
        with qbg.Graph(st.ctx) as g:
            st.ef.evaluate_async(st.c, st.h, forces=True, prec=case["prec"])
        st.graph = g
    return st


def run(st):
    case, ef, op = st.case, st.ef, st.case["op"]
    prec = case["prec"]
    if op == "gram":
        qbg.gram(st.ctx, st.c, ef.ngw, ef.ngw, case["bands"])
        return {"c": st.c.t}
    if op == "transforms":
        for b in (st.rho, st.h):
            st.ctx.check(st.ctx.lib.qbg_memset(st.ctx.h, b.p, 0, b.t.nbytes))
        omega = case["a0"] * case["a1"] * case["a2"]
        st.grid.compute_density(st.c, ef.ngw, case["bands"], st.sysdef.occ, 1.0, omega, st.rho,
                                prec)
        st.grid.rs_mul_add(st.v, st.c, ef.ngw, case["bands"], st.h, ef.ngw, prec)
        return {"rho": st.rho.t, "h": st.h.t}
    if op == "scf":
        ef.update_density(st.c, prec)
        st.mixer.update()
        ef.update_vhxc(False)
        st.stepper.preprocess()
        ef.energy_async(st.c, st.h, prec=prec, same_c=True)
        st.stepper.update(st.c, st.h)
        r = ef.results()
        s = st.stepper.results()
        return {"energies": np.array([r[t] for t in TERMS]), "eig": s["eigenvalue_sum"],
                "c": st.c.t, "direction": st.h.t}
    if op == "graph":
        st.graph.launch()
        r = ef.results()
    else:
        r = ef.evaluate(st.c, st.h, forces=True, stress=case["stress"], prec=prec)
    out = {"energies": np.array([r[t] for t in TERMS]), "fion": r["fion"], "h": st.h.t}
    if case["stress"]:
        out["sigma"] = r["sigma"]
    return out


# ------------------------------------------------------- what a pass cannot do without
def _sizes(case):
    """Basis size, grid, columns, active rows and projectors, from the volume."""
    L = [case["a0"], case["a1"], case["a2"]]
    omega = L[0] * L[1] * L[2]
    kf = math.sqrt(case["ecut"])                      # |G| of the cutoff (Ry -> sqrt(2 Ha))
    half = 1.0 if case["nkp"] > 1 else 0.5
    ngw = half * omega * kf ** 3 / (6.0 * PI ** 2)
    n = [2.0 * kf * x / PI + 2 for x in L]            # density grid: twice the sphere's width
    cols = L[0] * L[1] * kf ** 2 / (4.0 * PI)
    rows = n[1] / 2.0
    npr = 9 if case["proj"] == "spd" else 4
    return ngw, n, cols, rows, case["na"] * npr + case["nb"] * 4


def work(case):
    ngw, n, cols, rows, m = _sizes(case)
    nb, nk, op = case["bands"], case["nkp"], case["op"]
    N = n[0] * n[1] * n[2]
    c = 16.0 * ngw * nb * nk
    if op == "gram":
        return {"bytes": 2 * c, "flops": 2.0 * nb * nb * 2 * ngw}
    # one transform between coefficients and the real-space grid; two bands share one at Gamma
    def line(x):
        return 5.0 * x * math.log2(x)
    fft = (cols * line(n[2]) + rows * n[2] * line(n[0]) + n[0] * n[2] * line(n[1])) \
        * (nb * nk if nk > 1 else nb / 2.0)
    if op == "transforms":
        return {"bytes": 2 * c + 16.0 * N, "flops": 2 * fft}
    # projections and their part of H psi; one product more for forces or stress
    gemm = (8.0 if nk > 1 else 4.0) * m * ngw * nb * nk
    if op == "scf":
        # overlaps with H c and with the previous bands, the new overlap, two updates of c
        return {"bytes": 3 * c, "flops": 2 * fft + 2 * gemm + 9.0 * 2 * ngw * nb * nb}
    return {"bytes": 2 * c, "flops": 2 * fft + (4 if case["stress"] else 3) * gemm}


def tolerance(case):
    """About four times what two ways of rounding show (each against exact():
    1e-13 in FP64, 2e-7 with FP32 transforms and FP32 or split products)."""
    if case["op"] == "gram":
        return {"rel": 1e-12, "max": 1e-9}
    if case["op"] == "scf":       # the rounding of H c goes through the step and the mixing
        return {"rel": 1e-9, "max": 1e-6} if case["prec"] == "fp64" else {"rel": 2e-5, "max": 1e-2}
    if case["prec"] == "fp64":
        return {"rel": 2e-12, "max": 1e-9}
    return {"rel": 1.5e-6, "max": 2e-4}


# ------------------------------------------------------------------ 64-bit reference
def _radial(l, s, g2):
    """Transform of r^l exp(-r^2 / 2 sigma^2), without the factor |G|^l."""
    return (2.0 * PI) ** 1.5 * s.sigma ** (2 * l + 3) * torch.exp(-0.5 * g2 * s.sigma ** 2)


def _projectors(s, g):
    """(npr x ng) solid harmonics times radial part, phase (-i)^l apart, l and D of each."""
    x, y, z = g[:, 0], g[:, 1], g[:, 2]
    g2 = (g * g).sum(1)
    rows, ls = [math.sqrt(1 / (4 * PI)) * _radial(0, s, g2)], [0]
    f = math.sqrt(3 / (4 * PI)) * _radial(1, s, g2)
    rows += [f * x, f * y, f * z]
    ls += [1] * 3
    if s.lmax >= 2:
        f = math.sqrt(5 / (4 * PI)) * _radial(2, s, g2)
        q = math.sqrt(3.0)
        rows += [f * 0.5 * (3 * z * z - g2), f * 0.5 * q * (x * x - y * y), f * q * x * y,
                 f * q * y * z, f * q * x * z]
        ls += [2] * 5
    return torch.stack(rows), ls, [s.d[l] for l in ls]


def _exc(ru, rd):
    """Exchange-correlation energy per volume: Perdew-Zunger, interpolated in the spin."""
    r = ru + rd
    ok = r > 0
    r1 = torch.where(ok, r, torch.ones_like(r))
    rs = 0.6203504908994001 / r1 ** (1.0 / 3.0)

    def fit(cx, A, B, b1, b2, G):
        D = G / (1 + b1 + b2) - B
        C = -A - D - G * ((b1 / 2 + b2) / (1 + b1 + b2) ** 2)
        lr, q = torch.log(rs), torch.sqrt(rs)
        return 0.75 * cx / rs + torch.where(rs < 1, A * lr + B + C * rs * lr + D * rs,
                                            G / (1 + b1 * q + b2 * rs))

    e = fit(-0.610887057711, 0.0311, -0.048, 1.0529, 0.3334, -0.1423)
    if ru is not rd:
        zeta = torch.where(ok, (ru - rd) / r1, torch.zeros_like(r))
        f = ((1 + zeta) ** (4 / 3) + (1 - zeta) ** (4 / 3) - 2) / (2 * 2 ** (1 / 3) - 2)
        e = e + f * (fit(-0.769669463118, 0.01555, -0.0269, 1.3981, 0.2611, -0.0843) - e)
    return torch.where(ok, r * e, torch.zeros_like(r))


class _Model:
    """The system's energy at fixed bands as plain sums over plane waves."""

    def __init__(self, st):
        case, sd, ef = st.case, st.sysdef, st.ef
        self.case, self.sd = case, sd
        dev = dict(dtype=torch.float64, device="cuda")
        self.L = torch.tensor([case["a0"], case["a1"], case["a2"]], **dev)
        self.np = (ef.np0, ef.np1, ef.np2)
        self.N = ef.N
        # the lists of basis vectors are part of the inputs: they say what each coefficient is
        self.idx = [torch.from_numpy(ef.kset_basis(k)["idx"].astype(np.int64)).cuda()
                    for k in range(case["nkp"])]
        self.idxv = torch.from_numpy(ef.basis(1)["idx"].astype(np.int64)).cuda()
        kp, w = _kpoints(case)
        self.gamma = kp is None
        self.k = torch.zeros(1, 3, **dev) if kp is None else torch.from_numpy(kp).cuda()
        self.w = [1.0] if w is None else [float(x) for x in w]
        self.nst = case["bands"]
        self.c = [st.c.t[k * self.nst:(k + 1) * self.nst, :len(self.idx[k])].clone()
                  for k in range(case["nkp"])]
        self.occ = torch.tensor(sd.occ, **dev)
        self.tau = torch.tensor(sd.tau, **dev)
        self.sets = [(0, self.nst)] if case["nspin"] == 1 else [(0, sd.nst_up),
                                                               (sd.nst_up, self.nst)]

    def g(self, idx, k=0.0, strain=None):
        g = (idx + k) * (2 * PI / self.L)
        return g if strain is None else g @ torch.linalg.inv(torch.eye(3).to(g) + strain)

    def _slot(self, idx):
        n = self.np
        return ((idx[:, 2] % n[2]) * n[1] + idx[:, 1] % n[1]) * n[0] + idx[:, 0] % n[0]

    def grid(self, c, idx):
        f = torch.zeros(self.N, dtype=torch.complex128, device="cuda")
        if self.gamma:
            f[self._slot(-idx)] = c.conj()
        f[self._slot(idx)] = c
        n = self.np
        return torch.fft.ifftn(f.view(n[2], n[1], n[0]), norm="forward").reshape(-1)

    def coefficients(self, f, idx):
        n = self.np
        return torch.fft.fftn(f.view(n[2], n[1], n[0]), norm="forward").reshape(-1)[
            self._slot(idx)]

    def density(self):
        omega = float(self.L.prod())
        rho = [torch.zeros(self.N, dtype=torch.float64, device="cuda") for _ in self.sets]
        for k, idx in enumerate(self.idx):
            for r, (b0, b1) in zip(rho, self.sets):
                for b in range(b0, b1):
                    psi = self.grid(self.c[k][b], idx)
                    r += (self.w[k] * self.occ[b] / omega) * (psi.real ** 2 + psi.imag ** 2)
        return rho

    def local(self, rho, grads=True):
        """Energies of the density terms, the potential(s) on the grid and the
        derivatives with respect to the positions and to a strain per term."""
        eye = torch.eye(3, dtype=torch.float64, device="cuda")
        omega0 = self.L.prod()
        rhog = self.coefficients((sum(rho) + 0j) * omega0, self.idxv)    # electrons
        eps = torch.zeros(3, 3, dtype=torch.float64, device="cuda", requires_grad=True)
        det = torch.linalg.det(eye + eps)
        g = self.g(self.idxv, strain=eps)
        g2 = (g * g).sum(1)
        g2i = torch.cat([torch.zeros_like(g2[:1]), 1 / g2[1:]])
        g0 = self.g(self.idxv)
        first = np.cumsum([0] + self.sd.na)
        s = []
        for a0, a1 in zip(first[:-1], first[1:]):
            t = torch.zeros(len(g0), dtype=torch.complex128, device="cuda")
            for a in range(a0, a1):
                t += torch.exp(-1j * (g0 @ self.tau[a]))
            s.append(t.requires_grad_(True))
        omega = omega0 * det
        vps = rps = 0
        for q, sf in zip(self.sd.species, s):
            # the local potential less that of the Gaussian pseudocharge
            v = -4 * PI * q.zval * (torch.exp(-g2 * q.rc ** 2 / 4)
                                    - torch.exp(-g2 * q.rcps ** 2 / 4)) * g2i
            v = torch.cat([v[:1] + PI * q.zval * (q.rc ** 2 - q.rcps ** 2), v[1:]])
            vps = vps + sf * (v / omega)
            rps = rps + sf * (-q.zval * torch.exp(-g2 * q.rcps ** 2 / 4) / omega)
        re = rhog / omega
        wt = torch.full_like(g2, 2.0)
        wt = torch.cat([wt[:1] - 1.0, wt[1:]])
        e = dict(eps=omega * (wt * (re.conj() * vps).real).sum(),
                 ehart=omega * 2 * PI * (wt * g2i * (re + rps).abs() ** 2).sum())
        up = (rho[0] if len(rho) == 2 else 0.5 * rho[0]).clone().requires_grad_(True)
        dn = rho[1].clone().requires_grad_(True) if len(rho) == 2 else up
        fx = omega0 / self.N * _exc(up, dn).sum()
        v = torch.autograd.grad(fx, [up] if dn is up else [up, dn])
        v = [x * self.N / omega0 * (0.5 if dn is up else 1.0) for x in v]
        vg = (vps + 4 * PI * g2i * (re + rps)).detach()
        f = torch.zeros(self.N, dtype=torch.complex128, device="cuda")
        f[self._slot(-self.idxv)] = vg.conj()
        f[self._slot(self.idxv)] = vg
        n = self.np
        vl = torch.fft.ifftn(f.view(n[2], n[1], n[0]), norm="forward").reshape(-1).real
        vr = [x + vl for x in v]
        u = up.detach() / det
        e["exc"] = omega / self.N * _exc(u, u if dn is up else dn.detach() / det).sum()
        e["esr"] = self.esr(eps)
        fion = strain = None
        if grads:
            strain = {t: torch.autograd.grad(x, eps, retain_graph=True)[0] for t, x in e.items()}
            gs = torch.autograd.grad(e["eps"] + e["ehart"], s)
            fion = torch.zeros_like(self.tau)
            for (a0, a1), gr in zip(zip(first[:-1], first[1:]), gs):
                for a in range(a0, a1):    # d exp(-i G tau) = -i G exp(-i G tau)
                    ph = torch.exp(-1j * (g0 @ self.tau[a]))
                    fion[a] = -((gr.conj() * (-1j) * ph).real[:, None] * g0).sum(0)
            tau = self.tau.clone().requires_grad_(True)
            fion = fion - torch.autograd.grad(self.esr(None, tau), tau)[0]
        return {k: float(x) for k, x in e.items()}, vr, fion, strain

    def esr(self, strain=None, tau=None):
        """Overlap correction of the Gaussian pseudocharges, all images in reach."""
        tau = self.tau if tau is None else tau
        z = torch.tensor(np.repeat([q.zval for q in self.sd.species], self.sd.na)).to(tau)
        rc = math.sqrt(2) * self.sd.species[0].rcps
        nat, tot = len(tau), 0.0
        m = [int(math.ceil(8 * rc / float(x) + 0.5)) for x in self.L]
        d0 = tau[:, None] - tau[None]
        with torch.no_grad():
            wrap = torch.round(d0 / self.L) * self.L
        pair = z[:, None] * z[None]
        eye = torch.eye(nat, device="cuda", dtype=torch.bool)
        for i in range(-m[0], m[0] + 1):
            for j in range(-m[1], m[1] + 1):
                for k in range(-m[2], m[2] + 1):
                    d = d0 - wrap + torch.tensor([i, j, k]).to(tau) * self.L
                    if strain is not None:
                        d = d + d @ strain.t()
                    skip = eye if i == j == k == 0 else torch.zeros_like(eye)
                    r = torch.sqrt((d * d).sum(-1) + skip)
                    t = pair * torch.special.erfc(r / rc) / r
                    tot = tot + 0.5 * torch.where(skip, torch.zeros_like(t), t).sum()
        return tot

    def bands_part(self, h=None, grads=True):
        """Kinetic and nonlocal energy, their derivatives; adds their H psi to h."""
        omega0 = self.L.prod()
        strain = {t: torch.zeros(3, 3, dtype=torch.float64, device="cuda")
                  for t in ("ekin", "enl")}
        fion = torch.zeros_like(self.tau)
        e = dict(ekin=0.0, enl=0.0)
        first = np.cumsum([0] + self.sd.na)
        for k, idx in enumerate(self.idx):
            c = self.c[k]
            eps = torch.zeros(3, 3, dtype=torch.float64, device="cuda", requires_grad=grads)
            g = self.g(idx, self.k[k], eps)
            g0 = self.g(idx, self.k[k])
            den = ((self.occ * self.w[k])[:, None] * (c.real ** 2 + c.imag ** 2)).sum(0)
            kin = ((1.0 if self.gamma else 0.5) * den * (g * g).sum(1)).sum()
            e["ekin"] += float(kin.detach())
            if grads:
                strain["ekin"] += torch.autograd.grad(kin, eps)[0]
            if h is not None:
                h[k] += 0.5 * (g0 * g0).sum(1) * c
            for q, a0, a1 in zip(self.sd.species, first[:-1], first[1:]):
                for b0 in range(a0, a1, 16):
                    tau = self.tau[b0:min(a1, b0 + 16)].clone().requires_grad_(grads)
                    eb = torch.zeros(3, 3, dtype=torch.float64, device="cuda",
                                     requires_grad=grads)
                    t, ls, d = _projectors(q, self.g(idx, self.k[k], eb))
                    ph = torch.exp(-1j * (tau @ g0.t()))
                    il = torch.tensor([(-1j) ** x for x in ls], device="cuda")
                    p = (ph[:, None, :] * (il[:, None] * t)[None]).reshape(-1, len(idx))
                    f = p.conj() @ c.t()                       # <beta|psi>
                    if self.gamma:
                        f = 2 * f.real - (p[:, :1].conj() * c[:, 0]).real
                    dm = torch.tensor(d).to(self.tau).repeat(len(tau))[:, None]
                    ob = (self.occ * self.w[k])[None]
                    enl = (dm * ob * f.abs() ** 2).sum() / (omega0 * torch.linalg.det(
                        torch.eye(3).to(eb) + eb))
                    e["enl"] += float(enl.detach())
                    if grads:
                        gt, ge = torch.autograd.grad(enl, [tau, eb])
                        fion[b0:b0 + len(tau)] -= gt
                        strain["enl"] += ge
                    if h is not None:
                        with torch.no_grad():
                            h[k] += ((dm / omega0) * f).t().to(p.dtype) @ p
        return e, fion, strain

    def add_local(self, vr, h):
        for k, idx in enumerate(self.idx):
            for v, (b0, b1) in zip(vr, self.sets):
                for b in range(b0, b1):
                    h[k][b] += self.coefficients(v * self.grid(self.c[k][b], idx), idx)


def _overlap(a, b):
    p, q = (torch.view_as_real(x.contiguous()).reshape(len(x), -1) for x in (a, b))
    return 2.0 * (p @ q.t()) - torch.outer(p[:, 0], q[:, 0])


def _mix(m, c):
    return m.to(c.dtype) @ c


def exact(case, seed):
    st = prepare(dict(case, op="evaluate") if case["op"] == "graph" else case, seed)
    m = _Model(st)
    if case["op"] == "gram":
        c = m.c[0]
        return {"c": _mix(torch.linalg.inv(torch.linalg.cholesky(_overlap(c, c))), c)}
    if case["op"] == "transforms":
        h = [torch.zeros_like(m.c[0])]
        m.add_local([st.v.t], h)
        return {"rho": m.density()[0], "h": h[0]}
    rho = m.density()
    charge = float(sum(rho).sum()) * float(m.L.prod()) / m.N
    grads = case["op"] != "scf"
    e, vr, f1, s1 = m.local(rho, grads)
    h = [torch.zeros_like(c) for c in m.c]
    eb, f2, s2 = m.bands_part(h, grads)
    m.add_local(vr, h)
    e.update(eb)
    e["eself"] = sum(n * q.zval ** 2 / (math.sqrt(2 * PI) * q.rcps)
                     for q, n in zip(m.sd.species, m.sd.na))
    e["etotal"] = sum(e[t] for t in ("ekin", "eps", "enl", "ehart", "exc", "esr")) - e["eself"]
    e["total_charge"] = charge
    energies = np.array([e[t] for t in TERMS])
    if case["op"] == "scf":
        # one PSDA step without extrapolation: residual, preconditioner, step,
        # then the orthonormal bands closest to the previous ones
        c, d = m.c[0], h[0]
        eig = float(_overlap(c, d).trace())
        d = d - _mix(_overlap(d, c), c)
        g2 = (m.g(m.idx[0]) ** 2).sum(1)
        n2 = c.real ** 2 + c.imag ** 2
        ekin = (n2 * g2).sum(1) / (2 * n2.sum(1) - n2[:, 0])
        d = -d * torch.where(0.5 * g2 < ekin[:, None], 0.5 / ekin[:, None],
                             0.5 / (0.5 * g2).clamp_min(1e-300))
        new = c + d
        new[:, 0] = new[:, 0].real.to(new.dtype)
        inv = torch.linalg.inv(torch.linalg.cholesky(_overlap(new, new)))
        new = _mix(inv, new)
        u, _, vh = torch.linalg.svd(_overlap(new, c))
        return {"energies": energies, "eig": eig, "c": _mix((u @ vh).t().contiguous(), new),
                "direction": d}
    hp = torch.zeros_like(st.h.t)
    for k, x in enumerate(h):
        hp[k * m.nst:(k + 1) * m.nst, :x.shape[1]] = x
    out = {"energies": energies, "fion": (f1 + f2).cpu().numpy(), "h": hp}
    if case["stress"]:
        s1.update(s2)
        rows = []
        for t in ("ekin", "eps", "enl", "ehart", "exc", "esr"):
            s = -s1[t] / m.L.prod()
            s = 0.5 * (s + s.t())
            rows.append([float(s[i, j]) for i, j in ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2),
                                                     (0, 2))])
        out["sigma"] = np.array([np.sum(rows, 0)] + rows)
    return out
