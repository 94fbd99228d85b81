"""Parity of the pass kernels of every further line length that a grid can
have (csrc/fft4_g.hip ... fft4_o.hip) on every axis, with an odd band count
and a last plane block that is not full, against numpy's FFT on the full grid:
single transforms, SlaterDet::compute_density and rs_mul_add
(src/SlaterDet.cpp:225-298, 410-477).  FP64 to 1e-12 relative, FP32 to 2e-5,
the bounds of the neighbouring length test.
"""
import math

import numpy as np
import pytest

from qbg import configs as cf

TOL = {"fp64": 1e-12, "fp32": 2e-5}

LENGTHS = (16, 18, 20, 30, 32, 36, 40, 42, 44, 48, 56, 60, 66, 70, 72, 80, 84, 88, 110, 120, 132,
           140, 154, 176, 180, 192, 220, 240, 252, 256, 264, 280, 288, 308, 320, 330, 336, 352,
           360, 384, 396)


def grid_system(k, nst=3):
    """Grid k puts a short, a middle and a long length on the three axes, and
    over all k each length on each axis; the sphere fills its natural share."""
    n = len(LENGTHS)
    pick = [LENGTHS[k], LENGTHS[(k + 14) % n], LENGTHS[(k + 27) % n]]
    h, x = 0.3, 0.45
    ecut_ha = (2.0 * math.pi * x / h) ** 2 / 8.0
    s = cf.SystemDef(f"grid {pick}", np.diag([h * m for m in pick]), 2.0 * ecut_ha,
                     [cf.SPECIES_A], [1], nst, 700 + k, 0.0, tau=np.zeros((1, 3)))
    return s, tuple(pick)


def test_compiled_lengths():
    """Every even length to 396 that Basis::factorizable admits is compiled."""
    import qbg
    for n in range(16, 398, 2):
        m = n
        for f in (11, 7, 5, 3, 3):
            if m % f == 0:
                m //= f
        while m % 2 == 0:
            m //= 2
        assert (len(qbg.fft_splits(n)) > 0) == (m == 1), n


@pytest.mark.gpu
@pytest.mark.parametrize("k", range(len(LENGTHS)))
def test_grid_lengths(oracle_mod, k):
    import qbg
    s, grid = grid_system(k)
    o = oracle_mod.Oracle(s, grid=grid)
    print(f"[case] {s.name} ngw {o.ngw}", flush=True)
    b = o.basis(0)
    ctx = qbg.Context(0)
    g = qbg.Grid(ctx, *grid, b["ip"], b["im"], b["zvec_to_val"])
    assert g.four_step
    idx = np.asarray(b["idx"]).reshape(-1, 3) % np.array(grid)
    neg = -np.asarray(b["idx"]).reshape(-1, 3) % np.array(grid)
    at, an = tuple(idx[:, ::-1].T), tuple(neg[:, ::-1].T)

    def synth(c):
        f = np.zeros(grid[::-1], dtype=np.complex128)
        f[an] = c.conj()
        f[at] = c
        return np.fft.ifftn(f, norm="forward")

    rng = np.random.default_rng(k)
    c = cf.random_coefficients(800 + k, np.asarray(b["g2"]), s.nst)
    psi = [synth(x) for x in c]
    occ = np.linspace(2.0, 0.5, s.nst)
    omega = abs(np.linalg.det(s.cell))
    rho = sum(f / omega * p.real ** 2 for f, p in zip(occ, psi)).ravel()
    v = rng.standard_normal(o.N)
    h = np.stack([np.fft.fftn(v.reshape(p.shape) * p.real, norm="forward")[at] for p in psi])
    x = rng.standard_normal(o.N) + 1j * rng.standard_normal(o.N)
    xf = np.fft.fftn(x.reshape(grid[::-1]), norm="forward")[at]
    dc, dv = ctx.to_device(c), ctx.to_device(v)
    for prec, tol in TOL.items():
        print(f"[case] {s.name} {prec}", flush=True)

        def close(a, r, what):
            assert np.abs(a - r).max() < tol * np.abs(r).max(), (prec, what)

        f = ctx.array(o.N, np.complex128)
        g.fft_backward(dc, f, prec)
        close(f.download(), psi[0].ravel(), "backward")
        out = ctx.array(o.ngw, np.complex128)
        g.fft_forward(ctx.to_device(x), out, prec)
        close(out.download(), xf, "forward")
        dr = ctx.array(o.N).zero()
        g.compute_density(dc, o.ngw, s.nst, occ, 1.0, omega, dr, prec)
        close(dr.download(), rho, "density")
        hp = ctx.to_device(np.zeros_like(c))
        g.rs_mul_add(dv, dc, o.ngw, s.nst, hp, o.ngw, prec)
        close(hp.download(), h, "rs_mul_add")
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("edge,ecut,grid,bound", [(43.2, 22.2, 140, 8.0e-8),
                                                  (67.2, 22.2, 220, 8.0e-8),
                                                  (48.0, 22.2, 160, 9.0e-8)])
def test_fp32_density_rounding(edge, ecut, grid, bound):
    """The density of smooth bands in FP32 on lines with factors 5, 7 and 11.  Sums
    over bands average the rounding of single operations, not that of the DFT
    constants, which acts on every line and band alike, so this shows it: with every sine
    and cosine rounded once 7.6e-8 (140^3) and 7.1e-8 (220^3) in the 2-norm, with
    products of rounded constants 8.8e-8 and 8.5e-8; 160^3 as 16 x 10 8.5e-8, as
    10 x 16 9.7e-8.  The bounds lie between."""
    import qbg
    s = cf.SystemDef(f"cube {grid}", np.diag([edge] * 3), ecut, [cf.SPECIES_A], [1], 24, 1, 0.0,
                     tau=np.zeros((1, 3)))
    print(f"[case] {s.name}", flush=True)
    ctx = qbg.Context(0)
    ef = qbg.EnergyFunctional(ctx, s)
    assert (ef.np0, ef.np1, ef.np2) == (grid,) * 3
    c = cf.gram_numpy(cf.random_coefficients(5, ef.basis(0)["g2"], s.nst))
    dc, rho = ctx.to_device(c), {}
    for prec in ("fp64", "fp32"):
        ef.update_density(dc, prec)
        rho[prec] = ef.get(0)
    err = np.linalg.norm(rho["fp32"] - rho["fp64"]) / np.linalg.norm(rho["fp64"])
    assert err < bound, err
    ctx.close()


def test_splits_of_saved_plans():
    """qbg_grid_plan takes every split that a plan kept by a caller may name."""
    import qbg
    for n, n1 in ((90, (10, 18)), (96, (12, 16)), (112, (16, 14)), (126, (14, 18)),
                  (128, (16, 32)), (144, (16, 12)), (160, (16, 20)), (168, (21, 14)),
                  (198, (18, 22)), (210, (15, 14)), (224, (16, 32))):
        assert set(n1) <= set(qbg.fft_splits(n)), n


def test_default_splits_by_error():
    """Lengths whose default is the split with the smaller FP32 error (fft4_reg.cpp)
    where the times differ by 4 % at most."""
    import qbg
    for n, n1 in ((96, 12), (128, 16), (160, 16), (168, 14)):
        assert qbg.fft_splits(n)[0] == n1, n
