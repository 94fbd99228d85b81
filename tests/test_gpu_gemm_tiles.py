"""The dense products (csrc/gemm.hip) at the edges of their tiles: the overlap
(symmetric, split over the reduction), its factors and the update of the
coefficients through SlaterDet::gram at band counts around the 32-column steps
of the tiles, coefficient counts around the 16-deep chunks and a leading
dimension and base address that are only 8-byte aligned; and the projections
and the H psi and force products of the nonlocal part at ragged projector and
band counts, against the oracle.

Bounds: gram against numpy's Cholesky of the same bands to 1e-11 (sums of at most 3000
products of condition below 100 in FP64); the nonlocal part as the neighbouring energy
tests (1e-10 in FP64, 1e-6 Ha in FP32).
"""
import dataclasses

import numpy as np
import pytest

from qbg import configs as cf

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import qbg
    c = qbg.Context(0)
    yield c
    c.close()


# (no more bands than the basis spans)
@pytest.mark.parametrize("nst,ngw,shift",
                         [(n, g, s) for g, s in ((7, 0), (8, 1), (129, 0), (1500, 1))
                          for n in (1, 2, 31, 32, 33, 63, 65, 96, 97, 128, 129, 161, 257)
                          if n <= 2 * g - 1])
@pytest.mark.parametrize("which", ["gram", "gram_noalloc"])
def test_gram_ragged(ctx, nst, ngw, shift, which):
    import qbg
    print(f"[case] {which} nst {nst} ngw {ngw} shift {shift}", flush=True)
    rng = np.random.default_rng(nst * 10000 + ngw)
    ldc = ngw + 1
    c = rng.standard_normal((nst, ldc)) + 1j * rng.standard_normal((nst, ldc))
    # orthonormal bands and a perturbation keep the overlap well conditioned
    q, _ = np.linalg.qr(rng.standard_normal((2 * ngw - 1, nst)))
    p = np.zeros((nst, 2 * ngw))
    p[:, 0], p[:, 2:] = q[0], q[1:].T / np.sqrt(2.0)
    p[:, 2:] += 0.05 / np.sqrt(ngw) * rng.standard_normal((nst, 2 * ngw - 2))
    c[:, :ngw] = np.ascontiguousarray(p).view(np.complex128)
    ref = cf.gram_numpy(np.ascontiguousarray(c[:, :ngw]))
    # one double into the allocation: the coefficients are then 8-byte aligned
    buf = np.zeros(2 * c.size + 1)
    buf[shift:shift + 2 * c.size] = c.view(np.float64).ravel()
    d = ctx.to_device(buf)

    class View:
        p = d.offset(8 * shift)

    getattr(qbg, which)(ctx, View, ldc, ngw, nst)
    got = d.download()[shift:shift + 2 * c.size].copy().view(np.complex128).reshape(nst, ldc)
    assert np.abs(got[:, :ngw] - ref).max() < 1e-11
    assert np.array_equal(got[:, ngw:], c[:, ngw:])     # padding untouched


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("na,nst", [((1, 0), 1), ((3, 5), 33), ((8, 1), 47), ((9, 16), 97)])
def test_nonlocal_products_ragged(ctx, oracle_mod, prec, na, nst):
    import qbg
    sp = [cf.SPECIES_D] + ([cf.SPECIES_B] if na[1] else [])
    s = cf.SystemDef(f"ragged {na} {nst}", np.diag([11.0, 12.0, 13.5]), 14.0, sp,
                     [n for n in na if n], nst, 77 + nst, 1.6).build_positions()
    print(f"[case] {s.name} {prec}", flush=True)
    o = oracle_mod.Oracle(s)
    c = cf.gram_numpy(cf.random_coefficients(5 + nst, o.basis(0)["g2"], nst))
    ref = o.evaluate(c, hpsi=True, forces=True)
    ef = qbg.EnergyFunctional(ctx, s)
    hp = ctx.array(c.shape, np.complex128)
    r = ef.evaluate(ctx.to_device(c), hp, forces=True, prec=prec)
    h = hp.download()
    tol, ftol, htol = (1e-10, 1e-10, 1e-10) if prec == "fp64" else (1e-6 * s.nat, 1e-5, 1e-5)
    assert abs(r["enl"] - ref["enl"]) < tol * max(1.0, abs(ref["enl"]) if prec == "fp64" else 1.0)
    fref = np.asarray(ref["fion"]).reshape(-1, 3)
    fs = np.abs(fref).max() if prec == "fp64" else 1.0
    assert np.abs(r["fion"] - fref).max() < ftol * fs
    assert np.abs(h - ref["hpsi"]).max() < htol * np.abs(ref["hpsi"]).max()
    ef.release()


def test_fp32_chain_length(ctx):
    """The nonlocal H psi of FP32 products at a long reduction (K = 108672), whose
    error is that of its chains of FP32 sums.  Adding term k rounds a partial sum of
    variance k; the mean square of that, relative to the sum, is 2^-46 / 12 times the
    mean of 1 / m^2 over the leading digits m (0.54), so a chain of n terms is off by
    sqrt(0.045 / 2) 2^-23 sqrt(n) = 0.15 2^-23 sqrt(n), and a sum of independent
    chains of that length by the same.  The projections may use chains of K / 32 terms
    (the splits are added in FP64), the product with the projectors has M: 10 % above
    both is 1.26e-6, and 1.08e-6 is measured; projections in chains of twice that
    length take it to 1.43e-6."""
    import qbg
    nst = 300
    s = cf.SystemDef("long reduction", np.diag([24.0, 24.0, 24.0]), 60.0, [cf.SPECIES_A], [175],
                     nst, 77, 1.6).build_positions()
    print(f"[case] {s.name}", flush=True)
    ef = qbg.EnergyFunctional(ctx, s)
    nl = qbg.NonLocalPotential(ef)
    rng = np.random.default_rng(3)
    c = rng.standard_normal((nst, ef.ngw)) + 1j * rng.standard_normal((nst, ef.ngw))
    c[:, 0] = c[:, 0].real
    dc, h = ctx.to_device(c), {}
    for prec in ("fp64", "fp32"):
        dh = ctx.to_device(np.zeros_like(c))
        nl.energy(dc, dh, prec=prec)
        h[prec] = dh.download()
        dh.release()
    err = np.linalg.norm(h["fp32"] - h["fp64"]) / np.linalg.norm(h["fp64"])
    assert err < 1.1 * 0.15 * 2.0 ** -23 * np.sqrt(2 * ef.ngw / 32 + 4 * s.nat), err
    dc.release()
    nl.release()
    ef.release()
