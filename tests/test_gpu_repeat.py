"""A functional used again: what an evaluation writes first (the density of its
first batch, the nonlocal forces, the sums of two passes in one launch) must not
hold anything of the evaluation before it.  Each evaluation of a used
functional equals, bit by bit, the same evaluation of a fresh one: after other
bands, after one without forces, on a grid of the generic transforms (a line longer
than the compiled lengths) and of the compiled ones, with more bands than one
batch of the density, with k-points, and with a spin that lost its bands.
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


def _long_cell():
    return cf.SystemDef("long line", np.diag([140.0, 6.0, 6.5]), 26.0, [cf.SPECIES_A], [2], 3, 900,
                        0.0, tau=np.array([[0.3, 0.1, 0.2], [40.0, 2.0, 3.0]]))


@pytest.mark.parametrize("what", ["compiled", "generic", "batches", "kset", "spin"])
@pytest.mark.parametrize("prec", ["fp64", "bf16x2"])
def test_used_equals_fresh(ctx, what, prec):
    import qbg
    print(f"[case] repeat {what} {prec}", flush=True)
    kw, s = {}, cf.config(11)
    if what == "generic":
        s = _long_cell()
    elif what == "batches":
        s = dataclasses.replace(cf.config(0), nst=150)
    elif what == "kset":
        kw = dict(kpoints=[[0.25, 0.1, -0.2], [-0.25, 0.35, 0.1]], weights=[0.25, 0.75])
    elif what == "spin":
        s = cf.spin_polarized(s, 12, 1, 1)

    def functional():
        ef = qbg.EnergyFunctional(ctx, s, **kw)
        if what == "generic":
            assert ef.np0 > 396
        return ef

    used, fresh = functional(), functional()
    rng = np.random.default_rng(8)

    def bands():
        n = used.kngw if what == "kset" else [used.ngw]
        out = []
        for m in n:
            c = (rng.standard_normal((s.nst, m)) + 1j * rng.standard_normal((s.nst, m)))
            if what != "kset":
                c[:, 0] = c[:, 0].real
            out.append(c / np.sqrt(m))
        return used.kset_pack(out) if what == "kset" else out[0]

    def evaluate(ef, c, forces):
        dc, dh = ctx.to_device(c), ctx.to_device(np.zeros_like(c))
        r = dict(ef.evaluate(dc, dh, forces=forces, stress=forces, prec=prec))
        r["h"], r["rho"] = dh.download(), ef.get(0)
        for d in (dc, dh):
            d.release()
        return r

    if what == "spin":
        evaluate(used, bands(), True)
        used.set_nspin(2, s.nst)            # the density of the second spin is zero now
        fresh.set_nspin(2, s.nst)
    evaluate(used, bands(), True)
    evaluate(used, bands(), False)
    c = bands()
    got, ref = evaluate(used, c, True), evaluate(fresh, c, True)
    for k in ref:
        assert np.array_equal(np.asarray(got[k]), np.asarray(ref[k])), k
    assert np.abs(ref["fion"]).max() > 0.0
    used.release()
    fresh.release()
