"""Evaluations above the size from which the kinetic and nonlocal part runs on a
second stream beside the transforms, against the same evaluation in order (which
an enabled profiler selects): the same kernels on the same operands, joined
before anything adds to their results, so every result is equal bit by bit.

Three sets of bands and two sets of positions take turns and H psi is overwritten
before each call, so that nothing left by the call before it can pass for a result;
the evaluations are checked one by one, then enqueued behind one another
without a wait or a copy in between, through evaluate_async and through the calls of a host loop.
The count of evaluations beside the transforms shows which of them were.
"""
import dataclasses

import numpy as np
import pytest

from qbg import configs as cf

pytestmark = pytest.mark.gpu

SETS = 3


@pytest.fixture(scope="module")
def ctx():
    import qbg
    c = qbg.Context(0)
    yield c
    c.close()


def _same(a, b):
    assert a.keys() == b.keys()
    for k in a:
        assert np.array_equal(np.asarray(a[k]), np.asarray(b[k])), k


def _system(what):
    if what == "kset":                      # the full sphere of 3 k-points, about 11400 each
        return dataclasses.replace(cf.config(0), nst=100), dict(
            kpoints=np.array([[0.25, 0.1, 0.0], [0.0, 0.3, 0.2], [0.4, 0.0, 0.1]]),
            weights=np.array([0.5, 0.25, 0.25]))
    s = cf.config(1)
    return cf.spin_polarized(s, 128, 1, 1) if what == "spin" else s, {}


@pytest.mark.parametrize("what,prec", [("gamma", "bf16x2"), ("gamma", "bf16x3"), ("gamma", "fp32"),
                                       ("gamma", "fp64"), ("kset", "bf16x2"), ("kset", "fp64"),
                                       ("spin", "bf16x2")])
def test_beside_equals_in_order(ctx, what, prec):
    import qbg
    print(f"[case] side stream {what} {prec}", flush=True)
    s, kw = _system(what)
    ef = qbg.EnergyFunctional(ctx, s, **kw)
    assert ef.ngw * s.nst * ef.nkp >= 3 << 20
    rng = np.random.default_rng(5)

    def bands(n):
        x = rng.standard_normal((s.nst, n)) + 1j * rng.standard_normal((s.nst, n))
        if what != "kset":
            x[:, 0] = x[:, 0].real
        return x / np.sqrt(n)

    cs = [ef.kset_pack([bands(n) for n in ef.kngw]) if what == "kset" else bands(ef.ngw)
          for _ in range(SETS)]
    dcs = [ctx.to_device(c) for c in cs]
    stale = np.full_like(cs[0], 7.25 - 3.5j)
    dhs = [ctx.to_device(stale) for _ in cs]
    tau = [np.asarray(s.tau), np.asarray(s.tau) + rng.uniform(-0.1, 0.1, np.shape(s.tau))]
    prof = qbg.Profiler(ctx)

    def evaluate(i, forces=True):
        dhs[i].upload(stale)
        r = dict(ef.evaluate(dcs[i], dhs[i], forces=forces, stress=forces, prec=prec))
        r["h"] = dhs[i].download()
        return r

    evaluate(0)                             # the launch choices are timed here
    prof.enable(True)
    n0 = ctx.beside_count()
    ref = []
    for t in tau:
        ef.set_positions(t)
        ref.append([evaluate(i) for i in range(SETS)])
    assert ctx.beside_count() == n0         # in order under the profiler
    prof.enable(False)
    for a in ref[0] + ref[1]:               # all differ, so that each check means something
        for b in ref[0] + ref[1]:
            assert a is b or (a["enl"] != b["enl"] and a["etotal"] != b["etotal"] and
                              not np.array_equal(a["h"], b["h"]))
    assert ref[0][0]["ekin"] != ref[0][1]["ekin"]

    for p in (0, 1):
        ef.set_positions(tau[p])
        for i in (1, 0, 2, 1):
            _same(evaluate(i), ref[p][i])
            n0 += 1
            assert ctx.beside_count() == n0

    def check_queue(enqueue, p, order):
        nonlocal n0
        ef.set_positions(tau[p])
        for d in dhs:
            d.upload(stale)
        ctx.sync()
        for i in order:
            enqueue(i)
        r = dict(ef.results())
        n0 += len(order)
        assert ctx.beside_count() == n0
        last = order[-1]
        _same(r, {k: v for k, v in ref[p][last].items() if k != "h"})
        for i in order:
            assert np.array_equal(dhs[i].download(), ref[p][i]["h"]), i

    def one_call(i):
        ef.evaluate_async(dcs[i], dhs[i], forces=True, stress=True, prec=prec)

    def host_loop(i):
        ef.update_density(dcs[i], prec)
        ef.update_vhxc(True)
        ef.energy_async(dcs[i], dhs[i], forces=True, stress=True, prec=prec, same_c=True)

    check_queue(one_call, 1, (2, 0, 1))
    check_queue(one_call, 0, (0, 1, 2))
    check_queue(host_loop, 1, (1, 2, 0))
    # H psi over the bands themselves stays in order
    prof.enable(True)
    dc = ctx.to_device(cs[0])
    ef.evaluate(dc, dc, forces=False, stress=False, prec=prec)
    own = dc.download()
    prof.enable(False)
    dc.upload(cs[0])
    ef.evaluate(dc, dc, forces=False, stress=False, prec=prec)
    assert np.array_equal(dc.download(), own)
    assert ctx.beside_count() == n0
    for d in dcs + dhs + [dc]:
        d.release()
    ef.release()


@pytest.mark.parametrize("k,captured", [(0, False), (1, True)])
def test_small_and_captured_stay_in_order(ctx, k, captured):
    import qbg
    s = cf.config(k)
    print(f"[case] in order {s.name} captured {captured}", flush=True)
    ef = qbg.EnergyFunctional(ctx, s)
    c = cf.random_coefficients(3, ef.basis(0)["g2"], s.nst)
    dc, dh = ctx.to_device(c), ctx.to_device(np.zeros_like(c))
    n0 = ctx.beside_count()
    ref = [ef.evaluate(dc, dh, forces=True, prec="fp64") for _ in range(2)][1]
    assert (ctx.beside_count() > n0) == captured        # this size would run beside
    n0 = ctx.beside_count()
    if captured:
        with qbg.Graph(ctx) as g:
            ef.evaluate_async(dc, dh, forces=True, prec="fp64")
        for _ in range(3):
            dh.zero()
            g.launch()
            assert ef.results()["etotal"] == ref["etotal"]
        g.release()
    assert ctx.beside_count() == n0
    for d in (dc, dh):
        d.release()
    ef.release()
