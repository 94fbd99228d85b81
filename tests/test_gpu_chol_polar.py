"""The dense steps of csrc/chol.hip and the mixer's eigensolver at the edges of
their blocks: the polar iteration around the 16-row tiles, the 64-column panels
and the largest matrix of the one-launch form, in both branches; a pivot that
fails in the first, last and middle columns of a panel; and Anderson mixing with
an odd and the full number of past vectors.

Bounds: the polar factor of a matrix with singular values in [0.3, 2.5] has a
perturbation bound of 2 / (2 x 0.3) times the rounding of a few products of n <= 160
terms, below 1e-12, and what the iteration leaves at its stop is of third order in 1e-6;
mixing as the neighbouring tests (1e-12), times the condition of the normal equations
of densities that differ in every call (below 100).
"""
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


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 63, 64, 65, 80, 90, 127, 128, 129, 160])
@pytest.mark.parametrize("branch", ["bjorck", "higham"])
def test_polar_sizes(ctx, oracle_mod, n, branch):
    import qbg
    print(f"[case] polar n {n} {branch}", flush=True)
    rng = np.random.default_rng(10 * n)
    u0, _ = np.linalg.qr(rng.standard_normal((n, n)))
    v0, _ = np.linalg.qr(rng.standard_normal((n, n)))
    sv = (1.0 + 0.4 * rng.uniform(-1, 1, n) / np.sqrt(n) if branch == "bjorck"
          else np.concatenate([[2.5], rng.uniform(0.3, 2.5, n - 1)]))
    x = u0 @ np.diag(sv) @ v0
    assert (np.linalg.norm(np.eye(n) - x.T @ x) < 1.0) == (branch == "bjorck")
    u, it = qbg.polar(ctx, x)
    _, ito = oracle_mod.polar(x)
    assert it == ito
    assert np.abs(u - u0 @ v0).max() < 1e-11
    assert np.abs(u.T @ u - np.eye(n)).max() < 1e-12


@pytest.mark.parametrize("n,col", [(5, 4), (64, 0), (64, 63), (100, 40), (100, 70), (128, 64),
                                   (150, 149)])
def test_polar_singular(ctx, n, col):
    import qbg
    print(f"[case] singular polar n {n} column {col}", flush=True)
    x = 2.0 * np.eye(n)
    x[:, col] = 0.0                        # its pivot is exactly 0
    with pytest.raises(qbg.QbgError) as e:
        qbg.polar(ctx, x)
    assert e.value.code == -4              # QBG_E_NOT_SPD
    u, _ = qbg.polar(ctx, 2.0 * np.eye(n))
    assert np.abs(u - np.eye(n)).max() < 1e-13


@pytest.mark.parametrize("nst,col", [(1, 0), (64, 0), (64, 63), (65, 64), (130, 100), (200, 15)])
@pytest.mark.parametrize("which", ["gram", "gram_noalloc"])
def test_gram_pivot(ctx, nst, col, which):
    import qbg
    print(f"[case] {which} nst {nst} zero band {col}", flush=True)
    rng = np.random.default_rng(nst + col)
    ngw = 400
    c = rng.standard_normal((nst, ngw)) + 1j * rng.standard_normal((nst, ngw))
    c[col] = 0.0
    d = ctx.to_device(c)
    with pytest.raises(qbg.QbgError) as e:
        getattr(qbg, which)(ctx, d, ngw, ngw, nst)
    assert e.value.code == -4
    c[:, 0] = c[:, 0].real
    assert np.array_equal(d.download(), c)


@pytest.mark.parametrize("ndim", [1, 2, 5, 8])
def test_mixer_dimensions(ctx, oracle_mod, ndim):
    import qbg
    print(f"[case] mixer ndim {ndim}", flush=True)
    s = cf.config(11)
    ef = qbg.EnergyFunctional(ctx, s)
    o = oracle_mod.Oracle(s)
    b = ef.basis(0)
    mx = qbg.Mixer(ef, 0.4, 6.0, ndim, 3.0)
    mo = o.mixer(0.4, 6.0, ndim, 3.0)
    for it in range(ndim + 3):
        c = cf.gram_numpy(cf.random_coefficients(170 + it, b["g2"], s.nst))
        dc = ctx.to_device(c)
        ef.update_density(dc)
        mx.update()
        o.update_density(c)
        mo.update()
        for k in (0, 3):
            got, ref = np.asarray(ef.get(k)), np.asarray(o.get(k))
            assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max(), (it, k)
        dc.release()
    mx.release()
    ef.release()
