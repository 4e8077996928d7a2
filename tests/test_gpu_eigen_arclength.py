"""GPU: stability eigenvalues (LOBPCG on J) and arc-length continuation,
checked with the oracle: eigenpairs against a dense symmetric
eigendecomposition of the oracle's Jacobian, every continuation state
against the oracle's F, and the folds of the Meissner branch against the
eigenvalue that must cross zero there."""
import numpy as np
import pytest

from nosh_amd import meshgen as mg

pytestmark = pytest.mark.gpu

NEWTON = dict(tol=1e-10, max_iters=10, minres_rtol=1e-12, minres_max_iters=3000)


def _setup(ncell=16):
    import nosh_amd as nosh
    from oracle import oracle as O
    c, t = mg.square_tri(ncell)
    mesh = nosh.Mesh(c, t)
    mvp = nosh.VectorFieldExplicitValues(mesh, mg.magnetic_potential(c), 0.0)
    model = nosh.Nls(mesh, mvp, nosh.ScalarFieldConstant(mesh, -1.0), 1.0,
                     nosh.ScalarFieldConstant(mesh, 1.0))
    om = O.Model(O.Mesh(c, t), mg.magnetic_potential(c))
    return c, t, model, om


def _meissner(model, n, mu):
    """The Meissner state at mu by natural continuation from psi = 1 at 0."""
    import nosh_amd as nosh
    psi0 = np.zeros(2 * n)
    psi0[0::2] = 1.0
    psi, rec = nosh.continuation(model, psi0, {"g": 1.0}, "mu", 0.0, mu, 5, predictor=1,
                                 tol=1e-11, max_iters=20, minres_rtol=1e-12,
                                 minres_max_iters=3000)
    assert all(r["converged"] for r in rec)
    return psi


def _dense_jac(om, psi, mu):
    om.set_params(1.0, mu)
    om.jac_rebuild(psi)
    m = psi.size
    J = np.empty((m, m))
    e = np.zeros(m)
    for i in range(m):
        e[i] = 1.0
        J[:, i] = om.jac(e)
        e[i] = 0.0
    return 0.5 * (J + J.T)


def _gauge(psi):
    q = np.empty_like(psi)
    q[0::2], q[1::2] = -psi[1::2], psi[0::2]
    return q / np.linalg.norm(q)


def _dense_spectrum(om, psi, mu):
    """(all eigenvalues, the eigenvalues without the phase mode, eigvecs)."""
    w, V = np.linalg.eigh(_dense_jac(om, psi, mu))
    g = int(np.argmax(np.abs(V.T @ _gauge(psi))))
    assert abs(w[g]) < 1e-9 * np.abs(w).max()  # i psi is in the null space
    return w, np.delete(w, g), V


def test_eigenpairs_match_dense_oracle():
    """16x16 square, Meissner state at mu = 0.25: the 4 smallest eigenvalues
    with the phase mode deflated, the 3 smallest without (the first is the
    phase mode's zero) and the 2 largest agree with numpy's eigh of the
    oracle's dense Jacobian; the vectors are eigenvectors of the oracle's J."""
    import nosh_amd as nosh
    c, t, model, om = _setup()
    n = c.shape[0]
    mu = 0.25
    psi = _meissner(model, n, mu)
    w, wd, _ = _dense_spectrum(om, psi, mu)
    scale = np.abs(w).max()
    ev, vec, st = nosh.jacobian_eigenpairs(model, psi, {"g": 1.0, "mu": mu}, nev=4,
                                           vectors=True, tol=1e-10)
    print("deflated", ev, "dense", wd[:4], st)
    assert st["converged"] == 4
    assert np.allclose(ev, wd[:4], rtol=1e-8, atol=1e-11 * scale)
    om.set_params(1.0, mu)
    om.jac_rebuild(psi)
    q = _gauge(psi)
    for j in range(4):
        v = vec[j]
        assert abs(np.linalg.norm(v) - 1.0) < 1e-10
        assert np.linalg.norm(om.jac(v) - ev[j] * v) <= 1e-9 * scale
        assert abs(v @ q) < 1e-8
    ev0, _, st0 = nosh.jacobian_eigenpairs(model, psi, {"g": 1.0, "mu": mu}, nev=3,
                                           deflate_gauge=0, tol=1e-10)
    print("not deflated", ev0, "dense", w[:3], st0)
    assert abs(ev0[0]) < 1e-9 * scale
    assert np.allclose(ev0[1:], w[1:3], rtol=1e-8, atol=1e-11 * scale)
    evl, _, stl = nosh.jacobian_eigenpairs(model, psi, {"g": 1.0, "mu": mu}, nev=2, which=1,
                                           use_prec=0, tol=1e-10, max_iters=3000)
    print("largest", evl, "dense", w[-2:], stl)
    assert np.allclose(evl, w[::-1][:2], rtol=1e-9)


def test_arclength_turns_at_folds_where_an_eigenvalue_crosses_zero():
    """Arc-length continuation of the Meissner branch of the 16x16 square from
    mu = 0.25 (ds = 0.02): every state solves F = 0 (oracle); the parameter
    turns back near mu = 0.304 and forward again near mu = 0.289 (two folds,
    which natural continuation cannot pass), and across each fold exactly one
    stability eigenvalue changes sign (det J changes sign with p'), the
    eigenvalues there agreeing with the oracle's dense spectrum."""
    import nosh_amd as nosh
    c, t, model, om = _setup()
    n = c.shape[0]
    psi0 = _meissner(model, n, 0.25)
    psi, rec, states = nosh.arclength(model, psi0, {"g": 1.0, "mu": 0.25}, "mu", start=0.25,
                                      max_steps=18, states=True, initial_step=0.02,
                                      max_step=0.02, eigenvalues=5, newton_kw=NEWTON)
    for r in rec:
        print(round(r["param"], 6), round(r["param_dot"], 4), r["newton_iters"],
              r["minres_iters"], r["num_negative"], [f"{e:+.3e}" for e in r["eigs"]])
    assert len(rec) == 19 and all(r["converged"] for r in rec)
    for r, x in zip(rec, states):
        om.set_params(1.0, r["param"])
        assert np.linalg.norm(om.f(x)) <= 1e-9
    mus = np.array([r["param"] for r in rec])
    pd = np.array([r["param_dot"] for r in rec])
    neg = np.array([r["num_negative"] for r in rec])
    f1 = int(np.argmax(pd < 0))
    assert f1 > 0 and pd[f1] < 0
    f2 = f1 + int(np.argmax(pd[f1:] > 0))
    assert f2 > f1 and pd[f2] > 0
    assert 0.302 < mus.max() < 0.307
    assert 0.286 < mus[f1:f2 + 1].min() < 0.292
    assert neg[f1] - neg[f1 - 1] == 1
    assert neg[f2] - neg[f2 - 1] == -1
    # Dense check of the spectrum just past the first fold.
    _, wd, _ = _dense_spectrum(om, states[f1], mus[f1])
    assert np.allclose(rec[f1]["eigs"], wd[:5], rtol=1e-7, atol=1e-9)


def test_arclength_adaptive_steps_and_bound():
    """From psi = 1 at mu = 0 with a small first step: the accepted step sizes
    follow the adaptive rule ds' = min(max, ds (1 + a ((N - k)/(N - 1))^2)),
    the run stops exactly on max_value = 0.1 with a natural step there, and the
    final state equals the natural-parameter continuation's at mu = 0.1 (up to
    the phase); the secant predictor ends on the same state."""
    import nosh_amd as nosh
    from conftest import phase_align
    c, t, model, om = _setup()
    n = c.shape[0]
    psi0 = np.zeros(2 * n)
    psi0[0::2] = 1.0
    finals = {}
    for pred in (1, 2):
        psi, rec = nosh.arclength(model, psi0, {"g": 1.0, "mu": 0.0}, "mu", start=0.0,
                                  max_steps=40, initial_step=0.002, max_step=0.03,
                                  aggressiveness=2.0, max_value=0.1, predictor=pred,
                                  newton_kw=NEWTON)
        print(pred, [(round(r["param"], 5), r["step"], r["newton_iters"]) for r in rec])
        assert all(r["converged"] for r in rec)
        assert rec[-1]["param"] == 0.1 and len(rec) < 41
        N = NEWTON["max_iters"]
        for a, b in zip(rec[1:-2], rec[2:-1]):
            if b["failures"] == 0 and a["failures"] == 0:
                q = (N - a["newton_iters"]) / (N - 1)
                assert b["step"] == pytest.approx(min(0.03, a["step"] * (1 + 2.0 * q * q)),
                                                  rel=1e-12)
        assert max(r["step"] for r in rec) == 0.03
        om.set_params(1.0, 0.1)
        assert np.linalg.norm(om.f(psi)) <= 1e-9
        finals[pred] = psi
    ref, rn = nosh.continuation(model, psi0, {"g": 1.0}, "mu", 0.0, 0.1, 5, predictor=1,
                                tol=1e-11, max_iters=20, minres_rtol=1e-12, minres_max_iters=3000)
    assert all(r["converged"] for r in rn)
    for pred in (1, 2):
        d = np.linalg.norm(phase_align(finals[pred], ref) - ref) / np.linalg.norm(ref)
        assert d < 1e-9, (pred, d)


def test_arclength_run_written_by_the_observers(tmp_path):
    """An arclength run with eigenvalues, written as the reference's drivers
    write it: the observer CSV (Gibbs energy and scaled norm from the library
    agree with their formulas over the oracle's control volumes), the eigen
    data CSV and one state file per step (read back bit-exact)."""
    import nosh_amd as nosh
    from nosh_amd import io as nio
    from oracle import oracle as O
    c, t, model, om = _setup(12)
    n = c.shape[0]
    psi0 = np.zeros(2 * n)
    psi0[0::2] = 1.0
    psi, rec, states = nosh.arclength(model, psi0, {"g": 1.0, "mu": 0.0}, "mu", start=0.0,
                                      max_steps=5, states=True, initial_step=0.05,
                                      max_step=0.05, eigenvalues=3, newton_kw=NEWTON)
    assert len(rec) == 6 and all(r["converged"] for r in rec)
    obs = nio.ContinuationObserver(str(tmp_path / "cont.dat"), "mu", model=model)
    eig = nio.EigenDataSaver(str(tmp_path / "eig.dat"))
    saver = nio.ContinuationDataSaver(c, t, str(tmp_path), "mu")
    for r, x in zip(rec, states):
        obs.observe(x, r["param"])
        eig.save(r["eigs"])
        saver.save_solution(x, r["param"])
    obs.close()
    eig.close()
    cv = O.Mesh(c, t).control_volumes()
    labels, rows = nio.read_csv(str(tmp_path / "cont.dat"))
    assert labels[1] == "(1) mu" and rows.shape == (6, 4)
    for k, (r, x) in enumerate(zip(rec, states)):
        a2 = x[0::2] ** 2 + x[1::2] ** 2
        assert rows[k, 0] == k and rows[k, 1] == pytest.approx(r["param"], rel=1e-14)
        assert rows[k, 2] == pytest.approx(-np.sum(cv * a2 * a2) / cv.sum(), rel=1e-12)
        assert rows[k, 2] == pytest.approx(r["gibbs"], rel=1e-12)
        assert rows[k, 3] == pytest.approx(np.sqrt(np.sum(cv * a2) / cv.sum()), rel=1e-12)
        p, fd = nio.read_state(str(tmp_path / f"out{k:04d}.vtu"))
        assert np.array_equal(p, x) and fd["mu"] == r["param"]
    labels, erows = nio.read_csv(str(tmp_path / "eig.dat"))
    assert erows.shape == (6, 7)
    assert np.allclose(erows[:, 4:], [r["eigs"] for r in rec], rtol=1e-14)


def test_invalid_options_are_errors_not_crashes():
    """Bad eigensolver / arclength options come back as errors (ValueError
    for NOSH_ERR_INVALID) and leave the model usable; a bound crossed on the
    first step ends the run on the bound."""
    import nosh_amd as nosh
    c, t, model, om = _setup(8)
    n = c.shape[0]
    psi0 = np.zeros(2 * n)
    psi0[0::2] = 1.0
    p = {"g": 1.0, "mu": 0.0}
    for bad in (dict(nev=0), dict(nev=17), dict(nev=2, which=2), dict(nev=2, tol=0.0),
                dict(nev=2, max_iters=0)):
        with pytest.raises(ValueError):
            nosh.jacobian_eigenpairs(model, psi0, p, **bad)
    with pytest.raises(KeyError):
        nosh.jacobian_eigenpairs(model, psi0, {"mu": 0.0}, nev=2)
    for bad in (dict(max_steps=0), dict(initial_step=0.0), dict(min_value=1.0, max_value=0.0),
                dict(predictor=3), dict(eigenvalues=9)):
        with pytest.raises(ValueError):
            nosh.arclength(model, psi0, p, "mu", start=0.0, **bad)
    with pytest.raises(ValueError):
        nosh.arclength(model, psi0, p, "V", start=0.0)
    psi, rec = nosh.arclength(model, psi0, p, "mu", start=0.0, max_steps=5, initial_step=0.5,
                              max_value=0.05, newton_kw=NEWTON)
    assert len(rec) == 2 and rec[-1]["param"] == 0.05 and rec[-1]["converged"]
    om.set_params(1.0, 0.05)
    assert np.linalg.norm(om.f(psi)) <= 1e-9
    ev, _, st = nosh.jacobian_eigenpairs(model, psi, {"g": 1.0, "mu": 0.05}, nev=2, tol=1e-9)
    assert st["converged"] == 2 and ev[0] > 0


@pytest.mark.parametrize("nev,block", [(1, 1), (2, 3), (5, 8), (16, 16)])
def test_eigenvalues_at_other_block_sizes(nev, block):
    """Block products of 1 to 48 columns (every width of the combination kernel,
    the padded ones, and blocks above 8, whose X and P are combined apart):
    the smallest eigenvalues of the 8x8 square's J, phase mode deflated, against
    numpy's eigh of the oracle's dense J."""
    import nosh_amd as nosh
    c, t, model, om = _setup(8)
    psi = _meissner(model, c.shape[0], 0.2)
    w, wd, _ = _dense_spectrum(om, psi, 0.2)
    ev, _, st = nosh.jacobian_eigenpairs(model, psi, {"g": 1.0, "mu": 0.2}, nev=nev,
                                         block_size=block, tol=1e-10, max_iters=2000)
    assert st["converged"] == nev
    assert np.allclose(ev, wd[:nev], rtol=1e-8, atol=1e-11 * np.abs(w).max())


@pytest.mark.parametrize("ncell", [446, 447])
def test_eigenvectors_at_the_column_split(ncell):
    """199809 and 200704 rows, the two sides of the line between two and eight
    columns a thread: the pairs of J at psi = 1, mu = 0 are pairs of the
    oracle's J. The solver ends at 1e-8 of the largest Rayleigh quotient of its
    start, random vectors; |J x| / |x| of one such vector is no smaller."""
    import nosh_amd as nosh
    c, t, model, om = _setup(ncell)
    psi = np.zeros(2 * c.shape[0])
    psi[0::2] = 1.0
    ev, vec, st = nosh.jacobian_eigenpairs(model, psi, {"g": 1.0, "mu": 0.0}, nev=2, vectors=True,
                                           tol=1e-8, max_iters=1000)
    assert st["converged"] == 2
    om.set_params(1.0, 0.0)
    om.jac_rebuild(psi)
    x = np.random.default_rng(5).standard_normal(psi.size)
    scale = np.linalg.norm(om.jac(x)) / np.linalg.norm(x)
    for j in range(2):
        assert np.linalg.norm(om.jac(vec[j]) - ev[j] * vec[j]) <= 2e-8 * scale
