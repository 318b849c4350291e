"""The lane-group engine against the wave engine on the same walkers: every
compiled electron-count shape, walker counts that leave lanes and groups
idle, with and without Pade series terms.  Both run the FP64 arithmetic in
another order; the bounds are those of the engines' other trajectory tests
(1e-9, from FP64 rounding amplified by the Slater inverses)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 0), (1, 1), (2, 1), (2, 2), (3, 2), (3, 3), (4, 4), (5, 5)]


@pytest.fixture(scope="module")
def Q():
    import rust_qmc_amd

    return rust_qmc_amd


def _system(Q, nu, nd, precision, series):
    """Two nuclei with two s shells and a p shell each, random orthonormal
    MOs that differ between the spins."""
    rng = np.random.default_rng(11)
    aos, ex, co = [], [], []
    for c in range(2):
        for l, m, n in [(0, 0, 3), (0, 0, 1), (1, 0, 2), (1, 1, 2), (1, 2, 2)]:
            aos.append((0, c, l, m, n, len(ex)))
            if l == 1 and m > 0:  # one radial part for the three p components
                ex += ex[-n:]
                co += co[-n:]
            else:
                ex += list(0.25 * 3.0 ** np.arange(n) * (1 + 0.3 * c))
                co += list(rng.uniform(0.3, 0.8, n))
    mo = [np.linalg.qr(rng.normal(size=(10, 10)))[0][:5] for _ in range(2)]
    s = Q.System.from_desc(dict(
        spins=[1, -1] * nd + [1] * (nu - nd), nuclei=[[0.0, 0.0, 0.0], [0.3, 0.2, 1.9]], charges=[4.0, 3.0], aos=aos,
        prim_exp=ex, prim_coef=co, mo_up=mo[0], mo_dn=mo[1], jastrow_kind=2, b_ee=1.2, b_en=1.7,
        init_nuc=[i % 2 for i in range(nu + nd)]), precision)
    if series:
        s.set_jastrow_series(3, 0)
        p = s.get_params()
        p[4:] = 0.05 * rng.normal(size=p.size - 4)
        s.set_params(p)
    return s


def _chain(Q, s, engine, W, steps, step, **kw):
    s.set_engine(engine)
    ens = Q.Ensemble(s, W, 7)
    es, e2, acc, tr = ens.sweeps(steps, step, trace=True, **kw)
    return es, acc, tr, ens.positions(), ens.state()


@pytest.mark.parametrize("W", [1, 67])
@pytest.mark.parametrize("nu,nd", SHAPES)
def test_all_electron_matches_wave_engine(Q, nu, nd, W):
    s = _system(Q, nu, nd, "fp64", series=nu == nd)
    a = _chain(Q, s, "auto", W, 6, 0.2, move=Q.QMC_MOVE_ALL, steps_per_launch=4)
    b = _chain(Q, s, "wave", W, 6, 0.2, move=Q.QMC_MOVE_ALL)
    assert np.array_equal(a[1], b[1]) and b[1].sum() > 0
    np.testing.assert_allclose(a[3], b[3], rtol=0, atol=1e-12)
    for x, y in zip((a[0], a[2], *a[4]), (b[0], b[2], *b[4])):
        np.testing.assert_allclose(x, y, rtol=1e-9, atol=1e-9)


def test_all_electron_mixed_follows_the_wave_engine(Q):
    """FP32 positions; the lane-group energies run in FP64 on them, the wave
    engine's in FP32 (its bound: 2e-4 relative + 1e-3 Ha)."""
    s = _system(Q, 5, 5, "mixed", series=False)
    a = _chain(Q, s, "auto", 67, 4, 0.2, move=Q.QMC_MOVE_ALL)
    b = _chain(Q, s, "wave", 67, 4, 0.2, move=Q.QMC_MOVE_ALL)
    assert np.array_equal(a[1], b[1])
    np.testing.assert_array_equal(a[3], b[3])
    np.testing.assert_allclose(a[2], b[2], rtol=2e-4, atol=1e-3)


@pytest.mark.parametrize("move", ["single", "drift"])
@pytest.mark.parametrize("W", [1, 5, 67, 130])
@pytest.mark.parametrize("name", ["h2", "li", "li-ref", "ch4-sto3g", "ch4-631g"])
def test_fp64_sweeps_match_register_engine(Q, name, W, move):
    """Metropolis and drift-diffusion sweeps of every compiled structure
    against the one-walker-per-lane kernels: the same decisions, positions
    and energies to FP64 rounding (1e-9, as above)."""
    s = {"h2": lambda: Q.H2MoleculeMO(), "li": lambda: Q.Lithium(0), "li-ref": lambda: Q.Lithium(),
         "ch4-sto3g": lambda: Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0), "ch4-631g": lambda: Q.MethaneGTO()}[name]()
    kw = dict(move=Q.QMC_MOVE_SINGLE if move == "single" else Q.QMC_MOVE_DRIFT, steps_per_launch=3, refresh_interval=5,
              max_drift=0.5)
    step = 0.3 if move == "single" else 0.02
    a = _chain(Q, s, "auto", W, 8, step, **kw)
    b = _chain(Q, s, "register", W, 8, step, **kw)
    assert np.array_equal(a[1], b[1]) and b[1].sum() > 0
    np.testing.assert_allclose(a[3], b[3], rtol=0, atol=1e-9)
    for x, y in zip((a[0], a[2], *a[4]), (b[0], b[2], *b[4])):
        np.testing.assert_allclose(x, y, rtol=1e-9, atol=1e-9)


def test_fp64_sweeps_of_an_en_jastrow_on_h2(Q):
    """H2's two lanes hold the electrons, so its nuclei take a second partner
    round: a Pade Jastrow on the H2 shell structure."""
    s = Q.System.from_desc(dict(
        spins=[1, -1], nuclei=[[0, 0, 0.7], [0, 0, -0.7]], charges=[1.0, 1.0], aos=[(2, 0, 0, 0, 1, 0), (2, 1, 0, 0, 1, 1)],
        prim_exp=[1.3, 1.3], prim_coef=[1.0, 1.0], prim_pow=[0, 0], mo_up=[[1.0, 1.0]], jastrow_kind=2, b_ee=1.1, b_en=1.6,
        init_nuc=[0, 1]))
    assert s.engine_name() == "register/h2-slater1s"
    for move in (Q.QMC_MOVE_SINGLE, Q.QMC_MOVE_DRIFT):
        a = _chain(Q, s, "auto", 67, 6, 0.05, move=move)
        b = _chain(Q, s, "register", 67, 6, 0.05, move=move)
        assert np.array_equal(a[1], b[1])
        np.testing.assert_allclose(a[2], b[2], rtol=1e-9, atol=1e-9)
        np.testing.assert_allclose(a[3], b[3], rtol=0, atol=1e-9)


@pytest.mark.parametrize("W", [1, 3, 67])
@pytest.mark.parametrize("name", ["h2", "li", "li-ref", "ch4-sto3g", "ch4-631g"])
def test_derivatives_match_register_engine(Q, name, W):
    """E_L, O, dE_L/dp, F and Omega of every compiled structure against the
    one-walker-per-lane kernels, 1e-9 of each output's scale."""
    s = {"h2": lambda: Q.H2MoleculeMO(), "li": lambda: Q.Lithium(0), "li-ref": lambda: Q.Lithium(),
         "ch4-sto3g": lambda: Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0), "ch4-631g": lambda: Q.MethaneGTO()}[name]()
    pos = 0.8 * np.random.default_rng(W).normal(size=(W, s.n_elec, 3))
    s.set_engine("auto")
    a = s.derivatives_batch(pos)
    s.set_engine("register")
    b = s.derivatives_batch(pos)
    for k in b:
        if b[k].size:
            assert np.abs(a[k] - b[k]).max() <= 1e-9 * max(1.0, np.abs(b[k]).max()), k


@pytest.mark.parametrize("W", [1, 3, 67])
@pytest.mark.parametrize("name", ["h2", "li", "li-ref", "ch4-sto3g", "ch4-631g"])
def test_evaluation_matches_register_engine(Q, name, W):
    """ln|psi|, sign, gradients, Laplacians and E_L, 1e-9 of each output's scale."""
    s = {"h2": lambda: Q.H2MoleculeMO(), "li": lambda: Q.Lithium(0), "li-ref": lambda: Q.Lithium(),
         "ch4-sto3g": lambda: Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0), "ch4-631g": lambda: Q.MethaneGTO()}[name]()
    pos = 0.8 * np.random.default_rng(W).normal(size=(W, s.n_elec, 3))
    s.set_engine("auto")
    a = s.evaluate_batch(pos)
    s.set_engine("register")
    b = s.evaluate_batch(pos)
    for k in b:
        assert np.abs(a[k] - b[k]).max() <= 1e-9 * max(1.0, np.abs(b[k]).max()), k


def test_singular_configuration_is_reported(Q):
    s = Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0)
    pos = 0.8 * np.random.default_rng(5).normal(size=(6, 10, 3))
    pos[4, 0] = 1e4  # every orbital of this electron underflows to zero
    s.set_flags(0)
    with pytest.raises(Q.QmcError, match="1 configurations with a singular"):
        s.evaluate_batch(pos)
    s.set_flags(Q.QMC_FLAGS_REFERENCE)
    o = s.evaluate_batch(pos)
    assert o["logabs"][4] == -np.inf and o["sign"][4] == 0.0 and np.isfinite(o["logabs"][:4]).all()


@pytest.mark.parametrize("distance", [0.0, 1e-9, 1e-4])
@pytest.mark.parametrize("name", ["li", "ch4-sto3g", "ch4-631g"])
def test_laplacian_next_to_a_nucleus_or_an_electron(Q, name, distance):
    """Where 1/r is many orders larger than the Laplacian, the Laplacian keeps
    its own digits: electron 0 at a nucleus, and the last electron on electron
    1, against the one-walker-per-lane kernel (1e-9 of the finite values'
    scale, as above)."""
    s = {"li": lambda: Q.Lithium(0), "ch4-sto3g": lambda: Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0),
         "ch4-631g": lambda: Q.MethaneGTO()}[name]()
    rng = np.random.default_rng(9)
    pos = 0.8 * rng.normal(size=(5, s.n_elec, 3))
    R, d = s.get_nuclei(), distance * np.array([2.0, -1.0, 2.0]) / 3.0
    for w in range(4):
        pos[w, 0] = R[w % len(R)] + d
    pos[4, -1] = pos[4, 1] + d
    res = []
    for engine in ("auto", "register"):
        s.set_engine(engine)
        res.append(s.evaluate_batch(pos, ("lap",))["lap"])
    ok = np.isfinite(res[1])
    assert np.array_equal(np.isfinite(res[0]), ok) and ok[4].all()
    for a, b, k in zip(*res, ok):
        assert np.abs(a - b)[k].max() <= 1e-9 * max(1.0, np.abs(b[k]).max())
