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
