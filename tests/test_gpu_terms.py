"""The one-electron-per-lane evaluation and derivative kernels of benzene
against the wave engine's on the same configurations: walker counts on both
sides of a workgroup's three, singular Slater matrices, a perturbed geometry
(the C-H MOs follow it).  Both are FP64 in another order; 1e-9 of each
output's scale, from FP64 rounding amplified by the Slater inverses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Q():
    import rust_qmc_amd

    return rust_qmc_amd


def _configs(Q, s, W, seed):
    d = np.random.default_rng(seed)
    nuc = s.get_nuclei()
    e = np.array([[i % 6, i % 12] for i in range(42)])[:, 1]
    return nuc[e] + 0.8 * d.normal(size=(W, 42, 3))


def _both(Q, s, f):
    s.set_engine("auto")
    a = f()
    s.set_engine("wave")
    return a, f()


def _same(a, b):
    for k in b:
        scale = np.abs(b[k]).max() or 1.0
        assert np.abs(a[k] - b[k]).max() <= 1e-9 * scale, k


@pytest.mark.parametrize("W", [1, 2, 3, 4, 64, 100])
def test_evaluate_and_derivatives_match_wave_engine(Q, W):
    s = Q.BenzeneGTO(1.5, 2.0, 2.64, 2.05, precision="fp64")
    R = s.get_nuclei()
    s.set_nuclei(R + 0.02 * np.random.default_rng(3).normal(size=R.shape))
    pos = _configs(Q, s, W, W)
    _same(*_both(Q, s, lambda: s.evaluate_batch(pos)))
    _same(*_both(Q, s, lambda: s.derivatives_batch(pos)))


def test_ensemble_measure_matches_wave_engine(Q):
    for precision, tol in (("fp64", 1e-9), ("mixed", 2e-3)):  # the wave engine's mixed terms run in FP32
        s = Q.BenzeneGTO(1.5, 2.0, 2.64, 2.05, precision=precision)
        ens = Q.Ensemble(s, 100, 3)

        def moments():
            ens.measure(reset=True)
            m = ens.moments()
            return {k: np.asarray(m[k], dtype=float) for k in ("o_mean", "S", "f", "de_mean", "f_hf", "f_zv", "energy")}

        a, b = _both(Q, s, moments)
        for k in b:
            assert np.abs(a[k] - b[k]).max() <= tol * max(1.0, np.abs(b[k]).max()), (precision, k)


def test_singular_matrix_is_reported(Q):
    s = Q.BenzeneGTO(1.5, 2.0, 2.64, 2.05, precision="fp64")
    pos = _configs(Q, s, 5, 1)
    pos[3, 0] = 1e4  # every orbital of this electron underflows to zero
    s.set_flags(0)
    with pytest.raises(Q.QmcError, match="1 configurations with a singular"):
        s.evaluate_batch(pos)
    s.set_flags(Q.QMC_FLAGS_REFERENCE)
    o = s.evaluate_batch(pos)
    assert o["logabs"][3] == -np.inf and o["sign"][3] == 0.0
    assert np.isfinite(o["logabs"][[0, 1, 2, 4]]).all() and np.isfinite(o["eloc"]).all()
