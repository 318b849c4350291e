"""Ensembles and batches past the limits at which launches, staging buffers
and scratch are divided: nothing may change at a seam."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Q():
    import rust_qmc_amd

    return rust_qmc_amd


def test_all_electron_past_one_row_of_workgroups(Q):
    """65,536 workgroups of four CH4 walkers are one row of the grid: the
    walkers around its end move as the wave engine moves them."""
    s = Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0, precision="mixed")
    W = 4 * 65536 + 6
    out = []
    for engine in ("auto", "wave"):
        s.set_engine(engine)
        ens = Q.Ensemble(s, W, 3)
        p0 = ens.positions()
        es, _, acc = ens.sweeps(2, 0.2, move=Q.QMC_MOVE_ALL)
        out.append((acc, ens.positions(), ens.state()[2], es))
    (acc, pos, el, es), (acc_w, pos_w, _, _) = out
    assert np.array_equal(acc, acc_w)
    np.testing.assert_array_equal(pos, pos_w)
    np.testing.assert_allclose(es[-1], el.sum(), rtol=1e-11)  # every partial sum counted once
    # E_L of the walkers that moved is FP64 at the FP32 positions; 1e-8 leaves
    # FP64 rounding a factor of 1e7 for the worst-conditioned Slater matrix
    moved = (pos != p0).any(axis=(1, 2))
    ref = Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0).evaluate_batch(pos[moved], ("eloc",))["eloc"]
    np.testing.assert_allclose(el[moved], ref, rtol=1e-8, atol=1e-8)


@pytest.mark.parametrize("asked", [0, 16, 40])
def test_partial_sums_of_a_large_ensemble_stay_bounded(Q, asked):
    """All-electron CH4 moves have a partial-sum row per four walkers; a launch
    takes as many steps as 32 MiB of them hold."""
    s = Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0, precision="mixed")
    W, n = 500_000, 40
    ens = Q.Ensemble(s, W, 3)
    ens.set_timing()
    es, _, acc = ens.sweeps(n, 0.2, move=Q.QMC_MOVE_ALL, steps_per_launch=asked)
    per = (32 << 20) // (24 * (W // 4))
    assert ens.timing()[1] == -(-n // per)
    np.testing.assert_allclose(es[-1], ens.state()[2].sum(), rtol=1e-11)
    assert (0 < acc).all() and (acc < W).all()
