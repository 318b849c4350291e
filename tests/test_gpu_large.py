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


def _system(Q, name, precision):
    return {"h2": lambda: Q.H2MoleculeMO(precision=precision), "ch4": lambda: Q.MethaneGTO(precision=precision),
            "benzene": lambda: Q.BenzeneGTO(precision=precision)}[name]()


# 1, 64 and 65 walkers; 512 KiB (10,922 of H2's 48 bytes, 2,184 of CH4's 240, 520
# of benzene's 1,008) and 32 MiB (699,008 walkers of H2, 139,776 of CH4, 33,280
# of benzene) are where the way of the copy changes
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name,W", [("h2", 1), ("h2", 65), ("h2", 10_922), ("h2", 10_923), ("h2", 699_008), ("h2", 699_010),
                                    ("ch4", 64), ("ch4", 2_185), ("ch4", 139_777 + 64), ("benzene", 65),
                                    ("benzene", 521), ("benzene", 33_281)])
def test_positions_round_trip(Q, name, W, precision):
    """Positions set from the host and from the device come back exactly
    (rounded to FP32 in mixed precision), and the state is theirs."""
    s = _system(Q, name, precision)
    n, rng = s.n_elec, np.random.default_rng(W)
    pos = s.get_nuclei()[np.arange(n) % s.n_nuc] + rng.normal(size=(W, n, 3))
    want = pos if precision == "fp64" else pos.astype(np.float32).astype(np.float64)
    ens = Q.Ensemble(s, W, 1)
    ens.set_positions(pos)
    np.testing.assert_array_equal(ens.positions(), want)
    some = np.unique(np.r_[0, W // 2, W - 1])
    ref = s.evaluate_batch(want[some])
    np.testing.assert_allclose(ens.state()[0][some], ref["logabs"], rtol=1e-9, atol=1e-9)
    with Q.DeviceBuffer(pos.nbytes) as buf:
        buf.upload(pos[::-1])
        Q.check(Q.lib().qmc_ensemble_set_positions(ens._h, buf.ptr))
        np.testing.assert_array_equal(ens.positions(), want[::-1])
        Q.check(Q.lib().qmc_ensemble_get_positions(ens._h, buf.ptr))
        np.testing.assert_array_equal(buf.download(np.float64, pos.size).reshape(pos.shape), want[::-1])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_benzene_refresh_in_parts(Q, precision):
    """The tile refresh takes 65,536 walkers at a time: ln|psi| after it, and
    E_L of one sweep from its inverses, are those of the positions on both
    sides of the seam (1e-9 in FP64, the engines' bound; mixed: the FP32 E_L's
    2e-4 + 1e-2 Ha)."""
    s = _system(Q, "benzene", precision)
    W = 65536 + 21
    ens = Q.Ensemble(s, W, 2)
    some = np.r_[0:8, 65536 - 8 : W]
    ens.sweeps(2, 0.2, refresh_interval=2)  # the inverses are refreshed after the second sweep
    ref = s.evaluate_batch(ens.positions()[some])
    np.testing.assert_allclose(ens.state()[0][some], ref["logabs"], rtol=1e-9, atol=1e-9)
    el = ens.sweeps(1, 0.2, refresh_interval=0, trace=True)[3][0][some]
    ref = s.evaluate_batch(ens.positions()[some], ("eloc",))["eloc"]
    np.testing.assert_allclose(el, ref, rtol=1e-9 if precision == "fp64" else 2e-4, atol=1e-9 if precision == "fp64" else 1e-2)


# 131,072 a part; the kernel AUTO takes depends on the call's size and not on a
# part's (77 mixed CH4 configurations alone would go to the FP64 lane groups)
@pytest.mark.parametrize("name,precision", [("h2", "fp64"), ("ch4", "mixed")])
def test_derivatives_in_parts(Q, name, precision):
    """A call past the size of one part equals, to the bit, two calls that
    share its configurations and lie within one part."""
    s = _system(Q, name, precision)
    W, rng = 131072 + 77, np.random.default_rng(4)
    pos = s.get_nuclei()[np.arange(s.n_elec) % s.n_nuc] + 0.7 * rng.normal(size=(W, s.n_elec, 3))
    out = s.derivatives_batch(pos)
    for a, b in ((0, 100_000), (100_000, W)):
        ref = s.derivatives_batch(pos[a:b])
        for k in ref:
            np.testing.assert_array_equal(out[k][a:b], ref[k], err_msg=k)


# host calls of up to 2 MiB share one allocation, inputs or outputs of up to 1 MiB
# one copy each way, and derivatives of up to 128 KiB of features are unpacked on
# the host: W on both sides of each for CH4 (240 + 416 bytes, 48 features) and H2
# (48 + 88 bytes, 16 features, no parameters)
@pytest.mark.parametrize("name,W", [("ch4", 341), ("ch4", 342), ("ch4", 2520), ("ch4", 2600), ("ch4", 3196), ("ch4", 3197),
                                    ("ch4", 4369), ("ch4", 4370), ("h2", 1024), ("h2", 1025), ("h2", 15_420),
                                    ("h2", 15_421), ("h2", 21_846)])
def test_host_calls_around_the_copy_limits(Q, name, W):
    """Whatever way the arrays take, the results are those of batches of 100
    (which share one allocation and one copy each way), to the bit: the same
    kernel runs on both."""
    s = _system(Q, name, "fp64")
    rng = np.random.default_rng(W)
    pos = s.get_nuclei()[np.arange(s.n_elec) % s.n_nuc] + 0.7 * rng.normal(size=(W, s.n_elec, 3))
    for f in (s.evaluate_batch, s.derivatives_batch):
        out = f(pos)
        for a in (0, W // 2, W - 100):
            ref = f(pos[a : a + 100])
            for k in ref:
                np.testing.assert_array_equal(out[k][a : a + 100], ref[k], err_msg=k)
