"""The half-wave engine (FP64 benzene sweeps, 32 lanes per walker) against
the tile engine on the same walkers: both workgroup sizes, walker counts
that leave half a wavefront or a workgroup idle, MOs that differ between the
spins, a run without an e-n Jastrow.  FP64 in another order: the same
decisions, positions and energies to 1e-9, the engines' other trajectory
bound."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Q():
    import rust_qmc_amd

    return rust_qmc_amd


def _chain(Q, s, engine, W, move, n):
    s.set_engine(engine)
    ens = Q.Ensemble(s, W, 5)
    es, e2, acc, tr = ens.sweeps(n, 0.2 if move == Q.QMC_MOVE_SINGLE else 0.005, move=move, trace=True, max_drift=0.3,
                                 refresh_interval=3, steps_per_launch=2)
    return es, acc, tr, ens.positions(), ens.state()


def _compare(Q, s, W, n=5):
    for move in (Q.QMC_MOVE_SINGLE, Q.QMC_MOVE_DRIFT):
        a, b = _chain(Q, s, "auto", W, move, n), _chain(Q, s, "tile", W, move, n)
        assert np.array_equal(a[1], b[1]) and b[1].sum() > 0
        np.testing.assert_allclose(a[3], b[3], rtol=0, atol=1e-9)
        for x, y in zip((a[0], a[2], *a[4]), (b[0], b[2], *b[4])):
            np.testing.assert_allclose(x, y, rtol=1e-9, atol=1e-9)


@pytest.mark.parametrize("W", [1, 2, 9, 35, 2051])
def test_matches_tile_engine(Q, W):
    _compare(Q, Q.BenzeneGTO(1.5, 2.0, 2.64, 2.05), W, 5 if W < 100 else 2)


def test_spin_dependent_mos_and_other_shell_patterns(Q):
    d = json.loads(Q.BenzeneGTO(1.5, 2.0, 2.64, 2.05).to_json())
    rng = np.random.default_rng(2)
    del d["mo_rule"]
    d["mo_dn"] = (np.array(d["mo_dn"]) + 0.02 * rng.normal(size=(21, 66))).tolist()
    for a in d["aos"][:9]:  # the first carbon with five instead of six core primitives
        if len(a["exp"]) == 6:
            a["exp"], a["coef"], a["pow"] = a["exp"][:5], a["coef"][:5], a["pow"][:5]
    s = Q.System.from_json(json.dumps(d))
    _compare(Q, s, 9, 3)
    pos = s.get_nuclei()[np.arange(42) % 12] + 0.8 * rng.normal(size=(5, 42, 3))
    s.set_engine("auto")
    a = s.evaluate_batch(pos), s.derivatives_batch(pos)
    s.set_engine("wave")
    b = s.evaluate_batch(pos), s.derivatives_batch(pos)
    for x, y in zip(a, b):
        for k in y:
            assert np.abs(x[k] - y[k]).max() <= 1e-9 * max(1.0, np.abs(y[k]).max()), k


def test_without_jastrow(Q):
    d = json.loads(Q.BenzeneGTO(1.5, 2.0, 2.64, 2.05).to_json())
    d["jastrow"] = {"kind": "none"}
    _compare(Q, Q.System.from_json(json.dumps(d)), 3, 3)
