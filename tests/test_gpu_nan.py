"""One configuration of a batch with a NaN coordinate: its ln|psi| and E_L are
NaN, and every other configuration keeps its bits (kernels that invert the
matrices of several walkers in one workgroup share its LDS)."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Q():
    import rust_qmc_amd

    return rust_qmc_amd


def _no_jastrow(Q, s):
    d = json.loads(s.to_json())
    d["jastrow"] = {"kind": "none"}
    return Q.System.from_json(json.dumps(d))


def _configs(s, W):
    d = json.loads(s.to_json())
    return np.array(d["nuclei"])[d["init_nuc"]] + 0.7 * np.random.default_rng(W).normal(size=(W, s.n_elec, 3))


@pytest.mark.parametrize("electron", [0, 1, -1])
@pytest.mark.parametrize("name", ["li", "ch4-sto3g", "ch4-631g", "benzene"])
def test_evaluate_and_derivatives(Q, name, electron):
    s = _no_jastrow(Q, {"li": lambda: Q.Lithium(0),
                        "ch4-sto3g": lambda: Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0), "ch4-631g": lambda: Q.MethaneGTO(),
                        "benzene": lambda: Q.BenzeneGTO()}[name]())
    pos, bad = _configs(s, 19), 4
    ref, dref = s.evaluate_batch(pos), s.derivatives_batch(pos)
    pos[bad, electron, 1] = np.nan
    out, dout = s.evaluate_batch(pos), s.derivatives_batch(pos)
    assert np.isnan(out["logabs"][bad]) and np.isnan(out["eloc"][bad]) and np.isnan(dout["eloc"][bad])
    rest = np.arange(19) != bad
    for a, b in ((out, ref), (dout, dref)):
        for k in b:
            assert np.array_equal(a[k][rest], b[k][rest]), k


@pytest.mark.parametrize("electron", [0, 16, 41])
def test_benzene_ensemble_build(Q, electron):
    """The FP64 ensemble's matrices are inverted 16 walkers per workgroup."""
    s = _no_jastrow(Q, Q.BenzeneGTO())
    pos, bad = _configs(s, 35), 18
    ens = Q.Ensemble(s, 35, 1)
    ens.set_positions(pos)
    ref = ens.state()
    tref = ens.sweeps(2, 0.2, trace=True)[3]
    pos[bad, electron, 2] = np.nan
    ens = Q.Ensemble(s, 35, 1)
    ens.set_positions(pos)
    out = ens.state()
    tout = ens.sweeps(2, 0.2, trace=True)[3]
    assert np.isnan(out[0][bad]) and np.isnan(out[2][bad])
    rest = np.arange(35) != bad
    for a, b in zip(out, ref):
        assert np.array_equal(a[rest], b[rest])
    assert np.array_equal(tout[:, rest], tref[:, rest])
