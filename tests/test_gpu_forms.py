"""The kernels AUTO takes for few walkers and for benzene against the general
engine of the same system, over the forms of a description that reach them:
every kind of Jastrow factor and its flags, MOs that differ between the spins,
spins in any order.  Evaluations, derivatives, moments and all three kinds of
move, FP64 in another order: the engines' 1e-9 of each output's scale."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def Q():
    import rust_qmc_amd

    return rust_qmc_amd


def _form(d, form):
    rng = np.random.default_rng(3)
    if form in ("no jastrow", "pair", "pair with quirks", "pade"):
        d["jastrow"] = {"no jastrow": {"kind": "none"},
                        "pade": {"kind": "pade", "b_ee": 1.3, "b_en": 0.9, "a_anti": 0.45, "a_para": 0.3}}.get(
                            form, {"kind": "pair", "F": 1.7})
    if form in ("pair with quirks", "no flags"):
        d["flags"] = 15 if form == "pair with quirks" else 0
    if form == "spin-dependent MOs":
        d.pop("mo_rule", None)
        d["mo_dn"] = (np.array(d["mo_dn"]) + 0.05 * rng.normal(size=np.shape(d["mo_dn"]))).tolist()
    if form == "shuffled spins":
        d["spins"] = rng.permutation(d["spins"]).tolist()
    return d


@pytest.mark.parametrize("form", ["as built", "no jastrow", "pair", "pair with quirks", "pade", "no flags",
                                  "spin-dependent MOs", "shuffled spins"])
@pytest.mark.parametrize("name", ["h2", "li", "li-ref", "ch4-sto3g", "ch4-631g", "benzene"])
def test_auto_matches_the_general_engine(Q, name, form):
    base = {"h2": lambda: Q.H2MoleculeMO(), "li": lambda: Q.Lithium(0), "li-ref": lambda: Q.Lithium(),
            "ch4-sto3g": lambda: Q.MethaneGTO(1.5, 2.0, 2.06, "STO-3G", 0), "ch4-631g": lambda: Q.MethaneGTO(),
            "benzene": lambda: Q.BenzeneGTO()}[name]()
    d = _form(json.loads(base.to_json()), form)
    n = len(d["spins"])
    pos = np.array(d["nuclei"])[d["init_nuc"]] + 0.6 * np.random.default_rng(5).normal(size=(13, n, 3))
    res = []
    for engine in ("auto", "wave" if name == "benzene" else "register"):
        s = Q.System.from_json(json.dumps(d))
        s.set_engine(engine)
        r = {"evaluate " + k: v for k, v in s.evaluate_batch(pos).items()}
        r.update({"derivatives " + k: v for k, v in s.derivatives_batch(pos).items()})
        for move, step in ((Q.QMC_MOVE_SINGLE, 0.25), (Q.QMC_MOVE_DRIFT, 0.01), (Q.QMC_MOVE_ALL, 0.05)):
            ens = Q.Ensemble(s, 13, 4)
            ens.set_positions(pos)
            acc, tr = ens.sweeps(3, step, move, refresh_interval=2, trace=True)[2:]
            la, sg, _ = ens.state()
            for k, v in dict(accepted=acc, trace=tr, positions=ens.positions(), logabs=la, sign=sg).items():
                r[f"move {move} {k}"] = v
        ens.measure(reset=True)
        m = ens.moments()
        r.update({"moments " + k: m[k] for k in ("o_mean", "S", "f", "f_hf", "f_zv")})
        res.append(r)
    for k, b in res[1].items():
        if np.size(b):
            assert np.abs(res[0][k] - b).max() <= 1e-9 * max(1.0, np.abs(b).max()), k
