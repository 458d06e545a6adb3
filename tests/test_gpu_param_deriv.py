"""Parameter derivatives against the float64 oracle at the engine's own
coordinates and sensitivities (needs a GPU): central differences of the
oracle's edge values and node potentials, which are smooth in the parameters.
Bar: 1e-4 of the norm, as against the compiled reference (a float32 sum over
the edges of a type pair, or over the residues)."""
import numpy as np
import pytest

from conftest import read_pos

import upside_oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-4


@pytest.fixture(scope="module")
def ue():
    import upside_engine
    upside_engine.load_upside_library()
    return upside_engine


def engines(ue, path, n_res):
    pos0 = read_pos(path)
    pos = (pos0 + np.random.default_rng(n_res).normal(scale=0.1, size=pos0.shape)).astype(np.float32)
    eng = ue.Upside(path, quiet=True)
    eng.deriv(pos)
    return eng, O.Engine(path, dtype=np.float64)


@pytest.mark.parametrize("n_res", [2, 31, 64, 211])
@pytest.mark.parametrize("name", ["hbond_coverage", "hbond_coverage_hydrophobe"])
def test_coverage_param_deriv(ue, chain_file, name, n_res):
    """Rows of no edge, of a few and of many, and row counts off a multiple of
    the workgroup."""
    eng, ora = engines(ue, chain_file(n_res, 9), n_res)
    node = ora.nodes[name]
    ig = node.ig
    for n in (ig.node1, ig.node2):
        n.output[:] = eng.get_output(n.name)
    ig.edges()
    p = ig.params_of_edges()
    row = ig.type1[ig.i1] * ig.n_type2 + ig.type2[ig.i2]
    shape = (ig.param.shape[0], ig.n_param)
    sens = eng.get_sens(name)[:, 0].astype(np.float64)
    on = ig.i1 if len(sens) == len(ig.loc1) else ig.i2
    want = np.zeros(shape)
    h = 1e-4
    for k in range(ig.n_param):
        if not len(row):
            break
        hi, lo = p.copy(), p.copy()
        hi[:, k] += h
        lo[:, k] -= h
        dv = (ig.it.compute(hi, ig.x1, ig.x2)[0] - ig.it.compute(lo, ig.x1, ig.x2)[0]) / (2 * h)
        np.add.at(want[:, k], row, sens[on] * dv)
    got = eng.get_param_deriv(shape, name).astype(np.float64)
    assert np.linalg.norm(got - want) <= TOL * max(np.linalg.norm(want), 1e-6)
    assert n_res < 31 or np.linalg.norm(want) > 0


@pytest.mark.parametrize("n_res", [2, 63, 65, 300])
@pytest.mark.parametrize("name", ["sigmoid_coupling_environment", "bb_sigmoid_coupling_environment", "hbond_energy"])
def test_coupling_param_deriv(ue, chain_file, name, n_res):
    """Fewer residues than a wave, one more than a wave, and several workgroups."""
    eng, ora = engines(ue, chain_file(n_res, 10), n_res)
    node = ora.nodes[name]
    for a in node.args:
        ora.nodes[a].output[:] = eng.get_output(a)
    if name == "hbond_energy":
        node.params = node.params.astype(np.float64)
        parts, zeros = [(node, "params", 4)], 8   # the energies; no derivative of the shapes (src/hbond.cpp:655-720)
    elif name.startswith("bb"):
        parts, zeros = [(node, "scale", 0)], 3    # of the scale alone (src/environment.cpp:1054-1138)
    else:
        parts, zeros = [(node, k, len(getattr(node, k))) for k in ("scale", "center", "sharp")], 0
    want = []
    h = 1e-5

    def potential():
        node.compute(0)
        return float(node.potential)

    for obj, attr, n in parts:
        base = getattr(obj, attr)
        for k in range(max(n, 1)):
            e = []
            for s in (h, -h):
                v = np.array(base, np.float64)
                v[k if n else ()] += s
                setattr(obj, attr, v)
                e.append(potential())
            want.append((e[0] - e[1]) / (2 * h))
        setattr(obj, attr, base)
    if name == "sigmoid_coupling_environment":
        # 20 independent weights (the file's number_independent_weights): a
        # weight is shared by all types, each of which reports its derivative
        base, col = node.w, np.zeros(node.nt)
        for k in range(node.nt):
            e = []
            for s in (h, -h):
                v = base.astype(np.float64).reshape(node.nt, node.nt)
                v[:, k] += s
                node.w = v.ravel()
                e.append(potential())
            col[k] = (e[0] - e[1]) / (2 * h)
        node.w = base
        want += list(np.tile(col, node.nt))
    want = np.array(want + [0.0] * zeros)
    got = eng.get_param_deriv(want.shape, name).astype(np.float64)
    assert np.linalg.norm(got - want) <= TOL * max(np.linalg.norm(want), 1e-6)
