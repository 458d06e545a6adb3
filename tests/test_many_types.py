"""Environment coverage with the most residue types that a file may have: the
bins of all lanes then take more than the LDS staging area."""
import ctypes as ct
import os

import numpy as np
import pytest

from conftest import PKG

N_TYPE = 79


def chain(path, n_res, n_type):
    """A chain whose residue types are moved to the last 20 of n_type types."""
    import upconfig
    rng = np.random.default_rng(3)
    seq = upconfig.random_sequence(n_res, rng)
    g = upconfig.build_ff21(seq, upconfig.random_initial_config(n_res, rng))
    cov, coup = "/input/potential/environment_coverage_sc", "/input/potential/sigmoid_coupling_environment"
    first = n_type - 20
    g.groups[cov]["num_aa_types"] = n_type
    g.dsets[cov + "/aa_types"] = g.dsets[cov + "/aa_types"] + first
    w = np.zeros((n_type, n_type), np.float32)
    w[:20, first:] = np.asarray(g.dsets[coup + "/weights"]).reshape(20, 20)
    g.dsets[coup + "/weights"] = w.reshape(-1)
    for name in ("scale", "center", "sharpness"):
        g.dsets["%s/%s" % (coup, name)] = np.concatenate([g.dsets["%s/%s" % (coup, name)], np.ones(first)])
    upconfig.write_up(path, g)
    return path


def test_types_accepted(tmp_path):
    lib = ct.CDLL(os.path.join(PKG, "lib", "libupside.so"))
    buf = ct.create_string_buffer(1024)
    for n, ok in ((N_TYPE, True), (N_TYPE + 1, False)):
        path = chain(str(tmp_path / ("t%d.up" % n)), 20, n)
        assert (lib.upside_check_program(path.encode(), buf, len(buf)) == 0) == ok, buf.value


@pytest.mark.gpu
@pytest.mark.parametrize("n_res,team", [(20, 1), (150, 1), (150, 4)])
def test_many_types_as_twenty(tmp_path, monkeypatch, n_res, team):
    """Same bits as with twenty types: the others only add zeros."""
    import upside_engine as ue
    from conftest import read_pos
    monkeypatch.setenv("UPSIDE_TEAM", str(team))
    path = chain(str(tmp_path / "a.up"), n_res, 20)
    a = ue.Upside(path, quiet=True)
    b = ue.Upside(chain(str(tmp_path / "b.up"), n_res, N_TYPE), quiet=True)
    pos = read_pos(path)
    np.testing.assert_array_equal(a.deriv(pos), b.deriv(pos))
    cov = [e.get_output("environment_coverage_sc").reshape(n_res, -1) for e in (a, b)]
    assert cov[0].any() and not cov[1][:, :N_TYPE - 20].any()
    np.testing.assert_array_equal(cov[0], cov[1][:, N_TYPE - 20:])
