"""Pair-list rebuilds on every path of their scans (needs a GPU): the other
side in one LDS tile, in the LDS grid, or in several tiles, and rows that are
copied from their slab or scanned again because they outgrow it."""
import numpy as np
import pytest

from conftest import read_pos
from test_gpu_parity import oracle_edges_at

import upside_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ue():
    import upside_engine
    upside_engine.load_upside_library()
    return upside_engine


@pytest.mark.parametrize("n_res,nodes", [
    (2, ["rotamer", "environment_coverage_sc"]),                       # one tile, shorter than a lane group
    (100, ["rotamer", "hbond_coverage", "environment_coverage_sc"]),   # one tile
    (600, ["rotamer", "hbond_coverage", "environment_coverage_hb"]),   # grid
    (3000, ["environment_coverage_sc"])])                              # more than one tile
def test_scan_paths(ue, chain_file, monkeypatch, n_res, nodes):
    """Edge sets equal the oracle's at the engine's own coordinates, and
    derivatives do not depend on the capacities (small ones have rows longer
    than their slab)."""
    path = chain_file(n_res, 5)
    pos = read_pos(path)
    ora = O.Engine(path)
    got = []
    for scale in ("0.25", "4"):
        monkeypatch.setenv("UPSIDE_CAPACITY_SCALE", scale)
        e = ue.Upside(path, quiet=True)
        got.append(e.deriv(pos))
        for name in nodes:
            assert set(map(tuple, e.edge_pairs(name))) == oracle_edges_at(e, ora, name), (scale, name)
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("n_res,grid", [(1706, True), (1742, True), (1760, False)])
def test_grid_sizes(ue, tmp_path, n_res, grid):
    """Points that the LDS grid holds: with all its buckets, with half of them,
    and more than it holds.  The one pair graph of these files is the
    environment coverage; its edges equal the oracle's either way."""
    import upconfig
    rng = np.random.default_rng(5)
    seq = upconfig.random_sequence(n_res, rng)
    g = upconfig.build_ff21(seq, upconfig.random_initial_config(n_res, rng))
    keep = ["Dihedral_phi", "Dihedral_psi", "rama_coord", "affine_alignment", "placement_fixed_point_vector_only",
            "placement_scalar", "weighted_pos", "placement_fixed_point_vector_only_CB", "environment_coverage_sc"]
    kept = lambda p: not p.startswith("/input/potential/") or p.split("/")[3] in keep
    n_point = len(g.dsets["/input/potential/environment_coverage_sc/id2"])
    assert {1706: 7100, 1742: 7200, 1760: 7320}[n_res] < n_point < {1706: 7168, 1742: 7321, 1760: 7500}[n_res]
    g.order = [p for p in g.order if kept(p)]
    g.dsets = {p: a for p, a in g.dsets.items() if kept(p)}
    path = str(tmp_path / "coverage.up")
    upconfig.write_up(path, g)
    b = ue.Batch([path], [0.85], seed=1)
    b.enable_profile()
    b.energies()
    line = [x for x in b.profile_report(0).splitlines() if "LDS grid builds" in x]
    assert (float(line[0].split()[-2]) > 0) == grid, line
    e, ora = ue.Upside(path, quiet=True), O.Engine(path)
    e.deriv(read_pos(path))
    name = "environment_coverage_sc"
    assert set(map(tuple, e.edge_pairs(name))) == oracle_edges_at(e, ora, name)
