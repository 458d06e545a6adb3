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
