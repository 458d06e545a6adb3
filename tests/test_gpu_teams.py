"""Rules that choose how many workgroups work on a system (needs a GPU).

Every choice computes the same arithmetic in the same order, so comparisons
are bit for bit, but for energies: a sum over all threads depends on how many
there are (float32, 1e-5 as for every other comparison of teams)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ue():
    import upside_engine
    upside_engine.load_upside_library()
    return upside_engine


@pytest.mark.parametrize("n_res,team", [(2, 16), (150, 15), (150, 16), (165, 16), (180, 32)])
def test_rotamer_solve_by_edges(ue, chain_file, n_res, team):
    """The default layout of the rotamer solve around the number of edges where
    it changes from one workgroup to several."""
    path = chain_file(n_res, 12)
    b1 = ue.Batch([path], [0.85], seed=6)
    b1.run(3)
    bt = ue.Batch([path], [0.85], seed=6)
    if bt.max_team() < team:
        pytest.skip("no team of this size fits")
    bt.set_team(team)
    bt.run(3)
    assert b1.bp_stats(0)["total"] == bt.bp_stats(0)["total"]
    np.testing.assert_array_equal(bt.pos(0), b1.pos(0))
    np.testing.assert_array_equal(bt.mom(0), b1.mom(0))
