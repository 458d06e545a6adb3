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


@pytest.mark.parametrize("n_res", [25, 26, 55, 56, 125, 126])
def test_evaluation_on_a_team(ue, chain_file, monkeypatch, n_res):
    """Evaluations of a one-system engine, on both sides of each line of the
    rule for its team, against one workgroup."""
    import upconfig
    path = chain_file(n_res, 11)
    rng = np.random.default_rng(n_res)
    a = ue.Upside(path, quiet=True)
    monkeypatch.setenv("UPSIDE_TEAM", "1")
    b = ue.Upside(path, quiet=True)
    for _ in range(3):
        pos = np.ascontiguousarray(upconfig.random_initial_config(n_res, rng), np.float32)
        np.testing.assert_allclose(a.energy(pos), b.energy(pos), rtol=1e-5)
        np.testing.assert_array_equal(a.deriv(pos), b.deriv(pos))
        np.testing.assert_allclose(a.get_output("rotamer"), b.get_output("rotamer"), rtol=1e-5)
        for node in ("placement_fixed_point_vector_only", "hbond_coverage"):
            np.testing.assert_array_equal(a.get_output(node), b.get_output(node))
            np.testing.assert_array_equal(a.get_sens(node), b.get_sens(node))


@pytest.mark.parametrize("n_res,team", [(2, 16), (150, 15), (150, 16), (165, 16), (180, 32),
                                        (256, 16), (257, 16)])
def test_rotamer_solve_by_edges(ue, chain_file, n_res, team):
    """The default layout of the rotamer solve around the number of edges where
    it changes from one workgroup to several, and around the number of nodes
    that half the team can keep in registers."""
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


def test_evaluations_in_threads(ue, chain_file):
    """Engines of several threads, each with its own stream, whose teams ask
    for the same workgroup slots."""
    import threading

    import upconfig
    path = chain_file(126, 11)
    rng = np.random.default_rng(7)
    pos = [np.ascontiguousarray(upconfig.random_initial_config(126, rng), np.float32) for _ in range(4)]
    ref = ue.Upside(path, quiet=True)
    want = [ref.deriv(p) for p in pos]
    engines = [ue.Upside(path, quiet=True) for _ in range(4)]
    bad = []

    def work(k):
        for i in range(20):
            p = (i + k) % 4
            if not np.array_equal(engines[k].deriv(pos[p]), want[p]):
                bad.append((k, i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("n_res", [26, 126])
@pytest.mark.parametrize("spins", [0, 2, 4, 8, 30])
def test_evaluation_whose_team_cannot_meet(ue, chain_file, monkeypatch, capfd, n_res, spins):
    """Barriers that give up after a few polls (0: at the first workgroup that
    is not there yet; more: somewhere in the evaluation, or not at all): every
    workgroup leaves, and the evaluation is repeated on one.  Same bits."""
    import upconfig
    path = chain_file(n_res, 11)
    rng = np.random.default_rng(n_res)
    pos = [np.ascontiguousarray(upconfig.random_initial_config(n_res, rng), np.float32) for _ in range(4)]
    with monkeypatch.context() as m:
        m.setenv("UPSIDE_TEAM", "1")
        one = ue.Upside(path, quiet=True)
    with monkeypatch.context() as m:
        m.setenv("UPSIDE_BARRIER_SPINS", str(spins))
        eng = ue.Upside(path, quiet=True)
    want = [(one.deriv(p), one.energy(p)) for p in pos]
    capfd.readouterr()
    # 64 evaluations on one workgroup, then the team's second try
    for k in range(68 if spins == 0 else 4):
        d, e = want[k % 4]
        np.testing.assert_array_equal(eng.deriv(pos[k % 4]), d)
        if k < 4:
            np.testing.assert_allclose(eng.energy(pos[k]), e, rtol=1e-5)
    said = capfd.readouterr().err
    if spins == 0:
        assert "the next 64 evaluations" in said and "the next 128 evaluations" in said


@pytest.mark.parametrize("spins", [0, 8])
def test_run_whose_team_cannot_meet(ue, chain_file, monkeypatch, spins):
    """A run on such teams is an error, or (enough polls) the run; after the
    error the batch evaluates and runs like a new one."""
    path = chain_file(56, 11)
    monkeypatch.setenv("UPSIDE_BARRIER_SPINS", str(spins))
    b = ue.Batch([path], [0.85], seed=4)
    if b.max_team() < 8:
        pytest.skip("no team of this size fits")
    start = b.pos(0), b.mom(0)
    b.set_team(8)
    try:
        b.run(4)
        assert spins > 0
    except RuntimeError:
        pass
    b.set_team(1)
    b.set_pos(0, start[0])
    b.set_mom(0, start[1])
    new = ue.Batch([path], [0.85], seed=4)
    np.testing.assert_array_equal(b.energies(), new.energies())
    np.testing.assert_array_equal(b.deriv(0), new.deriv(0))


def test_exchange_whose_systems_cannot_meet(ue, chain_file, monkeypatch):
    """The same for the barrier of all systems around a replica exchange."""
    path = chain_file(30, 11)
    monkeypatch.setenv("UPSIDE_BARRIER_SPINS", "0")
    temps = [0.8, 0.85, 0.9, 0.95]
    b = ue.Batch([path] * 4, temps, seed=4)
    start = [b.pos(s) for s in range(4)]
    b.set_replica_exchange(2, [[(0, 1), (2, 3)], [(1, 2)]])
    with pytest.raises(RuntimeError):
        b.run_logged(6, 0)
    for s in range(4):
        b.set_pos(s, start[s])
    np.testing.assert_array_equal(b.energies(), ue.Batch([path] * 4, temps, seed=4).energies())


def test_every_evaluation_in_threads(ue, chain_file):
    """As test_evaluations_in_threads, where an evaluation that fails is a
    failure too: all of them are counted."""
    import concurrent.futures

    import upconfig
    path = chain_file(126, 11)
    rng = np.random.default_rng(8)
    pos = [np.ascontiguousarray(upconfig.random_initial_config(126, rng), np.float32) for _ in range(4)]
    ref = ue.Upside(path, quiet=True)
    want = [ref.deriv(p) for p in pos]
    engines = [ue.Upside(path, quiet=True) for _ in range(4)]

    def work(k):
        for i in range(20):
            np.testing.assert_array_equal(engines[k].deriv(pos[(i + k) % 4]), want[(i + k) % 4])
        return 20

    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        assert sum(f.result() for f in [pool.submit(work, k) for k in range(4)]) == 80


@pytest.mark.parametrize("n_res", [199, 200])
def test_evaluation_without_a_rotamer_solve(ue, tmp_path, monkeypatch, n_res):
    """Pair lists but no rotamer node, on both sides of the rule's line for them."""
    import upconfig
    rng = np.random.default_rng(n_res)
    seq = upconfig.random_sequence(n_res, rng)
    g = upconfig.build_ff21(seq, upconfig.random_initial_config(n_res, rng))
    keep = ["Distance3D", "Spring_bond", "Angle", "Spring_angle", "Dihedral_omega", "Spring_omega", "rama_map_pot",
            "rama_map_pot_ref", "backbone_pairs", "infer_H_O", "protein_hbond", "hbond_energy", "Dihedral_phi",
            "Dihedral_psi", "rama_coord", "affine_alignment"]
    kept = lambda p: not p.startswith("/input/potential/") or p.split("/")[3] in keep
    g.order = [p for p in g.order if kept(p)]
    g.dsets = {p: a for p, a in g.dsets.items() if kept(p)}
    path = str(tmp_path / "backbone.up")
    upconfig.write_up(path, g)
    a = ue.Upside(path, quiet=True)
    monkeypatch.setenv("UPSIDE_TEAM", "1")
    b = ue.Upside(path, quiet=True)
    for _ in range(3):
        pos = np.ascontiguousarray(upconfig.random_initial_config(n_res, rng), np.float32)
        np.testing.assert_allclose(a.energy(pos), b.energy(pos), rtol=1e-5)
        np.testing.assert_array_equal(a.deriv(pos), b.deriv(pos))
        np.testing.assert_array_equal(a.get_output("protein_hbond"), b.get_output("protein_hbond"))
