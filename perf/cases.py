"""What the engine is timed on: the calls a user's program makes, over the sizes it makes them at.

  evaluate    Upside.deriv and Upside.energy of separate conformations (scoring
              decoys, force calls from Python): one chain, the conformations
              far apart, so every one needs its pair lists anew.
  gradient    the training step of a force field: the forces of a conformation
              and the energy's derivatives by the parameters.
  dynamics    Batch.run of one chain from where the last call left it, then the
              positions and momenta back.
  exchange    replicas of one chain with replica exchange inside the run.
  batch       independent chains of uneven length in one launch.
  train, fit  the belief propagation warm-start network: Adam steps on batches
              of rows, and loss and gradient over all rows.

`solve` of a dynamics case picks the stopping rule of the rotamer solve: the
reference's (0), plain start to a tight residual (1), or warm start to a tight
residual (2).

The chains are seeded random sequences (upconfig.make_chain).  Their .up files
depend on length and number alone and are written once per process; the seed
of a state gives its positions, momenta and thermostat stream, or its rows.
"""
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "upside2-md_amd"))
import upconfig  # noqa: E402
import upside_engine  # noqa: E402

DT = 0.009
TEMP = 0.85
N_CONF = 4          # conformations of an evaluate pass
RELAX_ROUNDS = 10   # rounds run before a dynamics state is handed over
N_PARAM_ROTAMER = (20, 20, 54)

_dir = None
_files = {}


def listed():
    return [
        # a peptide the size of chignolin: launches, copies and synchronisations
        dict(name="evaluate 10", kind="evaluate", n_res=10),
        dict(name="evaluate 101", kind="evaluate", n_res=101),
        dict(name="evaluate 500", kind="evaluate", n_res=500),
        # contrastive-divergence training on a protein of ordinary size
        dict(name="gradient 210", kind="gradient", n_res=210),
        # a small protein alone on the GPU, an odd length
        dict(name="dynamics 67", kind="dynamics", n_res=67, rounds=20, solve=0),
        # the repository's headline chain, and the largest it is tested at
        dict(name="dynamics 500", kind="dynamics", n_res=500, rounds=10, solve=0),
        dict(name="dynamics 1000", kind="dynamics", n_res=1000, rounds=6, solve=0),
        # tight solves from the warm start
        dict(name="dynamics 300 warm", kind="dynamics", n_res=300, rounds=10, solve=2),
        # 16 temperatures, neighbours swapped every 7 rounds
        dict(name="exchange 16x150", kind="exchange", n_res=150, n_sys=16, rounds=14),
        # 64 runs of 16 chains between 50 and 400 residues
        dict(name="batch 64", kind="batch", n_min=50, n_max=400, n_chain=16, n_sys=64, rounds=6),
        # training of the warm-start network at its usual batch, and over all rows
        dict(name="train 4096", kind="train", rows=20000, batch=4096, steps=50),
        dict(name="fit 97801", kind="fit", rows=97801),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["evaluate", "evaluate", "gradient", "dynamics", "dynamics", "dynamics", "exchange", "batch",
                       "train", "fit"])
    if kind == "evaluate":
        return dict(kind=kind, n_res=_log_int(rng, 10, 500))
    if kind == "gradient":
        return dict(kind=kind, n_res=_log_int(rng, 20, 400))
    if kind == "dynamics":
        n = _log_int(rng, 30, 1000)
        return dict(kind=kind, n_res=n, rounds=rng.randint(3, 6 if n > 500 else 12), solve=rng.choice([0, 0, 1, 2]))
    if kind == "exchange":
        return dict(kind=kind, n_res=_log_int(rng, 30, 150), n_sys=rng.randint(4, 16), rounds=rng.randint(8, 14))
    if kind == "batch":
        lo = rng.randint(20, 120)
        return dict(kind=kind, n_min=lo, n_max=rng.randint(lo + 20, 400), n_chain=rng.randint(3, 12),
                    n_sys=rng.randint(12, 64), rounds=rng.randint(2, 5))
    if kind == "train":
        rows = _log_int(rng, 600, 20000)
        return dict(kind=kind, rows=rows, batch=min(rows, _log_int(rng, 100, 4096)), steps=rng.randint(5, 50))
    return dict(kind=kind, rows=_log_int(rng, 50, 97801))


# ------------------------------------------------------------------- inputs
def _up(n_res, k=0):
    """The .up file of the k-th chain of n_res residues, written on first use."""
    global _dir
    if _dir is None:
        _dir = tempfile.TemporaryDirectory(prefix="upside_cases_")
    if (n_res, k) not in _files:
        path = os.path.join(_dir.name, "chain%d_%d.up" % (n_res, k))
        upconfig.make_chain(path, n_res, seed=1000 * k + n_res)
        _files[n_res, k] = path
    return _files[n_res, k]


def _conformation(n_res, rng):
    return np.ascontiguousarray(upconfig.random_initial_config(n_res, rng), np.float32)


def _lengths(case):
    """Chain lengths of a batch case, evenly over [n_min, n_max], in mixed order."""
    n = np.linspace(case["n_min"], case["n_max"], case["n_chain"]).round().astype(int)
    return [int(x) for x in np.random.default_rng(7).permutation(n)]


def _rows(n, seed):
    """Training rows of the warm-start network as a first belief propagation
    pass gives them: max-normalised log probabilities, first beliefs and
    previous marginals of 3- or 6-state residues, the mask, degree, entropy and
    flags; the targets are the marginals the solve ends at."""
    rng = np.random.default_rng(seed)
    six = rng.random(n) < 0.4
    ok = np.arange(6)[None, :] < np.where(six, 6, 3)[:, None]

    def logs(z):
        z = np.where(ok, z, -np.inf)
        return np.where(ok, np.maximum(z - z.max(1, keepdims=True), -30.0), 0.0)

    z = rng.normal(0.0, 2.0, (n, 6))
    first = z + rng.normal(0.0, 0.7, (n, 6))
    last = first + 0.3 * rng.normal(0.0, 1.0, (n, 6)) - 0.1 * z
    f = np.zeros((n, 32), np.float32)
    f[:, 0:6], f[:, 6:12], f[:, 12:18] = logs(z), logs(first), logs(last + rng.normal(0.0, 0.1, (n, 6)))
    f[:, 18:24] = ok
    p = np.exp(logs(first)) * ok
    s = p.sum(1)
    f[:, 24] = rng.integers(0, 20, n) / 8.0
    f[:, 25] = six
    f[:, 26] = np.log(s) - (p * logs(first)).sum(1) / s
    f[:, 27] = 1.0 - 1.0 / s
    f[:, 28] = 1.0
    t = np.exp(logs(last)) * ok
    target = np.zeros((n, 8), np.float32)
    target[:, :6] = t / t.sum(1, keepdims=True)
    return f, target


def _params(seed):
    """Parameters of a network in training: He-normal hidden layers, a small output layer."""
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.normal(size=128 * 32) * np.sqrt(2 / 32), rng.normal(size=128) * 0.05,
                           rng.normal(size=128 * 128) * np.sqrt(2 / 128), rng.normal(size=128) * 0.05,
                           rng.normal(size=16 * 128) * 0.02, np.zeros(16)]).astype(np.float32)


def _tuned(batch, teams):
    """As a program does before a long run: settle, then let the engine choose its layout."""
    batch.run(RELAX_ROUNDS)
    batch.autotune_layout(3, teams, (0, 1, 3))
    return batch


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind in ("evaluate", "gradient"):
        n = case["n_res"]
        eng = upside_engine.Upside(_up(n), quiet=True)
        count = N_CONF if kind == "evaluate" else 1
        return dict(case=case, eng=eng, pos=[_conformation(n, rng) for _ in range(count)])
    if kind in ("train", "fit"):
        net = upside_engine.WarmStartNet(seed=1)
        net.set_params(_params(seed))
        net.set_data(*_rows(case["rows"], seed))
        return dict(case=case, net=net)
    if kind == "dynamics":
        b = upside_engine.Batch([_up(case["n_res"])], [TEMP], seed=seed % (1 << 31), dt=DT)
        b.set_pos(0, _conformation(case["n_res"], rng))
        if case["solve"] == 2:
            b.set_warm_start(_params(seed))
        b.set_bp_schedule(case["solve"])
        _tuned(b, (8, 16, 32))
    elif kind == "exchange":
        m = case["n_sys"]
        temps = [0.80 * (0.95 / 0.80) ** (i / (m - 1.0)) for i in range(m)]
        b = upside_engine.Batch([_up(case["n_res"])] * m, temps, seed=seed % (1 << 31), dt=DT)
        start = _conformation(case["n_res"], rng)
        for s in range(m):
            b.set_pos(s, start)
        _tuned(b, (b.max_team() // 2, b.max_team()))
        b.set_replica_exchange(7, [[(i, i + 1) for i in range(0, m - 1, 2)], [(i, i + 1) for i in range(1, m - 1, 2)]])
    else:
        n_res = _lengths(case)
        which = [s % len(n_res) for s in range(case["n_sys"])]
        b = upside_engine.Batch([_up(n_res[k], k) for k in which], [TEMP] * len(which), seed=seed % (1 << 31), dt=DT)
        for s, k in enumerate(which):
            b.set_pos(s, _conformation(n_res[k], rng))
        _tuned(b, (2, 0))
    return dict(case=case, batch=b)


# --------------------------------------------------------------------- runs
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "evaluate":
        eng = state["eng"]
        deriv = [eng.deriv(p) for p in state["pos"]]
        return dict(deriv=deriv, energy=[float(eng.energy(p)) for p in state["pos"]])
    if kind == "gradient":
        eng = state["eng"]
        out = dict(deriv=eng.deriv(state["pos"][0]))
        out["rotamer"] = eng.get_param_deriv(N_PARAM_ROTAMER, "rotamer")
        out["coverage"] = eng.get_param_deriv((8, 20, 50), "hbond_coverage")
        out["hydrophobe"] = eng.get_param_deriv((12, 20, 50), "hbond_coverage_hydrophobe")
        out["environment"] = eng.get_param_deriv((3 * 20 + 400,), "sigmoid_coupling_environment")
        out["hbond"] = eng.get_param_deriv((12,), "hbond_energy")
        return out
    if kind == "train":
        losses = state["net"].train(case["steps"], case["batch"])
        return dict(losses=losses, params=state["net"].params())
    if kind == "fit":
        loss, grad = state["net"].loss_grad()
        return dict(loss=loss, grad=grad)
    b = state["batch"]
    if kind == "exchange":
        b.run_logged(case["rounds"], 0)
    else:
        b.run(case["rounds"])
    out = dict(pos=np.concatenate([b.pos(s) for s in range(b.n_sys)]),
               mom=np.concatenate([b.mom(s) for s in range(b.n_sys)]))
    if kind == "exchange":
        out["replica"] = b.replica_stats()[0].astype(np.int64)
    return out


# --------------------------------------------------------------------- work
# A force evaluation per residue, counted on relaxed random chains: about 25
# rotamer and 20 coverage spline edges (250 operations), 60 environment and 15
# backbone or hydrogen-bond edges (60), and 16 belief propagation passes over
# 3 residue pairs (2 * 36 multiply-adds and 12 renormalisations each way).
FLOPS_PER_RESIDUE = 45 * 250 + 75 * 60 + 16 * 3 * 300
# Positions in and derivatives out.
EVAL_BYTES_PER_RESIDUE = 2 * 3 * 12
# Positions and momenta, in and out.
STATE_BYTES_PER_RESIDUE = 4 * 3 * 12
# The interaction tables (rotamer, coverage), read once.
TABLE_BYTES = 4 * (20 * 20 * 54 + 8 * 20 * 50 + 12 * 20 * 50)
MLP_MACS = 32 * 128 + 128 * 128 + 128 * 16
MLP_PARAMS = MLP_MACS + 128 + 128 + 16


def work(case):
    kind = case["kind"]
    if kind in ("evaluate", "gradient"):
        n = case["n_res"]
        evals = 2 * N_CONF if kind == "evaluate" else 1
        grad = TABLE_BYTES if kind == "gradient" else 0
        return dict(bytes=evals * n * EVAL_BYTES_PER_RESIDUE + TABLE_BYTES + grad, flops=evals * n * FLOPS_PER_RESIDUE)
    if kind in ("train", "fit"):
        rows = case["batch"] * case["steps"] if kind == "train" else case["rows"]
        steps = case["steps"] if kind == "train" else 1
        # forward, gradient of the activations, gradient of the weights; Adam's three vectors in and out
        per_step = MLP_PARAMS * 4 * (6 if kind == "train" else 2)
        return dict(bytes=rows * 40 * 4 + steps * per_step, flops=6 * rows * MLP_MACS)
    if kind == "batch":
        n_res = _lengths(case)
        total = sum(n_res[s % len(n_res)] for s in range(case["n_sys"]))
    else:
        total = case["n_res"] * case.get("n_sys", 1)
    return dict(bytes=total * STATE_BYTES_PER_RESIDUE + TABLE_BYTES, flops=3 * case["rounds"] * total * FLOPS_PER_RESIDUE)


# -------------------------------------------------------------------- exact
def _forward64(p, x):
    """The network in 64 bits: 32 -> 128 -> 128 -> 16, ReLU; p is the flat parameter vector."""
    shapes = [(128, 32), (128,), (128, 128), (128,), (16, 128), (16,)]
    parts, at = [], 0
    for s in shapes:
        n = int(np.prod(s))
        parts.append(p[at:at + n].reshape(s))
        at += n
    w1, b1, w2, b2, w3, b3 = parts
    return torch.relu(torch.relu(x @ w1.T + b1) @ w2.T + b2) @ w3.T + b3


def _loss64(p, feat, target):
    """Mean over rows of -sum_r t_r log softmax(first log beliefs + output) over the row's states."""
    z = feat[:, 6:12] + _forward64(p, feat)[:, :6]
    logp = torch.log_softmax(z.masked_fill(feat[:, 18:24] < 0.5, -float("inf")), 1)
    return -(target[:, :6] * logp.masked_fill(feat[:, 18:24] < 0.5, 0.0)).sum(1).mean()


def exact(case, seed):
    """The network's loss and gradient in 64 bits.  Forces and energies have no
    64-bit value to compare with: they depend on where the reference's rule
    stops the loopy belief propagation and the residue frames' eigen-iteration
    (1e-4 of the forces); a training run of Adam steps takes the sign of
    gradients near zero."""
    if case["kind"] != "fit":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    feat, target = (torch.from_numpy(a).to(dev, torch.float64) for a in _rows(case["rows"], seed))
    p = torch.from_numpy(_params(seed)).to(dev, torch.float64).requires_grad_(True)
    loss = _loss64(p, feat, target)
    loss.backward()
    return dict(loss=float(loss), grad=p.grad.cpu().numpy())
