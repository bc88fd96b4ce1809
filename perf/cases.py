"""Workloads of the framework for measuring it: simulations advanced through
``api.Simulation`` and the rate surrogate trained, differentiated and
evaluated through ``surrogate.MLP``.

A case is a dict of plain values; ``prepare`` builds what a program holds
before the call (a network laid out on the device and past its cold start; a
model with its weights and data set), ``run`` is one pass through the public
entry points.  A simulation keeps its state from pass to pass, as a program
that advances it piece by piece does, and returns its neurons' state and its
delivery count; training goes on from the weights that it has.
"""
import math

import numpy as np
import torch

from bsim_amd import api, netspec, surrogate, sweep

DT = 1e-4
SIMS = ("random", "plain", "standard", "sweep")


def listed():
    return [
        # an interactive session: a few dozen neurons of every kind of source,
        # advanced 20 cycles at a time, the fired ids and some membrane traces read back
        dict(name="step_small", kind="random", n_lif=40, n_arr=5, n_bern=3, dmax=5, cycles=20),
        # the plain method's network, 2 x 1,000 neurons joined all to all, 0.1 s with its raster recorded
        dict(name="plain_2x1000", kind="plain", n=1000, cycles=1000),
        # a feed-forward network of a size that nobody rounded
        dict(name="standard_ragged", kind="standard", npop=7, n=1237, fanout=333, dmax=6, refrac=2e-3,
             drive=20.0, cycles=400, preroll=1000, hz=100.0),
        # the standard feed-forward network at ~100 Hz with half of its 64 populations
        dict(name="standard_100hz", kind="standard", npop=32, n=10000, fanout=1000, dmax=6, refrac=2e-3,
             drive=20.0, cycles=200, preroll=1000, hz=100.0),
        # the high-activity network (~2,000 Hz, delays up to 50 steps) with a tenth of its populations
        dict(name="stress_2000hz", kind="standard", npop=10, n=10000, fanout=2200, dmax=50, refrac=0.35e-3,
             drive=20.0, cycles=60, preroll=600, hz=1600.0),
        # a batched sweep: many independent small chains advanced together, at the tile a tuner picks
        dict(name="sweep_96", kind="sweep", nets=96, min_size=100, max_size=1000, tile=384, cycles=400,
             preroll=256, hz=54.0),
        # the surrogate as it is trained for screening: a few steps of an epoch
        dict(name="train_4096", kind="train", n_in=8, hidden=512, layers=4, n_out=200, batch=4096, steps=12),
        # a small surrogate on few rows: every launch is short
        dict(name="train_256", kind="train", n_in=6, hidden=192, layers=2, n_out=37, batch=256, steps=32),
        # the gradient of one batch of a wide model, for a program with its own optimiser
        dict(name="gradients_2048", kind="gradients", n_in=17, hidden=1024, layers=3, n_out=333, batch=2048),
        # a handful of sweep points scored
        dict(name="predict_37", kind="predict", n_in=8, hidden=512, layers=4, n_out=200, rows=37),
        # screening: very many candidates scored in one call
        dict(name="predict_100003", kind="predict", n_in=8, hidden=512, layers=4, n_out=200, rows=100003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("random", "plain", "standard", "standard", "stress", "sweep", "train", "train",
                       "gradients", "predict"))
    if kind == "random":
        return dict(kind="random", n_lif=_log(rng, 10, 200), n_arr=rng.randint(1, 12),
                    n_bern=rng.randint(1, 8), dmax=rng.randint(1, 30), cycles=_log(rng, 1, 63))
    if kind == "plain":
        return dict(kind="plain", n=_log(rng, 100, 1000), cycles=_log(rng, 100, 1000))
    if kind == "standard":
        n = _log(rng, 300, 10000)
        fanout = _log(rng, 50, min(1000, n))
        npop = _log(rng, 2, max(2, min(32, int(3.2e8 / (n * fanout)))))
        return dict(kind="standard", npop=npop, n=n, fanout=fanout, dmax=rng.randint(2, 20), refrac=2e-3,
                    drive=float(rng.randint(5, 50)), cycles=rng.randint(64, 200), preroll=1000, hz=100.0)
    if kind == "stress":
        n = _log(rng, 1000, 9000)
        return dict(kind="standard", npop=rng.randint(3, 9), n=n, fanout=int(0.22 * n),
                    dmax=rng.randint(25, 60), refrac=0.35e-3, drive=20.0, cycles=rng.randint(20, 60),
                    preroll=600, hz=1600.0)
    if kind == "sweep":
        return dict(kind="sweep", nets=_log(rng, 4, 90), min_size=100, max_size=_log(rng, 300, 1000),
                    tile=rng.choice((0, 192, 384, 768)), cycles=rng.randint(64, 400), preroll=256, hz=54.0)
    c = dict(kind=kind, n_in=rng.randint(1, 64), hidden=64 * rng.randint(1, 8), layers=rng.randint(1, 5),
             n_out=_log(rng, 1, 256))
    if kind == "predict":
        c.update(rows=_log(rng, 1, 100000))
    elif kind == "gradients":
        c.update(batch=256 * rng.randint(1, 8))
    else:
        c.update(batch=256 * rng.randint(1, 16), steps=rng.randint(1, 12))
    return c


# ---- the networks ----------------------------------------------------------

def _network(case, seed):
    kind = case["kind"]
    if kind == "random":
        return api.Network.from_spec(netspec.random_net(seed, n_lif=case["n_lif"], n_arr=case["n_arr"],
                                                        n_bern=case["n_bern"], dmax=case["dmax"]))
    if kind == "plain":
        return api.Network.from_spec(netspec.c0(seed, n=case["n"]))
    if kind == "standard":
        stress = case["refrac"] < 1e-3
        # weights scaled so that a neuron's expected input does not depend on the fan-in
        w0 = netspec.C2["w0"] * 2200.0 / case["fanout"] if stress else netspec.C1["w0"] * 1000.0 / case["fanout"]
        return api.Network.standard(npop=case["npop"], n=case["n"], fanout=case["fanout"], w0=w0,
                                    inh_frac=0.2 if stress else 0.25, dmax=case["dmax"], remote_frac=0.2,
                                    drive_rate_hz=case["drive"], n_drive=case["n"], drive_w=1.0,
                                    drive_fanout=min(100, case["fanout"]), seed=seed + 1,
                                    tau_refrac=case["refrac"], i_offset=(14.5, 16.5))
    # the same population sizes whatever the seed, other networks and drives of those sizes
    points = sweep.sample(case["nets"], seed=case["nets"], size=(case["min_size"], case["max_size"]))
    for p, q in zip(points, sweep.sample(case["nets"], seed=seed + 1)):
        p.w0, p.inh_frac, p.drive_rate_hz, p.seed = q.w0, q.inh_frac, q.drive_rate_hz, q.seed
    return sweep.build(points).net


def _prepare_sim(case, seed):
    net = _network(case, seed)
    rec, ids = 0, ()
    if case["kind"] in ("random", "plain"):
        rec = case["cycles"]
        ids = [int(i) for i in np.random.default_rng(seed).integers(0, net.n, 8)]
    sim = api.Simulation(net, DT, tile=case.get("tile", 0), rec_steps=rec, rec_ids=ids)
    if case.get("preroll"):
        sim.step(case["preroll"])       # past the cold start, in the regime that a run spends its time in
        sim.sync()
    return dict(case=case, sim=sim)


def _run_sim(state):
    case, sim = state["case"], state["sim"]
    sim.run(case["cycles"] * DT)
    out = dict(sim.state(), events=sim.events())
    if case["kind"] in ("random", "plain"):
        counts, fired, _ = sim.raster()
        raster = np.zeros((len(counts), sim.n), np.bool_)
        raster[np.repeat(np.arange(len(counts)), counts), fired] = True
        out.update(raster=raster, trace=sim.trace())
    return out


# ---- the surrogate -----------------------------------------------------------

def _dims(case):
    return [64] + [case["hidden"]] * case["layers"] + [-(-case["n_out"] // 64) * 64]


def _mlp_inputs(case, seed):
    """Weights (He-uniform, zero past the valid widths), inputs in [-1, 1],
    targets as rates come (many zeros, the others skewed), minibatch rows."""
    rng = np.random.default_rng(seed)
    dims = _dims(case)
    valid = [case["n_in"]] + [case["hidden"]] * case["layers"] + [case["n_out"]]
    flat = []
    for l in range(len(dims) - 1):
        w = np.zeros((dims[l + 1], dims[l]), np.float32)
        bound = math.sqrt(6.0 / valid[l])
        w[:valid[l + 1], :valid[l]] = rng.uniform(-bound, bound, (valid[l + 1], valid[l]))
        b = np.zeros(dims[l + 1], np.float32)
        b[:valid[l + 1]] = rng.uniform(-0.05, 0.05, valid[l + 1])
        flat += [w.ravel(), b]
    d = dict(params=np.concatenate(flat))
    n = case.get("rows") or (4 if case["kind"] == "train" else 1) * case["batch"]
    d["x"] = rng.uniform(-1.0, 1.0, (n, case["n_in"])).astype(np.float32)
    if case["kind"] != "predict":
        y = rng.exponential(2.0, (n, case["n_out"])).astype(np.float32)
        y[rng.random((n, case["n_out"]), np.float32) < 0.4] = 0.0
        d["y"] = y
    if case["kind"] == "train":
        d["rows"] = rng.integers(0, n, (case["steps"], case["batch"])).astype(np.int32)
    return d


def _prepare_mlp(case, seed):
    d = _mlp_inputs(case, seed)
    batch = case.get("batch", 4096)
    m = surrogate.MLP(in_dim=case["n_in"], hidden=case["hidden"], layers=case["layers"],
                      out_dim=case["n_out"], max_batch=batch)
    m.set_params(d["params"])
    if case["kind"] == "train":
        m.set_data(d["x"], d["y"])
    return dict(case=case, mlp=m, data=d)


def _run_mlp(state):
    case, m, d = state["case"], state["mlp"], state["data"]
    if case["kind"] == "train":
        loss = m.train(d["rows"], case["batch"], 1e-3)
        return dict(loss=loss, params=m.get_params())
    if case["kind"] == "gradients":
        grad, loss = m.gradients(d["x"], d["y"])
        return dict(grad=grad, loss=np.float32(loss))
    return dict(y=m.predict(d["x"]))


def _forward64(layers, x):
    acts = [x]
    for i, (w, b) in enumerate(layers):
        z = acts[-1] @ w.T + b
        acts.append(torch.relu(z) if i + 1 < len(layers) else z)
    return acts


def exact(case, seed):
    if case["kind"] in SIMS:
        # a spiking network's state is what its 32-bit sums, one by one in order,
        # make of it: in 64 bits other neurons fire
        return None
    d = _mlp_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    dims = _dims(case)
    flat = torch.from_numpy(d["params"]).to(dev).double()
    layers, spans, off = [], [], 0
    for l in range(len(dims) - 1):
        nw, nb = dims[l + 1] * dims[l], dims[l + 1]
        spans += [(off, off + nw), (off + nw, off + nw + nb)]
        layers.append([flat[off:off + nw].view(dims[l + 1], dims[l]), flat[off + nw:off + nw + nb]])
        off += nw + nb
    x = torch.zeros((d["x"].shape[0], 64), dtype=torch.float64, device=dev)
    x[:, :case["n_in"]] = torch.from_numpy(d["x"]).to(dev).double()
    n_out = case["n_out"]
    if case["kind"] == "predict":
        return dict(y=_forward64(layers, x)[-1][:, :n_out].cpu().numpy())
    y = torch.from_numpy(d["y"]).to(dev).double()

    def loss_grad(xb, yb):
        acts = _forward64(layers, xb)
        err = acts[-1][:, :n_out] - yb
        dz = torch.zeros_like(acts[-1])
        dz[:, :n_out] = err * (2.0 / err.numel())
        grad = torch.zeros_like(flat)
        for l in range(len(layers) - 1, -1, -1):
            (a, b), (c, e) = spans[2 * l], spans[2 * l + 1]
            grad[a:b] = (dz.T @ acts[l]).reshape(-1)
            grad[c:e] = dz.sum(0)
            if l:
                dz = (dz @ layers[l][0]) * (acts[l] > 0)
        return float((err * err).mean()), grad

    if case["kind"] == "gradients":
        loss, grad = loss_grad(x, y)
        return dict(grad=grad.cpu().numpy(), loss=np.float64(loss))
    m, v = torch.zeros_like(flat), torch.zeros_like(flat)
    losses = []
    for t, rows in enumerate(torch.from_numpy(d["rows"]).to(dev).long(), 1):
        loss, g = loss_grad(x[rows], y[rows])
        losses.append(loss)
        m.mul_(0.9).add_(g, alpha=0.1)
        v.mul_(0.999).add_(g * g, alpha=0.001)
        flat -= 1e-3 * (m / (1.0 - 0.9 ** t)) / ((v / (1.0 - 0.999 ** t)).sqrt() + 1e-8)
    return dict(loss=np.array(losses), params=flat.cpu().numpy())


# ---- the measured interface ---------------------------------------------------

def prepare(case, seed):
    return _prepare_sim(case, seed) if case["kind"] in SIMS else _prepare_mlp(case, seed)


def run(state):
    return _run_sim(state) if state["case"]["kind"] in SIMS else _run_mlp(state)


def work(case):
    """A delivery reads 8 bytes (32-bit weight and target) and adds once; a
    neuron's update moves about 52 bytes of state and constants each cycle.
    Linear layers count 2 operations per product, three products in training."""
    kind = case["kind"]
    if kind in SIMS:
        if kind == "random":
            n, syn, hz = case["n_lif"] + case["n_arr"] + case["n_bern"], 0.2 * case["n_lif"] ** 2, 300.0
        elif kind == "plain":
            n, syn, hz = 2 * case["n"], float(case["n"]) ** 2, 10.0
        elif kind == "standard":
            n = (case["npop"] + 1) * case["n"]
            syn, hz = float(case["npop"]) * case["n"] * case["fanout"], case["hz"]
        else:
            # 2 to 8 populations of log-uniform size, fan-in 100 to 1,000 but at most the source's size
            lo, hi = case["min_size"], case["max_size"]
            size = (hi - lo) / math.log(hi / lo)
            n = case["nets"] * 6 * size
            syn, hz = case["nets"] * 4 * size * min(550.0, 0.8 * size), case["hz"]
        events = syn * hz * DT
        return dict(bytes=case["cycles"] * (8.0 * events + 52.0 * n), flops=case["cycles"] * (events + 10.0 * n))
    w = [case["n_in"]] + [case["hidden"]] * case["layers"] + [case["n_out"]]
    kn = [w[l] * w[l + 1] for l in range(len(w) - 1)]
    params = sum(kn) + sum(w[1:])
    if kind == "predict":
        return dict(bytes=4.0 * case["rows"] * (w[0] + w[-1]) + 4.0 * params, flops=2.0 * case["rows"] * sum(kn))
    batch = case["batch"]
    flops = 2.0 * batch * (3 * sum(kn) - kn[0])
    data = 4.0 * batch * (w[0] + w[-1])
    if kind == "gradients":
        return dict(bytes=data + 8.0 * params, flops=flops)
    return dict(bytes=case["steps"] * (data + 24.0 * params), flops=case["steps"] * flops)
