"""Workloads of the framework for timing: what a user's program has in hand
(prepare), one pass through the public entry points (run) and the work that
pass cannot do without (work).

Kinds of case:

  sim       one simulation handle, set up and snapshotted once; a pass is one
            whole run from the snapshot (restore, run, generation tallies)
  steps     the same handle advanced day by day, as an interactive or coupled
            program does, with interventions and the agent state read back
  program   one constants row from nothing to its results: create, set up,
            seed, run, tallies, close (what a sweep does per run when it does
            not batch)
  batch     a replicate batch of constants rows of mixed sizes
  ensemble  a replicate batch of intervention scenarios, as the surrogate's
            training set is generated
  train     Adam steps of the surrogate's MLP ensemble, then its weights
  predict   surrogate predictions of scenario vectors on host arrays
  table     a stand-alone location table on the caller's device buffers
"""
import functools
import math

import numpy as np
import torch

import pandemicthrust_amd as pt
from pandemicthrust_amd import api, ensemble, scenarios, surrogate

AGENTS_PER_SCALE = 2.354e6      # agents at people_scaling_factor 1
DIMS = (16, 512, 512, 512, 512, 720)


def listed():
    return [
        # The reference's own headline run: scale 21.24 (50.0M agents), 100
        # days, R 1.8 / 1.3 (the benchmark's default workload).
        dict(name="sim 50M x 100 days", kind="sim", people=21.24, locations=21.24, days=100, r_p=1.8, r_s=1.3,
             init_p=10, init_s=10, pct=1.0, asymp=0.0, vaccination=0.0, closure=0),
        # The default constants.csv scale (2.35M agents).
        dict(name="sim 2.4M x 100 days", kind="sim", people=1.0, locations=1.0, days=100, r_p=1.8, r_s=1.3,
             init_p=10, init_s=10, pct=1.0, asymp=0.0, vaccination=0.0, closure=0),
        # The batcher's sweep also scales locations ten times the people
        # (10, 100): 23.5M agents over ten times as many, emptier locations.
        dict(name="sim 24M 10x locations", kind="sim", people=10.0, locations=100.0, days=60, r_p=1.8, r_s=1.3,
             init_p=60, init_s=60, pct=1.0, asymp=0.0, vaccination=0.0, closure=0),
        # Day by day with interventions and the state read back: 235k agents
        # in a 10x location grid (the sweep's 0.1, 1), asymptomatic cases.
        dict(name="steps 235k x 35 days", kind="steps", people=0.1, locations=1.0, days=35, r_p=2.2, r_s=1.5,
             init_p=30, init_s=60, pct=0.7, asymp=0.3, vaccination=0.1, closure=14),
        # One small run from nothing to its results (100k agents): host and
        # launch costs, allocations, set-up.
        dict(name="program 100k x 60 days", kind="program", people=0.0425, locations=0.0425, days=60, r_p=1.8,
             r_s=1.3, init_p=10, init_s=10, pct=1.0, asymp=0.0, vaccination=0.0, closure=0),
        # The replicate set's first 48 rows (50k to 2M agents each).
        dict(name="batch 48 rows", kind="batch", rows=48, first=0, days=180, people=1.0),
        # 3 scenarios x 8 seeds at 1M agents, 120 days, with interventions.
        dict(name="ensemble 3 x 8 at 1M", kind="ensemble", rows=3, replicates=8, agents=1000000, days=120),
        # The surrogate as it is trained: 5 members, batch 1024.
        dict(name="train 5 x 1024", kind="train", members=5, batch=1024, steps=100, lr=1e-3, rows=7936),
        # Screening predictions of an odd number of vectors.
        dict(name="predict 5 x 3001", kind="predict", members=5, batch=1024, rows=3001),
        # A handful of scenarios asked of a small ensemble.
        dict(name="predict 2 x 7", kind="predict", members=2, batch=64, rows=7),
        # A large location table: as many buckets as the 50M-agent weekday.
        dict(name="table 20M to 61597", kind="table", pairs=20000000, buckets=61597, noalloc=False),
        # A small one, allocation-free, as a captured or tight loop calls it.
        dict(name="table 29919 to 545", kind="table", pairs=29919, buckets=545, noalloc=True),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _epidemic(rng, kind, agents, days):
    people = round(agents / AGENTS_PER_SCALE, 6)
    ratio = rng.choice([1.0, 1.0, 1.0, 10.0, round(_log(rng, 0.3, 3.0), 3)])
    return dict(kind=kind, people=people, locations=round(people * ratio, 6), days=days,
                r_p=round(rng.uniform(1.2, 2.5), 4), r_s=round(rng.uniform(1.0, 1.8), 4), init_p=rng.randint(5, 60),
                init_s=rng.randint(5, 60), pct=rng.choice([1.0, 1.0, round(rng.uniform(0.5, 1.0), 3)]),
                asymp=rng.choice([0.0, round(rng.uniform(0.05, 0.5), 3)]),
                vaccination=rng.choice([0.0, 0.0, round(rng.uniform(0.05, 0.4), 3)]),
                closure=rng.choice([0, 0, rng.randint(7, 42)]))


def draw(rng):
    kind = rng.choice(["sim", "sim", "sim", "steps", "program", "batch", "ensemble", "train", "predict", "table"])
    if kind == "sim":
        agents = _log(rng, 20e3, 50e6)
        return _epidemic(rng, kind, agents, int(min(rng.randint(30, 180), max(20, 4.8e9 / agents))))
    if kind == "steps":
        return _epidemic(rng, kind, _log(rng, 20e3, 2e6), rng.randint(8, 40))
    if kind == "program":
        return _epidemic(rng, kind, _log(rng, 20e3, 3e6), rng.randint(20, 120))
    if kind == "batch":
        return dict(kind=kind, rows=rng.randint(5, 36), first=rng.randint(0, 200), days=rng.randint(60, 180),
                    people=round(_log(rng, 0.1, 1.0), 4))
    if kind == "ensemble":
        agents = int(_log(rng, 50e3, 1e6))
        return dict(kind=kind, rows=rng.randint(1, 3), replicates=rng.randint(2, 8), agents=agents,
                    days=rng.randint(40, 120))
    if kind == "train":
        return dict(kind=kind, members=rng.randint(1, 6), batch=64 * rng.randint(1, 20), steps=rng.randint(10, 100),
                    lr=round(_log(rng, 1e-4, 1e-3), 6), rows=rng.randint(2000, 7936))
    if kind == "predict":
        return dict(kind=kind, members=rng.randint(1, 6), batch=64 * rng.randint(1, 20), rows=int(_log(rng, 1, 4000)))
    noalloc = rng.random() < 0.5
    return dict(kind=kind, pairs=int(_log(rng, 1e3, 4.1e6 if noalloc else 2e7)), buckets=int(_log(rng, 29, 1.3e6)),
                noalloc=noalloc)


def _params(case):
    return pt.Params(int(case["days"]), case["r_p"], case["r_s"], case["init_p"], case["init_s"], case["people"],
                     case["locations"], case["pct"], case["asymp"])


def _core_seed(seed):
    return 1 + int(seed) % 2000000011


def _simulation(case, seed):
    s = pt.PandemicSim(_params(case), _core_seed(seed))
    if case["vaccination"] or case["closure"]:
        s.set_interventions(api.Interventions(
            latent=(1, 0), infectious=(8, 10), school_close_start=7, school_close_days=int(case["closure"]),
            workplace_reduction=0.25 if case["closure"] else 0.0, errand_reduction=0.1 if case["closure"] else 0.0,
            vaccination=(case["vaccination"], case["vaccination"])))
    s.setup_sim()
    return s


def _batch_rows(case):
    rows = scenarios.load_replicate_set()
    out = []
    for i in range(case["rows"]):
        f = list(rows[(case["first"] + i) % len(rows)][1])
        f[0] = str(case["days"])
        f[5] = f[6] = "%.6f" % (float(f[5]) * case["people"])
        out.append(pt.Params.from_row(f))
    return out


@functools.lru_cache(maxsize=1)
def _training_set():
    """(scaled inputs, targets) of the committed training set."""
    X, Y, _ = ensemble.load_training_set(surrogate.DATA)
    return surrogate.normalize(X), surrogate.targets(Y)


def _weights(case, seed):
    """Glorot-uniform weights, small biases: members x parameters."""
    rng = np.random.default_rng([int(seed), 77])
    members = []
    for _ in range(case["members"]):
        parts = []
        for a, b in zip(DIMS[:-1], DIMS[1:]):
            lim = math.sqrt(6.0 / (a + b))
            parts += [rng.uniform(-lim, lim, a * b), rng.uniform(-0.05, 0.05, b)]
        members.append(np.concatenate(parts))
    return np.stack(members).astype(np.float32)


def _rows(case, seed):
    X, Y = _training_set()
    take = np.random.default_rng([int(seed), 78]).permutation(len(X))[:case["rows"]]
    return X[take], Y[take]


def _device_keys(case, seed):
    """Bucket keys as errands have them: 62% of the pairs in 38% of the buckets."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n, K = case["pairs"], case["buckets"]
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    crowd = torch.rand(n, generator=g, device="cuda") < 0.62
    cut = max(1, int(0.38 * K))
    key = torch.where(crowd, u * cut, cut + u * (K - cut))
    return key.to(torch.int32).clamp_(0, K - 1)


def _padded(a, shape):
    """`a` at the start of an array of -1 (sizes that depend on the seed)."""
    out = np.full(shape, -1, np.int32)
    out[tuple(slice(0, n) for n in a.shape)] = a
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("sim", "steps"):
        s = _simulation(case, seed)
        s.snapshot()
        return dict(case=case, sim=s)
    if kind == "program":
        return dict(case=case, seed=seed)
    if kind == "batch":
        params = _batch_rows(case)
        b = pt.PandemicBatch(params, [_core_seed(seed + 131 * i) for i in range(len(params))])
        b.setup()
        b.snapshot()
        return dict(case=case, batch=b)
    if kind == "ensemble":
        vectors = ensemble.sample_scenarios(case["rows"], 1 + int(seed))
        params, ivs = [], []
        for v in vectors:
            p, iv = ensemble.scenario_inputs(v, case["agents"], case["days"])
            params += [p] * case["replicates"]
            ivs += [iv] * case["replicates"]
        b = pt.PandemicBatch(params, [_core_seed(seed + 131 * i) for i in range(len(params))])
        b.set_interventions(ivs)
        b.setup()
        b.snapshot()
        return dict(case=case, batch=b)
    if kind in ("train", "predict"):
        sur = surrogate.Surrogate(members=case["members"], batch=case["batch"], seed=1)
        sur.set_params(_weights(case, seed))
        X, Y = _rows(case, seed)
        if kind == "train":
            sur.set_data(X, Y)
        return dict(case=case, surrogate=sur, X=X, seed=int(seed) % (1 << 31))
    keys = _device_keys(case, seed)
    return dict(case=case, keys=keys, people=torch.empty(case["pairs"], dtype=torch.int32, device="cuda"),
                offsets=torch.empty(case["buckets"] + 1, dtype=torch.int32, device="cuda"))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sim":
        s = state["sim"]
        s.restore()
        counts, infected = s.run()
        gp, gs = s.generation_offsets()
        return dict(counts=_padded(counts, (case["days"], 16)), infected=_padded(infected, (case["days"],)),
                    generations_p=gp, generations_s=gs)
    if kind == "steps":
        s = state["sim"]
        s.restore()
        days = []
        for _ in range(case["days"]):
            ended, counts, infected = s.step()
            days.append(np.append(counts, infected))
            if ended:
                break
        names = ("status_p", "status_s", "day_p", "day_s", "gen_p", "gen_s")
        state = {k: s.array(which) for which, k in enumerate(names)}    # PT_STATUS_P .. PT_GEN_S
        agents = int(1.05 * case["people"] * AGENTS_PER_SCALE) + 1000
        return dict({k: _padded(a, (agents,)) for k, a in state.items()},
                    days=_padded(np.stack(days), (case["days"], 17)))
    if kind == "program":
        s = _simulation(case, state["seed"])
        counts, infected = s.run()
        gp, gs = s.generation_offsets()
        s.close()
        return dict(counts=_padded(counts, (case["days"], 16)), infected=_padded(infected, (case["days"],)),
                    generations_p=gp, generations_s=gs)
    if kind in ("batch", "ensemble"):
        b = state["batch"]
        b.restore()
        res = b.run()
        return dict(counts=np.stack([_padded(c, (case["days"], 16)) for c, _ in res]),
                    infected=np.stack([_padded(i, (case["days"],)) for _, i in res]))
    if kind == "train":
        sur = state["surrogate"]
        loss = sur.train(case["steps"], lr=case["lr"], seed=state["seed"])
        return dict(loss=loss, weights=sur.params())
    if kind == "predict":
        return state["surrogate"].predict(state["X"])
    entry = "pt_location_table_noalloc" if case["noalloc"] else "pt_location_table"
    rc = getattr(pt.lib(), entry)(state["keys"].data_ptr(), case["pairs"], case["buckets"], state["people"].data_ptr(),
                                  state["offsets"].data_ptr(), state["keys"].device.index,
                                  torch.cuda.current_stream().cuda_stream)
    if rc:
        raise RuntimeError(pt.lib().pt_last_error().decode())
    return dict(people=state["people"], offsets=state["offsets"])


def work(case):
    """A simulation reads every agent's two statuses and age each day and
    writes its six state bytes once; its operations are the errand draws that
    every agent makes each day (a 20-round Threefry2x64 block per two agents
    and two location walks on weekdays, two blocks and three walks on
    weekends).  A table reads its keys and writes its ids and offsets."""
    kind = case["kind"]
    if kind in ("sim", "steps", "program"):
        agents, days = case["people"] * AGENTS_PER_SCALE, case["days"]
    elif kind == "batch":
        agents, days = sum(p.people_scaling for p in _batch_rows(case)) * AGENTS_PER_SCALE, case["days"]
    elif kind == "ensemble":
        agents, days = case["agents"] * case["rows"] * case["replicates"], case["days"]
    elif kind in ("train", "predict"):
        macs = sum(a * b for a, b in zip(DIMS[:-1], DIMS[1:]))
        count = macs + sum(DIMS[1:])
        m = case["members"]
        if kind == "predict":
            return dict(bytes=4.0 * m * count + 4.0 * case["rows"] * (DIMS[0] + m * DIMS[-1]),
                        flops=2.0 * macs * m * case["rows"])
        steps, batch = case["steps"], case["batch"]
        return dict(bytes=steps * (4.0 * m * count * 7 + 4.0 * batch * (DIMS[0] + DIMS[-1])),
                    flops=2.0 * steps * batch * m * (3 * macs - DIMS[0] * DIMS[1]))
    else:
        return dict(bytes=8.0 * case["pairs"] + 4.0 * (case["buckets"] + 1), flops=0.0)
    return dict(bytes=agents * (3.0 * days + 6.0), flops=agents * days * (5 * 110.0 + 2 * 370.0) / 7)


def _split(flat):
    """[(W, b)] of one member's parameter block."""
    out, o = [], 0
    for a, b in zip(DIMS[:-1], DIMS[1:]):
        out.append((flat[o:o + a * b].reshape(a, b), flat[o + a * b:o + a * b + b]))
        o += a * b + b
    return out


def _forward(x, layers):
    acts, pres = [x], []
    for i, (w, b) in enumerate(layers):
        z = acts[-1] @ w + b
        if i < len(layers) - 1:
            pres.append(z)
            z = 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0)))
        acts.append(z)
    return acts, pres


def exact(case, seed):
    """64-bit results of the surrogate's passes; a simulation's and a table's
    outputs are whole numbers."""
    if case["kind"] not in ("train", "predict"):
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = dict(dtype=torch.float64, device=dev)
    P = torch.tensor(_weights(case, seed), **f64)
    X, Y = _rows(case, seed)
    if case["kind"] == "predict":
        x = torch.tensor(X, **f64)
        return torch.stack([_forward(x, _split(P[k]))[0][-1] for k in range(case["members"])]).cpu()
    X, Y = torch.tensor(X, **f64), torch.tensor(Y, **f64)
    steps, batch = case["steps"], case["batch"]
    rng = np.random.default_rng(int(seed) % (1 << 31))
    parts, have = [], 0
    while have < steps * batch:
        parts.append(rng.permutation(len(X)))
        have += len(X)
    order = torch.as_tensor(np.concatenate(parts)[:steps * batch].astype(np.int64), device=dev).reshape(steps, batch)
    losses = torch.zeros(steps, case["members"], dtype=torch.float64)
    for k in range(case["members"]):
        p = P[k]
        m, v = torch.zeros_like(p), torch.zeros_like(p)
        for t in range(steps):
            x, y = X[order[t]], Y[order[t]]
            layers = _split(p)
            acts, pres = _forward(x, layers)
            err = acts[-1] - y
            losses[t, k] = float((err * err).mean())
            d = err * (2.0 / err.numel())
            grads = []
            for i in range(len(layers) - 1, -1, -1):
                grads = [(acts[i].T @ d).reshape(-1), d.sum(0)] + grads
                if i:
                    z = pres[i - 1]
                    cdf = 0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))
                    d = (d @ layers[i][0].T) * (cdf + z * torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi))
            g = torch.cat(grads)
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            p = p - case["lr"] * (m / (1 - 0.9 ** (t + 1))) / (torch.sqrt(v / (1 - 0.999 ** (t + 1))) + 1e-8)
        P[k] = p
    return dict(loss=losses, weights=P.cpu())
