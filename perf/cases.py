"""The work that a user of this package has the GPU do, as timed cases.

A sampler case is one print block of a simulation: advance the context by
`steps` sweeps, check the energy against a recompute where the driver program
does, read the counters and download the particles (what PatchyParticles_hip
does at every Print_every step, csrc/host/pp_main.c).  The others are the
snapshot energies of an analysis script and the training of the proposal
network.  Sizes are those of the bench workloads, the tests and the reference
program's own input files.
"""
import math

import numpy as np
import torch

import patchyparticles_amd as pp

DELTA, COSMAX = 0.12, 0.92  # the package's default patch geometry

# layers of the proposal network (include/pp.h): inputs x outputs as stored,
# and the entries that are not padding
LAYERS = ((96, 128, 84, 128), (128, 128, 128, 128), (128, 128, 128, 128), (128, 32, 128, 26))


def listed():
    run = dict(kind="run", ensemble="nvt", copies=1, uneven=False, trials=0, tune=False, trace=False, check=True, equil=200)
    return [
        # the smallest ordinary job: the reference program's N=1000 example
        # with its own schedule (one trial per particle and sweep), printed
        # every 100 sweeps; launches and latency count
        dict(run, name="nvt_n1000", n=1000, rho=0.1, T=0.1, steps=100),
        # the bench's liquid with the reference's schedule, the default of the
        # driver program and of System
        dict(run, name="nvt_n32768_members", n=32768, rho=0.5, T=0.12, steps=100),
        # the same liquid with the bench's 16 trials per cell and pass
        dict(run, name="nvt_n32768_s16", n=32768, rho=0.5, T=0.12, trials=16, steps=100),
        # a decorrelation run: 8 copies of one state in a batch, the energy
        # recorded after every sweep
        dict(run, name="nvt_8x4096_trace", n=4096, rho=0.5, T=0.2, copies=8, trials=16, steps=200, trace=True,
             check=False),
        # many uneven independent replicas in one context, launch shape tuned
        dict(run, name="nvt_256_uneven", n=8000, rho=0.6, T=0.2, copies=256, uneven=True, trials=16, tune=True,
             steps=100, check=False, equil=50),
        # the gel with the learned proposal in 80 % of the colour passes
        dict(run, name="learned_n65536", ensemble="learned", n=65536, rho=0.3, T=0.09, trials=1, steps=50),
        # a small constant-pressure run, one volume move per sweep
        dict(run, name="npt_n1331", ensemble="npt", n=1331, rho=0.3, T=0.2, P=0.2, steps=100),
        # the largest job: 16 big dilute constant-pressure replicas
        dict(run, name="npt_16x131072", ensemble="npt", n=131072, rho=0.05, T=0.11, P=0.02, copies=16, trials=16,
             tune=True, steps=16, check=False, equil=10),
        # insertions and removals in the reference's grand-canonical example
        dict(run, name="gc_box10", ensemble="gc", n=100, rho=0.1, T=0.2, activity=0.2, gc_n_max=1000, steps=100),
        # analysis of a saved configuration: per-particle bonds and overlaps
        dict(kind="snapshot", name="snapshot_n32768", n=32768, rho=0.5, T=0.12),
        # the network's loss and gradients on one training batch
        dict(kind="loss_grad", name="loss_grad_m4096", m=4096),
        # denoising training on the sampler's states, one sweep between steps
        dict(kind="train", name="train_n32768_b4096", n=32768, rho=0.5, T=0.12, trials=8, batch=4096, steps=40),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["nvt", "nvt", "nvt", "batch", "batch", "learned", "npt", "npt", "gc", "snapshot", "loss_grad", "train"])
    T, rho = round(rng.uniform(0.08, 0.20), 3), round(rng.uniform(0.05, 0.60), 3)
    run = dict(kind="run", ensemble="nvt", copies=1, uneven=False, trials=rng.choice([0, 0, 1, 2, 4, 8, 16, 16]), tune=False,
               trace=rng.random() < 0.25, check=rng.random() < 0.5, equil=rng.randrange(20, 200), rho=rho, T=T)
    if kind == "nvt":
        return dict(run, n=_log_uniform(rng, 400, 65536), steps=rng.randrange(20, 120))
    if kind == "batch":
        copies = _log_uniform(rng, 2, 200)
        return dict(run, n=_log_uniform(rng, 500, max(600, min(8000, 500000 // copies))), copies=copies,
                    uneven=rng.random() < 0.5, tune=rng.random() < 0.5, steps=rng.randrange(20, 100))
    if kind == "learned":
        return dict(run, ensemble="learned", n=_log_uniform(rng, 500, 65536), trials=rng.choice([0, 1, 16]),
                    steps=rng.randrange(10, 50))
    if kind == "npt":
        copies = rng.choice([1, 1, 2, 5, 16])
        return dict(run, ensemble="npt", n=_log_uniform(rng, 700, 131072 if copies == 1 else 32768),
                    rho=round(rng.uniform(0.05, 0.35), 3), P=round(rng.uniform(0.02, 0.3), 3), copies=copies,
                    tune=rng.random() < 0.5, steps=rng.randrange(10, 40))
    if kind == "gc":
        n = _log_uniform(rng, 100, 3000)
        return dict(run, ensemble="gc", n=n, rho=0.1, T=0.2, activity=round(rng.uniform(0.05, 0.2), 3),
                    gc_n_max=n * 10, steps=rng.randrange(20, 100))
    if kind == "snapshot":
        return dict(kind="snapshot", n=_log_uniform(rng, 100, 100000), rho=rho, T=T)
    if kind == "loss_grad":
        return dict(kind="loss_grad", m=_log_uniform(rng, 1, 16384))
    return dict(kind="train", n=_log_uniform(rng, 500, 65536), rho=rho, T=T, trials=rng.choice([0, 8, 16]),
                batch=_log_uniform(rng, 64, 16384), steps=rng.randrange(10, 40))


# ---------------------------------------------------------------- inputs


def _start(n, rho, seed):
    return pp.generate(n, rho, 1 + seed % 1000000007)


def _params(c):
    p = dict(T=c["T"], kf_delta=DELTA, kf_cosmax=COSMAX)
    if c["ensemble"] == "npt":
        p.update(ensemble=pp.NPT, P=c["P"], rescale_factor_max=0.01)
    if c["ensemble"] == "gc":
        p.update(ensemble=pp.GC, activity=c["activity"], gc_n_max=c["gc_n_max"])
    return p


def _sizes(c):
    """Particles, temperature and density of every replica."""
    if not c["uneven"]:
        return [(c["n"], c["T"], c["rho"])] * c["copies"]
    g = np.random.default_rng(c["n"] * 1009 + c["copies"])
    n = np.exp(g.uniform(math.log(500), math.log(max(c["n"], 501)), c["copies"])).astype(int)
    return list(zip(n.tolist(), g.uniform(0.08, max(c["T"], 0.081), c["copies"]).tolist(),
                    g.uniform(0.05, max(c["rho"], 0.051), c["copies"]).tolist()))


def _network(seed):
    """Weights as a new network has them: Glorot-uniform, a last layer that
    proposes small moves along four random axes."""
    g = np.random.default_rng(seed + 77)
    w, b = [], []
    for k, (rows, cols, fan_in, fan_out) in enumerate(LAYERS):
        m = np.zeros((rows, cols), np.float32)
        lim = math.sqrt(6.0 / (fan_in + fan_out)) * (0.1 if k == 3 else 1.0)
        m[:fan_in, :fan_out] = g.uniform(-lim, lim, (fan_in, fan_out))
        v = np.zeros(cols, np.float32)
        if k == 3:
            v[3:6] = math.log(0.03)
            v[6:26] = np.concatenate([np.append(g.uniform(-1, 1, 3), (math.log(0.1), 0.0)) for _ in range(4)])
        w.append(m.reshape(-1))
        b.append(v)
    return np.concatenate(w), np.concatenate(b)


def _bf16(a):
    return torch.from_numpy(np.asarray(a, np.float32)).bfloat16().float().numpy()


def _unit(g, *shape):
    v = g.normal(size=shape)
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def _training_rows(m, seed):
    """Descriptors of up to 12 neighbours, nearest first (separation and
    relative quaternion, BF16 values), and small moves as targets."""
    g = np.random.default_rng(seed + 5)
    dist = np.sort(g.uniform(1.0, 1.5, (m, 12)), axis=1)
    q = _unit(g, m, 12, 4)
    q[q[..., 3] < 0] *= -1
    x = np.concatenate([_unit(g, m, 12, 3) * dist[..., None], q], axis=-1)
    x[np.arange(12)[None, :] >= g.integers(3, 13, (m, 1))] = 0.0
    target = np.concatenate([g.normal(size=(m, 3)) * 0.03, _unit(g, m, 3)], axis=1)
    return _bf16(x.reshape(m, 84)), np.ascontiguousarray(target, np.float32)


def prepare(case, seed):
    c = case
    if c["kind"] == "loss_grad":
        net = pp.ProposalNet(seed=1)
        net.set(*_network(seed))
        x, target = _training_rows(c["m"], seed)
        return dict(c=c, net=net, x=x, target=target)
    if c["kind"] in ("snapshot", "train"):
        r, O, box = _start(c["n"], c["rho"], seed)
        if c["kind"] == "snapshot":
            with pp.System(r, O, box, T=c["T"], seed=seed, trials_per_cell=16) as s:
                s.do_ensemble(100)  # a bonded state
                r, O, box = s.state()
            return dict(c=c, r=r, O=O, box=box)
        s = pp.System(r, O, box, T=c["T"], seed=seed, trials_per_cell=c["trials"])
        s.do_ensemble(50)
        net = pp.ProposalNet(seed=1)
        net.set(*_network(seed))
        return dict(c=c, s=s, net=net)
    starts, prm = [], []
    for k, (n, T, rho) in enumerate(_sizes(c)):
        # copies of one state share their start; uneven replicas have their own
        starts.append(_start(n, rho, seed * 1009 + k) if c["uneven"] or k == 0 else starts[0])
        prm.append(dict(_params(c), T=T))
    s = pp.System.batch([x[0] for x in starts], [x[1] for x in starts], [x[2] for x in starts], prm, seed=seed,
                        trials_per_cell=c["trials"])
    s.do_ensemble(c["equil"])
    state = dict(c=c, s=s)
    if c["ensemble"] == "learned":
        state["net"] = pp.ProposalNet(seed=1)
        state["net"].set(*_network(seed))
        s.attach(state["net"], 0.8)
    if c["tune"]:
        s.autotune(2)
    s.reset_counters()
    return state


# ---------------------------------------------------------------- one pass


def run(state):
    c = state["c"]
    if c["kind"] == "snapshot":
        return pp.energy_snapshot(state["r"], state["O"], state["box"], DELTA, COSMAX)
    if c["kind"] == "loss_grad":
        return state["net"].loss_grad(state["x"], state["target"])
    s = state["s"]
    if c["kind"] == "train":
        losses = s.train(state["net"], steps=c["steps"], batch=c["batch"], lr=1e-3, pos_noise=0.03)
        return losses, state["net"].get()
    if c["trace"]:
        s.set_trace(c["steps"])
    s.do_ensemble(c["steps"])
    out = dict(counters=s.counters_all())
    if c["trace"]:
        out["trace"] = np.stack([s.trace(k) for k in range(s.R)])
    parts = [s.state(k) for k in range(s.R)]
    out["r"], out["O"], out["box"] = (np.concatenate([p[k] for p in parts]) for k in range(3))
    if c["ensemble"] == "gc":
        # arrays for the most particles the run may hold, as the driver has
        for k in ("r", "O"):
            full = np.zeros((c["gc_n_max"],) + out[k].shape[1:])
            full[:len(out[k])] = out[k]
            out[k] = full
    if c["check"]:
        out["energy"] = s.check_energy()
    return out


# ---------------------------------------------------------------- what a pass needs


def work(case):
    """One pass, without what the present kernels add: the state read and
    written once, and per attempted move the separations of the particles in
    the 27 cells around it, the new patches and the angular tests of the pairs
    in range (rough counts of FP64 operations)."""
    c = case
    mac = sum(fi * fo for _, _, fi, fo in LAYERS)
    if c["kind"] == "loss_grad":
        return dict(bytes=c["m"] * 90 * 4.0 + 3 * 50000 * 4.0, flops=6.0 * mac * c["m"])
    if c["kind"] == "snapshot":
        return dict(bytes=c["n"] * (96.0 + 5.0), flops=c["n"] * (27 * 1.5 * c["rho"] * 9 + 400.0))
    if c["kind"] == "train":
        return dict(bytes=2 * 96.0 * c["n"] + 6 * 50000 * 4.0,
                    flops=c["steps"] * (6.0 * mac * c["batch"] + 400.0 * c["n"] * max(1, c["trials"])))
    attempts, particles = 0.0, 0.0
    for n, _, rho in _sizes(c):
        side = (n / rho) ** (1 / 3)
        cells = (2 * math.floor(side / (2 * (1 + DELTA)))) ** 3
        per = n if c["trials"] == 0 else c["trials"] * cells * (1 - math.exp(-n / cells))
        attempts += c["steps"] * per * (27 * n / cells * 9 + 400)
        particles += n
    if c["ensemble"] == "learned":
        attempts += 0.8 * c["steps"] * particles * 0.7 * 4.0 * mac
    return dict(bytes=2 * 96.0 * particles, flops=attempts)


# ---------------------------------------------------------------- 64-bit values


def _snapshot_exact(r, O, box):
    """Bonds, overlaps and totals of a configuration from the definition of
    the model: spheres of diameter 1, a bond when a patch of each particle of
    a pair closer than 1 + delta points at the other within cosmax."""
    n, rc = len(r), 1.0 + DELTA
    m = np.maximum((box / (rc * (1 + 1e-9))).astype(int), 3)
    cell = np.minimum(np.floor((r / box - np.floor(r / box)) * m).astype(int), m - 1)
    flat = (cell[:, 0] * m[1] + cell[:, 1]) * m[2] + cell[:, 2]
    order = np.argsort(flat, kind="stable")
    first = np.searchsorted(flat[order], np.arange(m.prod() + 1))
    base = np.array([[-1, -1, 1], [1, -1, -1], [1, 1, 1], [-1, 1, -1]]) / math.sqrt(3.0)
    patches = np.einsum("nij,bj->nbi", O, base)
    bonds, overlap = np.zeros(n, np.int64), np.zeros(n, bool)
    for off in np.ndindex(3, 3, 3):
        other = (cell + np.array(off) - 1) % m
        oc = (other[:, 0] * m[1] + other[:, 1]) * m[2] + other[:, 2]
        lo, hi = first[oc], first[oc + 1]
        for k in range(int((hi - lo).max())):
            i = np.nonzero(lo + k < hi)[0]
            j = order[lo[i] + k]
            i, j = i[i != j], j[i != j]
            d = r[j] - r[i]
            d -= box * np.rint(d / box)
            d2 = (d * d).sum(1)
            overlap[i[d2 < 1.0]] = True
            near = (d2 >= 1.0) & (d2 < rc * rc)
            i, j, u = i[near], j[near], d[near] / np.sqrt(d2[near])[:, None]
            hit = (np.einsum("pbi,pi->pb", patches[i], u).max(1) > COSMAX) & (
                np.einsum("pbi,pi->pb", patches[j], -u).max(1) > COSMAX)
            np.add.at(bonds, i[hit], 1)
    bonds[overlap] = 0
    return bonds, overlap, int(bonds.sum()) // 2, bool(overlap.any())


def _loss_grad_exact(w, b, x, target):
    """Mean -log q and its gradients by automatic differentiation."""
    w = torch.tensor(w, dtype=torch.float64, requires_grad=True)
    b = torch.tensor(b, dtype=torch.float64, requires_grad=True)
    h = torch.zeros(len(x), 96, dtype=torch.float64)
    h[:, :84] = torch.from_numpy(x).double()
    t = torch.from_numpy(target).double()
    wo = bo = 0
    for k, (rows, cols, _, _) in enumerate(LAYERS):
        h = h @ w[wo:wo + rows * cols].view(rows, cols) + b[bo:bo + cols]
        h = torch.relu(h) if k < 3 else h
        wo, bo = wo + rows * cols, bo + cols
    log_sigma = h[:, 3:6].clamp(-6.2, -0.5)
    gauss = (-0.5 * ((t[:, :3] - h[:, :3]) * torch.exp(-log_sigma)) ** 2 - log_sigma - 0.5 * math.log(2 * math.pi)).sum(1)
    comp = h[:, 6:26].view(-1, 4, 5)
    axis = comp[..., :3] / torch.sqrt((comp[..., :3] ** 2).sum(-1, keepdim=True) + 1e-12)
    log_kappa = comp[..., 3].clamp(-3.0, 8.0)
    kappa = torch.exp(log_kappa)
    vmf = log_kappa - math.log(2 * math.pi) - kappa - torch.log(-torch.expm1(-2 * kappa)) + kappa * (axis * t[:, None, 3:]).sum(-1)
    loss = -(gauss + torch.logsumexp(torch.log_softmax(comp[..., 4], 1) + vmf, 1)).mean()
    loss.backward()
    return loss.item(), w.grad.numpy(), b.grad.numpy()


def exact(case, seed):
    if case["kind"] == "snapshot":
        s = prepare(case, seed)
        return _snapshot_exact(s["r"], s["O"], s["box"])
    if case["kind"] == "loss_grad":
        return _loss_grad_exact(*_network(seed), *_training_rows(case["m"], seed))
    # a trajectory has no value but the sampler's own: its random moves are
    # part of it, and any other arithmetic ends in another state
    return None
