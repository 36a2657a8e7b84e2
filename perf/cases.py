"""The work a user of su2hip has it do, as timed cases.

Every case goes through the package's public handles (su2higgs_amd.lattice
and su2higgs_amd.serve), the calls the `su2hip` driver and bench.py make:

- "sweeps": chains advanced by compound sweeps, measured every `every`
  sweeps, their fields downloaded once at the end as a checkpoint does;
- "muca": the same for the multicanonical adjoint model;
- "measure": the FP64 volume sums of resident configurations;
- "flow": the RK3 gradient flow of one configuration, measured on the way;
- "serve": a queue of scan points run to completion by the request loop.

Sizes, couplings and sweep mixes are those of bench.py, the tests and the
driver's sample configurations, or generic extents between them.
"""
import numpy as np

from su2higgs_amd import abi, serve
from su2higgs_amd.lattice import Batch

# field content by model name: fundamental doublets, U(1), adjoint, singlet
MODELS = {
    "h": dict(nhiggs=1),
    "hu": dict(nhiggs=1, u1=1),
    "hsu": dict(nhiggs=1, u1=1, singlet=1),
    "ht": dict(nhiggs=1, triplet=1),
    "t": dict(nhiggs=0, triplet=1),
    "du": dict(nhiggs=2, u1=1),
}

# couplings of the workloads (bench.py); the others take make_params' values,
# the reference's sample configuration
COUPLINGS = {
    "h": dict(betasu2=8.0, msq_phi=-0.20, lambda_phi=0.02),
    "hu": dict(betasu2=9.0, betau1=27.0, r_u1=1.0, msq_phi=-0.20, lambda_phi=0.015),
}


def listed():
    def sweeps(name, L, model, fp32, n, every, overrelax=4, chains=1, graph=True):
        return dict(name=name, job="sweeps", L0=L[0], L1=L[1], L2=L[2], model=model, fp32=fp32,
                    sweeps=n, every=every, overrelax=overrelax, chains=chains, graph=graph)

    return [
        # one sweep of the smallest lattice of the tests, launched kernel by
        # kernel: a first try of a set-up, all latency
        sweeps("tiny-8", (8, 8, 8), "h", False, 1, 1, graph=False),
        # the driver's default field content at a ragged box, the reference's
        # own mix (no link overrelaxation): a plain run of the driver
        sweeps("box-hsu-fp64", (18, 14, 26), "hsu", False, 50, 10, overrelax=0),
        # one scan point on its own, as a user explores couplings
        sweeps("chain-32-fp32", (32, 32, 32), "h", True, 200, 20),
        # an elongated box, for a correlation length along z
        sweeps("box-hu-fp64", (30, 22, 70), "hu", False, 100, 20),
        # the flagship workload in both precisions
        sweeps("chain-96-fp32", (96, 96, 96), "hu", True, 200, 50),
        sweeps("chain-96-fp64", (96, 96, 96), "hu", False, 100, 50),
        # a volume beyond the flagship, the largest fields
        sweeps("chain-144-fp32", (144, 128, 144), "hu", True, 100, 50),
        # a scan over volumes and couplings in one handle
        dict(name="scan-32-fp32", job="sweeps", L0=0, L1=0, L2=0, model="h", fp32=True, sweeps=200,
             every=50, overrelax=4, chains=32, graph=True),
        # multicanonical production of the adjoint model
        dict(name="muca-48-fp64", job="muca", L0=48, L1=48, L2=48, model="t", fp32=False, sweeps=60,
             every=10, overrelax=4, chains=4, graph=True),
        # measurement of stored configurations
        dict(name="measure-96-fp64", job="measure", L0=96, L1=96, L2=96, model="hu", fp32=False,
             chains=1),
        # smearing of one configuration for topology and correlators
        dict(name="flow-64-fp32", job="flow", L0=64, L1=64, L2=64, model="h", fp32=True, steps=50,
             every=10),
        # the request loop of a scan service
        dict(name="serve-24", job="serve", requests=24, largest=40, sweeps=100, flow_every=8),
    ]


def _even(rng, lo, hi):
    """An even extent, uniform in the logarithm."""
    x = lo * (hi / lo) ** rng.random()
    return max(2, 2 * round(x / 2))


def draw(rng):
    job = rng.choices(["sweeps", "muca", "measure", "flow", "serve"], [8, 2, 1.5, 1.5, 1])[0]
    if job == "serve":
        return dict(job=job, requests=rng.randint(6, 24), largest=_even(rng, 24, 40),
                    sweeps=rng.randint(40, 100), flow_every=rng.choice([0, 6, 8]))
    fp32 = rng.random() < 0.5
    if job == "flow":
        L = [_even(rng, 12, 64) for _ in range(3)]
        return dict(job=job, L0=L[0], L1=L[1], L2=L[2], model=rng.choice(["h", "hu", "t"]), fp32=fp32,
                    steps=rng.randint(10, 50), every=10)
    if job == "measure":
        L = [_even(rng, 16, 96) for _ in range(3)]
        return dict(job=job, L0=L[0], L1=L[1], L2=L[2], model=rng.choice(["h", "hu", "t", "hsu"]),
                    fp32=fp32, chains=rng.choice([1, 1, 4]))
    if job == "muca":
        L = [_even(rng, 16, 48) for _ in range(3)]
        return dict(job=job, L0=L[0], L1=L[1], L2=L[2], model="t", fp32=fp32, sweeps=rng.randint(20, 60),
                    every=10, overrelax=rng.choice([0, 4]), chains=rng.choice([1, 4]), graph=True)
    top = _even(rng, 8, 128)
    L = [max(4, 2 * round(top * (0.6 + 0.4 * rng.random()) / 2)) for _ in range(3)]
    chains = 1 if max(L) > 48 else rng.choice([1, 1, 4, 12])
    return dict(job="sweeps", L0=L[0], L1=L[1], L2=L[2], model=rng.choice(["h", "hu", "hu", "hsu", "ht", "du"]),
                fp32=fp32, sweeps=rng.randint(20, 100), every=20, overrelax=rng.choice([0, 4, 4]),
                chains=chains, graph=rng.random() < 0.8)


def _extents(case):
    """The extents of each chain; L0 = 0 stands for a scan over volumes."""
    n = case.get("chains", 1)
    if case["L0"]:
        return [(case["L0"], case["L1"], case["L2"])] * n
    vols = np.random.default_rng(96).choice([16, 24, 32, 48], size=n)
    return [(int(L),) * 3 for L in vols]


def _params(case, seed):
    model = MODELS[case["model"]]
    ps = []
    ext = _extents(case)
    for k, L in enumerate(ext):
        kw = dict(model, **COUPLINGS.get(case["model"], {}))
        if len(ext) > 1 and case["model"] == "h":  # the scan's mass range
            kw["msq_phi"] = -0.30 + 0.15 * k / (len(ext) - 1)
        ps.append(abi.make_params(L=L, precision=abi.FP32 if case.get("fp32") else abi.FP64,
                                  link_overrelax=case.get("overrelax", 4),
                                  seed=1000003 * (seed + 1) + k, **kw))
    return ps


def _fields(p, rng):
    """A configuration like a thermalised one: links and angles spread about
    the identity by their couplings, scalars about a common value."""
    V = abi.volume(p)
    f = {}
    q = np.empty((V, 3, 4))
    q[..., 0] = 1.0
    q[..., 1:] = rng.standard_normal((V, 3, 3), dtype=np.float32) * (1.0 / np.sqrt(p.betasu2))
    q /= np.sqrt((q * q).sum(-1, keepdims=True))
    f["su2link"] = q
    if p.u1:
        f["u1link"] = rng.standard_normal((V, 3)) / np.sqrt(2.0 * p.betau1)
    if p.nhiggs:
        shape = (2, V, 4) if p.nhiggs == 2 else (V, 4)
        d = 0.45 * rng.standard_normal(shape)
        d[..., 0] += 0.5
        f["doublet"] = d
    if p.triplet:
        f["triplet"] = 0.5 * rng.standard_normal((V, 3))
    if p.singlet:
        f["singlet"] = 0.4 * rng.standard_normal(V)
    return f


class _State:
    """A handle with its chains, and the host arrays they are downloaded to."""

    def __init__(self, case, seed):
        self.case = case
        self.params = _params(case, seed)
        self.batch = Batch(self.params)
        names = [k for k, v in abi.field_arrays(abi.make_params(L=(2, 2, 2), **MODELS[case["model"]])).items()
                 if v is not None]
        vols = [abi.volume(p) for p in self.params]
        dofs = {"su2link": 12, "u1link": 3, "doublet": 4 * max(1, self.params[0].nhiggs), "triplet": 3,
                "singlet": 1}
        self.host = {k: np.zeros(sum(vols) * dofs[k]) for k in names}
        self.part = []
        at = 0
        for V in vols:
            self.part.append({k: self.host[k][at * dofs[k]:(at + V) * dofs[k]] for k in names})
            at += V

    def __del__(self):
        self.batch.close()

    def download(self):
        """The chains' fields in the reference's host layout, one after the
        other, in arrays the program keeps."""
        lib, h = self.batch.lib, self.batch.h
        for i, f in enumerate(self.part):
            abi.check(lib.su2hip_get_fields(h, i, *[abi.ptr(f[k]) if k in f else None for k in (
                "su2link", "u1link", "doublet", "triplet", "singlet")]))
        return self.host


def _weight(bins=200, lo=0.0, hi=2.0):
    """The multicanonical workload's weight: slopes in [-5, 5]."""
    rng = np.random.default_rng(48)
    edges = np.linspace(lo, hi, bins + 1)
    W = np.concatenate([[0.0], np.cumsum(rng.uniform(-5, 5, bins) * (hi - lo) / bins)])
    m = abi.Muca()
    m.enabled, m.orderparam, m.mode, m.checks_per_sweep = 1, abi.SIGMASQ, abi.READONLY, 1
    m.bins, m.do_acceptance, m.delta, m.min, m.max, m.wrk_min, m.wrk_max = bins, 1, 1e-3, lo, hi, lo, hi
    return m, np.concatenate([[lo - 1000.0 * (hi - lo)], edges]), np.concatenate([[W[0]], W])


def _requests(case, seed):
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(case["requests"]):
        flow = int(bool(case["flow_every"]) and (i + 1) % case["flow_every"] == 0)
        rows.append(dict(id=i, sweeps=int(rng.integers(case["sweeps"] // 4, case["sweeps"] + 1)), arrival=0.0,
                         betasu2=float(rng.uniform(6, 12)), msq_phi=float(rng.uniform(-0.3, -0.1)),
                         lambda_phi=float(rng.uniform(0.005, 0.03)), seed=int(rng.integers(1 << 40)),
                         L=int(2 * rng.integers(12, case["largest"] // 2 + 1)), flow=flow))
    return serve.requests(rows)


def prepare(case, seed):
    if case["job"] == "serve":
        cfg = serve.config(realtime=0, flow_t_max=0.5)
        return dict(case=case, cfg=cfg, reqs=_requests(case, seed))
    s = _State(case, seed)
    rng = np.random.default_rng(seed)
    if case["job"] in ("sweeps", "muca"):
        # chains begin from a cold start, as the driver's do
        for i in range(len(s.params)):
            s.batch.cold_start(i, phi0=1.0, sigma0=0.5, singlet0=0.2)
        if case["job"] == "muca":
            for i in range(len(s.params)):
                s.batch.muca_set(i, *_weight())
        s.batch.use_graph(case["graph"])
        s.batch.update(2)
        s.batch.sync()
    else:
        for i, p in enumerate(s.params):
            s.batch.set_fields(i, _fields(p, rng))
    return s


def run(state):
    if isinstance(state, dict):
        res, _ = serve.serve(state["cfg"], state["reqs"])
        return {"sums": np.array([r.sums[:] for r in res]), "flow": np.array([r.flow_sums[:] for r in res]),
                "passes": np.array([r.pass_ for r in res], dtype=np.int64),
                "status": np.array([r.status for r in res], dtype=np.int64)}
    case, b = state.case, state.batch
    if case["job"] == "measure":
        return {"sums": b.measure_all()}
    if case["job"] == "flow":
        return {"rows": b.flow(0, abi.FLOW_RK3, 0.01, 0.01 * case["steps"], case["every"], max_rows=64)}
    out, left = {"sums": []}, case["sweeps"]
    while left > 0:
        n = min(left, case["every"])
        b.update(n)
        out["sums"].append(b.measure_all())
        left -= n
    out["sums"] = np.array(out["sums"])
    out["fields"] = state.download()
    if case["job"] == "muca":
        out["muca"] = np.array([b.muca_orderparam(i, recompute=False) for i in range(len(state.params))])
    c = [b.counters(i) for i in range(len(state.params))]
    out["counters"] = np.array([[x[k] for k in sorted(x)] for x in c], dtype=np.int64)
    return out


def work(case):
    """Bytes and operations of one pass: a sweep of a checkerboard kind reads
    every field its updates depend on once and writes the updated variables
    once; a measurement reads every field once."""
    if case["job"] == "serve":
        reqs = _requests(case, 0)
        byts = flops = 0.0
        for r in reqs:
            one = work(dict(job="sweeps", L0=r.L, L1=r.L, L2=r.L, model="h", fp32=True, sweeps=r.sweeps,
                            every=r.sweeps, overrelax=4, chains=1))
            byts += one["bytes"] - 16 * 8 * r.L ** 3  # the fields stay on the device
            flops += one["flops"]
            if r.flow:
                one = work(dict(job="flow", L0=r.L, L1=r.L, L2=r.L, model="h", fp32=True, steps=50, every=50))
                byts += one["bytes"]
                flops += one["flops"]
        return {"bytes": byts, "flops": flops}
    p = _params(case, 0)[0]
    w = 4 if case.get("fp32") else 8
    V = float(sum(L[0] * L[1] * L[2] for L in _extents(case)))
    lw = 9 if case.get("fp32") else 12  # words of a site's links: unit quaternions, three words suffice in FP32
    scal = 4 * p.nhiggs + 3 * p.triplet + p.singlet
    words = lw + 3 * p.u1 + scal
    meas_bytes, meas_flops = words * V * w, (330 + 60 * p.u1 + 180 * p.nhiggs + 600 * p.triplet) * V
    if case["job"] == "measure":
        return {"bytes": meas_bytes, "flops": meas_flops}
    if case["job"] == "flow":
        stages, rows = 3 * case["steps"], case["steps"] // case["every"] + 1
        return {"bytes": stages * (2 * lw + 18 + (6 + 3 if p.triplet else 0)) * V * w + rows * meas_bytes,
                "flops": stages * 3 * 270.0 * V + rows * meas_flops}
    # links: the two other directions, the direction itself in and out, and
    # what the scalars' hopping terms need
    rounds = 1 + case["overrelax"]
    link = rounds * 3 * ((lw + lw / 3) + 4 * p.nhiggs + p.u1 + 3 * p.triplet)
    u1 = 3 * (3 + 1 + lw / 3 + 4 * p.nhiggs) if p.u1 else 0
    scalar = 5 * p.nhiggs * (8 + lw + 3 * p.u1 + 3 * p.triplet + p.singlet)
    scalar += 5 * p.triplet * (6 + lw + 4 * p.nhiggs) + 5 * p.singlet * (2 + 4 * p.nhiggs)
    flops = rounds * 3 * 300.0 + (3 * 120.0 if p.u1 else 0) + 5 * p.nhiggs * 330.0 + 5 * p.triplet * 380.0 + \
        5 * p.singlet * 60.0
    n = case["sweeps"]
    meas = -(-n // case["every"])
    down = (12 + 3 * p.u1 + scal) * 8 * V
    return {"bytes": n * (link + u1 + scalar) * V * w + meas * meas_bytes + down,
            "flops": n * flops * V + meas * meas_flops}


# ---------------------------------------------------------------------------
# results in 64 bits by plain numpy: fields on a [z, y, x] grid, links as
# quaternions u0 + i u.sigma

def _grid(p, f):
    """The fields on the grid from the checkerboarded host order."""
    L0, L1, L2 = p.L
    z, y, x = np.meshgrid(np.arange(L2), np.arange(L1), np.arange(L0), indexing="ij")
    par = ((x + y + z) & 1).ravel()
    order = np.concatenate([np.nonzero(par == 0)[0], np.nonzero(par == 1)[0]])
    g = {}
    for k, a in f.items():
        if a.ndim == 1:
            a = a[:, None]
        o = np.empty_like(a)
        o[order] = a
        g[k] = np.moveaxis(o.reshape((L2, L1, L0) + a.shape[1:]), (0, 1, 2), (-3, -2, -1))
    return g


def _mul(x, y):
    a, b, c, d = x
    e, f, g, h = y
    return np.stack([a * e - b * f - c * g - d * h, a * f + b * e - (c * h - d * g),
                     a * g + c * e - (d * f - b * h), a * h + d * e - (b * g - c * f)])


def _conj(x):
    return np.stack([x[0], -x[1], -x[2], -x[3]])


def _up(a, d, n=1):
    """a at the neighbour n steps along d (grid axes z, y, x last)."""
    return np.roll(a, -n, axis=-1 - d)


def _plaquette(U, i, j):
    return _mul(_mul(U[i], _up(U[j], i)), _mul(_conj(_up(U[i], j)), _conj(U[j])))


def _sums(p, g):
    """The volume sums of a configuration of one doublet, with or without U(1)."""
    s = np.zeros(abi.NSUMS)
    U = g["su2link"]
    wil = p.betasu2 * sum((1.0 - _plaquette(U, i, j)[0]).sum() for j in range(3) for i in range(j))
    f = g["doublet"]
    mod = 0.5 * (f * f).sum(0)
    cov, u1w = 6.0 * mod.sum(), 0.0
    for d in range(3):
        t = _mul(_mul(_conj(f), U[d]), _up(f, d))
        if p.u1:
            al = g["u1link"][d]
            cov -= (t[0] * np.cos(al) + t[3] * np.sin(al)).sum()
        else:
            cov -= t[0].sum()
    if p.u1:
        A = g["u1link"]
        u1w = p.betau1 * sum((1.0 - np.cos(p.r_u1 * (A[i] + _up(A[j], i) - _up(A[i], j) - A[j]))).sum()
                             for j in range(3) for i in range(j))
    s[abi.SUM["wilson"]], s[abi.SUM["u1wilson"]] = wil, u1w
    s[abi.SUM["cov_phi"]], s[abi.SUM["phi2"]], s[abi.SUM["phi4"]] = cov, mod.sum(), (mod * mod).sum()
    s[abi.SUM["action"]] = wil + u1w + cov + p.msq_phi * mod.sum() + p.lambda_phi * (mod * mod).sum()
    return s


def _force(U, d):
    """The flow force of direction d: the vector part of -(U staple)."""
    W = 0.0
    for n in range(3):
        if n != d:
            W = W + _mul(_mul(_up(U[n], d), _conj(_up(U[d], n))), _conj(U[n]))
            lo = _mul(_mul(_conj(_up(U[n], d)), _conj(U[d])), U[n])
            W = W + _up(lo, n, -1)
    return -_mul(U[d], W)[1:]


def exact(case, seed):
    if case["job"] not in ("measure", "flow") or case["model"] not in ("h", "hu"):
        return None
    if case["job"] == "flow" and case["L0"] * case["L1"] * case["L2"] * case["steps"] > 1_000_000:
        return None
    rng = np.random.default_rng(seed)
    ps = _params(case, seed)
    grids = [_grid(p, _fields(p, rng)) for p in ps]
    if case["job"] == "measure":
        return {"sums": np.array([_sums(p, g) for p, g in zip(ps, grids)])}
    p, g = ps[0], grids[0]
    U = g["su2link"].copy()
    dt, rows = 0.01, [np.concatenate([[0.0], _sums(p, g)])]
    for step in range(1, case["steps"] + 1):
        Z = np.zeros((3, 3) + U.shape[2:])
        for c, e in ((0.25, 0.0), (8.0 / 9.0, 17.0 / 9.0), (0.75, 1.0)):
            Z = np.stack([c * dt * _force(U, d) for d in range(3)]) - e * Z
            mod = np.sqrt((Z * Z).sum(1))
            sn = np.sinc(mod / np.pi)
            U = np.stack([_mul(np.stack([np.cos(mod[d]), *(sn[d] * Z[d])]), U[d]) for d in range(3)])
        if step % case["every"] == 0 or step == case["steps"]:
            rows.append(np.concatenate([[dt * step], _sums(p, dict(g, su2link=U))]))
    return {"rows": np.array(rows)}
