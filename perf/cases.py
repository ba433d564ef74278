"""Timed workloads of the package: whole solves, surveys, batches and FWI
gradients through the public entry points, with their inputs, the least work
they need and their results in plain FP64.

    listed()           the fixed cases
    draw(rng)          one more case of the same ranges
    prepare(case, s)   inputs and plans made from the seed s, on the GPU
    run(state)         one pass and its outputs
    work(case)         bytes and operations of one pass
    exact(case, s)     the outputs of run in FP64, by plain torch

Kinds of case:
  solve   solve2D / solve3D, the drop-in call: host setup, plan, time loop,
          final field and seismograms.
  survey  a plan kept between solves: reset, the time loop, every shot's
          traces (one-shot plans: the final field too).
  batch   several models of different sizes in one Batch: run, all traces.
  fwi     misfit and gradient of a plan's shots (fwi.misfit_gradient), or
          of a velocity tensor through torch autograd (fwi.solve_traces).

Grids count every node: interior + 2 * (halo + 1) per axis.  The velocity
rises with depth (the second axis) and carries smooth seeded anomalies;
sources sit a few nodes below the top slab, receivers on a line or a grid.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "acousticwavecpml.jl_amd"))
import awcpml  # noqa: E402

DX = 10.0
RCOEF = 1e-3
VMIN, VMAX = 1500.0, 3000.0


def listed():
    return [
        # the smallest drop-in call, the size of a unit test or a first try:
        # setup, launch latency and copies
        _case("solve2d_f64_121x101", "solve", (121, 101), 20, "f64", 1, 220, freetop=True),
        # 256^2 interior, FP64, one shot, kept plan: the plain 2D workload
        _case("plan2d_f64_298", "survey", (298, 298), 20, "f64", 1, 1000, graph=True, steps=2),
        # the large single 2D run of the published benchmark tables (4097^2)
        _case("plan2d_f64_4097", "survey", (4097, 4097), 20, "f64", 1, 200, graph=True,
              steps=2),
        # many shots on one 2D model in FP32: the survey workload
        _case("survey2d_f32_1066x64", "survey", (1066, 1066), 20, "f32", 64, 400, graph=True,
              steps=2),
        # an odd wide model, a few shots, free top, no tuning knob set
        _case("survey2d_f32_701x333x7", "survey", (701, 333), 15, "f32", 7, 500, freetop=True),
        # a mid-size 3D drop-in call, FP64
        _case("solve3d_f64_101x91x83", "solve", (101, 91, 83), 20, "f64", 1, 160, freetop=True),
        # 256^3 interior, FP64, one shot: the plain 3D workload
        _case("plan3d_f64_298", "survey", (298, 298, 298), 20, "f64", 1, 400, freetop=True,
              graph=True, steps=2),
        # the same model, 8 shots in FP32: the 3D survey workload
        _case("survey3d_f32_298x8", "survey", (298, 298, 298), 20, "f32", 8, 100, freetop=True,
              graph=True, steps=2),
        # an odd 3D model with a thin halo, a few shots
        _case("survey3d_f32_187x131x223x3", "survey", (187, 131, 223), 12, "f32", 3, 200,
              steps=2),
        # models of different sizes advanced together
        _case("batch3d_f32_170_to_298", "batch", (170, 234, 298), 20, "f32", 1, 100, graph=True,
              steps=2),
        # one FWI iteration's gradient, 32 shots on 512^2 interior nodes
        _case("fwi2d_f32_554x32", "fwi", (554, 554), 20, "f32", 32, 400, steps=2),
        # a small 3D inversion through torch autograd, FP64
        _case("fwi3d_f64_81x73x69x2", "fwi", (81, 73, 69), 12, "f64", 2, 120, autograd=True),
    ]


def _case(name, kind, n, halo, dtype, shots, nt, freetop=False, graph=False, steps=0,
          autograd=False):
    """n: nodes per axis (batch: the cube edges of its models).  steps: the
    time blocking the program asks for (0: none)."""
    return {"name": name, "kind": kind, "ndim": 3 if kind == "batch" else len(n), "nx": n[0],
            "ny": n[1], "nz": n[2] if len(n) > 2 else 1, "halo": halo, "dtype": dtype,
            "shots": shots, "nt": nt, "freetop": freetop, "graph": graph, "steps": steps,
            "autograd": autograd}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "survey", "survey", "survey", "survey", "batch", "fwi"])
    ndim = 3 if kind == "batch" else rng.choice([2, 3])
    dtype = rng.choice(["f64", "f32"])
    halo = rng.choice([8, 12, 15, 20, 20, 20])
    low = 2 * halo + 24
    shots = 1
    if kind == "batch":
        n = tuple(_log_int(rng, max(low, 90), 298) for _ in range(3))
    elif ndim == 2:
        top = {"solve": 1200, "survey": 1100, "fwi": 560}[kind]
        n = (_log_int(rng, low, top), _log_int(rng, low, top))
        if kind == "survey" and rng.random() < 0.15:
            n = (_log_int(rng, 1100, 4000), _log_int(rng, 1100, 4000))
        elif kind != "solve":
            shots = _log_int(rng, 1, 64 if kind == "survey" else 32)
    else:
        top = {"solve": 150, "survey": 298, "fwi": 90}[kind]
        n = tuple(_log_int(rng, low, max(top, low + 6)) for _ in range(3))
        if kind != "solve":
            shots = _log_int(rng, 1, 8 if kind == "survey" else 3)
    nodes = shots * math.prod(n) if kind != "batch" else sum(e ** 3 for e in n)
    most = {"solve": 4e8, "survey": 8e9, "batch": 4e9, "fwi": 2e9}[kind]
    nt = int(max(30, min(rng.uniform(120, 600), most / nodes)))
    return {k: v for k, v in _case(
        "", kind, n, halo, dtype, shots, nt, freetop=rng.random() < 0.5,
        graph=kind in ("survey", "batch") and rng.random() < 0.6,
        steps=2 if kind != "solve" and rng.random() < 0.6 else 0,
        autograd=kind == "fwi" and shots <= 3 and rng.random() < 0.5).items() if k != "name"}


# ---------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------

def _shape(case):
    return (case["nx"], case["ny"], case["nz"])[:case["ndim"]]


def _models(case):
    """(nodes per axis) of each model of the case."""
    if case["kind"] == "batch":
        return [(e, e, e) for e in (case["nx"], case["ny"], case["nz"])]
    return [_shape(case)]


def _f0(ndim):
    return 12.0 if ndim == 2 else 10.0


def _velocity(n, rng):
    """Depth gradient plus three smooth anomalies, in VMIN..VMAX with the
    maximum attained exactly (so that dt does not depend on the seed)."""
    dims = tuple(reversed(n))                      # x fastest
    x = [np.linspace(0.0, 1.0, v).reshape([-1 if a == b else 1 for b in reversed(range(len(n)))])
         for a, v in enumerate(n)]
    v = np.empty(dims)
    v[...] = VMIN + (VMAX - VMIN) * 0.7 * x[1]
    for _ in range(3):
        term = rng.uniform(60.0, 120.0)
        for xa in x:
            term = term * np.cos(2 * np.pi * (rng.uniform(0.5, 2.5) * xa + rng.uniform()))
        v += term
    np.clip(v, VMIN, VMAX, out=v)
    v = v.T
    v[tuple(k // 2 for k in n)] = VMAX
    return v


def _spread(n, count, margin):
    """`count` 1-based node indices spread over an axis, `margin` from its ends."""
    lo, hi = margin, max(margin, n - 1 - margin)
    return [1 + int(round(lo + (q + 0.5) * (hi - lo) / count)) for q in range(count)]


def _model(case, n, rng):
    """One model and its acquisition: velocity, 1-based source node of every
    shot, receiver nodes (shared by the shots), wavelet delay."""
    h, nd = case["halo"], len(n)
    depth = 1 + (h + 2 if not case["freetop"] else 6)
    jitter = int(rng.integers(0, 3))
    src = []
    for q, i in enumerate(_spread(n[0], case["shots"], h + 4)):
        pos = [i, depth + jitter] + ([1 + n[2] // 2 + (q % 3) - 1] if nd == 3 else [])
        src.append(np.array([pos], dtype=np.int64))
    if nd == 2:
        rec = [[i, depth + 1] for i in _spread(n[0], min(128, n[0] // 3), h + 2)]
        rec += [[n[0] // 2, j] for j in _spread(n[1], 16, h + 2)]
    else:
        rec = [[i, depth + 1, k] for k in _spread(n[2], 8, h + 2) for i in _spread(n[0], 8, h + 2)]
        rec += [[n[0] // 2, j, n[2] // 2] for j in _spread(n[1], 16, h + 2)]
    return {"n": n, "vel": _velocity(n, rng), "src": src, "rec": np.array(rec, dtype=np.int64),
            "t0": 1.0 / _f0(nd) * (0.9 + 0.2 * rng.uniform())}


def _inputs(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return [_model(case, n, rng) for n in _models(case)]


def _dt(ndim):
    return math.sqrt(ndim) / (VMAX * ndim / DX) / 2


def _lt(case):
    return (case["nt"] - 0.5) * _dt(case["ndim"])


def _observed(case, m, rng):
    """Observed traces (shots, nt, receivers): a direct arrival at a
    mean velocity and a weaker later one, both of the wavelet's shape."""
    nd, dt = case["ndim"], _dt(case["ndim"])
    t = np.arange(case["nt"]) * dt
    out = np.empty((case["shots"], case["nt"], len(m["rec"])))
    for s, pos in enumerate(m["src"]):
        r = DX * np.sqrt((((m["rec"] - pos[0]) ** 2).sum(axis=1)).astype(float)) + DX
        amp = 3e-8 * (100.0 / r) ** 0.5 if nd == 2 else 2e-10 * (100.0 / r)
        for w, c in ((1.0, 1900.0), (0.3 + 0.2 * rng.uniform(), 1500.0)):
            u = (np.pi * _f0(nd) * (t[:, None] - m["t0"] - r[None, :] / c)) ** 2
            if c == 1900.0:
                out[s] = w * amp * (1 - 2 * u) * np.exp(-u)
            else:
                out[s] += w * amp * (1 - 2 * u) * np.exp(-u)
    return out


def _acquisition(m, nd):
    at = lambda p: (np.asarray(p, dtype=np.float64) - 1.0) * DX  # noqa: E731
    return (awcpml.Sources(at(m["src"][0]), [m["t0"]], [awcpml.rickersource1D], _f0(nd)),
            awcpml.Receivers(at(m["rec"])))


def _setup(case, m):
    srcs, recs = _acquisition(m, len(m["n"]))
    return awcpml.setup([(v - 1) * DX for v in m["n"]], _lt(case), m["vel"], srcs, recs,
                        halo=case["halo"], rcoef=RCOEF, freetop=case["freetop"])


def _plan(case, m):
    S = _setup(case, m)
    P = awcpml.Plan(S.n, S.halo, dtype=case["dtype"], nshots=case["shots"])
    P.set_model(S.fact, S.inv_d, S.inv_d2)
    for a in range(S.ndim):
        P.set_cpml(a, S.coef[a])
    for s in range(case["shots"]):
        P.set_sources(s, m["src"][s], S.dt2srctf)
        P.set_receivers(s, S.posrecs)
    if case["steps"]:
        P.set_time_block(case["steps"])
    if case["graph"] and case["kind"] != "batch":
        P.set_graph(True)
    return P


def prepare(case, seed):
    models = _inputs(case, seed)
    st = {"case": case}
    m = models[0]
    if case["kind"] == "solve":
        st["args"] = [(v - 1) * DX for v in m["n"]] + [_lt(case), m["vel"]]
        st["srcs"], st["recs"] = _acquisition(m, case["ndim"])
    elif case["kind"] == "survey":
        st["plan"] = _plan(case, m)
    elif case["kind"] == "batch":
        st["plans"] = [_plan(case, q) for q in models]
        st["batch"] = awcpml.Batch(st["plans"])
        if case["graph"]:
            st["batch"].set_graph(True)
    else:
        obs = _observed(case, m, np.random.Generator(np.random.PCG64([seed, 1])))
        if case["autograd"]:
            S = _setup(case, m)
            st["problem"] = awcpml.fwi.Problem(S, nshots=case["shots"], src_positions=m["src"],
                                               dtype=case["dtype"])
            if case["steps"]:
                st["problem"].plan.set_time_block(case["steps"])
            st["vel"] = torch.from_numpy(m["vel"])
            st["obs"] = torch.from_numpy(obs)
        else:
            st["plan"] = _plan(case, m)
            st["obs"] = list(obs)
    return st


def run(state):
    case = state["case"]
    if case["kind"] == "solve":
        solve = awcpml.solve2D if case["ndim"] == 2 else awcpml.solve3D
        field = solve(*state["args"], state["srcs"], state["recs"], halo=case["halo"],
                      rcoef=RCOEF, freetop=case["freetop"], dtype=case["dtype"])
        return {"field": field, "traces": state["recs"].seismograms}
    if case["kind"] == "survey":
        P = state["plan"]
        P.reset()
        P.advance(case["nt"])
        out = {"traces": np.stack([P.traces(s) for s in range(case["shots"])])}
        if case["shots"] == 1:
            out["field"] = P.field(0)
        return out
    if case["kind"] == "batch":
        state["batch"].run()
        return {"traces": [P.traces(0) for P in state["plans"]]}
    if case["autograd"]:
        vel = state["vel"].clone().requires_grad_(True)
        loss = 0.5 * (awcpml.fwi.solve_traces(vel, state["problem"]) - state["obs"]).pow(2).sum()
        loss.backward()
        return {"misfit": loss.detach(), "gradient": vel.grad}
    J, grad = awcpml.fwi.misfit_gradient(state["plan"], state["obs"])
    return {"misfit": J, "gradient": grad}


# ---------------------------------------------------------------------
# the least a pass needs
# ---------------------------------------------------------------------

def work(case):
    """Bytes: the model read once, the traces written once, for one-shot
    plans the final field, for gradients the observed traces read and the
    gradient written.  Operations: 12 (2D) or 16 (3D) per node, shot and
    step, and for a gradient the same again for the reverse step."""
    es = 8 if case["dtype"] == "f64" else 4
    total_b = total_f = 0.0
    for n in _models(case):
        N = math.prod(n)
        nrec = (min(128, n[0] // 3) + 16) if len(n) == 2 else 80
        traces = case["shots"] * case["nt"] * nrec
        whole = case["kind"] == "fwi" or (case["shots"] == 1 and case["kind"] != "batch")
        total_b += es * (N * (2 if whole else 1) + traces * (2 if case["kind"] == "fwi" else 1))
        total_f += (2 if case["kind"] == "fwi" else 1) * case["nt"] * case["shots"] * N * (
            12 if len(n) == 2 else 16)
    return {"bytes": total_b, "flops": total_f}


# ---------------------------------------------------------------------
# the same results in plain FP64 torch
# ---------------------------------------------------------------------

def _coefficients(case, n, dev):
    """Per axis: edge coefficients (n-1 edges) and node coefficients (n
    nodes), zero outside the absorbing sides, and the slab-node mask."""
    h, dt, nd = case["halo"], _dt(len(n)), len(n)
    amax = math.pi * _f0(nd)
    d0 = -3.0 * VMAX * math.log(RCOEF) / (2.0 * h * DX)

    def ab(dist):
        d = d0 * dist ** 2
        alpha = amax * (1.0 - dist)
        b = np.exp(-(d + alpha) * dt)
        return d * (b - 1.0) / (d + alpha), b

    on = ab(np.arange(h) / h)                     # from the inner edge outwards
    half_d = np.arange(h + 1) - 0.5
    half_d[0] = 0.0
    half = ab(half_d / h)
    out = []
    for a, v in enumerate(n):
        ae, be = np.zeros(v - 1), np.zeros(v - 1)
        an, bn, mask = np.zeros(v), np.zeros(v), np.zeros(v)
        if not (case["freetop"] and a == 1):      # low side: edges 0..h, nodes 1..h
            ae[:h + 1], be[:h + 1] = half[0][::-1], half[1][::-1]
            an[1:h + 1], bn[1:h + 1], mask[1:h + 1] = on[0][::-1], on[1][::-1], 1.0
        o = v - h - 2                             # high side: edges o..o+h, nodes o+1..o+h
        ae[o:o + h + 1], be[o:o + h + 1] = half
        an[o + 1:o + h + 1], bn[o + 1:o + h + 1], mask[o + 1:o + h + 1] = on[0], on[1], 1.0
        view = [1] * (nd + 1)
        view[nd - a] = -1                         # fields are (shot, [z,] y, x)
        out.append([torch.tensor(q, device=dev).reshape(view) for q in (ae, be, an[1:-1], bn[1:-1],
                                                                        mask[1:-1])])
    return out


def _inner(p, keep):
    """p without its first and last node along every axis except `keep`."""
    for d in range(1, p.dim()):
        if d != keep:
            p = p.narrow(d, 1, p.shape[d] - 2)
    return p


def _steps(it0, it1, fact, coef, srcs, wav, rec, state):
    """Time steps it0..it1-1 from state (pold, pcur, psi..., xi...)."""
    nd = fact.dim() - 1
    pold, pcur = state[0], state[1]
    psi, xi = list(state[2:2 + nd]), list(state[2 + nd:2 + 2 * nd])
    f = _inner(fact, -1)
    pad = (1, 1) * nd
    traces = []
    shot = torch.arange(pcur.shape[0], device=pcur.device)
    for it in range(it0, it1):
        lap = damp = 0.0
        for a in range(nd):
            ae, be, an, bn, mask = coef[a]
            dim = nd - a
            q = _inner(pcur, dim)
            m = q.shape[dim]
            e = q.narrow(dim, 1, m - 1) - q.narrow(dim, 0, m - 1)
            d2 = (e.narrow(dim, 1, m - 2) - e.narrow(dim, 0, m - 2)) * (1.0 / DX ** 2)
            psi[a] = be * psi[a] + ae * e * (1.0 / DX)
            dpsi = (psi[a].narrow(dim, 1, m - 2) - psi[a].narrow(dim, 0, m - 2)) * (mask / DX)
            xi[a] = bn * xi[a] + an * (d2 + dpsi)
            lap = lap + d2
            damp = damp + (dpsi + xi[a])
        new = 2.0 * _inner(pcur, -1) - _inner(pold, -1) + f * (lap + damp)
        new = torch.nn.functional.pad(new, pad)
        new = new.index_put((shot,) + srcs, wav[it].expand(len(shot)), accumulate=True)
        traces.append(new[(slice(None),) + rec])
        pold, pcur = pcur, new
    return (torch.stack(traces, dim=1), pold, pcur, *psi, *xi)


def _forward(case, m, fact, every=0):
    """Traces (shots, nt, receivers) and final field of one model; fact is
    (1, [z,] y, x).  every > 0: recomputed in pieces of `every` steps for
    the gradient."""
    from torch.utils.checkpoint import checkpoint
    n, nd, dev, S = m["n"], len(m["n"]), fact.device, case["shots"]
    coef = _coefficients(case, n, dev)
    t = np.arange(case["nt"]) * _dt(nd)
    u = (math.pi * _f0(nd) * (t - m["t0"])) ** 2
    wav = torch.tensor(_dt(nd) ** 2 / DX ** nd * (1.0 - 2.0 * u) * np.exp(-u), device=dev)
    src = np.concatenate(m["src"]) - 1
    srcs = tuple(torch.tensor(src[:, a].copy(), device=dev) for a in reversed(range(nd)))
    rec = tuple(torch.tensor(m["rec"][:, a] - 1, device=dev) for a in reversed(range(nd)))
    zero = lambda *s: torch.zeros((S,) + s, dtype=torch.float64, device=dev)  # noqa: E731
    dims = list(reversed(n))
    inner = [v - 2 for v in dims]
    state = [zero(*dims), zero(*dims)]
    for k in (1, 2):  # psi on the edges of its axis, xi on the inner nodes
        for a in range(nd):
            s = list(inner)
            s[nd - 1 - a] = n[a] - k
            state.append(zero(*s))
    traces, size = [], every or 50
    for it0 in range(0, case["nt"], size):
        args = (it0, min(case["nt"], it0 + size), fact, coef, srcs, wav, rec, tuple(state))
        got = checkpoint(_steps, *args, use_reentrant=False) if every else _steps(*args)
        traces.append(got[0])
        state = list(got[1:])
    return torch.cat(traces, dim=1), state[1]


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    models = _inputs(case, seed)
    traces, fields = [], []
    for m in models:
        nd = len(m["n"])
        vel = torch.tensor(np.ascontiguousarray(m["vel"].T), device=dev)[None]
        if case["kind"] == "fwi":
            obs = _observed(case, m, np.random.Generator(np.random.PCG64([seed, 1])))
            fact = (_dt(nd) ** 2 * vel ** 2).requires_grad_(True)
            tr, _ = _forward(case, m, fact, every=max(1, int(math.sqrt(case["nt"]))))
            loss = 0.5 * (tr - torch.tensor(obs, device=dev)).pow(2).sum()
            loss.backward()
            g = fact.grad * (2.0 * _dt(nd) ** 2 * vel) if case["autograd"] else fact.grad
            inside = torch.zeros_like(g)
            cut = (slice(None),) + (slice(1, -1),) * nd
            inside[cut] = g[cut]
            g = np.asfortranarray(inside[0].cpu().numpy().T)
            if case["autograd"]:
                return {"misfit": loss.detach().cpu(), "gradient": torch.from_numpy(g)}
            return {"misfit": float(loss.detach()), "gradient": g}
        with torch.no_grad():
            tr, p = _forward(case, m, _dt(nd) ** 2 * vel ** 2)
        traces.append(tr.cpu().numpy())
        fields.append(np.asfortranarray(p[0].cpu().numpy().T) if case["shots"] == 1 else None)
        del tr, p
    if case["kind"] == "solve":
        return {"field": fields[0], "traces": traces[0][0]}
    if case["kind"] == "batch":
        return {"traces": [t[0] for t in traces]}
    return {"traces": traces[0], "field": fields[0]} if case["shots"] == 1 else {"traces": traces[0]}
