"""The work a program has this framework do, as cases that can be timed and checked.

Four kinds of pass, each through the package's public entry points:

* solve: one `Solver.advance` of a mesh (`scenarios.build`), as the reference's time loop calls it; on small meshes the
  state is read back too (`Context.get_state`), as a run that ends in a checkpoint does.
* ensemble: one `Ensemble.advance` of many meshes together.
* predict: `Mlp.forward` of the surrogate network on rows it has not seen.
* train: a few epochs of `Mlp.train` and the weights after them.

Meshes, degrees, materials and the network are those of `scenarios.py` and `surrogate.py`, shortened in steps (and the
largest mesh and the ensemble in size, so that their inputs are quickly made).  A solve starts from a smooth wave field,
as a restarted run does, so that every receiver records a signal from the first step on.  The FP32 modes' rows are
returned as 32-bit values, which is what those modes compute in.
"""
import math

import numpy as np
import torch

import se2dr_fork_amd as S
from se2dr_fork_amd import scenarios as SC
from se2dr_fork_amd import surrogate as SG

L = 4000.0
BYTES_PER_NODE = {"fp64": 72, "fp32": 36, "fp32k": 52}  # read u, v, M (c), write u, v (c)
MEMBER_RECEIVERS = 8


def listed():
    return [
        # the reference program's own default mesh: a quick look, or a regression run
        {"name": "solve_8x8_p2_fp64", "kind": "solve", "mx": 8, "my": 8, "p": 2, "precision": "fp64", "steps": 100,
         "nr": 3, "state": True},
        # the reference's CPU-sized case, a homogeneous block at high degree
        {"name": "solve_64x64_p6_fp64", "kind": "solve", "mx": 64, "my": 64, "p": 6, "precision": "fp64", "steps": 100,
         "nr": 1, "state": True},
        # the headline workload, in the reference's arithmetic and in the compensated FP32 mode
        {"name": "solve_512x512_p4_fp64", "kind": "solve", "mx": 512, "my": 512, "p": 4, "precision": "fp64",
         "steps": 100, "nr": 16, "state": False},
        {"name": "solve_512x512_p4_fp32k", "kind": "solve", "mx": 512, "my": 512, "p": 4, "precision": "fp32k",
         "steps": 100, "nr": 16, "state": False},
        # an odd mesh at a middle degree, in plain FP32
        {"name": "solve_389x263_p5_fp32", "kind": "solve", "mx": 389, "my": 263, "p": 5, "precision": "fp32",
         "steps": 60, "nr": 16, "state": False},
        # high degree in the reference's arithmetic, element counts that divide into no tile
        {"name": "solve_389x301_p7_fp64", "kind": "solve", "mx": 389, "my": 301, "p": 7, "precision": "fp64",
         "steps": 30, "nr": 16, "state": False},
        # the largest mesh: degree 8, 16.8 million nodes
        {"name": "solve_512x512_p8_fp32", "kind": "solve", "mx": 512, "my": 512, "p": 8, "precision": "fp32",
         "steps": 40, "nr": 64, "state": False},
        # an uneven ensemble at degree 6
        {"name": "ensemble_24_p6_fp32", "kind": "ensemble", "members": 24, "lo": 64, "hi": 192, "p": 6,
         "precision": "fp32", "steps": 50},
        # the surrogate's training-data generator: equal meshes, many at a time
        {"name": "ensemble_64_p4_fp32", "kind": "ensemble", "members": 64, "lo": 96, "hi": 96, "p": 4,
         "precision": "fp32", "steps": 60},
        # one question to the trained surrogate, and a survey of many
        {"name": "predict_1", "kind": "predict", "rows": 1},
        {"name": "predict_512", "kind": "predict", "rows": 512},
        # ten epochs of the surrogate's training
        {"name": "train_2048", "kind": "train", "rows": 2048, "batch": 256, "epochs": 10},
    ]


def draw(rng):
    """One more case of the same ranges: meshes of 300 to 16 million nodes (FP32 from half a million, where its use
    begins), every degree from 2 to 8, uneven ensembles, any number of rows."""
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["solve", "solve", "solve", "solve", "ensemble", "predict", "train"])
    if kind == "solve":
        precision = rng.choice(["fp64", "fp64", "fp32", "fp32k"])
        p = rng.randint(2, 8)
        nodes = log_uniform(300, 6.0e6) if precision == "fp64" else log_uniform(5.0e5, 1.6e7)
        aspect = rng.uniform(0.5, 2.0)
        mx = max(3, int(round(math.sqrt(nodes * aspect) / p)))
        my = max(3, int(round(math.sqrt(nodes / aspect) / p)))
        nn = (p * mx + 1) * (p * my + 1)
        steps = max(10, min(100, int(2.0e8 / nn)))
        return {"kind": kind, "mx": mx, "my": my, "p": p, "precision": precision, "steps": steps,
                "nr": rng.randint(1, 64), "state": nn < 200000}
    if kind == "ensemble":
        lo = rng.randint(48, 128)
        return {"kind": kind, "members": rng.randint(9, 24), "lo": lo, "hi": lo + rng.randint(0, 64),
                "p": rng.randint(3, 6), "precision": rng.choice(["fp32", "fp32", "fp64"]), "steps": rng.randint(10, 30)}
    if kind == "predict":
        return {"kind": kind, "rows": int(round(log_uniform(1, 1000)))}
    return {"kind": kind, "rows": rng.randint(520, 2048), "batch": rng.choice([128, 192, 256]),
            "epochs": rng.randint(1, 8)}


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def gll(p):
    """GLL nodes, weights and derivative matrix D[q][i] = l_i'(x_q) of degree p."""
    leg = np.polynomial.legendre
    c = np.zeros(p + 1)
    c[p] = 1.0
    inner = np.sort(leg.legroots(leg.legder(c))) if p > 1 else np.zeros(0)
    for _ in range(3):  # Newton on P'_p
        d1, d2 = leg.legval(inner, leg.legder(c)), leg.legval(inner, leg.legder(c, 2))
        inner = inner - d1 / d2
    x = np.concatenate([[-1.0], inner, [1.0]])
    lp = leg.legval(x, c)
    w = 2.0 / (p * (p + 1) * lp * lp)
    D = np.zeros((p + 1, p + 1))
    for q in range(p + 1):
        for i in range(p + 1):
            if q != i:
                D[q, i] = lp[q] / (lp[i] * (x[q] - x[i]))
    D[0, 0], D[p, p] = -p * (p + 1) / 4.0, p * (p + 1) / 4.0
    return x, w, D


def scenario_of(rs, mx, my, p, steps, nr, ns):
    """A heterogeneous block of [0, L]^2, ns explosions and nr receivers.  Sources and receivers stand a hundredth of
    an element from an interior GLL node, so which node is nearest is beyond doubt; returns their elements and local
    node numbers too."""
    ne = mx * my
    vp = rs.uniform(4000.0, 6000.0, ne)
    rho = rs.uniform(2500.0, 3000.0, ne)
    x, _, _ = gll(p)
    hx, hy = L / mx, L / my

    def stand(n):
        ex, ey = rs.randint(1, mx - 1, n), rs.randint(1, my - 1, n)
        gi, gj = rs.randint(1, p, n), rs.randint(1, p, n)
        xy = np.stack([(ex + 0.5 * (1 + x[gi]) + 0.01) * hx, (ey + 0.5 * (1 + x[gj]) - 0.01) * hy], axis=1)
        return (ex, ey, gi, gj), xy

    src, src_xy = stand(ns)
    rec, rec_xy = stand(nr)
    f0 = rs.uniform(5.0, 20.0, ns)
    sc = SC.Scenario(name="case", mx=mx, my=my, p=p, scale=(L, L), shift=(0.0, 0.0), vp=vp, vs=vp / math.sqrt(3.0),
                     rho=rho, src_xy=src_xy, src_type=[S.SOURCE_MOMENT] * ns,
                     src_values=np.tile([1.0e9, 0.0, 0.0, 1.0e9], (ns, 1)),
                     stf=[("ricker", 0.0, float(f), 1.0) for f in f0], rec_xy=rec_xy, cfl_factor=0.2, nt=steps)
    return sc, src, rec


def field_of(rs, mx, my, p):
    """u, v, a in DMDA order: a few plane standing waves of some hundred metres (displacements of millimetres)."""
    x, _, _ = gll(p)

    def axis(m):
        return np.append((np.arange(m)[:, None] + 0.5 * (1 + x[:-1])[None, :]).reshape(-1), m) * (L / m)

    gx, gy = axis(mx), axis(my)
    out = []
    for size in (1.0e-3, 5.0e-2, 0.0):
        f = np.zeros((len(gy), len(gx), 2))
        if size:
            for c in range(2):
                for _ in range(2):
                    kx, ky = rs.uniform(0.5, 3.0, 2) * 2.0 * math.pi / 1000.0
                    f[:, :, c] += size * np.outer(np.cos(ky * gy + rs.uniform(0, 6)), np.cos(kx * gx + rs.uniform(0, 6)))
        out.append(f.reshape(-1))
    return out


def members_of(case, seed):
    """(scenario, sources, receivers, field) of every mesh of a solve (one) or an ensemble."""
    rs = np.random.RandomState(seed)
    if case["kind"] == "solve":
        sizes = [(case["mx"], case["my"])]
        nr, ns = case["nr"], 2
    else:
        sizes = [tuple(rs.randint(case["lo"], case["hi"] + 1, 2)) for _ in range(case["members"])]
        nr, ns = MEMBER_RECEIVERS, 1
    for mx, my in sizes:
        sc, src, rec = scenario_of(rs, int(mx), int(my), case["p"], case["steps"], nr, ns)
        yield sc, src, rec, field_of(rs, int(mx), int(my), case["p"])


def network_of(rs):
    """Weights of a network that has been trained a little: the uniform draw that training starts from, packed layer by
    layer, weights then biases."""
    p = []
    for i, o in zip(SG.WIDTHS[:-1], SG.WIDTHS[1:]):
        b = 1.0 / math.sqrt(i)
        p += [rs.uniform(-b, b, o * i), rs.uniform(-b, b, o)]
    return np.concatenate(p).astype(np.float32)


def rows_of(rs, n):
    """Inputs as `surrogate.encode` makes them, and outputs of unit size."""
    x = np.concatenate([rs.uniform(-16.0, 16.0, (n, 2)), SG.SIGMA * rs.normal(size=(n, 64))], axis=1).astype(np.float32)
    t = rs.normal(size=(n, SG.WIDTHS[-1])).astype(np.float32)
    return x, t


# ---------------------------------------------------------------------------
# the passes
# ---------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] in ("solve", "ensemble"):
        builts = []
        for sc, _, _, field in members_of(case, seed):
            b = SC.build(sc, precision=S.PRECISIONS[case["precision"]])
            b.solver.ctx.set_state(*field)
            b.solver.reserve(case["steps"])
            builts.append(b)
        ens = None
        if case["kind"] == "ensemble":
            ens = S.Ensemble([b.solver for b in builts])
            ens.autotune(steps=5, reps=2)
        return {"case": case, "builts": builts, "ens": ens}
    rs = np.random.RandomState(seed)
    net = S.Mlp(SG.WIDTHS, batch=case.get("batch", 256))
    net.set_params(network_of(rs))
    x, t = rows_of(rs, case["rows"])
    if case["kind"] == "train":
        net.set_data(x, t)
    return {"case": case, "net": net, "x": x}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "predict":
        return {"y": state["net"].forward(state["x"])}
    if kind == "train":
        losses = state["net"].train(case["epochs"], lr=1e-3, seed=7)
        return {"losses": losses, "params": state["net"].params()}
    rows = np.float64 if case["precision"] == "fp64" else np.float32
    if kind == "ensemble":
        res = state["ens"].advance(case["steps"], [b.dt for b in state["builts"]])
        return {"trace": np.stack([tr for _, tr in res]).astype(rows, copy=False)}
    b = state["builts"][0]
    _, trace = b.solver.advance(case["steps"], b.dt)
    out = {"trace": trace.astype(rows, copy=False)}
    if case["state"]:
        out["u"], out["v"], out["a"] = (f.astype(rows, copy=False) for f in b.solver.ctx.get_state())
    return out


def work(case):
    if case["kind"] in ("solve", "ensemble"):
        p, nb = case["p"], case["p"] + 1
        if case["kind"] == "solve":
            elements = case["mx"] * case["my"]
            nodes = (p * case["mx"] + 1) * (p * case["my"] + 1)
        else:
            mean = 0.5 * (case["lo"] + case["hi"])
            elements = case["members"] * mean * mean
            nodes = case["members"] * (p * mean + 1) ** 2
        return {"bytes": case["steps"] * nodes * BYTES_PER_NODE[case["precision"]],
                "flops": case["steps"] * elements * (16 * nb ** 3 + 20 * nb ** 2)}
    weights = sum(i * o for i, o in zip(SG.WIDTHS[:-1], SG.WIDTHS[1:]))
    io = 4 * (SG.WIDTHS[0] + SG.WIDTHS[-1]) * case["rows"]
    if case["kind"] == "predict":
        return {"bytes": 2 * weights + io, "flops": 2 * weights * case["rows"]}
    steps = case["epochs"] * (case["rows"] // case["batch"])
    # weights and both moments read and written each step; weights back to the host
    return {"bytes": steps * 24 * weights + 4 * weights + io, "flops": 6 * weights * case["batch"] * steps}


# ---------------------------------------------------------------------------
# the same in 64 bits, from the mathematics alone
# ---------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] in ("solve", "ensemble"):
        traces, fields = [], None
        for sc, src, rec, field in members_of(case, seed):
            trace, fields = wave(sc, src, rec, field, case["steps"])
            traces.append(trace)
        if case["kind"] == "ensemble":
            return {"trace": np.stack(traces)}
        out = {"trace": traces[0]}
        if case["state"]:
            out["u"], out["v"], out["a"] = fields
        return out
    rs = np.random.RandomState(seed)
    params, (x, t) = network_of(rs), rows_of(rs, case["rows"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    ws, o = [], 0
    for i, n in zip(SG.WIDTHS[:-1], SG.WIDTHS[1:]):
        for shape in ((n, i), (n,)):
            k = int(np.prod(shape))
            ws.append(torch.from_numpy(params[o:o + k].astype(np.float64).reshape(shape)).to(dev))
            o += k
    x, t = torch.from_numpy(x).double().to(dev), torch.from_numpy(t).double().to(dev)

    def forward(h):
        for k in range(0, len(ws), 2):
            h = h @ ws[k].t().contiguous() + ws[k + 1]
            if k + 2 < len(ws):
                h = torch.nn.functional.gelu(h)
        return h

    if case["kind"] == "predict":
        return {"y": forward(x).cpu().numpy()}
    n, batch = case["rows"], case["batch"]
    s, mask = 7, (1 << 64) - 1
    for w in ws:
        w.requires_grad_(True)
    opt = torch.optim.Adam(ws, lr=float(np.float32(1e-3)), betas=(0.9, 0.999), eps=1e-8)
    nb, losses = n // batch, []
    for _ in range(case["epochs"]):
        order, loss_sum = list(range(n)), 0.0
        for i in range(n - 1, 0, -1):  # Fisher-Yates on a splitmix64 stream
            s = (s + 0x9E3779B97F4A7C15) & mask
            z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            j = int(((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0) * (i + 1))
            order[i], order[j] = order[j], order[i]
        for k in range(nb):
            rows = torch.tensor(order[k * batch:(k + 1) * batch], device=dev)
            opt.zero_grad()
            loss = ((forward(x[rows]) - t[rows]) ** 2).mean()
            loss.backward()
            opt.step()
            loss_sum += float(loss.detach()) / nb
        losses.append(loss_sum)
    return {"losses": np.array(losses), "params": torch.cat([w.detach().reshape(-1) for w in ws]).cpu().numpy()}


def wave(sc, src, rec, field, steps):
    """`steps` velocity-Verlet steps of the spectral-element wave equation in 64 bits: receiver rows and final fields."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    mx, my, p, nb = sc.mx, sc.my, sc.p, sc.p + 1
    x, w, D = gll(p)
    jx, jy = 0.5 * L / mx, 0.5 * L / my
    mu = sc.vs ** 2 * sc.rho
    lam = sc.vp ** 2 * sc.rho - 2.0 * mu
    # the scenario's share of half the smallest node spacing over the fastest P wave
    dt = sc.cfl_factor * min(jx, jy) * float(np.diff(x).min()) / float(sc.vp.max())

    def cells(v):
        return torch.from_numpy(np.ascontiguousarray(v.reshape(my, mx, 1, 1))).to(dev)

    lam, mu, rho = cells(lam), cells(mu), cells(sc.rho)
    fac = torch.from_numpy(np.outer(w, w) * jx * jy).to(dev)
    Dt = torch.from_numpy(D).to(dev)
    DtT = Dt.t().contiguous()
    nx, ny = p * mx + 1, p * my + 1

    def add_up(fe):  # [my][mx][j][i] -> [ny][nx]
        out = torch.zeros(ny, nx, dtype=torch.float64, device=dev)
        for j in range(nb):
            for i in range(nb):
                out[j:j + p * (my - 1) + 1:p, i:i + p * (mx - 1) + 1:p] += fe[:, :, j, i]
        return out

    def elements(f):
        return f.unfold(0, nb, p).unfold(1, nb, p).contiguous()

    def d_x(e):
        return (e.reshape(-1, nb) @ DtT).reshape(e.shape) / jx

    def d_y(e):
        return (e.transpose(2, 3).contiguous().reshape(-1, nb) @ DtT).reshape(e.shape).transpose(2, 3) / jy

    def d_xt(s):
        return (s.contiguous().reshape(-1, nb) @ Dt).reshape(s.shape) / jx

    def d_yt(s):
        return (s.transpose(2, 3).contiguous().reshape(-1, nb) @ Dt).reshape(s.shape).transpose(2, 3) / jy

    mass = add_up(rho * fac)
    u, v, a = (list(torch.from_numpy(f.reshape(ny, nx, 2)).to(dev).unbind(2)) for f in field)
    u, v, a = [c.contiguous() for c in u], [c.contiguous() for c in v], [c.contiguous() for c in a]
    se_x, se_y, sgi, sgj = src
    re_x, re_y, rgi, rgj = rec
    ri = torch.from_numpy(re_x * p + rgi).to(dev)
    rj = torch.from_numpy(re_y * p + rgj).to(dev)
    k = torch.arange(nb, device=dev)
    row_i = torch.from_numpy(re_x * p).to(dev)[:, None] + k
    col_j = torch.from_numpy(re_y * p).to(dev)[:, None] + k
    Dgi, Dgj = Dt[torch.from_numpy(rgi).to(dev)], Dt[torch.from_numpy(rgj).to(dev)]
    rows, t = [], 0.0
    for _ in range(steps):
        t += dt
        for c in range(2):
            u[c] = u[c] + dt * v[c] + 0.5 * dt * dt * a[c]
            v[c] = v[c] + 0.5 * dt * a[c]
        ex, ey = elements(u[0]), elements(u[1])
        xx, yy, xy = d_x(ex), d_y(ey), d_y(ex) + d_x(ey)
        sxx, syy, sxy = fac * ((lam + 2 * mu) * xx + lam * yy), fac * (lam * xx + (lam + 2 * mu) * yy), fac * mu * xy
        f = [-add_up(d_xt(sxx) + d_yt(sxy)), -add_up(d_xt(sxy) + d_yt(syy))]
        for s in range(len(se_x)):
            arg = math.pi * sc.stf[s][2] * (t - sc.stf[s][1])
            psi = (1.0 - 2.0 * arg * arg) * math.exp(-arg * arg)
            i0, j0 = int(se_x[s]) * p, int(se_y[s]) * p
            m = sc.src_values[s]
            dx, dy = Dt[int(sgi[s])] / jx, Dt[int(sgj[s])] / jy
            for c in range(2):
                f[c][j0 + int(sgj[s]), i0:i0 + nb] += psi * m[2 * c] * dx
                f[c][j0:j0 + nb, i0 + int(sgi[s])] += psi * m[2 * c + 1] * dy
        for c in range(2):
            a[c] = f[c] / mass
            v[c] = v[c] + 0.5 * dt * a[c]
        curl = (v[1][rj[:, None], row_i] * Dgi).sum(1) / jx - (v[0][col_j, ri[:, None]] * Dgj).sum(1) / jy
        rows.append(torch.stack([f[rj, ri] for f in (u[0], u[1], v[0], v[1], a[0], a[1])] + [curl], dim=1))
    fields = [torch.stack(f, dim=2).reshape(-1).cpu().numpy() for f in (u, v, a)]
    return torch.stack(rows).cpu().numpy(), fields
