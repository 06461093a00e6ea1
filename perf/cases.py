"""Timed workloads of the ComputeUnit library, through its public entry points.

A case is one stretch of work as the programs of this repository do it between
two looks at the results: a stirred tank advanced and sampled (the accuracy
runs and the headline benchmark), the driver's loop with its output planes, the
per-call operators of the reference, a batch of tanks, a served stream of
requests.  Sizes are those of the benchmark, the tests and the example inputs,
and generic ones around them.

kind "tank"    run(steps), then the FP64 sums and the macroscopic field
kind "driver"  run(steps), then the exclusion mask, the two vorticity pictures
               and the XZ plane records that the driver writes every tenth step
kind "calls"   steps of the reference's operators with point lists from the host
kind "batch"   a batch of tanks of mixed edges advanced together, then each sampled
kind "serve"   requests submitted to a server and ticked until all have finished
"""
import math

import numpy as np
import torch

import tdlbcpp_amd as td

PRECISIONS = {"fp32": td.PREC_F32, "fp64": td.PREC_F64, "fp16": td.PREC_F16, "bf16": td.PREC_BF16,
              "e3m12": td.PREC_E3M12}
LAYOUTS = {"IJKL": td.LAYOUT_IJKL, "LIJK": td.LAYOUT_LIJK, "IJKL_SOA": td.LAYOUT_IJKL_SOA}
STREAMINGS = {"Simple": td.STREAM_SIMPLE, "Esotwist": td.STREAM_ESOTWIST}
POP_BYTES = {"fp32": 4, "fp64": 8, "fp16": 2, "bf16": 2, "e3m12": 2}
NU_BYTES = POP_BYTES
BATCH_EDGES = (48, 64, 96, 128, 160)  # the batched workload's grid edges
WARM = 20                             # steps a tank has taken before the first pass
STARTUP = 30                          # start-up ramp of the impeller (the example inputs)


def _case(name, kind, edge, steps, precision="fp32", streaming="Esotwist", layout="LIJK", tanks=1):
    return {"name": name, "kind": kind, "edge": edge, "steps": steps, "precision": precision,
            "streaming": streaming, "layout": layout, "tanks": tanks}


def listed():
    return [
        # the smallest tank that the tests and small studies run: launches and latency only
        _case("tank_24_fp32", "tank", 24, 20),
        # the example input: 60^3, pictures and plane records every tenth step, Simple streaming in the reference's layout
        _case("driver_60_simple_ijkl", "driver", 60, 10, streaming="Simple", layout="IJKL"),
        # the accuracy workload between two of its samples, in the format that meets its bar
        _case("tank_96_e3m12", "tank", 96, 62, "e3m12"),
        # a single tank of no round size, as requests bring them
        _case("tank_131_fp16", "tank", 131, 50, "fp16"),
        # the reference of the accuracy runs at their larger size
        _case("tank_192_fp64", "tank", 192, 62, "fp64"),
        # the reference's walls and layout at an ordinary size
        _case("tank_150_simple_ijkl", "tank", 150, 50, streaming="Simple", layout="IJKL"),
        # the reference's GPU layout
        _case("tank_256_ijkl", "tank", 256, 100, layout="IJKL"),
        # the headline tank, FP32 and 16-bit storage
        _case("tank_512_fp32", "tank", 512, 100),
        _case("tank_512_fp16", "tank", 512, 100, "fp16"),
        # the reference's loop call by call, lists from the host each step
        _case("calls_60_simple", "calls", 60, 5, streaming="Simple"),
        # independent tanks batched, edges of the benchmark's batch
        _case("batch_32_fp16", "batch", 0, 100, "fp16", tanks=32),
        # a few requests through the server, below its capacity
        _case("serve_6_fp16", "serve", 64, 200, "fp16", tanks=6),
    ]


def draw(rng):
    """A case of the listed ranges: edges log-uniform from 24 to 448 (odd ones as likely as even), the
    storage formats, streamings and layouts of the benchmark's variants."""
    kind = rng.choices(("tank", "driver", "calls", "batch", "serve"), (10, 2, 2, 2, 1))[0]

    def edge(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "batch":
        c = _case("", kind, 0, rng.randint(20, 60), rng.choice(("fp32", "fp16", "bf16", "e3m12")), "Esotwist",
                  rng.choice(("LIJK", "LIJK", "IJKL_SOA")), tanks=rng.randint(3, 24))
    elif kind == "serve":
        c = _case("", kind, edge(40, 90), rng.randint(100, 250), rng.choice(("fp16", "e3m12")), tanks=rng.randint(2, 6))
    elif kind == "calls":
        c = _case("", kind, edge(24, 100), rng.randint(2, 5), rng.choice(("fp32", "fp32", "fp64")),
                  rng.choice(("Simple", "Esotwist")), rng.choice(("IJKL", "LIJK")))
    elif kind == "driver":
        c = _case("", kind, edge(24, 200), rng.randint(5, 20), rng.choice(("fp32", "fp16")),
                  rng.choice(("Simple", "Esotwist")), rng.choice(("IJKL", "LIJK", "IJKL_SOA")))
    else:
        precision = rng.choice(("fp32", "fp32", "fp16", "e3m12", "bf16", "fp64"))
        e = edge(24, 448 if precision != "fp64" else 256)
        c = _case("", kind, e, rng.randint(20, 80), precision, rng.choice(("Esotwist", "Esotwist", "Simple")),
                  rng.choice(("LIJK", "LIJK", "IJKL", "IJKL_SOA")))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
def _conditions(case, seed):
    """Per tank: edge, tip speed, Reynolds number and impeller angle at the start, from the seed
    (the distributions of the batched and served workloads)."""
    rng = np.random.default_rng(seed)
    n = case["tanks"]
    if case["kind"] == "batch":  # the same edges whatever the seed: the work is the case's
        edges = np.random.default_rng(case["tanks"]).choice(BATCH_EDGES, size=n)
    elif case["kind"] == "serve":
        edges = np.round(case["edge"] * np.exp(np.linspace(0.0, math.log(2.0), n)))
    else:
        edges = [case["edge"]] * n
    return [{"edge": int(e), "tip": float(rng.uniform(0.05, 0.12)), "re": float(rng.uniform(2e3, 2e4)),
             "angle": float(rng.uniform(0.0, math.pi / 3))} for e in edges]


def _tank(case, cond, bind=True):
    precision = PRECISIONS[case["precision"]]
    flow = td.flow_for_tank(cond["edge"], re=cond["re"], uav=cond["tip"], cs0=0.1, use_les=1, precision=precision)
    cu = td.ComputeUnit(cond["edge"], layout=LAYOUTS[case["layout"]], streaming=STREAMINGS[case["streaming"]],
                        precision=precision, **flow)
    cu.initialise(1.0)
    rp = td.rushton_defaults(cond["edge"], tip_speed=cond["tip"], startup_steps=STARTUP)
    if bind:
        cu.bind_rushton(rp, step=1, angle=cond["angle"])
    return cu, rp


def _calls_step(state):
    """One iteration of the reference's main loop through its operators."""
    cu, rp = state["cu"], state["rp"]
    cu.step += 1
    delta = td.rushton_step_increment(rp, cu.step)
    cu.angle += delta
    points = np.concatenate([state["static"], td.rushton_generate(rp, td.GEOM_ROTATING, cu.angle, delta)])
    cu.collision()
    cu.bounce_back()
    cu.streaming_push()
    cu.moments()
    cu.forcing(points, 0.97, 1.9)


def prepare(case, seed):
    conds = _conditions(case, seed)
    state = {"case": case}
    if case["kind"] == "serve":
        state["requests"] = conds
        state["server"] = td.Server(PRECISIONS[case["precision"]], LAYOUTS[case["layout"]],
                                    STREAMINGS[case["streaming"]], tick_steps=50, keep_handles=True)
    elif case["kind"] == "batch":
        state["cus"] = [_tank(case, c)[0] for c in conds]
        batch = td.Batch(PRECISIONS[case["precision"]], LAYOUTS[case["layout"]], STREAMINGS[case["streaming"]])
        for cu in state["cus"]:
            batch.add(cu, 1 << 40)
        batch.run(WARM)
        state["batch"] = batch
    elif case["kind"] == "calls":
        cu, rp = _tank(case, conds[0], bind=False)
        cu.step, cu.angle = 1, conds[0]["angle"]
        delta = td.rushton_step_increment(rp, 1)
        state["static"] = np.concatenate([td.rushton_generate(rp, td.GEOM_FIXED),
                                          td.rushton_generate(rp, td.GEOM_ROTATING_NON_UPDATING, 0.0, delta)])
        cu.forcing(np.concatenate([state["static"], td.rushton_generate(rp, td.GEOM_ROTATING, cu.angle, delta)]),
                   0.97, 1.9)
        state["cu"], state["rp"] = cu, rp
        _calls_step(state)
    else:
        cu, state["rp"] = _tank(case, conds[0])
        cu.run(WARM)
        state["cu"] = cu
    return state


# ---------------------------------------------------------------- one pass
def _sums(cu):
    r = cu.reductions()
    return np.array([r["mass"], *r["momentum"], *r["force"], r["torque"]])


def run(state):
    case = state["case"]
    if case["kind"] == "serve":
        server, tickets = state["server"], []
        for q in state["requests"]:
            tickets.append((server.submit(q["edge"], q["tip"], q["re"], case["steps"], STARTUP), q["edge"]))
        done = {}
        while len(done) < len(tickets):
            server.tick()
            done.update((r["ticket"], r) for r in server.poll())
        out = {"results": np.array([[done[t][f] for f in ("mass", "mass_drift", "torque", "power_number")]
                                    for t, _ in tickets]),
               "errors": np.array([done[t]["error"] for t, _ in tickets])}
        for n, (ticket, edge) in enumerate(tickets):
            cu = server.take(ticket, edge)
            out["field%02d" % n] = cu.macroscopic()
            cu.close()
        return out
    if case["kind"] == "batch":
        state["batch"].run(case["steps"])
        return {"sums": np.array([_sums(cu) for cu in state["cus"]]),
                "fields": [cu.macroscopic() for cu in state["cus"]]}
    cu = state["cu"]
    if case["kind"] == "calls":
        for _ in range(case["steps"]):
            _calls_step(state)
        return {"field": cu.macroscopic(), "F": cu.get(td.FIELD_F), "Nu": cu.get(td.FIELD_NU),
                "Q": cu.get(td.FIELD_Q)}
    cu.run(case["steps"])
    if case["kind"] == "driver":
        exclude = cu.output_exclude()
        q, f = cu.plane_xz(2 * case["edge"] // 3, exclude)
        return {"exclude": exclude, "xy": cu.vorticity(1, case["edge"] // 2, exclude),
                "xz": cu.vorticity(0, 2 * case["edge"] // 3, exclude),
                "plane_q": np.ascontiguousarray(q["q"]), "plane_f": np.ascontiguousarray(f["q"]),
                "field": cu.macroscopic()}
    return {"sums": _sums(cu), "field": cu.macroscopic()}


def work(case):
    """Each population and eddy viscosity read and written once a step, the results written once; about
    400 operations a cell and step."""
    p = case["precision"]
    cell = 36 * POP_BYTES[p] + 2 * NU_BYTES[p]
    if case["kind"] == "calls":  # collision, push and moments are calls of their own
        cell += 2 * 36 * POP_BYTES[p]
    out = 32 if p == "fp64" else 16
    cells = sum(c["edge"] ** 3 for c in _conditions(case, 0))
    return {"bytes": cells * (cell * case["steps"] + out), "flops": 400.0 * cells * case["steps"]}


# ---------------------------------------------------------------- the same in 64 bits
DIRS = np.array([(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, -1, 0),
                 (1, 0, 1), (-1, 0, -1), (0, 1, 1), (0, -1, -1), (1, -1, 0), (-1, 1, 0), (1, 0, -1), (-1, 0, 1),
                 (0, 1, -1), (0, -1, 1)])


def _moment_matrix():
    x, y, z = DIRS.T.astype(np.float64)
    x2, y2, z2 = x * x, y * y, z * z
    e2 = x2 + y2 + z2
    return np.stack([np.ones(18), x, y, z, x2 + e2 - 2, x * y, y2 + e2 - 2, x * z, y * z, z2 + e2 - 2,
                     x * (3 * y2 - 1), y * (3 * x2 - 1), x * (3 * y2 + 6 * z2 - 3), y * (3 * x2 + 6 * z2 - 3),
                     z * (3 * x2 + 3 * y2 - 2), z * (3 * y2 - 3 * x2), np.where(x2 + y2 == 1, 0.5, -1.0),
                     1.5 * (x2 - y2) * (1 - 2 * z2)])


def _ring(T, r, j, omega, least):
    c = (T - 1.0) / 2.0
    if r <= 0.0:
        return [(c, c, j, 0.0, 0.0)]
    n = max(least, math.ceil(2 * math.pi * r))
    th = [2 * math.pi * a / n for a in range(n)]
    return [(c + r * math.cos(t), c + r * math.sin(t), j, -omega * r * math.sin(t), omega * r * math.cos(t)) for t in th]


def _centre(p):
    return math.floor(p[0] + 0.5), math.floor(p[1] + 0.5)


def _by_colour(points):
    return sorted(points, key=lambda p: 3 * (_centre(p)[0] % 3) + _centre(p)[1] % 3)


def _tank_points(T, omega):
    """Tank wall, baffles, disk, hub and shaft of the Rushton tank: (x, z, j, u, w) in list order."""
    c, D = (T - 1.0) / 2.0, T / 3.0
    disk, hb = min(int(D), T - 1), max(1, int(math.floor(D / 5.0 + 0.5)))
    lo = max(0, disk - hb // 2)
    hi = lo + min(hb + 1, T - lo)
    fixed = [p for j in range(T) for p in _ring(T, c, j, 0.0, 8)]
    for b in range(4):
        th = math.pi / 4 + math.pi / 2 * b
        for j in range(T):
            r = c - T / 10.0
            while r < c - 0.5:
                fixed.append((c + r * math.cos(th), c + r * math.sin(th), j, 0.0, 0.0))
                r += 1.0
    turning = [p for r in range(int(3.0 * D / 8.0) + 1) for p in _ring(T, float(r), disk, omega, 1)]
    turning += [p for j in range(lo, hi) if j != disk for p in _ring(T, D / 8.0, j, omega, 4)]
    turning += [p for j in range(hi, T) for p in _ring(T, D / 12.0, j, omega, 4)]
    return _by_colour(fixed) + _by_colour(turning), lo, hi


def _blade_points(T, lo, hi, angle, omega):
    c, D, outer = (T - 1.0) / 2.0, T / 3.0, float(int(T / 6.0))
    inner = outer - D / 4.0
    n_radial = int(math.floor(outer - inner + 1e-9)) + 1
    ncol = 6 if 2.0 * inner * math.sin(math.pi / 3) < 3.0 * math.sqrt(2.0) + 1e-9 else 2
    out = []
    for col in range(ncol):
        for rmod in range(5):
            for b in range(col, 6, ncol):
                th = angle + 2 * math.pi * b / 6
                for j in range(lo, hi):
                    for r in range(rmod, n_radial, 5):
                        rad = inner + r
                        out.append((c + rad * math.cos(th), c + rad * math.sin(th), j, -omega * rad * math.sin(th),
                                    omega * rad * math.cos(th)))
    return out


def _weight(x):
    a = x.abs()
    near = (1.0 + torch.sqrt((1.0 - 3.0 * a * a).clamp(min=0.0))) / 3.0
    far = (5.0 - 3.0 * a - torch.sqrt((1.0 - 3.0 * (1.0 - a) ** 2).clamp(min=0.0))) / 6.0
    return torch.where(a <= 0.5, near, torch.where(a <= 1.5, far, torch.zeros_like(a)))


class _Points:
    """A point list in order, as levels of points with disjoint stencils that give what the sequence gives."""

    def __init__(self, points, T, device):
        last, levels = {}, []
        for n, p in enumerate(points):
            i, k = _centre(p)
            cells = [((i + a) % T * T + p[2]) * T + (k + b) % T for b in (-1, 0, 1) for a in (-1, 0, 1)]
            level = 1 + max(last.get(q, -1) for q in cells)
            for q in cells:
                last[q] = level
            if level == len(levels):
                levels.append(([], []))
            levels[level][0].append(n)
            levels[level][1].append(cells)
        a = np.array(points, dtype=np.float64).reshape(-1, 5)
        frac = torch.tensor(a[:, :2] - np.floor(a[:, :2] + 0.5), device=device)
        off = torch.tensor([-1.0, 0.0, 1.0], dtype=torch.float64, device=device)
        w = _weight(off[None, None, :] - frac[:, :, None])  # per point and axis: the three weights
        w9 = (w[:, 1, :, None] * w[:, 0, None, :]).reshape(-1, 9)
        v = torch.tensor(np.stack([a[:, 3], np.zeros(len(a)), a[:, 4]], 1), device=device)
        self.levels = [(torch.tensor(c, device=device), w9[torch.tensor(n, device=device)],
                        v[torch.tensor(n, device=device)]) for n, c in levels]
        self.cells = torch.unique(torch.cat([c.reshape(-1) for c, _, _ in self.levels]))

    def force(self, rho, j, F, alfa=0.97, beta=1.9):
        for cells, w, v in self.levels:
            f = F[cells]
            wc = w[:, :, None]
            s = (wc * (j[cells] + 0.5 * f)).sum(1) - (w * rho[cells]).sum(1)[:, None] * v
            F[cells] = alfa * f - beta * wc * s[:, None, :]


def _increment(T, tip, step):
    full = tip / float(int(T / 6.0))
    return 0.5 * full * (1.0 - math.cos(math.pi * step / STARTUP)) if step < STARTUP else full


def _reference(case, cond, steps):
    """The tank after `steps` main-loop steps from rest: rho, j, F, Nu per interior cell, in 64 bits."""
    T, dev = cond["edge"], torch.device("cuda" if torch.cuda.is_available() else "cpu")
    M = torch.tensor(_moment_matrix(), device=dev)
    inverse = torch.linalg.inv(M)
    n = T ** 3
    m = torch.zeros(18, n, dtype=torch.float64, device=dev)
    m[0] = 1.0
    F = torch.zeros(n, 3, dtype=torch.float64, device=dev)
    nuc = torch.zeros(n, dtype=torch.float64, device=dev)
    nu0 = cond["tip"] * int(T / 6) / (cond["re"] * math.pi / 2.0)
    omega = _increment(T, cond["tip"], 1)
    angle = cond["angle"]
    static, lo, hi = _tank_points(T, omega)
    static = _Points(static, T, dev)

    def forcing(F, omega):
        blades = _Points(_blade_points(T, lo, hi, angle, omega), T, dev)
        new = torch.zeros_like(F)
        for cells in (static.cells, blades.cells):
            new[cells] = F[cells]
        j = m[1:4].T.contiguous()
        static.force(m[0], j, new)
        blades.force(m[0], j, new)
        return new

    F = forcing(F, omega)
    for step in range(2, steps + 2):
        omega = _increment(T, cond["tip"], step)
        angle += omega
        # collision with the Smagorinsky eddy viscosity
        rho = m[0]
        u = (m[1:4] + 0.5 * F.T) / rho
        fct = 3.0 / (rho * (1.0 + 6.0 * (nuc + nu0)))
        h = 0.5 * F.T
        normal = [fct * (m[1 + a] + h[a] * u[a] - m[r]) for a, r in ((0, 4), (1, 6), (2, 9))]
        shear = [2.0 * fct * (m[1 + a] + h[a] * u[b] - m[r]) for a, b, r in ((1, 0, 5), (2, 0, 7), (2, 1, 8))]
        div = normal[0] + normal[1] + normal[2]
        sh = 2.0 * sum(s * s for s in normal) + sum(s * s for s in shear) - (2.0 / 3.0) * div * div
        nuc = 0.1 * 0.1 * sh.abs().sqrt()
        nut6 = 6.0 * (nuc + nu0)
        b, c = 1.0 / (1.0 + nut6), 1.0 - nut6
        j2 = 2.0 * m[1:4] + F.T
        a = torch.empty_like(m)
        a[0] = rho
        a[1:4] = m[1:4] + F.T
        for r, p, q in ((4, 0, 0), (5, 0, 1), (6, 1, 1), (7, 0, 2), (8, 1, 2), (9, 2, 2)):
            a[r] = (j2[p] * u[q] - m[r] * c) * b
        a[10:16] = -0.8 * m[10:16]
        a[16:] = 0.0
        f = (inverse @ a).reshape(18, T, T, T)
        # streaming: periodic, or keeping the own value where the source lies outside the walls
        g = torch.empty_like(f)
        for d, e in enumerate(DIRS.tolist()):
            g[d] = torch.roll(f[d], e, (0, 1, 2))
            if case["streaming"] == "Simple":
                for axis, s in enumerate(e):
                    if s:
                        g[d].select(axis, 0 if s > 0 else T - 1).copy_(f[d].select(axis, 0 if s > 0 else T - 1))
        m = M @ g.reshape(18, n)
        F = forcing(F, omega)
    return m[0], m[1:4], F, nuc


def _exact_sums(T, rho, j, F):
    c, r = (T - 1.0) / 2.0, int(T / 6.0) + 2.0
    x = torch.arange(T, dtype=torch.float64, device=F.device) - c
    X, Z = x[:, None, None].expand(T, T, T).reshape(-1), x[None, None, :].expand(T, T, T).reshape(-1)
    inside = X * X + Z * Z <= r * r
    torque = torch.where(inside, X * F[:, 2] - Z * F[:, 0], torch.zeros_like(X)).sum()
    return torch.cat([rho.sum()[None], j.sum(1), F.sum(0), torque[None]]).cpu().numpy()


def exact(case, seed):
    if case["kind"] in ("batch", "serve") or case["edge"] > 200 or case["edge"] ** 3 * case["steps"] > 5e8:
        return None  # minutes in 64 bits
    cond, T = _conditions(case, seed)[0], case["edge"]
    calls = case["kind"] == "calls"
    rho, j, F, nuc = _reference(case, cond, case["steps"] + (1 if calls else WARM))
    field = torch.cat([rho[:, None], ((j + 0.5 * F.T) / rho).T], 1).reshape(T, T, T, 4).cpu().numpy()
    if case["kind"] == "tank":
        return {"sums": _exact_sums(T, rho, j, F), "field": field}
    if case["kind"] == "driver":
        return {"exclude": None, "xy": None, "xz": None, "plane_q": None, "plane_f": None, "field": field}
    full_f, full_nu = np.zeros((T + 2,) * 3 + (3,)), np.zeros((T + 2,) * 3)
    full_f[1:-1, 1:-1, 1:-1] = F.reshape(T, T, T, 3).cpu().numpy()
    full_nu[1:-1, 1:-1, 1:-1] = nuc.reshape(T, T, T).cpu().numpy()
    return {"field": field, "F": full_f.reshape(-1), "Nu": full_nu.reshape(-1), "Q": None}
