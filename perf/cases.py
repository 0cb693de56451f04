"""Performance cases of cubble_amd: the work a program has it do, timed through
its Python entry points.

Five kinds of call:

  run        Simulator.run_steps: a block of accepted steps on the device, then
             what a program reads at its end -- the printed row with every
             bubble's energy (Simulator.observe) or a snapshot of the whole
             state (Simulator.get_state).
  integrate  Simulator.integrate once per accepted step, the loop of a program
             that replaces the reference's step function and keeps its own
             driver, then a snapshot.
  batch      Batch.run_steps: many uneven 2D and 3D foams advanced together.
  attempt    Simulator.step + get_attempt: one uncommitted step attempt on a
             state the program brought itself.
  pairs      find_pairs: the pair list of caller-owned device arrays.

Foams are the benchmark's: normal radii (sd 0.1, clipped to [0.5, 1.5]) in 2D,
log-normal radii (sigma 0.15) in 3D, uniform positions, phi 0.84 to 0.9,
kappa 0.01, K 0.1, tolerance 1e-4.  A run leaves its foam advanced; a foam
loses a few percent of its bubbles over ten thousand steps, so repeated passes
do nearly the same work.
"""
import math

import numpy as np
import torch

import cubble_amd as ca

KAPPA, K_PARAM, TOL, DT0 = 0.01, 0.1, 1e-4, 1e-4
SKIN = 0.3
PRECISION = {"fp64": ca.PREC_FP64, "mixed": ca.PREC_MIXED}


def listed():
    return [
        # A parameter study of small foams, one at a time: launches and
        # latency are all there is.
        {"name": "run_2d_1e3", "kind": "run", "dim": 2, "bubbles": 1009, "precision": "fp64",
         "steps": 300, "walls": False, "flow": False, "read": "state"},
        # The same foam driven one accepted step per call from the host.
        {"name": "integrate_2d_4e3", "kind": "integrate", "dim": 2, "bubbles": 4001,
         "precision": "fp64", "steps": 60, "walls": False, "flow": False},
        # The ordinary 2D foam of the reference's input file size, a block of
        # steps between two printed rows.
        {"name": "run_2d_1e4", "kind": "run", "dim": 2, "bubbles": 10000, "precision": "fp64",
         "steps": 400, "walls": False, "flow": False, "read": "row"},
        # Channel flow between walls (the imposed flow option), with snapshots.
        {"name": "run_2d_flow_3e4", "kind": "run", "dim": 2, "bubbles": 30011,
         "precision": "fp64", "steps": 300, "walls": True, "flow": True, "read": "state"},
        # The ordinary 3D foam in mixed precision, rows between blocks.
        {"name": "run_3d_1e5_mixed", "kind": "run", "dim": 3, "bubbles": 100003,
         "precision": "mixed", "steps": 300, "walls": False, "flow": False, "read": "row"},
        # The large single foam of the benchmark, FP64.
        {"name": "run_3d_1e6", "kind": "run", "dim": 3, "bubbles": 1000000, "precision": "fp64",
         "steps": 100, "walls": False, "flow": False, "read": "row"},
        # The largest single foam, mixed precision.
        {"name": "run_3d_4e6_mixed", "kind": "run", "dim": 3, "bubbles": 4000037,
         "precision": "mixed", "steps": 100, "walls": False, "flow": False, "read": "row"},
        # The benchmark's batch: 256 uneven foams, 5e6 bubbles in all.
        {"name": "batch_256_mixed", "kind": "batch", "foams": 256, "smallest": 1000,
         "largest": 100000, "precision": "mixed", "steps": 50},
        # One attempt of a walled 3D foam, FP64, from the program's own arrays.
        {"name": "attempt_3d_2e5", "kind": "attempt", "dim": 3, "bubbles": 200003,
         "precision": "fp64", "walls": True},
        # The same in mixed precision, 2D, periodic.
        {"name": "attempt_2d_3e4_mixed", "kind": "attempt", "dim": 2, "bubbles": 30011,
         "precision": "mixed", "walls": False},
        # Pair lists for another program's foam: a small 2D one ...
        {"name": "pairs_2d_3e3", "kind": "pairs", "dim": 2, "bubbles": 3001, "walls": False,
         "ordered": False, "alloc": True},
        # ... and a large 3D one.
        {"name": "pairs_3d_5e5", "kind": "pairs", "dim": 3, "bubbles": 500009, "walls": False,
         "ordered": True, "alloc": False},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) | 1


def draw(rng):
    kind = rng.choice(["run", "run", "run", "integrate", "batch", "attempt", "pairs", "pairs"])
    dim = rng.choice([2, 3])
    if kind == "run":
        n = _log_uniform(rng, 1e3, 2e6)
        flow = rng.random() < 0.2
        return {"kind": kind, "dim": dim, "bubbles": n,
                "precision": rng.choice(["fp64", "mixed"]),
                "steps": rng.randint(50, 300 if n < 200000 else 100),
                "walls": flow or rng.random() < 0.2, "flow": flow,
                "read": "state" if n < 50000 and rng.random() < 0.5 else "row"}
    if kind == "integrate":
        return {"kind": kind, "dim": dim, "bubbles": _log_uniform(rng, 1e3, 2e5),
                "precision": rng.choice(["fp64", "mixed"]), "steps": rng.randint(20, 60),
                "walls": rng.random() < 0.2, "flow": False}
    if kind == "batch":
        lo = _log_uniform(rng, 1e3, 1e4)
        return {"kind": kind, "foams": rng.randint(4, 128), "smallest": lo,
                "largest": lo * rng.randint(2, 10), "precision": rng.choice(["fp64", "mixed"]),
                "steps": rng.randint(20, 60)}
    if kind == "attempt":
        return {"kind": kind, "dim": dim, "bubbles": _log_uniform(rng, 1e3, 3e5),
                "precision": rng.choice(["fp64", "mixed"]), "walls": rng.random() < 0.4}
    n = _log_uniform(rng, 1e3, 2e6)
    return {"kind": kind, "dim": dim, "bubbles": n, "walls": rng.random() < 0.3,
            "ordered": rng.random() < 0.5, "alloc": n > ca.FIND_PAIRS_NOALLOC_MAX or
            rng.random() < 0.5}


# ---- inputs -----------------------------------------------------------------
def _phi(dim):
    return 0.9 if dim == 2 else 0.84


def _walls(case):
    # walls on y: a channel (2D) or two plates (3D)
    return (0, 1, 0) if case["walls"] else (0, 0, 0)


def _config(case, seed, **over):
    dim = case["dim"]
    kw = dict(dim=dim, num_start=case["bubbles"], radius_dist=0 if dim == 2 else 1,
              r_std=0.1 if dim == 2 else 0.15, r_lo=0.5, r_hi=1.5, phi=_phi(dim), kappa=KAPPA,
              k_param=K_PARAM, error_tolerance=TOL, dt0=DT0, wall=_walls(case), seed=1 + seed,
              precision=PRECISION[case["precision"]])
    if case.get("flow"):
        kw.update(flow=1, flow_vel=(0.01, 0.0, 0.0), flow_lbb=(0.0, 0.475, 0.0),
                  flow_tfr=(0.4, 0.525, 1.0))
    kw.update(over)
    return ca.Config(**kw)


def _edge(dim, n):
    """Box edge of n bubbles of unit volume-mean radius at the gas fraction phi."""
    unit = math.pi if dim == 2 else math.pi * 1.33333333333333333333333333
    vol = float(np.cumsum(np.full(n, unit))[-1])
    t = vol / _phi(dim)
    return math.sqrt(t) if dim == 2 else float(np.cbrt(t))


def _arrays(dim, n, seed, edge):
    """A foam of n bubbles: uniform positions in the box, radii of the
    benchmark's distribution scaled to a volume mean of one, small velocities.
    Rows x, y, z, r."""
    rng = np.random.default_rng(77 + seed)
    z = rng.standard_normal(n)
    r = np.clip(1.0 + 0.1 * z, 0.5, 1.5) if dim == 2 else np.exp(0.15 * z)
    r /= np.mean(r ** dim) ** (1.0 / dim)
    x = np.zeros((4, n))
    x[:dim] = edge * rng.random((dim, n))
    x[3] = r
    v = np.zeros((2, 4, n))
    v[:, :dim] = 0.2 * rng.standard_normal((2, dim, n))
    v[:, 3] = 0.01 * rng.standard_normal((2, n))
    # velocities the mixed-precision buffers hold as they are
    return x, v.astype(np.float32).astype(np.float64)


def _cell_dims(edge, dim, max_r):
    q = max(1, int(math.floor(edge / (2 * (max_r + SKIN)))))
    return [q, q, q if dim == 3 else 1]


def _cell_order(x, dim, edge, cd):
    """Stable order of the bubbles by the cell holding them."""
    cid = np.zeros(x.shape[1], np.int64)
    for k in range(dim - 1, -1, -1):
        c = np.clip(np.floor(cd[k] * x[k] / edge), 0, cd[k] - 1).astype(np.int64)
        cid = cid * cd[k] + c
    return np.argsort(cid, kind="stable")


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "integrate"):
        # a foam well past seeding (dt has grown to the tolerance, bubbles
        # dissolve, searches come at their usual pace), resident on the GPU
        ip = ca.IntegrationParams(True, bool(case["flow"]), True)
        sim = ca.Simulator(_config(case, seed))
        sim.run_steps(1000 if case["bubbles"] < 300000 else 300, ip)
        return {"case": case, "sim": sim, "ip": ip}
    if kind == "batch":
        cfgs = ca.batch_workload(case["foams"], seed=2024 + seed,
                                 precision=PRECISION[case["precision"]], lo=case["smallest"],
                                 hi=case["largest"])
        batch = ca.Batch(cfgs)
        ip = ca.IntegrationParams()
        batch.run_steps(300, ip)
        return {"case": case, "batch": batch, "ip": ip}
    dim, n = case["dim"], case["bubbles"]
    edge = _edge(dim, n)
    x, v = _arrays(dim, n, seed, edge)
    if kind == "attempt":
        # equal unit radii give the box its edge; the arrays follow
        sim = ca.Simulator(_config(case, seed, radius_dist=1, r_std=0.0))
        sc = sim.scalars()
        sc.update(count=n, max_r_cell=float(x[3].max()), dt=DT0)
        st = {"x": x, "v": v[0], "vo": v[1], "saved": x, "path": np.zeros(n), "err": np.zeros(n),
              "wc": np.zeros((3, n), np.int32), "idx": np.arange(n, dtype=np.int32),
              "nbr_off": np.zeros(n + 1, np.int32), "nbr": np.zeros(0, np.int32)}
        sim.set_state(st, sc)
        sim.search_neighbors()
        return {"case": case, "sim": sim, "ip": ca.IntegrationParams()}
    if case["ordered"]:
        # as a foam that a simulation keeps in cell order
        order = _cell_order(x, dim, edge, _cell_dims(edge, dim, float(x[3].max())))
        x = x[:, order]
    cap = int(n * (4 if dim == 2 else 8)) + 64
    dev = [torch.tensor(x[k], dtype=torch.float64, device="cuda") for k in range(4)]
    return {"case": case, "x": dev, "cap": cap,
            "i": torch.full((cap,), -1, dtype=torch.int32, device="cuda"),
            "j": torch.full((cap,), -1, dtype=torch.int32, device="cuda"),
            "num": torch.zeros(1, dtype=torch.int64, device="cuda"),
            "box": ca.Box.of(dim, [0.0] * 3, [edge] * 3, _walls(case))}


# ---- one pass ---------------------------------------------------------------
def _fp32(state, keys):
    """The fields mixed precision holds in FP32, as FP32 (the host view is FP64)."""
    return {k: a.astype(np.float32) if k in keys else a for k, a in state.items()}


def _snapshot(sim, case):
    """The whole state, every field at the size the foam started with (bubbles
    that dissolved leave zeros), as a program's snapshot buffers are."""
    st, _ = sim.get_state()
    if case["precision"] == "mixed":
        st = _fp32(st, ("v", "vo", "saved", "err"))
    n = case["bubbles"]
    size = {"nbr": n * (10 if case["dim"] == 2 else 24), "nbr_off": n + 1}
    return {k: _padded(a, size.get(k, n)) for k, a in st.items()}


def _padded(a, n):
    if a.shape[-1] == n:
        return a
    out = np.zeros(a.shape[:-1] + (n,), a.dtype)
    out[..., :a.shape[-1]] = a
    return out


def run(state):
    case = state["case"]
    kind, ip = case["kind"], state.get("ip")
    if kind in ("run", "integrate"):
        sim = state["sim"]
        if kind == "run":
            result = sim.run_steps(case["steps"], ip)
        else:
            for _ in range(case["steps"]):
                result = sim.integrate(ip)
        if case.get("read") == "row":
            row = sim.observe(energy=True)
            row["energy"] = _padded(row["energy"], case["bubbles"])
            return {"result": result, "row": row}
        return {"result": result, "state": _snapshot(sim, case)}
    if kind == "batch":
        res = state["batch"].run_steps(case["steps"], ip)
        return {k: np.array([r[k] for r in res]) for k in res[0]}
    if kind == "attempt":
        result = state["sim"].step(ip)
        out = state["sim"].get_attempt()
        if case["precision"] == "mixed":
            out = _fp32(out, ("vp", "ov"))
        return {"too_large": result["error_too_large"], "attempt": out}
    x = state["x"]
    ca.find_pairs(x[0].data_ptr(), x[1].data_ptr(), x[2].data_ptr() if case["dim"] == 3 else 0,
                  x[3].data_ptr(), case["bubbles"], state["box"], SKIN, state["i"].data_ptr(),
                  state["j"].data_ptr(), state["cap"], state["num"].data_ptr(),
                  torch.cuda.current_stream().cuda_stream, noalloc=not case["alloc"])
    return {"i": state["i"], "j": state["j"], "num": state["num"]}


# ---- what a pass cannot do without ------------------------------------------
def _half_pairs(dim):
    """Expected pairs per bubble within r_i + r_j + skin at the gas fraction phi."""
    if dim == 2:
        return 0.5 * _phi(2) / math.pi * math.pi * (2 + SKIN) ** 2
    return 0.5 * _phi(3) / (4 / 3 * math.pi) * 4 / 3 * math.pi * (2 + SKIN) ** 3


def _step_work(dim, precision):
    """Bytes and operations of one accepted step per bubble: positions,
    velocities, saved positions, path and error read, the lists read once, the
    new state written; about 40 operations a pair and direction."""
    c, vb, p = dim + 1, 4 if precision == "mixed" else 8, _half_pairs(dim)
    return 16 * c + 4 * vb * c + 16 + 2 * vb + 8 * p, 80 * p + 60


def work(case):
    kind = case["kind"]
    if kind == "batch":
        a, b = case["smallest"], case["largest"]
        mean = (b - a) / math.log(b / a)
        each = [_step_work(d, case["precision"]) for d in (2, 3)]
        n = 0.5 * case["foams"] * mean * case["steps"]
        return {"bytes": n * (each[0][0] + each[1][0]), "flops": n * (each[0][1] + each[1][1])}
    dim, n = case["dim"], case["bubbles"]
    p = _half_pairs(dim)
    if kind in ("run", "integrate"):
        b, f = _step_work(dim, case["precision"])
        read = 8 if case.get("read") == "row" else 32 * (dim + 1) + 40 + 8 * p
        return {"bytes": n * (case["steps"] * b + read), "flops": n * case["steps"] * f}
    if kind == "attempt":
        b, f = _step_work(dim, case["precision"])
        return {"bytes": n * b, "flops": n * f}
    return {"bytes": n * (8 * (dim + 1) + 8 * p) + 8, "flops": n * p * 20}


# ---- the attempt in 64 bits -------------------------------------------------
def _pairs64(x, dim, edge, cd, wall):
    """All ordered pairs (i, j), i != j, within r_i + r_j + skin, and their
    minimum-image differences x_i - x_j.  x: (4, n) in cell order, on a device."""
    dev, n = x.device, x.shape[1]
    c = [torch.clamp(torch.floor(cd[k] * x[k] / edge), 0, cd[k] - 1).long() for k in range(dim)]
    if dim == 2:
        c.append(torch.zeros_like(c[0]))
    cid = (c[2] * cd[1] + c[1]) * cd[0] + c[0]
    ncell = cd[0] * cd[1] * cd[2]
    count = torch.bincount(cid, minlength=ncell)
    start = torch.cumsum(count, 0) - count
    most = int(count.max())
    slot = torch.arange(most, device=dev)
    offs = [(-1, 0, 1) if cd[k] > 2 else (0, 1)[:cd[k]] for k in range(3)]
    found = []
    for a in offs[2]:
        for b in offs[1]:
            for e in offs[0]:
                q, ok = [], torch.ones(n, dtype=torch.bool, device=dev)
                for k, o in enumerate((e, b, a)):
                    w = c[k] + o if cd[k] > 2 else torch.full_like(c[k], o)
                    if wall[k]:
                        ok &= (w >= 0) & (w < cd[k])
                    q.append(w % cd[k])
                cell = (q[2] * cd[1] + q[1]) * cd[0] + q[0]
                j = start[cell][:, None] + slot
                live = ok[:, None] & (slot < count[cell][:, None])
                i = torch.arange(n, device=dev)[:, None].expand_as(j)
                i, j = i[live], j[live]
                d = [x[k][i] - x[k][j] for k in range(dim)]
                d = [t if wall[k] else torch.where(
                    t.abs() > edge - t.abs(), t - torch.sign(t) * edge, t) for k, t in enumerate(d)]
                m = sum(t * t for t in d)
                near = (m < (x[3][i] + x[3][j] + SKIN) ** 2) & (i != j)
                found.append((i[near], j[near], [t[near] for t in d], m[near]))
    return (torch.cat([f[0] for f in found]), torch.cat([f[1] for f in found]),
            [torch.cat([f[2][k] for f in found]) for k in range(dim)],
            torch.cat([f[3] for f in found]))


def _touch(c, pos, rad, wall, edge, f0, keep):
    """Push and drag of the walls on the velocities c, axis after axis."""
    dim = len(c)
    drag = [torch.ones_like(rad) for _ in range(3)]
    out = list(c)
    for k in range(dim):
        if not wall[k]:
            continue
        lo, hi = pos[k], pos[k] - edge
        d = torch.where(lo * lo < hi * hi, lo, hi)
        hit = rad * rad >= d * d
        side = torch.where(d < 0, -1.0, 1.0)
        push = side * f0 * (1.0 - d * side / rad)
        for q in range(dim):
            if q == k:
                before = torch.ones_like(rad)
                for t in range(k):
                    before = before * drag[t]
                out[q] = torch.where(hit, out[q] + push * before, out[q])
            else:
                out[q] = torch.where(hit, out[q] * keep, out[q])
        drag[k] = torch.where(hit, keep, 1.0)
    return out


def exact(case, seed):
    """One attempt in 64 bits: predictor, pair velocities, overlap and gas
    flux, walls, liquid-mediated exchange, trapezoid corrector."""
    if case["kind"] != "attempt":
        return None
    dim, n, wall = case["dim"], case["bubbles"], _walls(case)
    edge, h, f0 = _edge(dim, n), 0.5 * DT0, 1.0
    x, v = _arrays(dim, n, seed, edge)
    cd = _cell_dims(edge, dim, float(x[3].max()))
    order = _cell_order(x, dim, edge, cd)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.tensor(x[:, order], device=dev)
    v, vo = (torch.tensor(u[:, order], device=dev) for u in v)
    i, j, _, _ = _pairs64(x, dim, edge, cd, wall)
    p = x + h * (3.0 * v - vo)  # predicted
    rad = p[3]
    d = [p[k][i] - p[k][j] for k in range(dim)]
    d = [t if wall[k] else torch.where(t.abs() > edge - t.abs(), t - torch.sign(t) * edge, t)
         for k, t in enumerate(d)]
    m = sum(t * t for t in d)
    ri, rj = rad[i], rad[j]
    on = (ri + rj) ** 2 >= m
    i, j, d, m, ri, rj = i[on], j[on], [t[on] for t in d], m[on], ri[on], rj[on]

    def total(t):
        return torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, i, t)

    pull = f0 * (1.0 / torch.sqrt(m) - 1.0 / (ri + rj))
    vel = [total(t * pull) for t in d]
    small, large = torch.minimum(ri, rj) ** 2, torch.maximum(ri, rj) ** 2
    lens = (rj * rj - (0.5 * (rj * rj - ri * ri + m)) ** 2 / m).abs()
    area = torch.where(m < large, small, lens)
    area = math.pi * area if dim == 3 else 2.0 * torch.sqrt(area)
    overlap, flux = total(area), total(area * (1.0 / rj - 1.0 / ri))
    if case["walls"]:
        vel = _touch(vel, p, rad, wall, edge, f0, 1.0 - 0.1)

    def surface(t):
        return 2.0 * math.pi * t * (2.0 * t if dim == 3 else 1.0)

    own = surface(rad)
    s_a, s_ar = own.sum(), (own / rad).sum()
    inv_rho = (s_ar - (overlap / rad).sum()) / (s_a - overlap.sum())
    mean_area = surface(1.0)
    dr = (inv_rho - 1.0 / rad) * (KAPPA * mean_area * n / s_a) * (own - overlap) + flux
    dr = dr * K_PARAM / own
    xc, vp = torch.zeros_like(x), torch.zeros_like(x)
    for k in range(dim):
        vp[k] = vel[k]
        xc[k] = x[k] + h * (v[k] + vel[k])
    vp[3] = dr
    xc[3] = x[3] + h * (v[3] + dr)
    path = torch.sqrt(sum((x[k] - xc[k]) ** 2 for k in range(dim)))
    return {"too_large": None, "attempt": {"xc": xc, "vp": vp, "ov": overlap, "path_new": path,
                                           "del": None}}
