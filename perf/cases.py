"""What a program asks of this engine, as timed cases: forces on host arrays, whole
leapfrog runs, forces and fields on device arrays, ensembles, and gradients of a run.

Every case goes through a public entry point (gravhopper_amd.grav, Simulation, the
methods of Context, Ensemble, autograd.leapfrog).  Particles are Plummer spheres for the
direct sum (star clusters of 1e6 Msun, b = 1 pc) and a halo with a disk for the octree
(1e12 and 5e10 Msun, 10 and 3 kpc), as in this repository's benchmark, sampled on the GPU.

The FP32 leapfrogs take 0.005 of a crossing time per step and eps = 0.02 b, the rule of
the benchmark's ensemble.
"""
import math

import numpy as np
import torch

import gravhopper_amd as gh
from gravhopper_amd import _native, autograd

# km/s/Myr per Msun/kpc^2 (G = 1), and kpc per km/s*Myr
ACCEL = 4.398600412921223e-09
DRIFT = 1.022712165045695e-03
G = ACCEL / DRIFT  # kpc (km/s)^2 / Msun

B, M = 1e-3, 1e6                                # the Plummer sphere: kpc, Msun
T_CR = math.sqrt(B ** 3 / (G * DRIFT ** 2 * M))  # its crossing time, Myr
THETA = 0.7


def listed():
    return [
        # one force evaluation of a small cluster on numpy arrays, the drop-in for the
        # reference's functions: transfers and launches count
        {"name": "grav_direct_500", "kind": "grav", "n": 500, "targets": 0},
        # the README's run: 2000 particles, FP64, with the history of every step (50 of its
        # 400 steps)
        {"name": "sim_direct_2000", "kind": "sim", "algorithm": "direct", "n": 2000,
         "steps": 50},
        # a larger FP64 direct sum on device arrays, at an odd size
        {"name": "force_direct_100003", "kind": "force", "algorithm": "direct", "n": 100003,
         "targets": 0},
        # the field of a cluster at a few thousand points (profiles, maps, tracers)
        {"name": "field_direct_65536_3001", "kind": "force", "algorithm": "direct",
         "n": 65536, "targets": 3001},
        # a short FP32 run of a small cluster: sorting and launches count
        {"name": "run_direct_fp32_3000", "kind": "run", "algorithm": "direct", "n": 3000,
         "steps": 16},
        # the FP32 direct sum at the benchmark's headline size
        {"name": "run_direct_fp32_262144", "kind": "run", "algorithm": "direct", "n": 262144,
         "steps": 2},
        # gradients of a run with respect to its initial state and masses
        {"name": "adjoint_16384", "kind": "adjoint", "n": 16384, "steps": 20},
        # a parameter study: independent spheres of uneven size advanced together
        {"name": "ensemble_32", "kind": "ensemble", "sims": 32, "lo": 1024, "hi": 16384,
         "steps": 4},
        # the default Simulation (octree, FP64) at the size of the documented merger example
        {"name": "sim_tree_40001", "kind": "sim", "algorithm": "tree", "n": 40001, "steps": 8},
        # the FP64 octree force at the benchmark's size
        {"name": "force_tree_1048576", "kind": "force", "algorithm": "tree", "n": 1048576,
         "targets": 0},
        # the octree's field at unsorted points: build and a walk of few targets
        {"name": "field_tree_300007_20011", "kind": "force", "algorithm": "tree",
         "n": 300007, "targets": 20011},
        # FP32 octree steps at the benchmark's size
        {"name": "run_tree_fp32_1048576", "kind": "run", "algorithm": "tree", "n": 1048576,
         "steps": 2},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grav", "sim_direct", "sim_tree", "force_direct", "force_tree",
                       "run_direct", "run_tree", "adjoint", "ensemble"])
    if kind == "grav":
        return {"kind": "grav", "n": _log_size(rng, 100, 8000),
                "targets": rng.choice([0, _log_size(rng, 1, 4000)])}
    if kind == "sim_direct":
        return {"kind": "sim", "algorithm": "direct", "n": _log_size(rng, 200, 8192),
                "steps": rng.randint(10, 50)}
    if kind == "sim_tree":
        return {"kind": "sim", "algorithm": "tree", "n": _log_size(rng, 1000, 60000),
                "steps": rng.randint(3, 8)}
    if kind == "force_direct":
        return {"kind": "force", "algorithm": "direct", "n": _log_size(rng, 2000, 100000),
                "targets": rng.choice([0, _log_size(rng, 30, 20000)])}
    if kind == "force_tree":
        return {"kind": "force", "algorithm": "tree", "n": _log_size(rng, 2000, 1048576),
                "targets": rng.choice([0, _log_size(rng, 30, 200000)])}
    if kind == "run_direct":
        n = _log_size(rng, 1000, 262144)
        return {"kind": "run", "algorithm": "direct", "n": n,
                "steps": 2 if n > 65536 else rng.randint(4, 16)}
    if kind == "run_tree":
        return {"kind": "run", "algorithm": "tree", "n": _log_size(rng, 2000, 1048576),
                "steps": rng.randint(2, 8)}
    if kind == "adjoint":
        return {"kind": "adjoint", "n": _log_size(rng, 1000, 16384), "steps": rng.randint(5, 20)}
    return {"kind": "ensemble", "sims": rng.randint(4, 32), "lo": rng.randint(500, 2000),
            "hi": rng.randint(4000, 16384), "steps": rng.randint(2, 4)}


# ------------------------------------------------------------------------------------
# particles, sampled on the GPU in FP64
# ------------------------------------------------------------------------------------
def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(g, n):
    """In the open interval (0, 1)."""
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    return u.clamp(1e-12, 1.0 - 1e-12)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _direction(g, n):
    d = _normal(g, n, 3)
    return d / d.norm(dim=1, keepdim=True)


def _plummer(g, n, b=B, mass=M):
    """Isotropic Plummer sphere; q^2 = (v / v_esc)^2 follows Beta(3/2, 9/2)."""
    r = b / torch.sqrt(_uniform(g, n) ** (-2.0 / 3.0) - 1.0)
    chi2 = _normal(g, n, 12) ** 2
    q = torch.sqrt(chi2[:, :3].sum(1) / chi2.sum(1))
    speed = q * math.sqrt(2.0 * G * mass / b) * (1.0 + (r / b) ** 2) ** -0.25
    pos, vel = r[:, None] * _direction(g, n), speed[:, None] * _direction(g, n)
    m = torch.full((n,), mass / n, dtype=torch.float64, device="cuda")
    return pos - pos.mean(0), vel - vel.mean(0), m


def _galaxy(g, n):
    """Hernquist halo (a = 10 kpc, 1e12 Msun, cut at 100 kpc) and exponential disk
    (Rd = 3 kpc, sech^2 height 0.3 kpc, 5e10 Msun), half of the particles each."""
    nh, nd = n - n // 2, n // 2
    a, mh, rd, md = 10.0, 1e12, 3.0, 5e10

    def speed(r):
        inside = mh * r ** 2 / (r + a) ** 2 + md * (1.0 - (1.0 + r / rd) * torch.exp(-r / rd))
        return torch.sqrt(G * inside / r)

    r = a / (1.0 / torch.sqrt(_uniform(g, nh) * (100.0 / 121.0)) - 1.0)
    halo_x = r[:, None] * _direction(g, nh)
    halo_v = _normal(g, nh, 3) * (speed(r) / math.sqrt(3.0))[:, None]
    # R / Rd of an exponential disk is the sum of two exponential variates
    R = -rd * (torch.log(_uniform(g, nd)) + torch.log(_uniform(g, nd)))
    phi = 2.0 * math.pi * _uniform(g, nd)
    z = 0.3 * torch.atanh(2.0 * _uniform(g, nd) - 1.0)
    disk_x = torch.stack([R * torch.cos(phi), R * torch.sin(phi), z], 1)
    vc = speed(R)
    disk_v = torch.stack([-vc * torch.sin(phi), vc * torch.cos(phi), torch.zeros_like(vc)], 1)
    disk_v = disk_v + _normal(g, nd, 3) * (0.1 * vc)[:, None]
    m = torch.cat([torch.full((nh,), mh / nh, dtype=torch.float64, device="cuda"),
                   torch.full((nd,), md / nd, dtype=torch.float64, device="cuda")])
    return torch.cat([halo_x, disk_x]), torch.cat([halo_v, disk_v]), m


def _inputs(case, seed):
    """Particles, softening, time step and field points (None without) of a case."""
    g = _rng(seed)
    if case.get("algorithm", "direct") == "tree":
        x, v, m = _galaxy(g, case["n"])
        eps, dt, span = 0.05, 0.1, 30.0
    else:
        x, v, m = _plummer(g, case["n"])
        eps, dt, span = 0.02 * B, 0.005 * T_CR, 3.0 * B
    nf = case.get("targets", 0)
    f = span * _normal(g, nf, 3) if nf else None
    if case["kind"] == "sim" and case["algorithm"] == "direct":
        eps, dt = 5e-5, 0.005  # the README's run
    return x, v, m, eps, dt, f


def _sizes(case):
    """The ensemble's particle counts, log-uniform: the same for every seed."""
    rng = np.random.default_rng(case["sims"])
    return np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]),
                              case["sims"])).astype(int).tolist()


def _spheres(case, seed):
    """The ensemble's simulations: b and M log-uniform, eps = 0.02 b, dt = 0.005 t_cr."""
    rng = np.random.default_rng(seed)
    sims = []
    for k, n in enumerate(_sizes(case)):
        b = float(np.exp(rng.uniform(np.log(0.5e-3), np.log(2e-3))))
        mass = float(np.exp(rng.uniform(np.log(1e5), np.log(1e7))))
        x, v, m = _plummer(_rng(1000 * seed + k), n, b, mass)
        sims.append({"pos": x, "vel": v, "mass": m, "eps": 0.02 * b,
                     "dt": 0.005 * math.sqrt(b ** 3 / (G * DRIFT ** 2 * mass))})
    return sims


# ------------------------------------------------------------------------------------
# preparing and running
# ------------------------------------------------------------------------------------
def prepare(case, seed):
    ctx = _native.default_context()
    state = {"case": case, "ctx": ctx}
    if case["kind"] == "ensemble":
        sims = [{k: v.cpu().numpy() if torch.is_tensor(v) else v for k, v in s.items()}
                for s in _spheres(case, seed)]
        state["ens"] = _native.Ensemble(ctx, sims, ipt=4, persistent=True)
        return state
    x, v, m, eps, dt, f = _inputs(case, seed)
    state.update(eps=eps, dt=dt)
    if case["kind"] in ("grav", "sim"):  # programs of the reference hold numpy arrays
        x, v, m = x.cpu().numpy(), v.cpu().numpy(), m.cpu().numpy()
        f = None if f is None else f.cpu().numpy()
        state.update(ic={"pos": x, "vel": v, "mass": m}, f=f)
        return state
    state.update(x=x, v=v, m=m, f=f)
    if case["kind"] == "force":
        state["acc"] = torch.empty_like(x if f is None else f)
    elif case["kind"] == "run":
        state["stream"] = torch.cuda.Stream()
    else:  # adjoint: fit the sphere to one displaced by b / 2
        state["x"] = x.requires_grad_()
        state["v"] = v.requires_grad_()
        # float32, as a torch parameter is by default; leapfrog works on FP64 masses
        state["m"] = m.float().requires_grad_()
        state["target"] = x.detach() + 0.5 * B * _direction(_rng(seed + 1), case["n"])
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "grav":
        if state["f"] is None:
            return gh.grav.direct_summation(state["ic"], state["eps"])
        return gh.grav.direct_summation_position(state["ic"], state["f"], state["eps"])
    if kind == "sim":
        sim = gh.Simulation(dt=state["dt"], eps=state["eps"], algorithm=case["algorithm"])
        sim.add_IC(state["ic"])
        sim.run(case["steps"])
        return sim.positions, sim.velocities
    if kind == "force":
        x, m, f, acc = state["x"], state["m"], state["f"], state["acc"]
        fp, nf = (0, 0) if f is None else (f.data_ptr(), len(f))
        if case["algorithm"] == "direct":
            ctx.direct_dev(x.data_ptr(), m.data_ptr(), len(m), state["eps"], _native.GH_FP64,
                           acc.data_ptr(), d_force_pos=fp, nf=nf)
        else:
            ctx.tree_dev(x.data_ptr(), m.data_ptr(), len(m), state["eps"], THETA,
                         _native.GH_FP64, acc.data_ptr(), d_force_pos=fp, nf=nf)
        return acc
    if kind == "run":
        algorithm = _native.GH_DIRECT if case["algorithm"] == "direct" else _native.GH_TREE
        with torch.cuda.stream(state["stream"]):
            x, v = state["x"].clone(), state["v"].clone()
            ctx.run_dev(x.data_ptr(), v.data_ptr(), state["m"].data_ptr(), case["n"],
                        state["dt"], state["eps"], case["steps"], algorithm=algorithm,
                        theta=THETA, precision=_native.GH_FP32,
                        stream=state["stream"].cuda_stream)
        return x, v
    if kind == "ensemble":
        state["ens"].run(case["steps"])
        return state["ens"].state()
    x, v, m = state["x"], state["v"], state["m"]
    xn, vn = autograd.leapfrog(x, v, m, state["dt"], state["eps"], case["steps"])
    loss = _loss(xn, state["target"])
    return (xn, vn, loss) + torch.autograd.grad(loss, (x, v, m))


def _loss(x, target):
    return ((x - target) ** 2).sum(-1).mean()


# ------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------
def work(case):
    """20 operations per interaction (3 differences, 6 for r^2 + eps^2, 1/r^3 in 4 and m/r^3
    in 1, 6 for the sums): every ordered pair of a direct sum, the accepted nodes of an
    octree walk.  Bytes: the inputs once and the outputs once."""
    def forces(n, algorithm, targets=0):
        t = targets or n
        if algorithm == "direct":
            return 20.0 * t * n
        # accepted nodes per target at theta = 0.7: 630 at n = 2^20, growing with log n
        return 20.0 * t * max(20.0, 33.0 * math.log2(n) - 30.0)

    kind = case["kind"]
    if kind == "ensemble":
        sizes = _sizes(case)
        return {"bytes": 104.0 * sum(sizes),
                "flops": case["steps"] * sum(forces(n, "direct") for n in sizes)}
    n, algorithm = case["n"], case.get("algorithm", "direct")
    if kind in ("grav", "force"):
        t = case["targets"]
        return {"bytes": 32.0 * n + 24.0 * (2 * t or n),
                "flops": forces(n, algorithm, t)}
    flops = case["steps"] * forces(n, algorithm)
    if kind == "sim":  # the history of every step goes out
        return {"bytes": 56.0 * n + 48.0 * n * (case["steps"] + 1), "flops": flops}
    if kind == "run":
        return {"bytes": 104.0 * n, "flops": flops}
    # a gradient: the forces, and per pair 36 operations of the transposed tidal field
    return {"bytes": 180.0 * n, "flops": flops + case["steps"] * 36.0 * n * n}


# ------------------------------------------------------------------------------------
# the same results from plain torch in 64 bits
# ------------------------------------------------------------------------------------
def _direct(x, m, f, eps, rows=None):
    """Accelerations at f (f is x: the particles' own) in G Msun / kpc^2."""
    rows = rows or max(1, (1 << 27) // len(m))
    out = []
    for k in range(0, len(f), rows):
        d = x[None, :, :] - f[k:k + rows, None, :]
        r2 = (d * d).sum(-1) + eps * eps
        w = m * r2 ** -1.5
        w = torch.where(r2 == 0.0, torch.zeros_like(w), w)
        out.append((d * w[..., None]).sum(1))
    return torch.cat(out)


def _octree(x, m, eps):
    """The octree level by level: (centre, size, mass, centre of mass, is leaf, first child
    in the next level, number of children) of each level's nodes."""
    lo, hi = x.min(0).values, x.max(0).values
    side = float(hi[0] - lo[0]) + eps
    for i in (1, 2):
        if float(hi[i] - lo[i]) > side:
            side = float(hi[i] - lo[i]) + eps
    centre = (0.5 * (lo + hi))[None, :]
    node = torch.zeros(len(x), dtype=torch.int64, device=x.device)
    levels = []
    while len(node):
        k = len(centre)
        count = torch.bincount(node, minlength=k)
        mass = torch.zeros(k, dtype=x.dtype, device=x.device).index_add_(0, node, m)
        com = torch.zeros(k, 3, dtype=x.dtype, device=x.device).index_add_(
            0, node, m[:, None] * x) / mass[:, None]
        leaf = count == 1
        alone = leaf[node]
        com[node[alone]] = x[alone]
        x, m, node = x[~alone], m[~alone], node[~alone]
        upper = x > centre[node]
        octant = (upper.long() << torch.arange(3, device=x.device)).sum(1)
        child, node = torch.unique(node * 8 + octant, return_inverse=True)
        children = torch.bincount(child // 8, minlength=k)
        levels.append((centre, side, mass, com, leaf, children.cumsum(0) - children, children))
        sign = (((child % 8)[:, None] >> torch.arange(3, device=x.device)) & 1) * 2 - 1
        centre = centre[child // 8] + sign.to(x.dtype) * 0.5 * (0.5 * side)
        side = 0.5 * side
    return levels


def _tree(x, m, f, eps, theta=THETA):
    """Monopole accelerations at f: a node is taken when it is a leaf or its size is less
    than theta times the distance of its centre, else opened."""
    levels, out = _octree(x, m, eps), []
    for k in range(0, len(f), 65536):
        p = f[k:k + 65536]
        acc = torch.zeros_like(p)
        t = torch.arange(len(p), device=p.device)
        node = torch.zeros_like(t)
        for centre, side, mass, com, leaf, first, children in levels:
            dist = (centre[node] - p[t]).norm(dim=1)
            take = leaf[node] | (side / dist < theta)
            a, b = t[take], node[take]
            d = com[b] - p[a]
            r2 = (d * d).sum(1) + eps * eps
            w = torch.where(r2 == 0.0, torch.zeros_like(r2), mass[b] * r2 ** -1.5)
            acc.index_add_(0, a, d * w[:, None])
            t, node = t[~take], node[~take]
            n = children[node]
            start = first[node] - (n.cumsum(0) - n)
            t = t.repeat_interleave(n)
            node = start.repeat_interleave(n) + torch.arange(len(t), device=p.device)
        out.append(acc)
    return torch.cat(out)


def _leapfrog(x, v, m, dt, eps, steps, force):
    """Drift-kick-drift; the state after every step and the half-step positions."""
    xs, vs, halves = [x], [v], []
    for _ in range(steps):
        h = xs[-1] + 0.5 * vs[-1] * dt * DRIFT
        v = vs[-1] + ACCEL * force(h, m, h, eps) * dt
        halves.append(h)
        vs.append(v)
        xs.append(h + 0.5 * v * dt * DRIFT)
    return xs, vs, halves


def _gradients(x, v, m, dt, eps, steps, target):
    """Final state, loss and its gradients, by reversing the steps."""
    xs, vs, halves = _leapfrog(x, v, m, dt, eps, steps, _direct)
    n = len(m)
    loss = _loss(xs[-1], target)
    lx, lv, lm = 2.0 * (xs[-1] - target) / n, torch.zeros_like(v), torch.zeros_like(m)
    rows = max(1, (1 << 24) // n)
    for h in reversed(halves):
        lv = lv + 0.5 * dt * DRIFT * lx
        u = ACCEL * dt * lv  # the force's cotangent
        src, mass = h.detach().requires_grad_(), m.detach().requires_grad_()
        own = torch.zeros_like(h)
        for k in range(0, n, rows):
            f = h[k:k + rows].detach().requires_grad_()
            a = _direct(src, mass, f, eps, rows)
            gs, gm, gf = torch.autograd.grad((a * u[k:k + rows]).sum(), (src, mass, f))
            lx, lm = lx + gs, lm + gm
            own[k:k + rows] = gf
        lx = lx + own
        lv = lv + 0.5 * dt * DRIFT * lx
    return xs[-1], vs[-1], loss, lx, lv, lm


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        pos, vel = [], []
        for s in _spheres(case, seed):
            x, v, _ = _leapfrog(s["pos"], s["vel"], s["mass"], s["dt"], s["eps"], case["steps"],
                                _direct)
            pos.append(x[-1])
            vel.append(v[-1])
        return pos, vel
    if kind == "run" and case["algorithm"] == "tree":
        # the FP32 walk may open more nodes than the opening angle asks for, so its sum has
        # no value in 64 bits apart from its own lists
        return None
    x, v, m, eps, dt, f = _inputs(case, seed)
    force = _tree if case.get("algorithm", "direct") == "tree" else _direct
    if kind in ("grav", "force"):
        return force(x, m, x if f is None else f, eps) * (ACCEL if kind == "grav" else 1.0)
    if kind == "adjoint":
        target = x + 0.5 * B * _direction(_rng(seed + 1), case["n"])
        return _gradients(x, v, m.float().double(), dt, eps, case["steps"], target)
    xs, vs, _ = _leapfrog(x, v, m, dt, eps, case["steps"], force)
    if kind == "sim":
        return torch.stack(xs), torch.stack(vs)
    return xs[-1], vs[-1]
