"""Performance cases: the work a molecular-dynamics program has this package do.

Every case goes through the public entry points: the one-call neighbour lists
(leaf-pair, point-query, cell list), the pair-list forces, `simulate_`, a
`Simulation` that is advanced in pieces with a frame recorded after each,
packed replicas, and the adjoint's forward and backward.  Positions are either
uniform at liquid density or in the unit cube (how the reference benchmarks
its searches) or jittered lattices at liquid density (how a dynamics run
starts: uniform points overlap and the Lennard-Jones force overflows).

Pair lists are compared as their 32-bit words (both ids and the distance's
bits): the lists are exact, order included.  Single-precision simulations
return single-precision arrays, double and mixed ones double.

`exact` restates the dynamics, the forces and the gradients in 64 bits with
plain torch.
"""
import ctypes
import math

import numpy as np
import torch

from __graft_entry__ import load_package

nd = load_package()

DENSITY = 0.8
KEYS = {"masked": nd.MORTON_MASKED, "interleave": nd.MORTON_INTERLEAVE}
PREDS = {"scalar": nd.PRED_SCALAR, "simd": nd.PRED_SIMD}
QUERIES = {"own": nd.QUERY_OWN_LEAF, "root": nd.QUERY_ROOT}


def listed():
    return [
        # a script's small list: host arrays in, host list out, the default
        # (masked) key and the 4 x 4 tile form; latency and launches count
        dict(name="list-host-1024", kind="list-host", n=1024, r=0.1, apl=4),
        # the search as the reference benchmarks it: unit cube, its own key
        dict(name="list-unit-65536", kind="list", n=65536, r=0.03, apl=4, key="masked", pred="scalar",
             points="unit"),
        # the list of a liquid-density system at the radius of a dynamics run
        dict(name="list-262144", kind="list", n=262144, r=2.8, apl=4, key="interleave", pred="scalar",
             points="uniform"),
        # the same search with odd sizes: 3 atoms per leaf, few neighbours
        dict(name="list-odd-30003", kind="list", n=30003, r=1.7, apl=3, key="interleave", pred="scalar",
             points="lattice"),
        # point queries (each atom walks from its own leaf)
        dict(name="point-100000", kind="point", n=100000, r=2.8, apl=5, key="interleave", query="own",
             points="uniform"),
        # the cell list a program calls when it needs the pairs only
        dict(name="cells-524287", kind="cells", n=524287, r=2.8, pred="simd", points="uniform"),
        # forces over a pair list kept from the last list build: both pair
        # terms and their sum, as the reference's step calls them
        dict(name="forces-131072", kind="forces", n=131072, r=2.8),
        # a whole simulate! call of a small system: list every step, frames
        # and the final state back on the host
        dict(name="simulate-4096", kind="simulate", n=4096, steps=100, rebuild=1, coul=False),
        # production: 100 steps of the 262,144-atom liquid between two frames
        dict(name="run-262144-fp32", kind="run", n=262144, steps=100, precision="fp32", apl=32, resort=200,
             points="lattice"),
        # droplets in vapour in the mixed form (voids, uneven lists)
        dict(name="run-blobs-262144-mixed", kind="run", n=262144, steps=50, precision="mixed", apl=16,
             resort=100, points="blobs"),
        # 96 ragged replicas packed into one launch sequence
        dict(name="batch-96", kind="batch", reps=96, lo=256, hi=8192, sizes=11, steps=50, apl=32),
        # loss and gradients of a 50-step trajectory in double precision
        dict(name="adjoint-32768-fp64", kind="adjoint", n=32768, steps=50, precision="fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _leaves(n, apl):
    return max(2, n // apl) * apl


def draw(rng):
    """One more case of the listed kinds: sizes over their logarithm, the
    options a program picks."""
    kind = rng.choice(["list-host", "list", "list", "point", "cells", "forces", "simulate", "run", "run",
                       "batch", "adjoint"])
    if kind == "list-host":
        return dict(kind=kind, n=_leaves(_log_int(rng, 64, 8192), 4), r=round(rng.uniform(0.03, 0.15), 3), apl=4)
    if kind == "list":
        apl = rng.choice([1, 2, 3, 4, 4, 4, 5, 8, 16])
        pred = rng.choice(["scalar", "simd"])
        if rng.random() < 0.4:
            n = _leaves(_log_int(rng, 2000, 65536), apl)
            # 4 to 12 neighbours within the radius
            r = (rng.uniform(4.0, 12.0) / n * 3.0 / (4.0 * math.pi)) ** (1.0 / 3.0)
            return dict(kind=kind, n=n, r=round(r, 4), apl=apl, key="masked", pred=pred, points="unit")
        return dict(kind=kind, n=_leaves(_log_int(rng, 2000, 262144), apl), r=round(rng.uniform(1.2, 2.8), 3),
                    apl=apl, key="interleave", pred=pred, points=rng.choice(["uniform", "lattice"]))
    if kind == "point":
        apl = rng.choice([1, 3, 4, 5, 8])
        return dict(kind=kind, n=_leaves(_log_int(rng, 2000, 262144), apl), r=round(rng.uniform(1.2, 2.8), 3),
                    apl=apl, key="interleave", query=rng.choice(["own", "root"]),
                    points=rng.choice(["uniform", "lattice"]))
    if kind == "cells":
        return dict(kind=kind, n=_log_int(rng, 1000, 524287), r=round(rng.uniform(1.2, 2.8), 3),
                    pred=rng.choice(["scalar", "simd"]), points=rng.choice(["uniform", "lattice"]))
    if kind == "forces":
        return dict(kind=kind, n=_log_int(rng, 1000, 131072), r=2.8)
    if kind == "simulate":
        return dict(kind=kind, n=_leaves(_log_int(rng, 500, 8192), 4), steps=10 * rng.randint(3, 10),
                    rebuild=rng.choice([1, 2, 5, 10]), coul=rng.random() < 0.5)
    if kind == "run":
        precision = rng.choice(["fp32", "mixed", "fp64"])
        apl = rng.choice([8, 16, 32])
        return dict(kind=kind, n=_leaves(_log_int(rng, 4000, 262144), apl), steps=10 * rng.randint(3, 5),
                    precision=precision, apl=apl, resort=rng.choice([0, 50, 200]),
                    points=rng.choice(["lattice", "lattice", "blobs"]))
    if kind == "batch":
        return dict(kind=kind, reps=rng.randint(4, 96), lo=256, hi=_log_int(rng, 1024, 8192),
                    sizes=rng.randrange(1 << 20), steps=50,
                    apl=rng.choice([16, 32]))
    return dict(kind=kind, n=_leaves(_log_int(rng, 1000, 32768), 4), steps=10 * rng.randint(2, 5),
                precision=rng.choice(["fp32", "fp64"]))


# ---- inputs --------------------------------------------------------------

def _points(case, seed):
    """(positions, box side) of a search case, FP32 on the host."""
    n = case["n"]
    if case["points"] == "unit":
        return nd.synth.uniform_positions(n, 1.0, seed), 1.0
    L = nd.synth.box_side(n, DENSITY)
    if case["points"] == "uniform":
        return nd.synth.uniform_positions(n, L, seed), L
    return nd.synth.lattice_positions(n, L, seed).astype(np.float32), L


def _dynamics(case, seed):
    """Initial state of a dynamics case: x, v, q (FP64, host), box side."""
    n = case["n"]
    if case.get("points") == "blobs":
        # liquid droplets: half the box's mean density, droplet spacing 1.1
        L = nd.synth.box_side(n, 0.4)
        x = nd.synth.blob_positions(n, L, seed, nblobs=16, std=2.0, spacing=1.1)
    else:
        L = nd.synth.box_side(n, DENSITY)
        x = nd.synth.lattice_positions(n, L, seed)
    return dict(x=x, v=nd.synth.gaussian_velocities(n, 1.0, seed), q=nd.synth.balanced_charges(n, seed), L=L)


def _run_spec(case, L):
    return nd.SimSpec(duration=0, stepwidth=0.001, rc=2.5, rc_coul=2.5, skin=0.4 if case["points"] == "blobs" else 0.3,
                      rebuild_every=10, lo=0.0, hi=L, precision=case["precision"], energy_every=10, walls=True,
                      atomsperleaf=case["apl"], resort_every=case["resort"])


def _replicas(case, seed):
    sizes = nd.batched.replica_sizes(case["reps"], case["lo"], case["hi"], case["sizes"])
    return nd.batched.make_replicas(sizes, seed)


def _target(case, seed):
    """A measured radial distribution to fit: one broad first shell."""
    rng = np.random.default_rng(seed + 31)
    r = (np.arange(50) + 0.5) * (2.5 / 50)
    g = 1.0 / (1.0 + np.exp(-(r - 0.95) / 0.04)) * (1.0 + 1.4 * np.exp(-((r - 1.1) / 0.15) ** 2))
    return g + rng.normal(0.0, 0.01, 50)


def _adjoint_inputs(case, seed):
    s = _dynamics(case, seed)
    s["target"] = _target(case, seed)
    return s


# ---- one pass ------------------------------------------------------------

def _ok(rc, what):
    nd._lib.check(rc, nd.default_context(), what)


def _ptr(tensor):
    return ctypes.c_void_p(tensor.data_ptr())


def _search_state(case, x, device):
    """What a program that builds lists keeps: the specification and a pair
    buffer with room for them (as 32-bit words)."""
    cap = int(1.3 * _pair_count(case, case["r"])) + 1024
    state = dict(kind=case["kind"], x=x, cap=cap, r=case["r"], count=ctypes.c_int64(0),
                 key=KEYS[case.get("key", "masked")], pred=PREDS[case.get("pred", "simd")],
                 query=QUERIES[case.get("query", "own")],
                 out=torch.zeros((cap, 3), dtype=torch.int32, device="cuda") if device else np.zeros((cap, 3), np.int32))
    if "apl" in case:
        state["spec"] = nd.SpheresBVHSpecs(neighbor_distance=case["r"], atom_count=case["n"], atomsperleaf=case["apl"])
    return state


def prepare(case, seed):
    kind = case["kind"]
    ctx = nd.default_context()
    if kind == "list-host":
        return _search_state(case, nd.synth.uniform_positions(case["n"], 1.0, seed), False)
    if kind in ("list", "point", "cells"):
        return _search_state(case, nd.DeviceArray.from_host(ctx, _points(case, seed)[0]), True)
    if kind == "forces":
        n = case["n"]
        s = _dynamics(case, seed)
        x = nd.DeviceArray.from_host(ctx, s["x"].astype(np.float32))
        # the list a program keeps between builds, its own copy
        spec = nd.SpheresBVHSpecs(neighbor_distance=case["r"], atom_count=n, atomsperleaf=1)
        found, count = nd.neighborlist_device(x, spec, nd.PRED_SCALAR, nd.MORTON_INTERLEAVE, ctx)
        pairs = nd.DeviceArray(ctx, (count,), nd.PAIR_DTYPE)
        nd._lib.check(nd.library().nd_memcpy_d2d(ctx.handle, pairs.ptr, found.ptr, pairs.nbytes), ctx, "copy")
        out = [torch.zeros((n, 3), dtype=torch.float32, device="cuda") for _ in range(3)]
        ctx.synchronize()
        return dict(kind=kind, x=x, q=nd.DeviceArray.from_host(ctx, s["q"].astype(np.float32)),
                    pairs=pairs, count=count, out=out, e_lj=ctypes.c_double(0), e_c=ctypes.c_double(0),
                    # eps, sigma, rc, k, rc_coul, no energy shifts
                    params=nd._lib.ForceParams(1.0, 1.0, 2.5, 1.0, 2.5, 0, 0))
    if kind == "simulate":
        s = _dynamics(case, seed)
        spec = nd.SimSpec(duration=case["steps"], stepwidth=0.001, rc=2.5, rc_coul=2.5 if case["coul"] else 0.0,
                          skin=0.0 if case["rebuild"] == 1 else 0.3, rebuild_every=case["rebuild"], lo=0.0,
                          hi=s["L"], precision="fp32", energy_every=10, record_every=10)
        return dict(kind=kind, spec=spec, x=s["x"].astype(np.float32), v=s["v"].astype(np.float32),
                    q=s["q"].astype(np.float32) if case["coul"] else None)
    if kind == "run":
        s = _dynamics(case, seed)
        sim = nd.Simulation(case["n"], _run_spec(case, s["L"]))
        sim.set_state(s["x"], s["v"], s["q"])
        sim.prepare()
        sim.energies()
        dtype = torch.float32 if case["precision"] == "fp32" else torch.float64
        return dict(kind=kind, sim=sim, steps=case["steps"],
                    frame=torch.empty((case["n"], 3), dtype=dtype, device="cuda"))
    if kind == "batch":
        spec = nd.SimSpec(duration=0, stepwidth=0.001, rc=2.5, rc_coul=0.0, skin=0.3, rebuild_every=10,
                          precision="fp32", energy_every=10, atomsperleaf=case["apl"], resort_every=500)
        b = nd.BatchedSimulation(_replicas(case, seed), spec)
        b.set_state()
        b.prepare()
        b.energies()
        return dict(kind=kind, batch=b, sim=b.sim, steps=case["steps"],
                    frame=torch.empty((b.packed["n"], 3), dtype=torch.float32, device="cuda"))
    s = _adjoint_inputs(case, seed)
    adj = nd.Adjoint(case["n"], case["steps"], dt=0.001, precision=case["precision"], checkpoint_every=50,
                     rebuild_every=10, nbins=50, rdf_rmax=2.5, rdf_h=0.1, volume=s["L"] ** 3)
    return dict(kind=kind, adj=adj, x=s["x"], v=s["v"], q=s["q"], target=s["target"],
                dtype=np.float32 if case["precision"] == "fp32" else np.float64)


def run(state):
    kind, lib, ctx = state["kind"], nd.library(), nd.default_context().handle
    if kind in ("list-host", "list", "point", "cells"):
        x, out, count = state["x"], state["out"], ctypes.byref(state["count"])
        if kind == "list-host":
            rc = lib.nd_leafbuild_traverse_bvh_host(ctx, nd._lib.ptr(x), ctypes.byref(state["spec"].c), state["pred"],
                                                    state["key"], nd._lib.ptr(out), state["cap"], count)
        elif kind == "list":
            rc = lib.nd_leafbuild_traverse_bvh(ctx, x.ptr, ctypes.byref(state["spec"].c), state["pred"], state["key"],
                                               _ptr(out), state["cap"], count)
        elif kind == "point":
            rc = lib.nd_build_traverse_bvh(ctx, x.ptr, ctypes.byref(state["spec"].c), state["query"], state["key"],
                                           _ptr(out), state["cap"], count)
        else:
            rc = lib.nd_cell_neighborlist(ctx, x.ptr, x.shape[0], state["r"], state["pred"], _ptr(out), state["cap"],
                                          count)
        _ok(rc, kind)
        return dict(pairs=out, count=state["count"].value)
    if kind == "forces":
        x, pairs, count, params = state["x"], state["pairs"], state["count"], ctypes.byref(state["params"])
        f_lj, f_c, f = state["out"]
        n, e_lj, e_c = x.shape[0], state["e_lj"], state["e_c"]
        _ok(lib.nd_force_lennardjones(ctx, _ptr(f_lj), pairs.ptr, count, x.ptr, n, params, ctypes.byref(e_lj)), kind)
        _ok(lib.nd_force_coulomb(ctx, _ptr(f_c), pairs.ptr, count, x.ptr, state["q"].ptr, n, params,
                                 ctypes.byref(e_c)), kind)
        _ok(lib.nd_sum_forces(ctx, _ptr(f), _ptr(f_lj), _ptr(f_c), n), kind)
        return dict(e_lj=e_lj.value, e_c=e_c.value, f_lj=f_lj, f_c=f_c, f=f)
    if kind == "simulate":
        sys = nd.ObjectCollection(position=state["x"].copy(), velocity=state["v"].copy(), charge=state["q"])
        poslog = nd.simulate_(sys, state["spec"])
        return dict(frames=np.stack(poslog).astype(np.float32), x=sys.position, v=sys.velocity,
                    energies=sys.energies[:, 1:4].astype(np.float32))
    if kind in ("run", "batch"):
        state["sim"].run(state["steps"])
        # a trajectory frame in original atom order, on the device
        _ok(lib.nd_sim_record_positions(state["sim"].handle, _ptr(state["frame"]),
                                        int(state["frame"].dtype == torch.float64)), kind)
        rows = state["sim"].energies()[:, 1:4]
        return dict(x=state["frame"],
                    energies=rows.astype(np.float32) if state["frame"].dtype == torch.float32 else rows.copy())
    adj, to = state["adj"], state["dtype"]
    loss, rdf = adj.forward(state["x"], state["v"], state["q"], state["target"])
    g = adj.backward()
    return dict(loss=to(loss), rdf=rdf.astype(to), deps=to(g["deps"]), dsigma=to(g["dsigma"]),
                dx0=g["dx0"].astype(to), dv0=g["dv0"].astype(to), dq=g["dq"].astype(to))


# ---- the work of one pass ------------------------------------------------

def _pair_count(case, r):
    """Unordered pairs within r (the mean of the distribution)."""
    density = case["n"] if case.get("points", "unit") == "unit" else DENSITY
    return 0.5 * case["n"] * density * 4.0 / 3.0 * math.pi * r ** 3


def _liquid_pairs(n, r):
    return _pair_count(dict(n=n, points="lattice"), r)


def work(case):
    kind = case["kind"]
    if kind in ("list", "list-host", "point", "cells"):
        pairs = _pair_count(case, case["r"])
        return {"bytes": 12.0 * case["n"] + 12.0 * pairs, "flops": 9.0 * pairs}
    if kind == "forces":
        pairs, inside = _liquid_pairs(case["n"], case["r"]), _liquid_pairs(case["n"], 2.5)
        # the list and the positions once for each term; three forces written
        return {"bytes": 2 * (12.0 * pairs + 12.0 * case["n"]) + (4 + 3 * 12 + 2 * 12) * case["n"],
                "flops": inside * 2 * 24.0 + 3.0 * case["n"]}
    if kind == "adjoint":
        # forward force, recomputed force and one Hessian product per step;
        # positions, velocities and two adjoints (FP64) read and written
        inside = _liquid_pairs(case["n"], 2.5)
        per = 8 if case["precision"] == "fp64" else 4
        return {"bytes": case["steps"] * case["n"] * (2 * 12.0 * per + 4 * 24.0),
                "flops": case["steps"] * inside * (2 * 32.0 + 90.0)}
    if kind == "batch":
        n = int(nd.batched.replica_sizes(case["reps"], case["lo"], case["hi"], case["sizes"]).sum())
        per, flops = 4, 26.0
    else:
        n = case["n"]
        per = 8 if case.get("precision") in ("fp64", "mixed") else 4
        flops = 32.0 if kind == "run" or case["coul"] else 26.0
    inside = _liquid_pairs(n, 2.5)
    # a step reads and writes each atom's position and velocity
    return {"bytes": case["steps"] * n * 4.0 * 3 * per, "flops": case["steps"] * (inside * flops + 18.0 * n)}


# ---- 64-bit values -------------------------------------------------------

def _pairs_within(x, r):
    """(i, j) of every unordered pair of x (n x 3, FP64) closer than r."""
    n, dev = len(x), x.device
    lo = x.min(0).values
    g = torch.clamp(((x.max(0).values - lo) / r).floor().long(), min=1)
    c = torch.minimum(((x - lo) / r).floor().long(), g - 1)
    key = (c[:, 2] * g[1] + c[:, 1]) * g[0] + c[:, 0]
    key, order = torch.sort(key, stable=True)
    xs, cs = x[order], c[order]
    start = torch.searchsorted(key, torch.arange(int(g.prod()) + 1, device=dev))
    half = [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1) if (dz, dy, dx) > (0, 0, 0)]
    at = torch.arange(n, device=dev)
    ii, jj = [], []
    for d in [(0, 0, 0)] + half:
        t = cs + torch.tensor(d, device=dev)
        ok = ((t >= 0) & (t < g)).all(1)
        k = torch.where(ok, (t[:, 2] * g[1] + t[:, 1]) * g[0] + t[:, 0], 0)
        b, e = start[k], torch.where(ok, start[k + 1], start[k])
        if d == (0, 0, 0):
            b = at + 1
        m = torch.clamp(e - b, min=0)
        i = torch.repeat_interleave(at, m)
        j = torch.arange(len(i), device=dev) - torch.repeat_interleave(torch.cumsum(m, 0) - m, m) + b[i]
        near = ((xs[i] - xs[j]) ** 2).sum(1) < r * r
        ii.append(order[i[near]])
        jj.append(order[j[near]])
    return torch.cat(ii), torch.cat(jj)


def _force(x, q, pairs, rc, coul, block=1 << 23):
    """Cut Lennard-Jones (+ Coulomb) forces, energy and virial in FP64."""
    f = torch.zeros_like(x)
    pe = torch.zeros((), dtype=x.dtype, device=x.device)
    vir = torch.zeros_like(pe)
    for i, j in zip(pairs[0].split(block), pairs[1].split(block)):
        d = x[i] - x[j]
        r2 = (d * d).sum(1)
        keep = r2 < rc * rc
        i, j, d, r2 = i[keep], j[keep], d[keep], r2[keep]
        i6 = 1.0 / r2 ** 3
        s = 24.0 * i6 * (2.0 * i6 - 1.0) / r2
        pe += (4.0 * i6 * (i6 - 1.0)).sum()
        if coul:
            e = q[i] * q[j] / torch.sqrt(r2)
            s = s + e / r2
            pe += e.sum()
        vir += (s * r2).sum()
        p = s[:, None] * d
        f.index_add_(0, i, p)
        f.index_add_(0, j, -p)
    return f, pe, vir


def _trajectory(x, v, q, dt, steps, lo, hi, coul, frame_every=0, energy_every=10):
    """Kick-drift-force-kick steps with reflecting walls (lo, hi: per axis or
    per atom and axis): positions, velocities, frames, energy rows."""
    skin, every = 0.6, 20
    frames, rows = [x.clone()], []
    pairs = _pairs_within(x, 2.5 + skin)
    f, pe, vir = _force(x, q, pairs, 2.5, coul)
    for k in range(steps):
        if k % energy_every == 0 and k > 0:
            rows.append(torch.stack([0.5 * (v * v).sum(), pe, vir]))
        v = v + 0.5 * dt * f
        x = x + dt * v
        low, high = x < lo, x > hi
        v = torch.where(low | high, -v, v)
        x = torch.where(low, lo, torch.where(high, hi, x))
        if (k + 1) % every == 0:
            pairs = _pairs_within(x, 2.5 + skin)
        f, pe, vir = _force(x, q, pairs, 2.5, coul)
        v = v + 0.5 * dt * f
        if frame_every and (k + 1) % frame_every == 0:
            frames.append(x.clone())
    rows.append(torch.stack([0.5 * (v * v).sum(), pe, vir]))
    return x, v, frames, torch.stack(rows)


def _adjoint_exact(case, seed):
    s = _adjoint_inputs(case, seed)
    dev = "cuda"
    x0, v0, q = (torch.tensor(s[k], device=dev, requires_grad=True) for k in ("x", "v", "q"))
    eps, sigma = (torch.tensor(1.0, dtype=torch.float64, device=dev, requires_grad=True) for _ in range(2))
    rc, dt, n = 2.5, 0.001, case["n"]

    def force(x, pairs):
        i, j = pairs
        d = x[i] - x[j]
        r = torch.sqrt((d * d).sum(1))
        lj = lambda u: 24.0 * eps * (2.0 * (sigma / u) ** 12 - (sigma / u) ** 6) / u  # noqa: E731
        s_ = (lj(r) - lj(torch.full_like(eps, rc))) / r + q[i] * q[j] * (1.0 / r ** 2 - 1.0 / rc ** 2) / r
        p = torch.where(r < rc, s_, torch.zeros_like(s_))[:, None] * d
        return torch.zeros_like(x).index_add(0, i, p).index_add(0, j, -p)

    x, v = x0, v0
    pairs = _pairs_within(x.detach(), 3.1)
    f = force(x, pairs)
    for k in range(case["steps"]):
        v = v + 0.5 * dt * f
        x = x + dt * v
        if (k + 1) % 20 == 0:
            pairs = _pairs_within(x.detach(), 3.1)
        f = force(x, pairs)
        v = v + 0.5 * dt * f
    i, j = _pairs_within(x.detach(), 2.7)
    r = torch.sqrt(((x[i] - x[j]) ** 2).sum(1))
    dr, h = 2.5 / 50, 0.1
    rb = (torch.arange(50, dtype=torch.float64, device=dev) + 0.5) * dr
    g = []
    for b in range(50):
        u = (r - rb[b]) / h
        g.append(torch.where(u.abs() < 1.0, (1.0 - u * u) ** 3, torch.zeros_like(u)).sum())
    g = torch.stack(g) * (s["L"] ** 3 / (0.5 * n * (n - 1) * 4.0 * math.pi * rb * rb * dr))
    loss = ((g - torch.tensor(s["target"], device=dev)) ** 2).sum()
    loss.backward()
    return dict(loss=loss.detach(), rdf=g.detach(), deps=eps.grad, dsigma=sigma.grad, dx0=x0.grad, dv0=v0.grad,
                dq=q.grad)


def exact(case, seed):
    """64-bit values of run()'s outputs; None for the pair lists, whose words
    are whole numbers."""
    kind = case["kind"]
    if kind in ("list", "list-host", "point", "cells"):
        return None
    if kind == "adjoint":
        return _adjoint_exact(case, seed)
    if kind == "batch":
        P = nd.batched.pack(_replicas(case, seed), 3.8, case["apl"])
        rep = torch.tensor(P["rep"], device="cuda").long()
        boxes = torch.tensor(np.concatenate([P["boxes"], [[-math.inf] * 3 + [math.inf] * 3]]), device="cuda")
        b = boxes[rep]  # padding atoms (replica -1) take the last row: no walls
        x, v, q = (torch.tensor(P[k], device="cuda") for k in ("x", "v", "q"))
        x, _, _, rows = _trajectory(x, v, q, 0.001, case["steps"], b[:, :3], b[:, 3:], False)
        return dict(x=x, energies=rows)
    s = _dynamics(case, seed)
    single = kind in ("forces", "simulate")  # their inputs are FP32 arrays
    x, v, q = (torch.tensor(s[k].astype(np.float32).astype(np.float64) if single else s[k], device="cuda")
               for k in ("x", "v", "q"))
    if kind == "forces":
        pairs = _pairs_within(x, case["r"])
        f_lj, e_lj, _ = _force(x, q, pairs, 2.5, False)
        f, e, _ = _force(x, q, pairs, 2.5, True)
        return dict(e_lj=e_lj, e_c=e - e_lj, f_lj=f_lj, f_c=f - f_lj, f=f)
    lo, hi = torch.zeros((), dtype=x.dtype, device="cuda"), torch.tensor(s["L"], dtype=x.dtype, device="cuda")
    if kind == "simulate":
        x, v, frames, rows = _trajectory(x, v, q, 0.001, case["steps"], lo, hi, case["coul"], frame_every=10)
        return dict(frames=torch.stack(frames), x=x, v=v, energies=None)
    x, _, _, rows = _trajectory(x, v, q, 0.001, case["steps"], lo, hi, True)
    return dict(x=x, energies=rows)
