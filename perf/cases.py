"""The workloads whose time is measured: what a program that uses this package has it do.

A friction-contact program solves problems (through the reference's driver, on a resident
problem, or many at once), assembles them, evaluates their residual, and trains the warm-start
network.  Every case goes through the package's Python surface or its C interface, and ends, as
such a program does, with the reactions and velocities on the host (the residual entry, which works
on the caller's device arrays, leaves its results there).

The problems come from the package's seeded generators (random sphere pairs, granular piles), at
the sizes of its tests and benchmark; the 2-D problems are granular layers made here, at the sizes
of the 2-D fixtures.
"""
import ctypes as C
import math

import numpy as np
import torch

from siconos_amd import capi, warmstart
from siconos_amd import numerics as N

FOCUS = dict(focus_passes=50, focus_every=16, focus_after=64, focus_count=256, focus_share=0.5,
             focus_omega=1.2)
FAST = dict(precision=1, fp32_tol=1e-6, fp32_local_solver=550, fp32_local_tol=1e-7)


def listed():
    return [
        # one call of the drop-in driver on a handful of contacts (a small mechanism), default
        # tolerance: the smallest call, all latency
        {"name": "driver_40", "kind": "driver", "nc": 40, "nbodies": 16, "tol": 1e-4},
        # the same driver on 1000 contacts of 300 spheres to 1e-8, hundreds of sweeps
        {"name": "driver_1000", "kind": "driver", "nc": 1000, "nbodies": 300, "tol": 1e-8},
        # plain FP64 solves of a resident problem: 50k random pairs to 1e-6, and a granular pile
        # of odd size to the reference's default tolerance
        {"name": "plain_pairs_50k", "kind": "plain", "gen": "pairs", "nc": 50_000,
         "nbodies": 20_000, "tol": 1e-6},
        {"name": "plain_pile_300k", "kind": "plain", "gen": "pile", "nc": 300_007,
         "nbodies": 120_001, "tol": 1e-4},
        # the fast method (velocity form, FP32 sweeps with FP64 refinement, focused passes) on
        # the 1M-contact pile
        {"name": "fast_pile_1m", "kind": "fast", "nc": 1_000_000, "nbodies": 400_000,
         "tol": 1e-6},
        # one step of a simulation: new values of W, q and mu on a kept contact set, then a solve
        # from the previous step's reactions
        {"name": "step_pile_50k", "kind": "step", "nc": 50_000, "nbodies": 20_000, "tol": 1e-4},
        # many independent problems at once, all FP64 and in mixed precision
        {"name": "batch_fp64_1024", "kind": "batch", "nprob": 1024, "lo": 8, "hi": 512,
         "mixed": False},
        {"name": "batch_mixed_4096", "kind": "batch", "nprob": 4096, "lo": 8, "hi": 512,
         "mixed": True},
        # a 2-D granular layer of about the largest 2-D fixture's size
        {"name": "fc2d_7k", "kind": "fc2d", "cols": 100, "rows": 50, "tol": 1e-5},
        # the residual on the caller's device arrays, as a caller with its own solver has it
        {"name": "residual_1m", "kind": "residual", "nc": 1_000_000, "nbodies": 400_000},
        # W = H M^-1 H^T and q = H v_free of one time step's contact set
        {"name": "assemble_200k", "kind": "assemble", "nc": 200_000, "nbodies": 80_000},
        # the warm-start network trained from a solved problem's contacts
        {"name": "train_20k", "kind": "train", "nc": 20_000, "nbodies": 8_000, "epochs": 4,
         "batch": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["driver", "plain", "fast", "step", "batch", "fc2d", "residual", "assemble",
                       "train"])
    if kind == "driver":
        nc = _log(rng, 8, 2000)
        return {"kind": kind, "nc": nc, "nbodies": max(8, int(nc * rng.uniform(0.3, 0.5))),
                "tol": rng.choice([1e-4, 1e-6, 1e-8])}
    if kind == "plain":
        nc = _log(rng, 2000, 300_000)
        return {"kind": kind, "gen": rng.choice(["pairs", "pile"]), "nc": nc,
                "nbodies": int(nc * rng.uniform(0.38, 0.5)),
                "tol": 1e-4 if nc > 50_000 else rng.choice([1e-4, 1e-6])}
    if kind == "fast":
        nc = _log(rng, 20_000, 1_000_000)
        return {"kind": kind, "nc": nc, "nbodies": int(nc * 0.4), "tol": 1e-6}
    if kind == "step":
        nc = _log(rng, 2000, 50_000)
        return {"kind": kind, "nc": nc, "nbodies": int(nc * rng.uniform(0.38, 0.5)), "tol": 1e-4}
    if kind == "batch":
        return {"kind": kind, "nprob": _log(rng, 16, 1024), "lo": 8, "hi": _log(rng, 32, 512),
                "mixed": rng.random() < 0.5}
    if kind == "fc2d":
        return {"kind": kind, "cols": _log(rng, 8, 100), "rows": _log(rng, 3, 50), "tol": 1e-5}
    if kind == "residual":
        nc = _log(rng, 100, 1_000_000)
        return {"kind": kind, "nc": nc, "nbodies": max(30, int(nc * rng.uniform(0.38, 0.5)))}
    if kind == "assemble":
        nc = _log(rng, 100, 200_000)
        return {"kind": kind, "nc": nc, "nbodies": max(30, int(nc * rng.uniform(0.38, 0.5)))}
    return {"kind": kind, "nc": _log(rng, 2000, 20_000), "nbodies": 8_000,
            "epochs": rng.randint(1, 4), "batch": 64 * rng.randint(2, 16)}


# ---- the problems -----------------------------------------------------------------------------

def _pairs(case, seed):
    return N.generate_random_pairs(case["nbodies"], case["nc"], 0.2, 0.5, seed)


def _pile(case, seed):
    return N.generate_granular_pile(case["nbodies"], case["nc"], 0.1, 0.9, seed)


def _layer(case, seed):
    """A 2-D granular layer: discs of radius 1 on a jittered hexagonal lattice over a floor, in
    contact with about half their neighbours (4.5 blocks a row of W, as in the 2-D fixtures) and
    with the floor.  Which ones is the case's; positions, velocities and friction are the seed's.
    Returns W's blocks (row, column, 2x2 values, row by row), q and mu."""
    rng = np.random.default_rng(seed)
    which = np.random.default_rng([case["cols"], case["rows"]])
    nx, ny = case["cols"], case["rows"]
    k = np.arange(nx * ny)
    i, j = k % nx, k // nx
    x = np.stack([2.0 * i + (j & 1) + 0.05 * rng.uniform(-1, 1, k.size),
                  math.sqrt(3.0) * j + 0.05 * rng.uniform(-1, 1, k.size)], 1)
    a, b = [], []
    right = k[i + 1 < nx]
    a.append(right)
    b.append(right + 1)
    for side in (0, 1):  # the two neighbours in the row above
        i2 = i + side - 1 + (j & 1)
        ok = (j + 1 < ny) & (i2 >= 0) & (i2 < nx)
        a.append(k[ok])
        b.append((i2 + nx * (j + 1))[ok])
    floor = k[j == 0]
    a, b = np.concatenate(a), np.concatenate(b)
    keep = which.random(a.size) < 0.47
    a = np.concatenate([a[keep], floor])
    b = np.concatenate([b[keep], np.full(floor.size, -1)])
    n = np.where((b >= 0)[:, None], x[a] - x[b], np.array([0.0, 1.0]))
    n /= np.linalg.norm(n, axis=1)[:, None]
    order = np.argsort(a, kind="stable")
    a, b, n = a[order], b[order], n[order]
    nc = a.size
    t = np.stack([-n[:, 1], n[:, 0]], 1)
    # rows (normal, tangent) of H for both bodies: (v, omega), lever arms -n and +n
    H = np.zeros((2, nc, 2, 3))
    H[0, :, 0, :2], H[0, :, 1, :2], H[0, :, 1, 2] = n, t, -1.0
    H[1, :, 0, :2], H[1, :, 1, :2], H[1, :, 1, 2] = -n, -t, -1.0
    H[1, b < 0] = 0.0
    minv = np.array([1.0, 1.0, 2.0])
    v = 0.3 * rng.standard_normal((nx * ny, 3)) * np.array([1.0, 1.0, 0.5])
    v[:, 1] -= 1.0
    q = np.einsum("cij,cj->ci", H[0], v[a]) + np.einsum("cij,cj->ci", H[1], v[np.maximum(b, 0)])
    # contacts of each body, padded, and every ordered pair of them
    body = np.concatenate([a, b[b >= 0]])
    cont = np.concatenate([np.arange(nc), np.arange(nc)[b >= 0]])
    side = np.concatenate([np.zeros(nc, int), np.ones(int((b >= 0).sum()), int)])
    order = np.argsort(body, kind="stable")
    body, cont, side = body[order], cont[order], side[order]
    start = np.searchsorted(body, np.arange(nx * ny + 1))
    most = int((start[1:] - start[:-1]).max())
    pos = np.arange(body.size) - start[body]
    table = np.full((nx * ny, most), -1)
    table[body, pos] = np.arange(body.size)
    p, r = np.broadcast_arrays(table[:, :, None], table[:, None, :])
    ok = (p >= 0) & (r >= 0)
    p, r = p[ok], r[ok]
    c, d = cont[p], cont[r]
    blocks = np.einsum("kil,l,kjl->kij", H[side[p], c], minv, H[side[r], d])
    key, where = np.unique(c.astype(np.int64) * nc + d, return_inverse=True)
    W = np.zeros((key.size, 2, 2))
    np.add.at(W, where, blocks)
    return key // nc, key % nc, W, q, rng.uniform(0.2, 0.7, nc)


def _fc2d_handle(case, seed):
    row, col, W, q, mu = _layer(case, seed)
    nc = mu.size
    # scalar rows: every block gives two entries to each of its two rows
    per = np.bincount(row, minlength=nc)
    rp = np.concatenate([[0], np.cumsum(np.repeat(2 * per, 2))]).astype(np.int64)
    first = np.concatenate([[0], np.cumsum(per)])[:-1]
    at = np.arange(row.size) - first[row]
    cols = np.zeros(rp[-1], np.int64)
    vals = np.zeros(rp[-1])
    for i in range(2):
        for k in range(2):
            e = rp[2 * row + i] + 2 * at + k
            cols[e] = 2 * col + k
            vals[e] = W[:, i, k]
    diag = np.ascontiguousarray(W[row == col].transpose(0, 2, 1)).reshape(-1)
    q = np.ascontiguousarray(q.reshape(-1))
    h = C.c_void_p()
    rc = capi.load().fc2d_hip_problem_create(nc, N.lptr(rp), N.lptr(cols), N.dptr(vals), 0, 0,
                                             N.dptr(diag), N.dptr(q), N.dptr(mu), 0, C.byref(h))
    if rc:
        raise RuntimeError(f"fc2d_hip_problem_create: {rc} {capi.last_error()}")
    p = N.Fc2dHipProblem.__new__(N.Fc2dHipProblem)
    p._lib, p.nc, p._h = capi.load(), nc, h
    return p


def _many(case, seed):
    """Independent random-pair problems, nc ~ U[lo, hi] (the case's sizes), bodies = nc / 2.5."""
    sizes = np.random.default_rng(case["nprob"]).integers(case["lo"], case["hi"] + 1,
                                                          case["nprob"])
    out = []
    for k, n in enumerate(sizes):
        nb = max(3, int(round(n * 0.4)))
        while n > nb * (nb - 1) // 2:
            nb += 1
        g = N.generate_random_pairs(nb, int(n), 0.1, 0.9, seed * 1000003 + k)
        out.append((g.W, g.q, g.mu))
    return out


def _factors(case, seed):
    """What a simulation hands to the assembly: a pile's contacts (which ones is the case's), with
    the seed's contact frames, masses and velocities.  Spheres of unit radius."""
    g = _pile_or_pairs(case, 1)
    rng = np.random.default_rng(seed)
    H = g.H.reshape(g.nc, 12, 3).copy()  # columns of both 3x6 blocks
    a = rng.uniform(0.0, 2.0 * math.pi, g.nc)  # the tangents turned about the normal
    c, s = np.cos(a)[:, None], np.sin(a)[:, None]
    H[:, :, 1], H[:, :, 2] = c * H[:, :, 1] + s * H[:, :, 2], c * H[:, :, 2] - s * H[:, :, 1]
    m = rng.uniform(0.5, 2.0, g.nbodies)
    minv = np.repeat(np.stack([1.0 / m, 2.5 / m], 1), 3, 1)
    v = rng.standard_normal((g.nbodies, 6))
    return g, np.ascontiguousarray(H.reshape(-1)), minv.reshape(-1), v.reshape(-1)


def _reaction(nc, seed):
    """Reactions of the kind a solver passes on the way: most inside the cone, some open."""
    rng = np.random.default_rng(seed + 1)
    r = np.empty((nc, 3))
    r[:, 0] = np.maximum(0.0, rng.standard_normal(nc))
    r[:, 1:] = 0.3 * r[:, :1] * rng.uniform(-1, 1, (nc, 2))
    return np.ascontiguousarray(r.reshape(-1))


# ---- prepare and run --------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "driver":
        g = _pairs(case, seed)
        s["problem"], s["nc"] = g.problem(), g.nc
        o = N.SolverOptions(N.SICONOS_FRICTION_3D_NSGS_HIP)
        o.dparam[N.SICONOS_DPARAM_TOL] = case["tol"]
        s["options"] = o
    elif kind == "plain":
        g = _pairs(case, seed) if case["gen"] == "pairs" else _pile(case, seed)
        s["H"] = N.HipProblem(g.W, g.q, g.mu)
        s["params"] = N.hip_params(tol=case["tol"], warm_start=1)
    elif kind == "fast":
        g = _pile(case, seed)
        s["H"] = N.HipProblem(g.W, g.q, g.mu)
        s["H"].set_bodies(g.nbodies, g.body_a, g.body_b, g.H, g.minv, g.vfree)
        s["params"] = N.hip_params(tol=case["tol"], max_iter=3000, warm_start=1, velocity_form=1,
                                   sweeps_per_launch=16, **FAST, **FOCUS)
    elif kind == "step":
        g = _pile(case, seed)
        rng = np.random.default_rng(seed)
        s["H"] = N.HipProblem(g.W, g.q, g.mu)
        s["H"].solve(N.hip_params(tol=case["tol"], warm_start=1))
        s["previous"] = s["H"].reaction()
        s["values"] = g.W.values * (1.0 + 1e-3 * float(rng.uniform(-1, 1)))
        s["q"] = g.q * (1.0 + 0.02 * rng.standard_normal(g.q.size))
        s["mu"] = g.mu
        s["params"] = N.hip_params(tol=case["tol"], warm_start=0)
    elif kind == "batch":
        s["B"] = N.Batch(_many(case, seed))
        s["params"] = N.hip_params(tol=1e-6, max_iter=1000, warm_start=1,
                                   **(FAST if case["mixed"] else {}))
    elif kind == "fc2d":
        s["P"] = _fc2d_handle(case, seed)
        s["zero"], s["tol"] = np.zeros(2 * s["P"].nc), case["tol"]
    elif kind == "residual":
        g = _pile_or_pairs(case, seed)
        dev = [torch.from_numpy(np.ascontiguousarray(v)).to("cuda")
               for v in (g.W.row_ptr, g.W.col_idx, g.W.values, g.q, g.mu,
                         _reaction(g.nc, seed))]
        s["in"], s["nc"], s["nnzb"] = dev, g.nc, g.W.nnzb
        s["norm"] = float(np.linalg.norm(g.q))
        s["u"] = torch.empty(3 * g.nc, dtype=torch.float64, device="cuda")
        s["error"] = torch.empty(1, dtype=torch.float64, device="cuda")
    elif kind == "assemble":
        g, H, minv, v = _factors(case, seed)
        s["args"] = (g.nbodies, g.body_a, g.body_b, H, minv, v)
    else:
        g = _pairs(case, seed)
        s["x"], s["t"], _ = warmstart.collect([(g.W, g.q, g.mu)], tol=1e-4)
        s["epochs"], s["batch"], s["seed"] = case["epochs"], case["batch"], seed & 0xffff
    return s


def _pile_or_pairs(case, seed):
    return _pile(case, seed) if case["nc"] >= 1000 else _pairs(case, seed)


def run(s):
    kind = s["kind"]
    if kind == "driver":
        r, u = np.zeros(3 * s["nc"]), np.zeros(3 * s["nc"])
        info = N.fc3d_driver(s["problem"], r, u, s["options"])
        return r, u, info
    if kind in ("plain", "fast"):
        st = s["H"].solve(s["params"])
        return s["H"].reaction(), s["H"].velocity(), st.iterations
    if kind == "step":
        H = s["H"]
        H.update(s["values"], s["q"], s["mu"])
        H.set_reaction(s["previous"])
        st = H.solve(s["params"])
        return H.reaction(), H.velocity(), st.iterations
    if kind == "batch":
        st, info, sweeps, res = s["B"].solve(s["params"])
        return s["B"].reaction(), s["B"].velocity(), sweeps
    if kind == "fc2d":
        s["P"].set_reaction(s["zero"])
        st = s["P"].solve(max_iter=2000, tol=s["tol"])
        return s["P"].reaction(), s["P"].velocity(), st.iterations
    if kind == "residual":
        rc = capi.load().fc3d_hip_compute_error_device(
            s["nc"], s["nnzb"], *(v.data_ptr() for v in s["in"]), s["norm"], s["u"].data_ptr(),
            s["error"].data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError(capi.last_error())
        return s["u"], s["error"]
    if kind == "assemble":
        W, q, _ = N.assemble(*s["args"])
        return W.row_ptr, W.col_idx, W.values, q
    m, loss = warmstart.train(s["x"], s["t"], seed=s["seed"], epochs=s["epochs"],
                              batch=s["batch"])
    params, mean, std = m.params()
    return params, mean, std, loss


# ---- what a pass cannot do without ------------------------------------------------------------

def _blocks(nc, nbodies):
    """Stored 3x3 blocks of W, about: every contact against the others of its two bodies."""
    per_body = 2.0 * nc / nbodies
    return nc * (2.0 * per_body - 1.0 + 0.5)


def work(case):
    """Inputs read once and outputs written once; a solve's products once per stored block (how
    many sweeps it takes is the problem's)."""
    kind = case["kind"]
    if kind == "batch":
        nc = case["nprob"] * (case["lo"] + case["hi"]) / 2.0
        nnzb = nc * 9.0
    elif kind == "fc2d":
        nc = case["cols"] * case["rows"] * 1.4
        return {"bytes": nc * (4.5 * 2 * 2 * 12 + 16 + 8 + 16 + 16), "flops": nc * 4.5 * 8}
    else:
        nc = float(case["nc"])
        nnzb = _blocks(nc, case["nbodies"])
    if kind in ("driver", "plain", "batch"):
        return {"bytes": nnzb * 76 + nc * (24 + 8 + 24 + 24), "flops": nnzb * 18}
    if kind == "fast":  # frames, lever arms, W_cc, q, mu; the FP64 residual reads W
        return {"bytes": nnzb * 76 + nc * (15 * 4 + 9 * 4 + 24 + 8 + 24 + 24),
                "flops": nnzb * 18 + nc * 200}
    if kind == "step":
        return {"bytes": nnzb * (72 + 76) + nc * (24 + 8 + 24 + 24 + 24), "flops": nnzb * 18}
    if kind == "residual":
        return {"bytes": nnzb * 80 + nc * (8 + 24 + 8 + 24 + 24), "flops": nnzb * 18 + nc * 40}
    if kind == "assemble":
        return {"bytes": nc * (288 + 8 + 24 + 8) + case["nbodies"] * 96 + nnzb * 80,
                "flops": nnzb * 108 + nc * 36}
    per = 2.0 * (22 * 128 + 2 * 128 * 128 + 128 * 3)
    return {"bytes": nc * 25 * 4 * case["epochs"] + 39312 * 4,
            "flops": 3 * per * nc * case["epochs"]}


# ---- 64-bit references ------------------------------------------------------------------------

def exact(case, seed):
    """The residual and the assembly have one right answer.  A solve stops at its tolerance, and
    the reactions of a hyperstatic problem are not unique; a training run's rounding goes through
    every later step: those have none."""
    if case["kind"] == "residual":
        g = _pile_or_pairs(case, seed)
        r = _reaction(g.nc, seed).reshape(-1, 3)
        u = g.q.reshape(-1, 3).copy()
        rows = np.repeat(np.arange(g.nc), np.diff(g.W.row_ptr))
        prod = np.einsum("kji,kj->ki", g.W.values.reshape(-1, 3, 3), r[g.W.col_idx])
        for e in range(3):
            u[:, e] += np.bincount(rows, weights=prod[:, e], minlength=g.nc)
        w = r - u
        w[:, 0] -= g.mu * np.hypot(u[:, 1], u[:, 2])
        nt = np.hypot(w[:, 1], w[:, 2])
        zero = g.mu * nt <= -w[:, 0]
        inside = ~zero & (nt <= g.mu * w[:, 0])
        slide = ~zero & ~inside
        p = np.where(inside[:, None], w, 0.0)
        pn = (g.mu * nt + w[:, 0]) / (g.mu ** 2 + 1.0)
        p[slide, 0] = pn[slide]
        p[slide, 1:] = (g.mu * pn / np.where(nt > 0, nt, 1.0))[slide, None] * w[slide, 1:]
        scale = max(np.linalg.norm(g.q), np.linalg.norm(r), np.linalg.norm(u))
        return u.reshape(-1), np.array([np.linalg.norm(r - p) / scale])
    if case["kind"] == "assemble":
        g, H, minv, v = _factors(case, seed)
        H = H.reshape(g.nc, 2, 6, 3)  # column-major 3x6 blocks: [side][column][row]
        minv, v = minv.reshape(-1, 6), v.reshape(-1, 6)
        ab = np.stack([g.body_a, g.body_b], 1)
        G = H * minv[ab][..., None]
        q = np.einsum("cslr,csl->cr", H, v[ab]).reshape(-1)
        rows = np.repeat(np.arange(g.nc), np.diff(g.W.row_ptr))
        W = np.zeros((g.W.nnzb, 3, 3))  # [block][column][row]
        for s1 in range(2):
            for s2 in range(2):
                k = np.nonzero(ab[rows, s1] == ab[g.W.col_idx, s2])[0]
                W[k] += np.einsum("kli,klj->kji", G[rows[k], s1], H[g.W.col_idx[k], s2])
        return g.W.row_ptr, g.W.col_idx, W.reshape(-1, 9), q
    return None
