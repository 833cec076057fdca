"""What is timed: the work a program using this library has it do, through the
public entry points.

A program builds a scene, initialises a `pdipc.Simulator` once and then, per
pass, restarts it from a state it holds on the host (`set_x`, `set_v`), runs a
few PD-IPC steps and reads the state back -- what a frame loop, a replay or a
trajectory search does -- or differentiates a rollout, or asks for the time of
impact of device-resident positions.  The scenes are the repository's own
(`scenes.py`): cloths dropped on a noisy sphere and a ground plane, tet blocks
under a cloth, stacked cloths; FP64 and FP32-split; one triangle patch to a
half million triangles; free fall, where a few outer iterations of the
local/global loop are the whole step, and contact, where the time-of-impact
and barrier passes run up to 30 times.

`exact` restates the step where nothing touches (the time of impact is 1 and
no barrier record is active) in plain torch, in 64 bits, for cloths and tet
blocks, with its derivative by autograd.
"""

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "pd-ipc-armadillodemo_amd"))

import pdipc  # noqa: E402
import scenes  # noqa: E402
from pdipc_autograd import PdIpcRollout  # noqa: E402


def listed():
    return [
        # the smallest scene in the tests' style: a 12 x 12 cloth reaching the sphere, default switches
        # (no graph replay): launches and host waits are all it costs
        dict(name="cloth12_fp64_contact", kind="step", scene="cloth", n=12, subdiv=2, fp32=False, graphs=False,
             contact=True, steps=2),
        # the 64^2 cloth over the subdivision-4 sphere, the small reference scene, in free fall
        dict(name="cloth64_fp64_fall", kind="step", scene="cloth", n=64, subdiv=4, fp32=False, graphs=True,
             contact=False, steps=4),
        # the same kind of scene at an odd size, landing, in the fast precision
        dict(name="cloth97_fp32_contact", kind="step", scene="cloth", n=97, subdiv=4, fp32=True, graphs=True,
             contact=True, steps=2),
        # the benchmark's 256^2 cloth while it falls, FP32-split
        dict(name="cloth256_fp32_fall", kind="step", scene="cloth", n=256, subdiv=6, fp32=True, graphs=True,
             contact=False, steps=4),
        # the benchmark's cloth landing on the sphere, both precisions
        dict(name="cloth256_fp32_contact", kind="step", scene="cloth", n=256, subdiv=6, fp32=True, graphs=True,
             contact=True, steps=2),
        dict(name="cloth256_fp64_contact", kind="step", scene="cloth", n=256, subdiv=6, fp32=False, graphs=True,
             contact=True, steps=2),
        # a cloth four times as large
        dict(name="cloth512_fp32_fall", kind="step", scene="cloth", n=512, subdiv=5, fp32=True, graphs=True,
             contact=False, steps=4),
        # a tet block on the ground under a cloth (15 local/global passes, SVD projections)
        dict(name="tets24_fp32_contact", kind="step", scene="tets", n=24, subdiv=0, fp32=True, graphs=True,
             contact=True, steps=2),
        # a falling tet block at an odd size, FP64
        dict(name="tets13_fp64_fall", kind="step", scene="tets", n=13, subdiv=0, fp32=False, graphs=True,
             contact=False, steps=2),
        # three stacked cloths on the ground, in contact with each other: many candidate records
        dict(name="layers139_fp32_contact", kind="step", scene="layers", n=139, subdiv=3, fp32=True, graphs=True,
             contact=True, steps=2),
        # a differentiable rollout of the 128^2 cloth: forward, and the gradient with respect to the
        # initial state, whole-run tape
        dict(name="grad128_fp64_fall", kind="grad", scene="cloth", n=128, subdiv=4, fp32=False, graphs=True,
             contact=False, steps=3),
        # the time of impact of device-resident positions, only enqueued (line searches, serving loops)
        dict(name="toi192", kind="toi", scene="cloth", n=192, subdiv=5, fp32=False, graphs=True, contact=True, steps=1),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step"] * 6 + ["grad", "autograd", "toi"])
    scene = rng.choice(["cloth"] * 3 + ["tets", "layers"]) if kind == "step" else "cloth"
    contact = rng.random() < 0.5 or scene == "layers" or kind == "toi"
    n = {"cloth": lambda: log_int(8, 220 if contact else 440), "tets": lambda: log_int(4, 24),
         "layers": lambda: log_int(12, 139)}[scene]()
    if kind == "grad":
        n = log_int(8, 128)
    if kind == "autograd":
        n = log_int(8, 48)
    return dict(kind=kind, scene=scene, n=n, subdiv=rng.randint(2, 5) if scene == "cloth" else 3 if scene == "layers" else 0,
                fp32=kind == "step" and rng.random() < 0.6, graphs=rng.random() < 0.7, contact=contact,
                steps=rng.randint(1, 3))


# ---------------------------------------------------------------- inputs

def _make_scene(case, seed):
    """The scene, its start velocity and the generator for what follows."""
    rng = np.random.default_rng(seed)
    n, contact = case["n"], case["contact"]
    if case["scene"] == "cloth":
        dim = n if n > 64 else min(n, 64)
        sc = scenes.cloth_over_sphere(n, case["subdiv"], ground=True, seed=seed % 100003, patch_dim=dim,
                                      sphere_patch_dim=max(8, 4 << case["subdiv"]))
        if n > 256:  # keep the 256^2 cloth's spacing: an edge below dHat would put barrier pairs inside the sheet
            sc["cloths"][0]["v"] = scenes.cloth_grid(n, side=0.5 * n / 256, height=0.2, seed=seed % 100003)[0]
        # contact: the lowest point of the cloth 1.5 mm above the top of the sphere
        top = float(sc["statics"][0]["v"][:, 1].max())
        v = sc["cloths"][0]["v"]
        v[:, 1] += (top + 1.5e-3 if contact else top + 0.1) - float(v[:, 1].min())
        if case["kind"] == "autograd":
            sc["cloths"][0]["tri_k"] = np.exp(rng.uniform(math.log(1e3), math.log(1e5), len(sc["cloths"][0]["f"])))
    elif case["scene"] == "tets":
        # cell size, cloth spacing and gaps of the 40^3-cell benchmark block (0.4 m) under its 128^2 cloth
        m = max(6, (16 * n) // 5)
        sc = scenes.config2(seed=seed % 100003, cells=n, cloth_n=m)
        t, c = sc["tets"][0], sc["cloths"][0]
        size = 0.01 * n
        tv, tt = scenes.tet_block(n, size=size, origin=(-size / 2, 0.0, -size / 2))
        tv[:, 1] += -0.2 + (1.5e-3 if contact else 0.2)
        t["v"], t["t"] = np.ascontiguousarray(tv), np.ascontiguousarray(tt)
        cv, cf = scenes.cloth_grid(m, side=1.5 * size, height=float(tv[:, 1].max()) + (4e-3 if contact else 0.1),
                                   jitter=min(2e-3, 0.2 * size / m), seed=seed % 100003)
        c["v"], c["f"] = cv, cf
    else:
        # three layers 5 mm apart at the scale run's grid spacing, the lowest just above the sphere
        sc = scenes.config4(seed=seed % 100003, n=n, side=2.0 * n / 1024)
        sv, sf = scenes.icosphere(case["subdiv"], radius=0.15, noise=0.015, seed=seed % 100003)
        sc["statics"][0] = dict(v=sv, f=sf, patch_dim=32)
        low = float(sc["cloths"][0]["v"][:, 1].min())
        for c in sc["cloths"]:
            c["v"][:, 1] += float(sv[:, 1].max()) + 1.5e-3 - low
    parts = [c["v"] for c in sc["cloths"]] + [t["v"] for t in sc["tets"]]
    vel = []
    for k, p in enumerate(parts):
        # a drift downwards (faster when landing; the upper layers faster still), a slow
        # tumble and a smooth wave, as a moving cloth or block has
        down = rng.uniform(0.6, 1.0) * (1.0 + 0.3 * k if contact else 0.5)
        spin = rng.normal(0.0, 0.3, 3)
        a = np.cross(spin[None, :], p - p.mean(0))
        ph, q = rng.uniform(0, 6.28, 3), rng.uniform(5, 15, (3, 3))
        a += 0.02 * np.sin(p @ q.T + ph)
        a[:, 1] -= down
        vel.append(a)
    return sc, np.concatenate(parts), np.concatenate(vel), rng


def prepare(case, seed):
    sc, x0, v0, rng = _make_scene(case, seed)
    sim = pdipc.Simulator.from_scene(sc, precision=pdipc.FP32_SPLIT if case["fp32"] else pdipc.FP64,
                                     use_graphs=1 if case["graphs"] else 0, skip_static_pairs=1)
    st = dict(kind=case["kind"], sim=sim, steps=case["steps"], x0=x0, v0=v0)
    if case["kind"] in ("grad", "autograd"):
        st["gx"] = rng.normal(0.0, 1.0, x0.shape)
        if case["kind"] == "autograd":
            st["k"] = torch.from_numpy(sc["cloths"][0]["tri_k"]).requires_grad_(True)
            st["v"] = torch.from_numpy(v0).requires_grad_(True)
    if case["kind"] == "toi":
        # the records of a broad phase over one step's motion, then positions inside that motion
        full = sim.x()
        dx = np.zeros_like(full)
        dx[: sim.sim] = 0.01 * v0 + rng.normal(0.0, 1e-4, v0.shape)
        sim.debug_broad_phase(full, dx)
        st["a"] = torch.from_numpy(full.reshape(-1)).cuda()
        st["b"] = torch.from_numpy((full + dx).reshape(-1)).cuda()
        st["toi"] = torch.zeros(1, dtype=torch.float64, device="cuda")
    return st


def run(st):
    sim = st["sim"]
    if st["kind"] == "toi":
        sim.toi_noalloc(st["a"].data_ptr(), st["b"].data_ptr(), st["toi"].data_ptr(),
                        torch.cuda.current_stream().cuda_stream)
        return st["toi"]
    if st["kind"] == "autograd":
        st["k"].grad = st["v"].grad = None
        x = PdIpcRollout.apply(st["k"], st["v"], sim, st["x0"], st["steps"], 0)
        x.backward(torch.from_numpy(st["gx"]))
        return dict(x=x.detach(), dv0=st["v"].grad, dk=st["k"].grad)
    sim.set_x(st["x0"])
    sim.set_v(st["v0"])
    if st["kind"] == "grad":
        sim.rollout(st["steps"], 0)
        x = sim.x()
        dx0, dv0, _ = sim.backward(dx=st["gx"])
        return dict(x=x, dx0=dx0, dv0=dv0)
    sim.run(st["steps"])
    return dict(x=sim.x(), v=sim.v())


# ---------------------------------------------------------------- work

def _counts(case):
    """(simulated points, off-diagonal system entries, static points)."""
    n = case["n"]
    if case["scene"] == "tets":
        m = max(6, (16 * n) // 5)
        return (n + 1) ** 3 + m * m, 15 * (n + 1) ** 3 + 18 * m * m, 4
    k = 3 if case["scene"] == "layers" else 1
    return k * n * n, 18 * k * n * n, 10 * 4 ** case["subdiv"] + 6


def work(case):
    """State in and out, and the system's entries (an 8-byte value, a 4-byte
    column) and the points' ring or element data (about 100 bytes a point), each
    once per pass; per outer iteration (two at least, one in a recorded step's
    reverse) 10 or 15 local/global passes of 15 sweeps, a sweep being two
    applications of the system to three coordinates, and about 300 operations a
    point for the local step.  A time of impact: two positions a point, and
    about 12 records a point of some 300 operations."""
    p, nnz, ns = _counts(case)
    if case["kind"] == "toi":
        return dict(bytes=48.0 * (p + ns) + 8, flops=300.0 * 12 * p)
    lg = 15 if case["scene"] == "tets" else 10
    per_outer = lg * (15 * 2 * 6 * nnz + 300 * p)
    k = 3 if case["kind"] != "step" else 1  # forward and reverse
    io = 8.0 * 3 * (2 * p + 2 * p + ns)
    return dict(bytes=io + 12.0 * nnz + 100.0 * p, flops=float(k * case["steps"] * 2 * per_outer))


# ---------------------------------------------------------------- the step where nothing touches, in 64 bits

class _Sym(torch.autograd.Function):
    """R x for a constant symmetric sparse R."""

    @staticmethod
    def forward(ctx, R, x):
        ctx.R = R
        return R @ x

    @staticmethod
    def backward(ctx, g):
        return None, ctx.R @ g


def _system(sc, dev):
    """The elastic system of the cloths and tets from first principles: springs,
    cotangent bending L^T diag(bend area) L, tet strain G^T G; returns its
    parts as torch tensors."""
    rows, cols, vals, masses = [], [], [], []
    cloths, tets = [], []
    base = 0

    def add(r, c, v):
        rows.append(r)
        cols.append(c)
        vals.append(v)

    for c in sc["cloths"]:
        v, f = c["v"], c["f"].astype(np.int64)
        nv = len(v)
        ar = 0.5 * np.linalg.norm(np.cross(v[f[:, 1]] - v[f[:, 0]], v[f[:, 2]] - v[f[:, 0]]), axis=1)
        area = np.zeros(nv)
        for k in range(3):
            np.add.at(area, f[:, k], ar / 3)
        i = np.concatenate([f[:, 0], f[:, 1], f[:, 2]])
        j = np.concatenate([f[:, 1], f[:, 2], f[:, 0]])
        o = np.concatenate([f[:, 2], f[:, 0], f[:, 1]])
        e1, e2 = v[i] - v[o], v[j] - v[o]
        cot = -0.5 * (e1 * e2).sum(1) / np.linalg.norm(np.cross(e1, e2), axis=1)
        key, inv = np.unique(np.minimum(i, j) * nv + np.maximum(i, j), return_inverse=True)
        a, b = key // nv, key % nv
        cw = np.bincount(inv, weights=cot, minlength=len(key))
        tri = np.concatenate([np.arange(len(f))] * 3)
        if c.get("tri_k") is not None:
            k0 = np.bincount(inv, weights=c["tri_k"][tri], minlength=len(key)) / np.bincount(inv, minlength=len(key))
        else:
            k0 = np.full(len(key), c["s0"])
        rest = np.linalg.norm(v[a] - v[b], axis=1)
        # L row i: cot / area_i to each neighbour, minus the sum on the diagonal
        li = np.concatenate([a, b])
        lj = np.concatenate([b, a])
        lv = np.concatenate([cw, cw]) / area[li]
        diag = -np.bincount(li, weights=lv, minlength=nv)
        t64 = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=dev)  # noqa: E731
        Li = np.concatenate([li, np.arange(nv)])
        Lj = np.concatenate([lj, np.arange(nv)])
        Lv = np.concatenate([lv, diag])
        L = torch.sparse_coo_tensor(t64(np.stack([Li, Lj])), t64(Lv), (nv, nv)).coalesce()
        h0 = torch.linalg.norm(L.to_sparse_csr() @ t64(v), dim=1)
        ba = t64(area * c["s1"])
        W = torch.sparse_coo_tensor(t64(np.stack([np.arange(nv)] * 2)), ba, (nv, nv))
        Lt = L.t().coalesce()
        B = torch.sparse.mm(Lt, torch.sparse.mm(W, L)).coalesce()
        add(base + B.indices()[0], base + B.indices()[1], B.values())
        cloths.append(dict(base=base, nv=nv, a=t64(a), b=t64(b), k=t64(k0), rest=t64(rest), L=L.to_sparse_csr(),
                           Lt=Lt.to_sparse_csr(), h0=h0, ba=ba, tri=t64(tri), inv=t64(inv),
                           deg=t64(np.bincount(inv, minlength=len(key)).astype(float)), nf=len(f)))
        masses.append(t64(area * c["density"]))
        base += nv
    for t in sc["tets"]:
        v, e = t["v"], t["t"].astype(np.int64)
        nv = len(v)
        t64 = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=dev)  # noqa: E731
        Dm = np.stack([v[e[:, k]] - v[e[:, 0]] for k in (1, 2, 3)], 2)
        vol = np.abs(np.linalg.det(Dm)) / 6
        Di = np.linalg.inv(Dm)
        H = np.concatenate([-Di.sum(1, keepdims=True), Di], 1)  # F = sum_c x_c H_c (row c of H)
        w = t["s0"] * vol
        K = np.einsum("tck,tdk->tcd", H, H) * w[:, None, None]
        add(base + t64(np.repeat(e, 4, 1).reshape(-1)), base + t64(np.tile(e, (1, 4)).reshape(-1)), t64(K.reshape(-1)))
        m = np.zeros(nv)
        for k in range(4):
            np.add.at(m, e[:, k], vol)
        tets.append(dict(base=base, e=base + t64(e), H=t64(H), w=t64(w)))
        masses.append(t64(m * t["density"]))
        base += nv
    mass = torch.cat(masses)
    return cloths, tets, rows, cols, vals, mass, base


def _split(n, rows, cols, vals, dev):
    """The summed entries as (diagonal, -offdiagonal in CSR)."""
    A = torch.sparse_coo_tensor(torch.stack([torch.cat(rows), torch.cat(cols)]), torch.cat(vals), (n, n)).coalesce()
    i, j, v = A.indices()[0], A.indices()[1], A.values()
    d = torch.zeros(n, dtype=torch.float64, device=dev).index_add(0, i[i == j], v[i == j])
    return d, i[i != j], j[i != j], -v[i != j]


def _free_step(p, cloths, tets, elastic, apply_r, mass, x, v):
    """One step of the method where the time of impact is 1 and no barrier
    record is active: prediction, then outer iterations of lg_iters local/global
    passes until the last one moves less than the tolerance."""
    dt, w = p["dt"], p["omega"]
    g = torch.zeros_like(x)
    g[:, 1] = p["gravity"]
    x0 = x
    s = x + dt * (v + dt * g)
    D = (elastic + mass / dt ** 2)[:, None]
    rhs0 = (mass / dt ** 2)[:, None] * s
    xold, x = x, s
    for outer in range(p["max_outer"]):
        for _ in range(p["lg_iters"]):
            b = rhs0
            for t in tets:
                F = torch.einsum("tci,tck->tik", x[t["e"]], t["H"])
                U, S, Vh = torch.linalg.svd(F)
                P = U @ torch.diag_embed(S.clamp(p["sigma_lo"], p["sigma_hi"])) @ Vh
                out = torch.einsum("tik,tck->tci", P, t["H"]) * t["w"][:, None, None]
                b = b.index_add(0, t["e"].reshape(-1), out.reshape(-1, 3))
            for c in cloths:
                xc = x[c["base"]: c["base"] + c["nv"]]
                d = xc[c["a"]] - xc[c["b"]]
                f = (c["k"] * c["rest"] / torch.linalg.norm(d, dim=1))[:, None] * d
                a = c["lap"](xc)
                nrm = torch.linalg.norm(a, dim=1, keepdim=True)
                a = torch.where(nrm >= 1e-10, a * (c["h0"][:, None] / nrm.clamp_min(1e-300)), a)
                y = c["lapT"](c["ba"][:, None] * a).index_add(0, c["a"], f).index_add(0, c["b"], -f)
                b = torch.cat([b[: c["base"]], b[c["base"]: c["base"] + c["nv"]] + y, b[c["base"] + c["nv"]:]])

            def M(y):
                return (1 - w) * y + w * apply_r(y) / D

            u = b / D
            cc = w * w * apply_r(u) / D + (2 - w) * w * u
            r = p["rho"] ** 2
            W = 2 / (2 - r)
            pre, cur = x, M(M(x)) + cc
            for _ in range(1, p["cheb_iters"]):
                pre, cur = cur, W * (M(M(cur)) + cc - pre) + pre
                W = 4 / (4 - r * W)
            x = cur
        if outer > 0 and float(((x - xold) ** 2).sum()) < p["residual_tol"]:
            break
        xold = x
    return x, (x - x0) * ((1 - dt) / dt)


def exact(case, seed):
    if case["contact"] or case["kind"] == "toi":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    sc, x0, v0, rng = _make_scene(case, seed)
    p = sc["params"]
    cloths, tets, rows, cols, vals, mass, n = _system(sc, dev)
    x = torch.as_tensor(x0, device=dev)
    v = torch.as_tensor(v0, device=dev)
    k = None
    if case["kind"] != "step":
        gx = torch.as_tensor(rng.normal(0.0, 1.0, x0.shape), device=dev)
        x.requires_grad_(True)
        v.requires_grad_(True)
    if case["kind"] == "autograd":
        k = torch.as_tensor(sc["cloths"][0]["tri_k"], device=dev).requires_grad_(True)
        c = cloths[0]
        c["k"] = torch.zeros_like(c["rest"]).index_add(0, c["inv"], k[c["tri"]]) / c["deg"]
    for c in cloths:
        lin = lambda A, At: (lambda y: _Lin.apply(A, At, y))  # noqa: E731
        c["lap"], c["lapT"] = lin(c["L"], c["Lt"]), lin(c["Lt"], c["L"])
        a, b = c["base"] + c["a"], c["base"] + c["b"]
        rows += [a, b, a, b]
        cols += [a, b, b, a]
        vals += [c["k"], c["k"], -c["k"], -c["k"]]
    if k is None:
        elastic, i, j, off = _split(n, rows, cols, vals, dev)
        R = torch.sparse_coo_tensor(torch.stack([i, j]), off, (n, n)).coalesce().to_sparse_csr()
        apply_r = lambda y: _Sym.apply(R, y)  # noqa: E731
    else:  # the entries carry the stiffness gradient
        i, j, val = torch.cat(rows), torch.cat(cols), torch.cat(vals)
        elastic = torch.zeros(n, dtype=torch.float64, device=dev).index_add(0, i[i == j], val[i == j])
        i, j, val = i[i != j], j[i != j], -val[i != j]
        apply_r = lambda y: torch.zeros_like(y).index_add(0, i, val[:, None] * y[j])  # noqa: E731
    y, u = x, v
    for _ in range(case["steps"]):
        y, u = _free_step(p, cloths, tets, elastic, apply_r, mass, y, u)
    if case["kind"] == "step":
        out = np.concatenate([y.cpu().numpy()] + [s["v"] for s in sc["statics"]])
        return dict(x=out, v=u.cpu().numpy())
    y.backward(gx)
    if case["kind"] == "autograd":
        return dict(x=y.detach(), dv0=v.grad, dk=k.grad)
    out = np.concatenate([y.detach().cpu().numpy()] + [s["v"] for s in sc["statics"]])
    return dict(x=out, dx0=x.grad, dv0=v.grad)


class _Lin(torch.autograd.Function):
    """A x for a constant sparse A whose transpose is at hand."""

    @staticmethod
    def forward(ctx, A, At, x):
        ctx.At, ctx.A = At, A
        return A @ x

    @staticmethod
    def backward(ctx, g):
        return None, None, ctx.At @ g
