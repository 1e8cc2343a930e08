"""Timing cases of the elastodynamics solver and of its surrogate network, each
through the entry points that a program calls.

Kinds of case (case["kind"]):

  step      one drop-in time step on host vectors (Context.time_step_matrix_free)
  loop      device-resident time loop (Context.step_n), state copied out at its end
  record    one solve from rest with a point source, receivers recorded
            (start_from_rest, step_n_record, traces) on a built operator
  run       the whole path of the driver: operator build, right-hand sides,
            projections, loop, error norms (make_matrices_free, run)
  ensemble  replay of a batched ensemble and its traces (Ensemble.run)
  train     Adam steps of a surrogate network (Mlp.train), then its parameters
  gradients one forward and backward on a host batch (Mlp.gradients)
  predict   forward of host inputs (Mlp.predict)

listed() gives the fixed cases, draw() one more of the same ranges; prepare()
makes what a program holds before the call, run() is one pass, work() the bytes
and operations of a pass, exact() its outputs from plain 64-bit numpy / torch.
"""
import copy
import functools
import math

import numpy as np
import torch

import lymph3d_apsc_amd as L
from lymph3d_apsc_amd import _lib, ensemble as E, mesh as M, mlp

DECKS = "tests/golden/decks"
SOME_NEUMANN = ("x0", "x1", "y0", "y1", "z0")  # Dirichlet there, traction-free z = 1


# ---- the cases -----------------------------------------------------------

def listed():
    return [
        # the drop-in TIME_STEP call of a host program on the smallest
        # agglomerated cube (125 polyhedra): latency of copies and launches
        dict(name="step_cube5_p2", kind="step", mesh="cube", n=5, p=2, bits=64, pairs=False),
        # 1000 steps of the same mesh, the CPU-runnable convergence set-up
        dict(name="loop_cube5_p2", kind="loop", mesh="cube", n=5, p=2, bits=64, pairs=False, steps=1000,
             tune=False),
        # the headline step: 64,000 polyhedra, 3.84 M unknowns, FP64
        dict(name="loop_cube40_p3_fp64", kind="loop", mesh="cube", n=40, p=3, bits=64, pairs=False, steps=60,
             tune=True),
        # its fastest form: 32-bit apply, every face pair stored once
        dict(name="loop_cube40_p3_fp32_pairs", kind="loop", mesh="cube", n=40, p=3, bits=32, pairs=True,
             steps=100, tune=False),
        # one block row per tet (the reference's own stepping), odd size, 48-bit apply
        dict(name="loop_tets17_p2_fp48", kind="loop", mesh="tets", n=17, p=2, bits=48, pairs=False, steps=200,
             tune=False),
        # uneven polyhedra of 4-40 tets, smooth lognormal material, Ricker
        # source and 64 receivers, the highest degree, 32-bit apply
        dict(name="record_uneven20_p4_fp32", kind="record", mesh="uneven", n=20, p=4, bits=32, steps=100, every=5,
             receivers=64),
        # the largest reference deck end to end (28,606 tets, p = 1)
        dict(name="run_deck625_p1", kind="run", mesh="deck", n=625, p=1, build="reference", steps=100),
        # set-up dominated run on an agglomerated cube, the reference's operand order
        dict(name="run_cube16_p3", kind="run", mesh="cube", n=16, p=3, build="reference", steps=20),
        # batched instances of both degrees replayed as one captured solve
        dict(name="ensemble16_fp32", kind="ensemble", instances=16, n_lo=10, n_hi=20, bits=32, steps=100, every=5,
             receivers=64),
        # the receiver network's training (the surrogate's default model)
        dict(name="train_receiver_b256", kind="train", n_in=32, width=512, hidden=5, n_out=64, batch=256, steps=256,
             samples=65536),
        # the network that gives all 64 receivers' traces at once
        dict(name="train_traces_b256", kind="train", n_in=8, width=512, hidden=3, n_out=38400, batch=256, steps=40,
             samples=1024),
        # evaluation of 256 parameter sets x 64 receivers, batches as trained
        dict(name="predict_receiver_16384", kind="predict", n_in=32, width=512, hidden=5, n_out=64, batch=256,
             rows=16384),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "loop", "loop", "loop", "record", "run", "run", "ensemble", "train", "train",
                       "gradients", "predict", "predict"])
    if kind in ("step", "loop", "run"):
        p = rng.choice([1, 2, 3, 4])
        mesh = rng.choice(["cube", "cube", "tets", "uneven"] + (["deck"] if kind == "run" else []))
        top = {"cube": {1: 40, 2: 40, 3: 32, 4: 20}, "tets": {1: 20, 2: 17, 3: 13, 4: 8},
               "uneven": {1: 24, 2: 24, 3: 20, 4: 16}, "deck": {1: 0, 2: 0, 3: 0, 4: 0}}[mesh][p]
        if kind == "run":
            top = min(top, {1: 24, 2: 20, 3: 14, 4: 8}[p] if mesh == "cube" else {1: 13, 2: 11, 3: 8, 4: 5}[p])
        n = _log_int(rng, 3, top) if top else rng.choice([25, 100, 125, 625])
        if mesh == "deck":
            p = rng.choice([1, 2])
        case = dict(kind=kind, mesh=mesh, n=n, p=p)
        if kind == "run":
            return dict(case, build=rng.choice(["reference", "factored"]), steps=rng.randint(5, 100))
        bits = rng.choice([64, 64, 32, 48])
        case.update(bits=bits, pairs=mesh != "uneven" and p <= 3 and rng.random() < 0.3)
        if kind == "loop":
            case.update(steps=_log_int(rng, 20, 100 if n * p > 40 else 1000), tune=False)
        return case
    if kind == "record":
        p = rng.choice([1, 2, 3, 4])
        return dict(kind=kind, mesh=rng.choice(["cube", "uneven"]), n=_log_int(rng, 4, 20 if p < 4 else 16), p=p,
                    bits=rng.choice([64, 32, 48]), steps=rng.randint(20, 200), every=rng.choice([1, 2, 5]),
                    receivers=_log_int(rng, 1, 64))
    if kind == "ensemble":
        lo = rng.randint(4, 12)
        return dict(kind=kind, instances=_log_int(rng, 2, 12), n_lo=lo, n_hi=lo + rng.randint(0, 6),
                    bits=rng.choice([64, 32, 48]), steps=rng.randint(20, 100), every=rng.choice([1, 5]),
                    receivers=_log_int(rng, 4, 64))
    net = dict(kind=kind, n_in=rng.choice([8, 16, 32, 40]), width=8 * _log_int(rng, 8, 64),
               hidden=rng.randint(1, 6), n_out=8 * _log_int(rng, 1, 1000), batch=8 * _log_int(rng, 1, 32))
    if kind == "train":
        net.update(steps=_log_int(rng, 4, 64), samples=_log_int(rng, 256, 4096))
    elif kind == "predict":
        net.update(rows=_log_int(rng, 1, 16384 if net["n_out"] <= 512 else 2048))
    return net


# ---- inputs --------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _shape(mesh, n):
    """Geometry of a case's mesh (the same for every seed)."""
    if mesh == "deck":
        return M.read_deck("%s/tet_%d" % (DECKS, n))
    if mesh == "uneven":
        return M.cube_mesh(n, dirichlet_faces=set(SOME_NEUMANN), poly_size=(4, 40), seed=3)
    return M.cube_mesh(n, agglomerate=mesh == "cube")


def _barycentres(m):
    return m.xyz[m.tet_vert].mean(axis=1)


def _mesh(case, seed):
    m = copy.copy(_shape(case["mesh"], case["n"]))
    if case["mesh"] == "uneven":  # smooth lognormal lambda and mu, uniform rho
        rng = np.random.default_rng(seed)
        bc = _barycentres(m)
        m.lam, m.mu = E.lognormal_field(rng, bc), E.lognormal_field(rng, bc)
        m.rho = rng.uniform(0.8, 1.2, m.n_tet)
    return m


def _dt(case, m):
    """0.2 h / (c_P p^2), h the cube's side (a quarter of it where every tet is
    an element of its own; decks bring their own step)."""
    if case["mesh"] == "deck":
        return m.dt if case["p"] == m.degree else 0.25 * m.dt
    speed = math.sqrt(float(((m.lam + 2 * m.mu) / m.rho).max()))
    return (0.05 if case["mesh"] == "tets" else 0.2) / case["n"] / (speed * case["p"] ** 2)


def _amplitudes(seed):
    """Seeded amplitudes of the initial displacement (two fields) and velocity."""
    return np.random.default_rng(seed + 77).uniform(0.5, 1.5, 3)


def _u0(x, a):
    """Initial displacement: standing wave and manufactured field, as the
    built-in fields LYMPH_FN_CUBE_U and LYMPH_FN_REF_UEX."""
    s, c = np.sin(np.pi * x), np.cos(np.pi * x)
    cube = np.repeat((s[..., 0] * s[..., 1] * s[..., 2])[..., None], 3, axis=-1)
    return a[0] * cube + a[1] * _uex(s, c)


def _uex(s, c):
    return np.stack([c[..., 0] * s[..., 1] * s[..., 2], s[..., 0] * c[..., 1] * s[..., 2],
                     s[..., 0] * s[..., 1] * c[..., 2]], axis=-1)


def _net_data(case, seed, rows):
    """Standardised inputs and smooth, correlated outputs, as traces have."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, case["n_in"]), dtype=np.float32)
    modes = rng.standard_normal((16, case["n_out"]), dtype=np.float32) / 4
    mix = rng.standard_normal((case["n_in"], 16), dtype=np.float32) / np.float32(math.sqrt(case["n_in"]))
    return x, np.sin(x @ mix) @ modes


def _widths(case):
    return [case["n_in"]] + [case["width"]] * case["hidden"] + [case["n_out"]]


def _order(case, seed):
    rng = np.random.default_rng(seed + 5)
    need = case["steps"] * case["batch"]
    parts = [rng.permutation(case["samples"]) for _ in range(-(-need // case["samples"]))]
    return np.concatenate(parts)[:need].astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "gradients", "predict"):
        net = mlp.Mlp(_widths(case), max_batch=case["batch"], seed=seed)
        s = dict(case=case, net=net)
        if kind == "train":
            net.set_data(*_net_data(case, seed, case["samples"]))
            s["order"] = _order(case, seed)
        else:
            s["x"], s["y"] = _net_data(case, seed, case.get("rows", case["batch"]))
        return s
    if kind == "ensemble":
        inst = [E.make_instance(1000 * (seed % 100000) + k, n_range=(case["n_lo"], case["n_hi"]),
                                n_receivers=case["receivers"]) for k in range(case["instances"])]
        dt = min(0.2 / i["n"] / (math.sqrt(float(((i["mesh"].lam + 2 * i["mesh"].mu) / i["mesh"].rho).max()))
                                 * i["p"] ** 2) for i in inst)
        return dict(case=case, ens=E.Ensemble(inst, dt, case["steps"], every=case["every"],
                                              apply_bits=case["bits"], autotune=False))
    m = _mesh(case, seed)
    ctx = L.Context(m, case["p"])
    s = dict(case=case, ctx=ctx, dt=_dt(case, m))
    if kind == "run":
        ctx.set_build(case["build"])
        s["dt"] *= 1 - 0.001 * _amplitudes(seed)[0]  # another seed, another time step
        return s
    ctx.set_keep_adg(False)
    ctx.set_build("factored")
    ctx.make_matrices_free()
    if case.get("pairs"):
        ctx.set_symmetric_storage(True, fp32=case["p"] == 3 and case["bits"] != 64)
    if case["bits"] != 64:
        ctx.set_apply_precision(case["bits"])
    if kind == "record":
        rng = np.random.default_rng(seed + 9)
        s.update(source=rng.uniform(0.3, 0.7, (1, 3)), force=np.array([[0.0, 0.0, 1.0]]),
                 receivers=rng.uniform(0.05, 0.95, (case["receivers"], 3)), f0=float(rng.uniform(4.0, 8.0)))
        return s
    a = _amplitudes(seed)
    ctx.make_rhs_free(_lib.PROB_NULL, _lib.SLOT_RHS_STAT)
    ctx.make_rhs_free(_lib.PROB_CUBE_WAVE, _lib.SLOT_RHS_DYN)
    u0 = a[0] * ctx.compute_modal_coefficients_free(_lib.FN_CUBE_U) \
        + a[1] * ctx.compute_modal_coefficients_free(_lib.FN_REF_UEX)
    v0 = a[2] * ctx.compute_modal_coefficients_free(_lib.FN_REF_VEL)
    u1 = u0 + s["dt"] * v0
    if kind == "step":
        s.update(u0=u0, u1=u1, g=_lib.time_function(_lib.PROB_CUBE_WAVE, s["dt"]))
        return s
    if case["tune"]:
        ctx.autotune(reps=20)
    ctx.set_slot(_lib.SLOT_U_PREV, u0)
    ctx.set_slot(_lib.SLOT_U_CUR, u1)
    s["t"] = s["dt"]
    return s


# ---- one pass --------------------------------------------------------------

def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "step":
        return state["ctx"].time_step_matrix_free(state["g"], state["dt"], state["u0"], state["u1"])
    if kind == "loop":
        ctx = state["ctx"]
        state["t"] = ctx.step_n(_lib.PROB_CUBE_WAVE, case["steps"], state["t"], state["dt"])
        return dict(prev=ctx.get_slot(_lib.SLOT_U_PREV), cur=ctx.get_slot(_lib.SLOT_U_CUR), t=state["t"])
    if kind == "record":
        ctx = state["ctx"]
        ctx.set_receivers(state["receivers"], max_records=case["steps"] // case["every"])
        t = ctx.start_from_rest(state["dt"], state["source"], state["force"], f0=state["f0"])
        ctx.step_n_record(_lib.PROB_RICKER, case["steps"], t, state["dt"], every=case["every"])
        return dict(traces=ctx.traces(), cur=ctx.get_slot(_lib.SLOT_U_CUR))
    if kind == "run":
        ctx = state["ctx"]
        ctx.make_matrices_free()
        problem = _lib.PROB_REF_MMS if case["mesh"] in ("deck", "uneven") else _lib.PROB_CUBE_WAVE
        r = ctx.run(problem, state["dt"], 1e9, case["steps"], want_u=True)
        return dict(u=r["u"], err_l2=float(r["err_l2"]), err_dg=float(r["err_dg"]))
    if kind == "ensemble":
        return state["ens"].run()
    net = state["net"]
    if kind == "train":
        losses = net.train(state["order"], case["batch"], 1e-3)
        return dict(losses=losses, params=net.params())
    if kind == "gradients":
        loss, g = net.gradients(state["x"], state["y"])
        return dict(loss=np.float32(loss), grads=g)
    return net.predict(state["x"])


# ---- what a pass cannot do without -------------------------------------------

@functools.lru_cache(maxsize=None)
def _sizes(mesh, n):
    """(tets, polyhedra, blocks, faces with a neighbour of another polyhedron)."""
    m = _shape(mesh, n)
    t, f = np.nonzero(m.neigh >= 0)
    a, b = m.tet_poly[t].astype(np.int64), m.tet_poly[m.neigh[t, f]].astype(np.int64)
    other = a != b
    pairs = np.unique(a[other] * m.n_poly + b[other]).size
    return m.n_tet, m.n_poly, m.n_poly + pairs, int(other.sum())


def _np(p):
    return (p + 1) * (p + 2) * (p + 3) // 6


def _step_work(n_poly, n_blk, p, bits, pairs=False):
    """Bytes and operations of one leapfrog step: each stored operator entry,
    the mass factors (64-bit apply) and five vectors once."""
    n3, Np = 3 * _np(p), _np(p)
    entries = n_blk * n3 * n3
    stored = entries
    if pairs and (bits == 64 or p == 3):
        stored = (n_blk - n_poly) // 2 * n3 * n3 + n_poly * n3 * (n3 + 1) // 2
    by = stored * bits // 8 + 5 * 8 * n_poly * n3 + (8 * n_poly * Np * (Np + 1) // 2 if bits == 64 else 0)
    return by, 2 * entries + 6 * n_poly * n3


def work(case):
    kind = case["kind"]
    if kind in ("train", "gradients", "predict"):
        w = _widths(case)
        params = sum(k * n + n for k, n in zip(w[:-1], w[1:]))
        gemm = 2 * sum(k * n for k, n in zip(w[:-1], w[1:]))
        B = case["batch"]
        if kind == "predict":
            return {"bytes": 4 * case["rows"] * (w[0] + w[-1]) + 2 * params, "flops": gemm * case["rows"]}
        back = 3 * gemm - 2 * w[0] * w[1]
        once = 4 * B * (w[0] + w[-1])
        if kind == "gradients":
            return {"bytes": once + 2 * params + 4 * params, "flops": back * B}
        # Adam reads and writes the parameters and both moments, once a step
        return {"bytes": case["steps"] * (once + 24 * params) + 4 * params, "flops": case["steps"] * back * B}
    if kind == "ensemble":
        by = fl = 0
        n = (case["n_lo"] + case["n_hi"]) // 2
        for p in (2, 3):  # half of the instances each
            b, f = _step_work(n ** 3, 7 * n ** 3 - 6 * n * n, p, case["bits"])
            by += case["instances"] / 2 * case["steps"] * b
            fl += case["instances"] / 2 * case["steps"] * f
        return {"bytes": by, "flops": fl}
    nt, n_poly, n_blk, faces = _sizes(case["mesh"], case["n"])
    p = case["p"]
    n3, Np = 3 * _np(p), _np(p)
    by, fl = _step_work(n_poly, n_blk, p, case.get("bits", 64), case.get("pairs", False))
    vec = 8 * n_poly * n3
    if kind == "step":
        return {"bytes": by + 3 * vec, "flops": fl}
    if kind in ("loop", "record"):
        return {"bytes": case["steps"] * by + 2 * vec, "flops": case["steps"] * fl}
    # run: both operators written, quadrature sums per basis pair (10 per
    # volume point, 14 per interior face point), then the loop
    build = 2 * Np * Np * (10 * nt * (p + 1) ** 3 + 14 * faces * (p + 1) ** 2)
    return {"bytes": case["steps"] * by + 16 * n_blk * n3 * n3 + 6 * vec, "flops": case["steps"] * fl + build}


# ---- 64-bit values from plain numpy / torch ------------------------------------

def _rules(p):
    x, w = np.polynomial.legendre.leggauss(p + 1)
    a, b, c = (v.ravel() for v in np.meshgrid(0.5 * x + 0.5, 0.5 * x + 0.5, 0.5 * x + 0.5, indexing="ij"))
    w3 = 0.125 * (w[:, None, None] * w[None, :, None] * w[None, None, :]).ravel()
    tet = np.stack([a, (1 - a) * b, (1 - a) * (1 - b) * c], axis=1)
    s, t = (v.ravel() for v in np.meshgrid(x, x, indexing="ij"))
    tri = np.stack([0.5 * (1 + s), 0.25 * (1 - s) * (1 + t)], axis=1)
    return tet, (1 - a) ** 2 * (1 - b) * w3, tri, 0.125 * (1 - s) * (w[:, None] * w[None, :]).ravel()


def _basis(x, bb, p):
    """phi (..., q, Np) and its gradient (..., 3, q, Np) at points x (..., q, 3)
    for bounding boxes bb (..., 6): products of Legendre polynomials of total
    degree <= p, q1 from p down, then q2, q3."""
    h, mid = (bb[..., 1::2] - bb[..., 0::2]) / 2, (bb[..., 1::2] + bb[..., 0::2]) / 2
    xi = (x - mid[..., None, :]) / h[..., None, :]
    one = np.ones_like(xi)
    Lg = [one, xi, (3 * xi ** 2 - 1) / 2, (5 * xi ** 3 - 3 * xi) / 2, (35 * xi ** 4 - 30 * xi ** 2 + 3) / 8]
    dL = [0 * one, one, 3 * xi, (15 * xi ** 2 - 3) / 2, (35 * xi ** 3 - 15 * xi) / 2]
    sq = np.sqrt(h)[..., None, :]
    V = [v / sq for v in Lg[:p + 1]]
    G = [g / (sq * h[..., None, :]) for g in dL[:p + 1]]
    idx = [(i, j, k) for i in range(p, -1, -1) for j in range(p - i, -1, -1) for k in range(p - i - j, -1, -1)]
    phi = np.stack([V[i][..., 0] * V[j][..., 1] * V[k][..., 2] for i, j, k in idx], axis=-1)
    d = [np.stack([G[i][..., 0] * V[j][..., 1] * V[k][..., 2] for i, j, k in idx], axis=-1),
         np.stack([V[i][..., 0] * G[j][..., 1] * V[k][..., 2] for i, j, k in idx], axis=-1),
         np.stack([V[i][..., 0] * V[j][..., 1] * G[k][..., 2] for i, j, k in idx], axis=-1)]
    return phi, np.stack(d, axis=-3)


# barycentric corners of a tet's four faces that the triangle rule's (s, t) run along
_FACE = ((0, 2, 1), (0, 1, 3), (3, 1, 2), (0, 3, 2))


class _Plain:
    """The discrete problem assembled with numpy: interior-penalty blocks K (and
    the DG norm's A), mass blocks, right-hand sides, projections."""

    def __init__(self, m, p, alpha=10.0, theta=-1.0):
        self.m, self.p, self.Np, self.n3 = m, p, _np(p), 3 * _np(p)
        tet, self.w3, tri, self.w2 = _rules(p)
        v = m.xyz[m.tet_vert]
        J = np.stack([v[:, k] - v[:, 0] for k in (1, 2, 3)], axis=2)
        self.aJ = np.abs(np.linalg.det(J))
        self.vx = v[:, None, 0] + np.einsum("qk,tdk->tqd", tet, J)
        self.bb = m.bbox[m.tet_poly]
        self.phi, dphi = _basis(self.vx, self.bb, p)
        self.fx = [v[:, None, a] + tri[:, 0, None] * (v[:, b] - v[:, a])[:, None] +
                   tri[:, 1, None] * (v[:, c] - v[:, a])[:, None] for a, b, c in _FACE]
        self.alpha, self.theta = alpha, theta
        P = m.tet_poly.astype(np.int64)
        wj = self.w3[None, :] * self.aJ[:, None]
        mass = np.einsum("tq,tqm,tqn->tmn", wj, self.phi, self.phi)
        self.Mm = np.zeros((m.n_poly, self.Np, self.Np))
        self.Mr = np.zeros_like(self.Mm)
        np.add.at(self.Mm, P, mass)
        np.add.at(self.Mr, P, mass * m.rho[:, None, None])
        D = np.einsum("tq,taqm,tbqn->tabmn", wj, dphi, dphi, optimize=True)
        rows, cols, Ks, As = [], [], [], []

        def add(r, c, k, a):
            rows.append(r)
            cols.append(c)
            Ks.append(k.transpose(0, 1, 3, 2, 4).reshape(len(r), self.n3, self.n3))
            As.append(a.transpose(0, 1, 3, 2, 4).reshape(len(r), self.n3, self.n3))

        l, u = (z[:, None, None] for z in (m.lam, m.mu))
        vol = np.zeros((m.n_tet, 3, 3, self.Np, self.Np))
        tr = D[:, 0, 0] + D[:, 1, 1] + D[:, 2, 2]
        for i in range(3):
            for j in range(3):
                vol[:, i, j] = (l + u) * D[:, i, i] + u * tr if i == j else l * D[:, i, j] + u * D[:, j, i]
        add(P, P, vol, vol)
        for f in range(4):
            nb = m.neigh[:, f]
            inner = nb >= 0
            Q = np.where(inner, P[nb], -1)
            at = np.nonzero((nb == -1) | (inner & (Q != P)))[0]
            for sel in (at[nb[at] >= 0], at[nb[at] < 0]):
                if sel.size:
                    self._face(f, sel, P[sel], Q[sel] if nb[sel[0]] >= 0 else None, add)
        key = np.concatenate([r * m.n_poly + c for r, c in zip(rows, cols)])
        uniq, inv = np.unique(key, return_inverse=True)
        self.row, self.col = uniq // m.n_poly, uniq % m.n_poly
        self.K, self.A = (self._sum(inv, v, uniq.size) for v in (Ks, As))

    def _sum(self, inv, parts, n):
        out, at = np.zeros((n, self.n3, self.n3)), 0
        for v in parts:
            np.add.at(out, inv[at:at + len(v)], v)
            at += len(v)
        return out

    def _traction(self, n, X, l, u):
        """T[i][j] = i == j: (l + 2u) n_i X_i + u sum_{a != i} n_a X_a, else l n_j X_i + u n_i X_j."""
        T = np.zeros((X.shape[0], 3, 3) + X.shape[2:])
        e = lambda z: z.reshape((-1,) + (1,) * (X.ndim - 2))  # noqa: E731
        tr = sum(e(n[:, a]) * X[:, a] for a in range(3))
        for i in range(3):
            for j in range(3):
                T[:, i, j] = (e(l + u) * e(n[:, i]) * X[:, i] + e(u) * tr) if i == j else \
                    e(l * n[:, j]) * X[:, i] + e(u * n[:, i]) * X[:, j]
        return T

    def _penalty(self, f, sel, hmin):
        m, n = self.m, self.m.normal[sel, f]
        sig = self.alpha * self.p ** 2 / hmin * (m.lam[sel] + 2 * m.mu[sel])
        C = 0.5 * n[:, :, None] * n[:, None, :]
        for i in range(3):
            C[:, i, i] = 0.5 * (n ** 2).sum(axis=1) + 0.5 * n[:, i] ** 2
        return n, (sig * m.area[sel, f])[:, None, None] * C

    def _face(self, f, sel, P, Q, add):
        m, w = self.m, self.w2
        n, C = self._penalty(f, sel, m.hk[P] if Q is None else np.minimum(m.hk[P], m.hk[Q]))
        ar, l, u = m.area[sel, f][:, None, None, None, None], m.lam[sel], m.mu[sel]
        ph, d = _basis(self.fx[f][sel], m.bbox[P], self.p)
        kk = 1.0 if Q is None else 0.5
        S = C[..., None, None] * np.einsum("q,tqm,tqn->tmn", w, ph, ph)[:, None, None]
        B = np.einsum("q,taqm,tqn->tamn", w, d, ph, optimize=True)
        T = self._traction(n, B, l, u)
        Tt = self._traction(n, B.transpose(0, 1, 3, 2), l, u).transpose(0, 2, 1, 3, 4)
        add(P, P, S + kk * ar * (self.theta * T - Tt), S)
        if Q is None:
            return
        qh, qd = _basis(self.fx[f][sel], m.bbox[Q], self.p)
        S = -C[..., None, None] * np.einsum("q,tqm,tqn->tmn", w, ph, qh)[:, None, None]
        Cp = self._traction(n, np.einsum("q,taqm,tqn->tamn", w, d, qh, optimize=True), l, u)
        # the neighbour's traction carries the indices of the test side's (as in the reference)
        Dq = self._traction(n, np.einsum("q,taqn,tqm->tamn", w, qd, ph, optimize=True), l, u)
        add(P, Q, S - 0.5 * ar * (self.theta * Cp + Dq), S)

    def load(self, values):
        """Sum over each polyhedron of w |J| values (t, q, 3) phi, (n_poly, 3, Np)."""
        b = np.einsum("q,t,tqi,tqm->tim", self.w3, self.aJ, values, self.phi, optimize=True)
        out = np.zeros((self.m.n_poly, 3, self.Np))
        np.add.at(out, self.m.tet_poly, b)
        return out

    def project(self, values):
        return np.linalg.solve(self.Mm[:, None], self.load(values)[..., None])[..., 0].reshape(-1, self.n3)

    def apply(self, blocks, x):
        y = np.matmul(blocks, x[self.col][..., None])[..., 0]
        out = np.zeros_like(x)
        np.add.at(out, self.row, y)
        return out

    def minv(self, r):
        return np.linalg.solve(self.Mr[:, None], r.reshape(-1, 3, self.Np)[..., None])[..., 0].reshape(-1, self.n3)

    def rhs(self, wave):
        """Right-hand side of the standing wave (zero Dirichlet data) or of the
        manufactured solution, with their Dirichlet and Neumann data."""
        m, pi = self.m, np.pi
        s, c = np.sin(pi * self.vx), np.cos(pi * self.vx)
        l, u, rho = (z[:, None] for z in (m.lam, m.mu, m.rho))
        if wave:
            a = (-3 * rho + 4 * u + l) * s[..., 0] * s[..., 1] * s[..., 2]
            cc = {(0, 1): c[..., 0] * c[..., 1] * s[..., 2], (0, 2): c[..., 0] * s[..., 1] * c[..., 2],
                  (1, 2): s[..., 0] * c[..., 1] * c[..., 2]}
            f = np.stack([a - (l + u) * (cc[min(i, j), max(i, j)] + cc[min(i, k), max(i, k)])
                          for i, j, k in ((0, 1, 2), (1, 0, 2), (2, 0, 1))], axis=-1)
            out = self.load(pi ** 2 * f)
        else:
            out = self.load(((-2 * rho + 3 * (l + 2 * u)) * pi ** 2)[..., None] * _uex(s, c))
        for f in range(4):
            s, c = np.sin(pi * self.fx[f]), np.cos(pi * self.fx[f])
            for kind in (-2,) if wave else (-1, -2):
                sel = np.nonzero(m.neigh[:, f] == kind)[0]
                if not wave:
                    sel = sel[np.isin(m.bc_space[sel, f], (1, 2, 3))]
                if not sel.size:
                    continue
                P = m.tet_poly[sel]
                ph, d = _basis(self.fx[f][sel], m.bbox[P], self.p)
                n, C = self._penalty(f, sel, m.hk[P])
                ar, S, Cs = m.area[sel, f], s[sel], c[sel]
                if kind == -1:
                    g = _uex(S, Cs)
                    T = self._traction(n, d, m.lam[sel], m.mu[sel])
                    b = self.theta * np.einsum("t,q,tijqm,tqj->tim", ar, self.w2, T, g, optimize=True) + \
                        np.einsum("q,tij,tqj,tqm->tim", self.w2, C, g, ph, optimize=True)
                else:
                    b = np.einsum("t,q,tqij,tj,tqm->tim", ar, self.w2,
                                  self._stress(wave, S, Cs, m.lam[sel, None], m.mu[sel, None]), n, ph, optimize=True)
                np.add.at(out, P, b)
        return out.reshape(-1, self.n3)

    @staticmethod
    def _stress(wave, s, c, l, u):
        """Stress (t, q, 3, 3) of the data set's displacement, sines s and cosines c."""
        if wave:
            g = np.pi * np.stack([c[..., 0] * s[..., 1] * s[..., 2], s[..., 0] * c[..., 1] * s[..., 2],
                                  s[..., 0] * s[..., 1] * c[..., 2]], axis=-1)
            st = u[..., None, None] * (g[..., :, None] + g[..., None, :])
            st[..., range(3), range(3)] += (l * g.sum(axis=-1))[..., None]
            return st
        st = np.zeros(s.shape + (3,))
        for i in range(3):
            st[..., i, i] = -np.pi * (3 * l + 2 * u) * s[..., 0] * s[..., 1] * s[..., 2]
            for j in range(3):
                if i != j:
                    st[..., i, j] = 2 * np.pi * u * c[..., i] * c[..., j] * s[..., 3 - i - j]
        return st


def _solver_exact(case, seed):
    nt, n_poly, n_blk, faces = _sizes(case["mesh"], case["n"])
    n3 = 3 * _np(case["p"])
    steps = case.get("steps", 1)
    if (n_blk + nt + faces) * n3 * n3 > 4e7 or n_blk * n3 * n3 * steps > 3e9:
        return None
    m = _mesh(case, seed)
    D = _Plain(m, case["p"])
    dt = _dt(case, m)
    s, c = np.sin(np.pi * D.vx), np.cos(np.pi * D.vx)
    a = _amplitudes(seed)
    mms = case["kind"] == "run" and case["mesh"] in ("deck", "uneven")
    F = D.rhs(not mms)
    g = (lambda t: math.sin(math.sqrt(2) * math.pi * t)) if mms else (lambda t: math.cos(math.sqrt(3) * math.pi * t))

    def step(prev, cur, t):
        return dt * dt * D.minv(F * g(t) - D.apply(D.K, cur)) + 2 * cur - prev

    vel = math.sqrt(2) * math.pi * _uex(s, c)
    if case["kind"] != "run":
        prev = D.project(_u0(D.vx, a))
        cur = prev + dt * a[2] * D.project(vel)
        if case["kind"] == "step":
            return step(prev, cur, dt).reshape(-1)
        t = dt
        for _ in range(case["steps"]):
            prev, cur = cur, step(prev, cur, t)
            t += dt
        return dict(prev=prev.reshape(-1), cur=cur.reshape(-1), t=t)
    dt *= 1 - 0.001 * a[0]
    prev = D.project(0 * vel if mms else _u0(D.vx, (1.0, 0.0)))
    v0 = D.project(vel) if mms else 0 * prev
    cur = prev + dt * v0 + 0.5 * dt * dt * D.minv(F * g(0.0) - D.apply(D.K, prev))
    t = dt
    for _ in range(case["steps"] - 1):
        prev, cur = cur, step(prev, cur, t)
        t += dt
    e = cur - g(t) * D.project(_uex(s, c) if mms else _u0(D.vx, (1.0, 0.0)))
    l2 = np.einsum("pim,pmn,pin->", e.reshape(-1, 3, D.Np), D.Mm, e.reshape(-1, 3, D.Np), optimize=True)
    return dict(u=cur.reshape(-1), err_l2=math.sqrt(l2), err_dg=math.sqrt(float((e * D.apply(D.A, e)).sum())))


def _net_exact(case, seed):
    w = _widths(case)
    rows = case.get("rows", case["batch"])
    macs = sum(k * n for k, n in zip(w[:-1], w[1:]))
    if macs * (rows if case["kind"] == "predict" else 3 * case["batch"] * case.get("steps", 1)) > 3e11:
        return None
    flat = torch.from_numpy(mlp.init_params(w, seed)).double().requires_grad_(case["kind"] != "predict")

    def forward(x):
        at = 0
        for i, (k, n) in enumerate(zip(w[:-1], w[1:])):
            W, b = flat[at:at + n * k].view(n, k), flat[at + n * k:at + n * k + n]
            at += n * k + n
            x = x @ W.T + b
            if i + 2 < len(w):
                x = 0.5 * x * (1 + torch.special.erf(x / math.sqrt(2)))
        return x

    x, y = (torch.from_numpy(v).double() for v in _net_data(case, seed, case.get("samples", rows)))
    if case["kind"] == "predict":
        return forward(x)
    if case["kind"] == "gradients":
        loss = ((forward(x) - y) ** 2).mean()
        return dict(loss=float(loss), grads=torch.autograd.grad(loss, flat)[0])
    order = torch.from_numpy(_order(case, seed)).long().view(case["steps"], case["batch"])
    m1, m2, losses = torch.zeros_like(flat), torch.zeros_like(flat), []
    for k, idx in enumerate(order):
        loss = ((forward(x[idx]) - y[idx]) ** 2).mean()
        g = torch.autograd.grad(loss, flat)[0]
        losses.append(float(loss.detach()))
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        with torch.no_grad():
            flat -= 1e-3 * (m1 / (1 - 0.9 ** (k + 1))) / ((m2 / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return dict(losses=np.array(losses), params=flat.detach())


def exact(case, seed):
    if case["kind"] in ("train", "gradients", "predict"):
        return _net_exact(case, seed)
    if case["kind"] in ("ensemble", "record"):
        return None  # whole operators per instance: beyond a plain evaluation's time
    return _solver_exact(case, seed)
