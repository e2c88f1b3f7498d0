"""Performance cases of the spark time-step library.

Each case is a piece of work that a program built on srs_amd does through the
public calls: stepping one spark or an ensemble of them and taking the fields
back, replaying a frozen channel trajectory, recording one, sampling a line
scan, and the loss and gradient of a line-scan fit.  ``prepare`` builds the
context a program keeps (mesh, realizations, scan line, initial state) and
``run`` makes the calls; ``exact`` restates the deterministic ones in plain
64-bit torch.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import srs_amd as S
from srs_amd import workloads as W


def listed():
    return [
        # The drop-in bridge on the smallest useful mesh: a host loop that sets
        # the channels, takes one step and reads channels and fields back.
        dict(name="bridge_small", kind="bridge", box="spark", n_xy=10, graded=False, order="rcm"),
        # The driver's loop on the plain spark: the loop body on the device,
        # states records drained and fields taken for a grid file at its end.
        dict(name="spark_protocol", kind="step", box="spark", n_xy=25, graded=False, order="morton", mode="protocol",
             physics="reference", steps=1000),
        # A spark mesh of another size in the default element order, with the
        # jSR diffusion coefficient and the SR binding sites on.
        dict(name="spark_physics", kind="step", box="spark", n_xy=37, graded=False, order="rcm", mode="plain",
             physics="extended", steps=555),
        # The flagship plain run: the 3M-element dyad box, gated steps.
        dict(name="dyad_plain", kind="step", box="dyad", n_xy=100, graded=False, order="block", mode="plain",
             physics="reference", steps=2000),
        # A dyad whose element rows all differ, as in a mesh from a mesher, in
        # the order the driver stores such meshes.
        dict(name="dyad_graded", kind="step", box="dyad", n_xy=75, graded=True, order="morton", mode="protocol",
             physics="reference", steps=700),
        # Monte Carlo ensembles: sparks on three meshes with clusters and SR
        # loads of their own, one at a time per tile and in groups of four.
        dict(name="ensemble", kind="ensemble", members=48, group=1, steps=200),
        dict(name="ensemble_groups", kind="ensemble", members=21, group=4, steps=150),
        # The frozen trajectories of a fit: one gated run of several members.
        dict(name="record", kind="record", box="dyad", n_xy=41, graded=False, order="block", members=12, steps=120),
        # Deterministic replay of a frozen trajectory.
        dict(name="replay", kind="replay", box="spark", n_xy=33, graded=False, order="rcm", steps=400),
        # One line scan of the current state (blurred fluorescence, nearest cells).
        dict(name="scan", kind="scan", box="dyad", n_xy=67, graded=False, order="block", points=96),
        # One fitting iteration on the spark box: forward, recomputation and
        # the reverse steps of a single realization.
        dict(name="grad_spark", kind="grad", box="spark", n_xy=25, graded=False, order="block", members=1, steps=2000,
             samples=10, points=64, grad=True),
        # One fitting iteration over a batch on the dyad box.
        dict(name="grad_batch", kind="grad", box="dyad", n_xy=67, graded=False, order="block", members=8, steps=64,
             samples=4, points=64, grad=True),
    ]


def draw(rng):
    kind = rng.choice(["bridge", "step", "step", "step", "ensemble", "record", "replay", "scan", "grad", "grad"])
    box = rng.choice(["spark", "dyad"])
    lo, hi = (9, 45) if box == "spark" else (24, 80)
    n_xy = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    mesh = dict(box=box, n_xy=n_xy, graded=rng.random() < 0.3, order=rng.choice(["rcm", "morton", "block"]))
    n = n_elements(mesh)

    def steps(cap, budget, members=1):  # spread over the logarithm, bounded by the element-steps
        top = max(8.0, min(cap, budget / (n * members)))
        return int(math.exp(rng.uniform(math.log(5.0), math.log(top))))

    if kind == "bridge":
        return dict(kind=kind, **mesh)
    if kind == "step":
        return dict(kind=kind, **mesh, mode=rng.choice(["plain", "protocol"]),
                    physics=rng.choice(["reference", "reference", "extended"]), steps=steps(3000, 3e9))
    if kind == "ensemble":
        members = int(math.exp(rng.uniform(math.log(2), math.log(49))))
        return dict(kind=kind, members=members, group=rng.choice([1, 1, 2, 4]), steps=rng.randint(10, 200))
    if kind == "record":
        members = rng.randint(1, 8)
        return dict(kind=kind, **mesh, members=members, steps=steps(1000, 1e9, members))
    if kind == "replay":
        return dict(kind=kind, **mesh, steps=steps(1000, 1e9))
    if kind == "scan":
        return dict(kind=kind, **mesh, points=rng.randint(8, 300))
    members = rng.randint(1, 6)
    k = max(6, steps(2000, 4e8, members))
    return dict(kind=kind, **mesh, members=members, steps=k, samples=rng.randint(1, min(6, k)),
                points=rng.randint(8, 120), grad=rng.random() < 0.7)


# ------------------------------------------------------------------- meshes
# dyad: plane counts below, in and above the cleft and jSR at spacing h
def _dyad_planes(n_xy):
    h = 2.0 / n_xy
    n_low = int(round(0.2 / h))
    return n_low, (50 - n_low - 3 if n_xy == 100 else int(round(0.745 / h)))


def n_elements(case):
    """Tetrahedra of a case's box (six per cube; the T-tubule takes out about
    1.6% of the dyad's)."""
    n = case["n_xy"]
    if case["box"] == "spark":
        return 6 * n * n * (2 + int(round(0.545 * n)) - 1)
    return int(0.984 * 6 * n * n * (sum(_dyad_planes(n)) + 3))


@functools.lru_cache(maxsize=6)
def _mesh(box, n_xy, graded, order):
    """(grid, aij, nij, element order, dt): the mesh files and operator a
    program has read and assembled."""
    spec = W.spark_box_spec(h=1.0 / n_xy, n_xy=n_xy) if box == "spark" else W.dyad_box_spec(h=2.0 / n_xy)
    if graded:  # planes drawn apart by up to a quarter of the spacing; the cleft and the jSR keep theirs
        rng = np.random.default_rng(n_xy)
        for name in ("xs", "ys", "zs"):
            p = np.array(getattr(spec, name))
            d = rng.uniform(-0.25, 0.25, len(p)) * np.min(np.diff(p))
            d[0] = d[-1] = 0.0
            if name == "zs":
                d[p < 0.256 if box == "dyad" else p < 0.056] = 0.0
            setattr(spec, name, p + d)
    g = S.box_grid(spec)
    aij, nij = S.assemble_operator(g)
    perm = dict(rcm=lambda: None, morton=lambda: S.morton_order(g), block=lambda: W.kuhn_block_order(g))[order]()
    return g, aij, nij, perm, W.stable_dt(aij, 0.22)


@functools.lru_cache(maxsize=1)
def _ensemble_meshes():
    return [m + (W.kuhn_block_order(m[0]),) for m in W.ensemble_meshes()]


def _case_mesh(case):
    return _mesh(case["box"], case["n_xy"], case["graded"], case["order"])


def _params(case, dt):
    p = W.spark_params(t_final=1e9, states_interval=0.01)
    p.setr(T_STEP=dt, INIT_RYR_HOLD=dt)
    p.seti(INIT_RYR=0)
    if case.get("physics") == "extended":
        p.setr(D_CA_JSR=W.CONFIG_D_JSR, T_STEP=0.6 * dt, INIT_RYR_HOLD=0.6 * dt)
    return p


def _state(g, p, rng):
    """Fields of a spark under way: the resting state, a Ca transient around
    the cluster with Ca-bound buffers following it, and noise."""
    X = S.equilibrium_state(g, p.reals)[0].reshape(6, -1)
    c = g.centroids()
    c0 = c[g.ryr_ele].mean(axis=0)
    bump = np.exp(-((c - c0) ** 2).sum(axis=1) / (2 * 0.12 ** 2))
    cyt = g.domain == 0
    X *= rng.uniform(0.97, 1.0, X.shape)
    X[S.CA] += cyt * bump * rng.uniform(5.0, 30.0)
    for s, top in ((S.ATP, 455.0), (S.CMDN, 24.0), (S.DYE, 50.0)):
        X[s] += cyt * bump * 0.3 * (top - X[s])
    return np.ascontiguousarray(X).reshape(-1)


def _channels(n_ryr, n_lcc, rng):
    return ((rng.random(n_ryr) < 0.2).astype(np.int32), rng.choice([1, 3, 6, 8], n_lcc).astype(np.int32),
            np.full(n_lcc, 2, np.int32), np.log(1.0 - rng.random(n_ryr + n_lcc)))


def _schedule(n_steps, n_ryr, rng):
    """RyR states per step: each RyR open and closed in turn for some hundreds
    of steps, starting where it is."""
    out = np.zeros((n_steps, n_ryr), np.int32)
    for i in range(n_ryr):
        k, s = 0, int(rng.random() < 0.25)
        while k < n_steps:
            m = 1 + int(rng.exponential(300.0))
            out[k:k + m, i] = s
            k, s = k + m, 1 - s
    return out


def _scan_desc(case, g):
    """A line of `points` along x through the cluster in a centred mesh, with
    the linescan program's PSF and padding around the box."""
    size = (1.0, 1.0, 0.6) if case["box"] == "spark" else (2.0, 2.0, 1.0)
    c0 = np.array(size) / 2
    d = S.read_scan_parameters(None)
    rc = g.centroids()[g.ryr_ele].mean(axis=0) - c0
    d.axis, d.offset1, d.offset2 = 0, float(rc[1]), float(rc[2])
    d.x_min, d.x_max = -0.48 * size[0], 0.48 * size[0]
    d.res_x_f = (d.x_max - d.x_min) / (case["points"] + 0.5)
    d.res_x_ca = 0.04
    for k in range(3):
        d.domain[k] = size[k]
    d.pad_min, d.pad_max, d.pad_res = -size[0] / 2 - 1.0, size[0] / 2 + 1.0, 0.15
    return d, g.centroids() - c0


def _samples(case):
    return np.linspace(max(1, case["steps"] // case["samples"]), case["steps"], case["samples"]).astype(np.int64)


def _target(case, rng):
    """A measured line scan: a transient that grows, with noise."""
    x = np.linspace(-1.0, 1.0, case["points"])
    t = np.linspace(0.3, 1.0, case["samples"])[:, None]
    return 0.4 * t * np.exp(-x * x / 0.18) + 0.02 * rng.standard_normal((case["samples"], case["points"]))


def _member_inputs(case, seed):
    """What each realization of a case on one mesh starts from."""
    g, _, _, _, dt = _case_mesh(case)
    out = []
    for m in range(case.get("members", 1)):
        rng = np.random.default_rng([seed, m])
        p = _params(case, dt)
        if case["kind"] == "grad":  # a fit's iterate, each member's own
            idx = S.adjoint_theta()
            p.reals[idx] *= rng.uniform(0.95, 1.05, len(idx))
        e = dict(p=p, X=_state(g, p, rng), ch=_channels(g.n_ryr, g.n_lcc, rng))
        if case["kind"] in ("replay", "grad"):
            e["sched"] = _schedule(case["steps"], g.n_ryr, rng)
        if case["kind"] == "grad":
            e["target"] = _target(case, rng)
        out.append(e)
    return out


def _start(ctx, r, e):
    ctx.state_set(r, e["X"])
    ctx.channels_set(r, *e["ch"])
    ctx.globals_set(r, 0.0, e["p"].reals[S.R["DEFAULT_CA_NSR"]])


def prepare(case, seed):
    if case["kind"] == "ensemble":
        return _prepare_ensemble(case, seed)
    g, aij, nij, perm, dt = _case_mesh(case)
    members = _member_inputs(case, seed)
    ctx = S.Context(0)
    mid = ctx.add_mesh_grid(g, aij, nij, perm=perm)
    for m, e in enumerate(members):
        ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, e["p"], seed=seed * 1000 + m, stream=m)
    ctx.finalize(4096 if case.get("mode") == "protocol" else 0)
    for m, e in enumerate(members):
        if case.get("physics") == "extended":
            ctx.extensions(m, **W.CONFIG_SR_SITES)
        _start(ctx, m, e)
    st = dict(case=case, ctx=ctx, members=members)
    if case["kind"] in ("scan", "grad"):
        d, cen = _scan_desc(case, g)
        st["scan"] = ctx.add_scan(mid, cen, d)[0]
    if case["kind"] == "grad":
        st["samples"] = _samples(case)
        st["scheds"] = [e["sched"] for e in members]
        st["targets"] = np.array([e["target"] for e in members])
    return st


def _prepare_ensemble(case, seed):
    meshes = _ensemble_meshes()
    ctx = S.Context(0)
    ctx.tune(group=case["group"])
    mids = [ctx.add_mesh_grid(g, aij, nij, perm=perm) for g, aij, nij, _, perm in meshes]
    members = []
    for r, mem in enumerate(W.ensemble_members(case["members"])):  # the clusters are the ensemble's, the rest the seed's
        g, _, _, dt, _ = meshes[mem["mesh"]]
        e = W.ensemble_member(mem, meshes[mem["mesh"]][:4], r, seed, with_state=False)
        ctx.add_realization(mids[mem["mesh"]], e["ryr_ele"], e["ryr_jsr"], e["ryr_nb"], e["lcc_ele"], e["p"],
                            seed=e["key"], stream=e["stream"])
        rng = np.random.default_rng([seed, r])
        members.append(dict(p=e["p"], X=_state(g, e["p"], rng), ch=_channels(e["n_ryr"], g.n_lcc, rng)))
    ctx.finalize()
    for r, e in enumerate(members):
        _start(ctx, r, e)
        e["X"] = None
    return dict(case=case, ctx=ctx, members=members)


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "bridge":  # one ExplicitStep of a host loop that owns the channels
        rs, ls, lvs, _ = ctx.channels_get(0)
        ctx.channels_set(0, rs, ls, lvs)
        ctx.globals_set(0, 0.0, state["members"][0]["p"].reals[S.R["DEFAULT_CA_NSR"]])
        ctx.explicit_step(1)
        return ctx.channels_get(0) + (ctx.state_get(0),)
    if kind == "step":
        if case["mode"] == "protocol":
            ctx.explicit_step(case["steps"], S.STEP_PROTOCOL | S.STEP_GRAPH)
            return (ctx.records(0, 4096), ctx.state_get(0)) + ctx.channels_get(0)
        ctx.explicit_step(case["steps"], S.STEP_GRAPH)
        return (ctx.state_get(0),) + ctx.channels_get(0)
    if kind == "ensemble":
        ctx.explicit_step(case["steps"], S.STEP_GRAPH)
        ch = [ctx.channels_get(r) for r in range(ctx.n_real)]
        return [ctx.state_get(r) for r in range(ctx.n_real)] + [np.concatenate(x) for x in zip(*ch)]
    if kind == "record":
        scheds = ctx.record_schedules(case["steps"])
        return np.stack(scheds), [ctx.state_get(r) for r in range(ctx.n_real)]
    if kind == "replay":
        ctx.replay(0, state["members"][0]["sched"])
        return ctx.state_get(0)
    if kind == "scan":
        return ctx.scan_sample(0, state["scan"])
    args = (state["scheds"], state["samples"], state["targets"])
    if case["members"] == 1 and case["grad"]:
        return ctx.loss_grad(0, state["scan"], args[0][0], args[1], args[2][0])
    return ctx.loss_grad_batch(range(case["members"]), state["scan"], *args, grad=case["grad"], scans=True)


# ----------------------------------------------------------------- the work
# A step reads and writes five live FP64 species per element (the four that
# diffuse, and TnC or CSQ) and takes about 130 operations; the operator row
# (five FP64, four int32) and the flags are read once per pass.  A reverse step
# reads a state and an adjoint and writes an adjoint.
def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        sizes = [6 * 25 * 25 * 15, 6 * 33 * 33 * 20, 6 * 40 * 40 * 24]
        n = sum(sizes[r % 3] for r in range(case["members"]))
        return dict(bytes=float(n * (80 * case["steps"] + 48) + 57 * sum(sizes)), flops=130.0 * n * case["steps"])
    e = n_elements(case)
    n = e * case.get("members", 1)
    if kind == "scan":
        return dict(bytes=float(e * 40), flops=8.0 * e * case["points"])
    steps = case.get("steps", 1)
    if kind != "grad":
        return dict(bytes=float(n * (80 * steps + 48) + 57 * e), flops=130.0 * n * steps)
    scans = 8.0 * n * case["points"] * case["samples"]
    per_b, per_f = (80.0, 130.0) if not case["grad"] else (80.0 + 120.0, 130.0 + 350.0)
    return dict(bytes=n * per_b * steps + 57.0 * e, flops=n * per_f * steps + (2.0 if case["grad"] else 1.0) * scans)


# ---------------------------------------------------------- 64-bit reference
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _T(a, **kw):
    return torch.as_tensor(np.ascontiguousarray(a), device=_device(), **kw)


class _Plain:
    """The frozen-channel step, the line scan and its loss, in torch."""

    def __init__(self, case):
        g, aij, nij, _, _ = _case_mesh(case)
        self.g, self.n = g, g.n_ele
        a, nb = aij.reshape(-1, 5), nij.reshape(-1, 4)
        self.a = [_T(a[:, k]) for k in range(5)]
        self.nb = [_T(nb[:, k]).long() for k in range(4)]
        self.jsr = _T(g.domain != 0)
        self.cyt = ~self.jsr
        self.trp = self.cyt & _T(g.tropc != 0)
        self.V0, self.tt = _T(g.V0), _T(g.tt_area)
        self.ryr_c, self.ryr_j = _T(g.ryr_ele).long(), _T(g.ryr_jsr).long()
        self.lcc = _T(g.lcc_ele).long()

    def step(self, X, P, open_ryr, open_lcc, nsr):
        """X: (6, n) -> (6, n); P: the parameter vector as 0-d tensors."""
        R = S.R
        ca, atp, cam, trn, csq, dye = X

        def diff(c):
            return c * self.a[0] + sum(c[self.nb[k]] * self.a[k + 1] for k in range(4))

        def bind(b, kon, koff, tot, mask):
            return torch.where(mask, P[R[kon]] * (P[R[tot]] - b) * ca - P[R[koff]] * b, torch.zeros_like(ca))

        r_trn = bind(trn, "K_ON_TRPN", "K_OFF_TRPN", "B_TOT_TRPN", self.trp)
        r_dye = bind(dye, "K_ON_DYE", "K_OFF_DYE", "B_TOT_DYE", self.cyt)
        r_atp = bind(atp, "K_ON_ATP", "K_OFF_ATP", "B_TOT_ATP", self.cyt)
        r_cam = bind(cam, "K_ON_CMDN", "K_OFF_CMDN", "B_TOT_CMDN", self.cyt)
        r_csq = bind(csq, "K_ON_CSQN", "K_OFF_CSQN", "B_T_JSR", self.jsr)
        ki, ks = (ca / P[R["K_D_I"]]) ** 2, (nsr / P[R["K_D_SR"]]) ** 2
        cyc = (0.104217 + 17.923 * ks) + ki * (1.75583e6 + ks * 7.61673e6) + ki * ki * (6.08463e11 + ks * 4.50544e11)
        serca = 2e-3 * P[R["A_P"]] * (ki * ki * 3.24873e12 + ki * (9.17846e6 - 11478.2 * ks) - 0.329904 * ks) / cyc
        rca = P[R["D_CA"]] * diff(ca) - r_trn - r_dye - r_atp - r_cam - r_csq
        rca = rca - torch.where(self.trp, serca, torch.zeros_like(ca))
        rca = rca + torch.where(self.jsr, (nsr - ca) * P[R["V_REFILL"]], torch.zeros_like(ca))
        J = open_ryr * P[R["V_RYR"]] * (ca[self.ryr_j] - ca[self.ryr_c]) * P[R["V_CELL"]]
        rca = rca.index_add(0, self.ryr_c, J / self.V0[self.ryr_c])
        rca = rca.index_add(0, self.ryr_j, -J / self.V0[self.ryr_j])
        v, k = 1e-6, 96.5 / (310 * 8.314)
        e2 = math.exp(2 * v * k)
        F = -(9.13e-13 * 1e12 * 1e-3) * v * 2 * k * (ca[self.lcc] * e2 - 0.34 * P[R["CA_0"]]) / (e2 - 1)
        rca = rca.index_add(0, self.lcc, open_lcc * F / self.V0[self.lcc])
        hi, lo = (self.tt * P[R[b]] / (self.V0 * 1e-15) for b in ("B_TOT_SL_HI", "B_TOT_SL_LO"))
        kh, kl = P[R["K_D_SL_HI"]], P[R["K_D_SL_LO"]]
        rca = rca / (1 + hi * kh / (kh + ca) ** 2 + lo * kl / (kl + ca) ** 2)
        dt = P[R["T_STEP"]]
        return torch.stack([ca + dt * rca, atp + dt * (P[R["D_ATP"]] * diff(atp) + r_atp),
                            cam + dt * (P[R["D_CMDN"]] * diff(cam) + r_cam), trn + dt * r_trn, csq + dt * r_csq,
                            dye + dt * (P[R["D_DYE"]] * diff(dye) + r_dye)])

    def start(self, e):
        rs, ls, lvs, _ = e["ch"]
        P = [torch.tensor(float(v), dtype=torch.float64, device=_device()) for v in e["p"].reals]
        lcc = _T((np.isin(ls, (6, 12)) & (lvs == 2)).astype(np.float64))
        return _T(e["X"].reshape(6, -1)), P, lcc, float(e["p"].reals[S.R["DEFAULT_CA_NSR"]])

    def scan_setup(self, case):
        d, cen = _scan_desc(case, self.g)
        self.d, s2 = d, np.array([d.var[0], d.var[1], d.var[2]])
        lo, hi = [-d.domain[k] / 2 for k in range(3)], [d.domain[k] / 2 for k in range(3)]
        a, b = d.pad_min, d.pad_max
        pts, vol = [], []
        for box in (((a, b), (a, b), (hi[2], b)), ((a, b), (a, b), (lo[2], a)), ((lo[0], a), (a, b), (lo[2], hi[2])),
                    ((hi[0], b), (a, b), (lo[2], hi[2])), ((lo[0], hi[0]), (lo[1], a), (lo[2], hi[2])),
                    ((lo[0], hi[0]), (hi[1], b), (lo[2], hi[2]))):
            ax = []
            for u, v in box:  # cells of the padding resolution from u towards v
                h = d.pad_res if v >= u else -d.pad_res
                ax.append(u + h * np.arange(int((v - u) / h)) + 0.5 * h)
            pts.append(np.stack(np.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3))
            vol.append(np.full(len(pts[-1]), d.pad_res ** 3))
        pad, vol = np.concatenate(pts), np.concatenate(vol)
        n_f, n_ca = (int((d.x_max - d.x_min) / r) for r in (d.res_x_f, d.res_x_ca))
        norm = 1.0 / (2 * 3.14159) ** 1.5 / math.sqrt(s2.prod())  # the program's pi
        cen, pad = _T(cen), _T(pad)

        def line(n, res):
            p = np.zeros((n, 3))
            p[:, 0], p[:, 1], p[:, 2] = d.x_min + res * np.arange(n), d.offset1, d.offset2
            return _T(p)

        def weights(c, p):
            r2 = (c - p) ** 2
            return torch.where(r2.sum(1) < 1.0, norm * torch.exp(-0.5 * (r2 / _T(s2)).sum(1)), 0.0)

        def nearest(p):  # first minimum over the mesh, then the padding cells
            m = ((cen - p) ** 2).sum(1).min(0)
            return -1 if len(pad) and float(((pad - p) ** 2).sum(1).min()) < float(m.values) else int(m.indices)

        pf = line(n_f, d.res_x_f)
        self.w = torch.stack([weights(cen, p) * self.V0 for p in pf])
        self.pad = torch.stack([(weights(pad, p) * _T(vol)).sum() * d.f0 for p in pf])
        self.near_f, self.near_ca = [nearest(p) for p in pf], [nearest(p) for p in line(n_ca, d.res_x_ca)]

    def blur(self, X):
        return self.w @ X[S.DYE] + self.pad


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("replay", "scan", "grad"):
        return None  # gated runs: the trajectory is one of random draws
    if work(case)["flops"] * (2.5 if case.get("grad") else 1.0) > 4e12 or case.get("steps", 0) > 2500:
        return None
    M = _Plain(case)
    members = _member_inputs(case, seed)
    if kind == "replay":
        X, P, lcc, nsr = M.start(members[0])
        sched = _T(members[0]["sched"]).double()
        for k in range(case["steps"]):
            X = M.step(X, P, sched[k], lcc, nsr)
        return X.reshape(-1)
    M.scan_setup(case)
    if kind == "scan":
        X = M.start(members[0])[0]
        ca = [float(X[S.CA, e]) if e >= 0 else M.d.c0 for e in M.near_ca]
        caf = [float(X[S.DYE, e]) if e >= 0 else M.d.f0 for e in M.near_f]
        return np.array(ca), np.array(caf), M.blur(X)
    out = [_exact_fit(M, case, e) for e in members]
    if case["members"] == 1 and case["grad"]:
        return out[0][0], out[0][1]
    res = (np.array([o[0] for o in out]),)
    if case["grad"]:
        res += (np.array([o[1] for o in out]),)
    return res + (np.array([o[2] for o in out]),)


def _exact_fit(M, case, e):
    """(loss, gradient, dF/F0 scans) of one member, differentiated by torch
    segment by segment from kept states."""
    X, P, lcc, nsr = M.start(e)
    sched, target = _T(e["sched"]).double(), _T(e["target"])
    samples = [int(k) for k in _samples(case)]
    idx = [int(i) for i in S.adjoint_theta()]
    seg = 40
    kept, scans = [], []

    def advance(X, a, b):
        loss, rows = 0.0, []
        for k in range(a, b):
            X = M.step(X, P, sched[k], lcc, nsr)
            if k + 1 in samples:
                rows.append(M.blur(X) / M.d.f0 - 1.0)
                loss = loss + ((rows[-1] - target[samples.index(k + 1)]) ** 2).sum()
        return X, loss, rows

    total = 0.0
    with torch.no_grad():
        for a in range(0, case["steps"], seg):
            kept.append(X)
            X, loss, rows = advance(X, a, min(a + seg, case["steps"]))
            total += float(loss)
            scans += [r.cpu().numpy() for r in rows]
    if not case["grad"]:
        return total, None, np.array(scans)
    theta = [P[i].requires_grad_(True) for i in idx]
    lam, grad = torch.zeros_like(X), np.zeros(len(idx))
    for q in reversed(range(len(kept))):
        x = kept[q].detach().requires_grad_(True)
        y, loss, _ = advance(x, q * seg, min((q + 1) * seg, case["steps"]))
        got = torch.autograd.grad((y * lam).sum() + loss, [x] + theta, allow_unused=True)
        lam = got[0]
        grad += np.array([0.0 if v is None else float(v) for v in got[1:]])
    return total, grad, np.array(scans)
