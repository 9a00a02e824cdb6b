"""The workloads whose speed is measured: what a user of hydra_amd has it do.

A case is a dict of plain values; "kind" says which calls it makes:

  step       a checkpoint loaded, then advect-loop steps called one by one
             with the scalars read back between them: the loop that a Fortran
             host drives itself
  run        a checkpoint loaded, then hyd_run for a number of steps and the
             state read out
  flow       hyd_run continuing a flow between two saves
  ensemble   hyd_run_batch over independent mixed-precision flows
  surgery    the drop-in surgery: contour tables in, surgery, tables out
  recontour  the end of a regularisation cycle: a checkpoint loaded, prepare
             and recontour, the new contours out
  dropin     con2grid, ptospc, main_invert and velint on host arrays, the
             calls that the drop-in Fortran modules delegate to
  train      one Adam step of the learned velocity correction

Flows start from the seeded random PV field of hydra_amd.ic (spectrum
k^3 exp(-2 (k/6)^2), rms 4 pi).  "ell_cells" 6.25 is the reference's own
node spacing dm, 1.0 the finer dm of the throughput benchmark.  "spin" is
the number of steps a flow has run before: contours stretch and fold, so a
developed flow has several times the nodes of a fresh one and fine cells
that many of them cross.

Node arrays are read out into arrays of a fixed capacity, as the module
arrays of a Fortran host are, zero beyond the nodes in use.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hydra_amd import Hydra, VelocityCNN
from hydra_amd.ic import random_pv

L = 2.0 * math.pi
CNN_CHANNELS = ((4, 32), (32, 32), (32, 32), (32, 2))
FLOPS_PER_PIXEL = 2 * 9 * sum(ci * co for ci, co in CNN_CHANNELS)


def _flow(kind, name, ng, ncontq=80, ell_cells=6.25, kd=0.0, precision=0, steps=1, spin=0):
    return dict(name=name, kind=kind, ng=ng, ncontq=ncontq, ell_cells=ell_cells, kd=kd,
                precision=precision, steps=steps, spin=spin)


def listed():
    return [
        # the smallest flow of the tests, advanced step by step by its host
        _flow("step", "step_ng32", 32, steps=8),
        # a small flow well into its run
        _flow("run", "run_ng64_developed", 64, steps=4, spin=200),
        # the 100-step parity workload's flow (80 levels, the reference's
        # dm), some 300 steps in
        _flow("run", "run_ng256_developed", 256, steps=10, spin=300),
        # QG with a deformation radius, an uneven number of levels and a dm
        # between the two standard ones, from its start
        _flow("run", "run_ng512_qg", 512, ncontq=55, ell_cells=2.5, kd=2.0, steps=20),
        # the throughput benchmark: plain FP64 at ng=1024, fine dm
        _flow("flow", "flow_ng1024_dm", 1024, ell_cells=1.0, steps=30),
        # the same flow in mixed precision
        _flow("flow", "flow_ng1024_mixed_dm", 1024, ell_cells=1.0, precision=1, steps=30),
        # the large QG flow in mixed precision (120 levels, kd = 2)
        _flow("flow", "flow_ng2048_mixed_qg", 2048, ncontq=120, kd=2.0, precision=1, steps=10),
        # an ensemble of uneven flows on one GPU
        dict(name="ensemble_8", kind="ensemble", flows=8, ng_min=128, ng_max=512, steps=5),
        # regularisation of a developed flow through the drop-in tables
        _flow("surgery", "surgery_ng256_developed", 256, spin=280),
        # recontouring of a developed flow
        _flow("recontour", "recontour_ng64_developed", 64, spin=150),
        # the host-array calls of one inversion in a Fortran host
        dict(name="dropin_ng512", kind="dropin", ng=512, nodes=150001, rings=120, kd=0.0),
        # training on the snapshots of an ng=512 flow, 60000 nodes each
        dict(name="train_n512", kind="train", ng=512, nodes=60000),
    ]


def draw(rng):
    kind = rng.choice(["step", "run", "run", "run", "mixed", "flow", "flow", "ensemble",
                       "surgery", "recontour", "dropin", "train"])
    levels = rng.randint(30, 80)
    ell = round(math.exp(rng.uniform(0.0, math.log(6.25))), 3)
    kd = rng.choice([0.0, 0.0, 1.0, 2.0])
    if kind == "step":
        c = _flow(kind, "", rng.choice([32, 64, 128]), levels, 6.25, kd, 0, rng.randint(2, 8))
    elif kind == "run":
        c = _flow(kind, "", rng.choice([32, 64, 128, 256, 512]), levels, max(ell, 2.0), kd, 0,
                  rng.randint(3, 12), rng.randint(0, 140))
    elif kind == "mixed":
        c = _flow("run", "", rng.choice([64, 128, 256, 512]), levels, max(ell, 2.0), kd, 1,
                  rng.randint(3, 12), rng.randint(0, 140))
    elif kind == "flow":
        ng = rng.choice([1024, 1024, 2048])
        c = _flow(kind, "", ng, levels, 6.25 if ng == 2048 else ell, kd,
                  1 if ng == 2048 else rng.choice([0, 1]), rng.randint(4, 8 if ng == 2048 else 24))
    elif kind == "ensemble":
        c = dict(kind=kind, flows=rng.randint(3, 8), ng_min=rng.choice([64, 128]),
                 ng_max=rng.choice([256, 512]), steps=rng.randint(2, 5))
    elif kind == "surgery":
        c = _flow(kind, "", rng.choice([64, 128, 256, 512]), levels, ell, kd, 0, 1,
                  rng.randint(0, 120))
    elif kind == "recontour":
        c = _flow(kind, "", rng.choice([64, 128, 256, 512]), levels, 6.25, kd, 0, 1,
                  rng.randint(0, 120))
    elif kind == "dropin":
        c = dict(kind=kind, ng=rng.choice([64, 128, 256, 512, 1024]),
                 nodes=int(math.exp(rng.uniform(math.log(2e3), math.log(5e5)))) | 1,
                 rings=rng.randint(10, 200), kd=kd)
    else:
        c = dict(kind="train", ng=rng.choice([64, 128, 256, 512]), nodes=rng.randint(2000, 60000))
    c.pop("name", None)
    return c


def _ensemble_flows(case):
    """(ng, levels) of each member: grid sizes in turn, levels 40..120."""
    sizes = [1 << p for p in range(int(math.log2(case["ng_min"])),
                                   int(math.log2(case["ng_max"])) + 1)]
    return [(sizes[i % len(sizes)], 40 + (37 * i) % 81) for i in range(case["flows"])]


def _capacity(case):
    """Nodes that the host's arrays and the flow's store hold."""
    return max(1 << 20, 3 * _nodes(case["ng"], case["ncontq"], case["ell_cells"]))


def _new_flow(case, seed):
    h = Hydra(case["ng"], ncontq=case["ncontq"], kd=case["kd"], ell_cells=case["ell_cells"],
              precision=case["precision"], node_capacity=2 * _capacity(case))
    h.set_field(random_pv(case["ng"], seed=seed))
    h.recontour()
    h.evolution_init()
    if case["spin"]:
        h.run(case["spin"])
    return h


class _Arrays:
    """A host program's contour arrays, of fixed capacity."""

    def __init__(self, nodes):
        self.xy = np.zeros((2, nodes))
        self.table = np.zeros((2, nodes // 8), np.int32)
        self.counts = (0, 0)

    def read(self, h):
        c = h.contours()
        counts = (len(c["x"]), len(c["npq"]))
        for a, old, n in ((self.xy, self.counts[0], counts[0]),
                          (self.table, self.counts[1], counts[1])):
            if n < old:
                a[:, n:old] = 0
        self.counts = counts
        self.xy[0, :counts[0]], self.xy[1, :counts[0]] = c["x"], c["y"]
        self.table[0, :counts[1]], self.table[1, :counts[1]] = c["npq"], c["indq"]
        return dict(x=self.xy[0], y=self.xy[1], npq=self.table[0], indq=self.table[1],
                    nptq=counts[0], nq=counts[1])


def _rings(case, seed):
    """Closed wavy rings, nodes in proportion to their lengths: the contours
    of a host program, with node numbers linked ring by ring."""
    rng = np.random.default_rng(seed)
    k = case["rings"]
    radius = np.exp(rng.uniform(np.log(0.05), np.log(1.2), k))
    count = 8 + (radius / radius.sum() * (case["nodes"] - 8 * k)).astype(np.int64)
    count[-1] += case["nodes"] - int(count.sum())
    xs, ys, nxt, n = [], [], [], 0
    for r, m in zip(radius, count):
        th = 2.0 * np.pi * np.arange(m) / m * rng.choice([-1.0, 1.0])
        rr = r * (1.0 + 0.25 * np.cos(rng.integers(2, 7) * th + rng.uniform(0.0, 6.0)))
        cx, cy = rng.uniform(-np.pi, np.pi, 2)
        for out, v in ((xs, cx + rr * np.cos(th)), (ys, cy + rr * np.sin(th))):
            out.append(np.clip(v - L * np.floor((v + np.pi) / L), -np.pi, np.nextafter(np.pi, 0)
                               * (1.0 - 1e-12)))
        nxt.append(np.r_[np.arange(n + 2, n + m + 1), n + 1])
        n += int(m)
    return (np.concatenate(xs), np.concatenate(ys), np.concatenate(nxt).astype(np.int32),
            float(rng.uniform(0.5, 1.5)))


def _weights(seed):
    """He-style random weights in the library's order: per layer
    W[out][in][tap] then the biases; the pad channel's weights are zero."""
    rng = np.random.default_rng(seed)
    out = []
    for i, (ci, co) in enumerate(CNN_CHANNELS):
        w = rng.normal(0.0, math.sqrt(2.0 / (9 * (3 if i == 0 else ci))), (co, ci, 9))
        if i == 0:
            w[:, 3] = 0.0
        out += [w.ravel(), rng.normal(0.0, 0.05, co)]
    return np.concatenate(out).astype(np.float32)


def _snapshot(case, seed):
    """A training pair of the shapes and scales that hydra_amd.learned makes:
    inputs u, v, q over their rms, targets over theirs."""
    n, m = case["ng"], case["nodes"]
    rng = np.random.default_rng(seed)
    in3 = np.stack([random_pv(n, seed=seed * 3 + j, rms=1.0) for j in range(3)], axis=-1)
    return (in3.reshape(n * n, 3).astype(np.float32), rng.uniform(-np.pi, np.pi, m),
            rng.uniform(-np.pi, np.pi, m), rng.normal(size=m).astype(np.float32),
            rng.normal(size=m).astype(np.float32))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "run", "flow", "recontour", "surgery"):
        h = _new_flow(case, seed)
        state = dict(case=case, h=h, arrays=_Arrays(_capacity(case)))
        if kind == "surgery":  # on to the step that regularises the flow
            while h.scalar("twist") <= 2.5:
                if h.advect_step() == 1:
                    h.recontour()
                    h.evolution_init()
        if kind != "flow":  # a checkpoint
            state.update(contours=h.contours(), qs=h.field("qs"), t=h.scalar("t"))
        return state
    if kind == "ensemble":
        flows = [_new_flow(dict(ng=ng, ncontq=levels, kd=0.0, ell_cells=6.25, precision=1,
                                spin=0), seed + 1000 * i)
                 for i, (ng, levels) in enumerate(_ensemble_flows(case))]
        return dict(case=case, flows=flows, arrays=[_Arrays(1 << 20) for _ in flows])
    if kind == "dropin":
        h = Hydra(case["ng"], kd=case["kd"], node_capacity=max(1 << 20, 2 * case["nodes"]))
        return dict(case=case, h=h, contours=_rings(case, seed))
    net = VelocityCNN(case["ng"], seed=1)
    net.set_weights(_weights(seed))
    return dict(case=case, net=net, pair=_snapshot(case, seed))


def _load(state):
    """The checkpoint into the flow, ready to step."""
    h = state["h"]
    h.set_contours(state["contours"])
    h.put_field("qs", state["qs"])
    h.set_scalar("t", state["t"])
    h.evolution_init()
    return h


def _read(h, arrays):
    return dict(arrays.read(h), qs=h.field("qs"), qd=h.field("qd"), t=h.scalar("t"))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        h = _load(state)
        clock = []
        for _ in range(case["steps"]):
            h.advect_step()
            clock.append(h.scalar("t"))
        return dict(_read(h, state["arrays"]), clock=clock)
    if kind == "run":
        h = _load(state)
        h.run(case["steps"])
        return _read(h, state["arrays"])
    if kind == "flow":
        state["h"].run(case["steps"])
        return _read(state["h"], state["arrays"])
    if kind == "ensemble":
        Hydra.run_batch(state["flows"], case["steps"])
        return [dict(a.read(h), qs=h.field("qs")) for h, a in zip(state["flows"], state["arrays"])]
    if kind == "surgery":
        state["h"].set_contours(state["contours"])
        state["h"].surgery()
        return state["arrays"].read(state["h"])
    if kind == "recontour":
        h = _load(state)
        h.prepare()
        h.recontour()
        return dict(state["arrays"].read(h), qr=h.field("qr"))
    if kind == "dropin":
        h, (x, y, nxt, qjump) = state["h"], state["contours"]
        qc = h.con2grid(x, y, nxt, qjump)
        qs = h.ptospc(qc)
        uu, vv, pp = h.main_invert(qs)
        uq, vq = h.velint(uu, vv, x, y)
        return dict(qc=qc, qs=qs, uu=uu, vv=vv, pp=pp, uq=uq, vq=vq)
    loss = state["net"].train_step(*state["pair"], lr=1e-3)
    return dict(weights=state["net"].weights(), loss=loss)


def _nodes(ng, ncontq, ell_cells):
    """About the node count of a freshly contoured flow, which a developed
    one exceeds several times."""
    return int(ncontq * (260 + 4.86 * ng * 6.25 / ell_cells))


def _step_bytes(ng, nodes, grid):
    """One RK4 step's logical traffic: each of the step's fields and node
    arrays read or written once per use, grid = bytes of a grid value."""
    return 137 * grid * ng * ng + 336 * nodes


def _step_flops(ng, nodes):
    """37 real 2-D transforms (2.5 n log2 n per vector and direction), about
    60 operations per grid point and 100 per node and stage."""
    return 37 * 2 * 2.5 * ng * ng * math.log2(ng) + 4 * (60 * ng * ng + 100 * nodes)


def work(case):
    kind, ng = case["kind"], case.get("ng")
    if kind in ("step", "run", "flow"):
        p = _nodes(ng, case["ncontq"], case["ell_cells"])
        g = 4 if case["precision"] else 8
        return dict(bytes=case["steps"] * _step_bytes(ng, p, g) + 20 * p + 16 * ng * ng,
                    flops=case["steps"] * _step_flops(ng, p))
    if kind == "ensemble":
        ps = [(n, _nodes(n, k, 6.25)) for n, k in _ensemble_flows(case)]
        return dict(bytes=sum(case["steps"] * _step_bytes(n, p, 4) + 20 * p + 8 * n * n
                              for n, p in ps),
                    flops=sum(case["steps"] * _step_flops(n, p) for n, p in ps))
    if kind == "surgery":
        p = _nodes(ng, case["ncontq"], case["ell_cells"])
        return dict(bytes=(72 + 40) * p, flops=300 * p)
    if kind == "recontour":
        p = _nodes(ng, case["ncontq"], case["ell_cells"])
        # the contours come from the field on a grid 16 times finer
        return dict(bytes=8 * 256 * ng * ng + 36 * p, flops=20 * 256 * ng * ng + 300 * p)
    if kind == "dropin":
        p = case["nodes"]
        return dict(bytes=8 * 9 * ng * ng + 68 * p,
                    flops=6 * 2.5 * ng * ng * math.log2(ng) + 100 * p)
    return dict(bytes=ng * ng * (12 + 3 * 2 * 2 * 32 + 8) + 24 * case["nodes"],
                flops=3 * FLOPS_PER_PIXEL * ng * ng)


# ---- the same results in 64 bits, without the library ----------------------
def exact(case, seed):
    """The drop-in calls and the training step; a run of the flow solver
    (thousands of lines of order-dependent contour work) has no short
    restatement."""
    if case["kind"] == "dropin":
        return _exact_dropin(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None


def _half_complex(x):
    """rfft along the last axis in stafft's order: Re X_k at k, Im X_k at n-k."""
    n = x.shape[-1]
    f = np.fft.rfft(x, axis=-1) / math.sqrt(n)
    return np.concatenate([f.real, f.imag[..., 1:n // 2][..., ::-1]], axis=-1)


def _average(f):
    """Nine-point average of a periodic field to every second point."""
    up = np.roll(f, 1, axis=0)[::2]
    dn, mid = f[1::2], f[::2]

    def rows(a):
        return np.roll(a, 1, axis=1)[:, ::2], a[:, ::2], a[:, 1::2]

    (ul, um, ur), (ml, mm, mr), (dl, dm, dr) = rows(up), rows(mid), rows(dn)
    return (0.0625 * (ul + ur + dl + dr) + 0.125 * (um + dm + ml + mr) + 0.25 * mm)


def _contour_field(ng, x, y, nxt, qjump):
    """The PV grid of the contours: level jumps at the crossings of a grid
    four times finer, summed up each column, averaged twice, mean removed."""
    nf = 4 * ng
    gi = nf / L
    xa, ya = x[nxt - 1], y[nxt - 1]
    dx = (xa - x) - L * np.trunc((xa - x) / np.pi)
    dy = (ya - y) - L * np.trunc((ya - y) / np.pi)
    ix = 1 + np.trunc(gi * (x + np.pi)).astype(np.int64)
    ixa = 1 + np.trunc(gi * (xa + np.pi)).astype(np.int64)
    d = ixa - ix
    nxc = d - nf * np.trunc(2 * d / nf).astype(np.int64)
    # the bottom row: segments that leave through y = ymin
    up = np.abs(ya - y) > np.pi
    cc = np.sign(dy[up])
    p = -(y[up] - np.pi * cc) / (dy[up] + 1e-12)
    jx = np.trunc(gi * np.fmod(L + np.pi + x[up] + p * dx[up], L)).astype(np.int64)
    bottom = np.bincount(jx, weights=-cc, minlength=nf)[:nf]
    bottom = np.r_[0.0, np.cumsum(bottom)[:-1]]
    # one entry per crossed grid line
    rep = np.abs(nxc)
    i = np.repeat(np.arange(len(x)), rep)
    k = np.arange(len(i)) - np.repeat(np.cumsum(rep) - rep, rep)
    jump = np.sign(nxc[i])
    col = (ix[i] + (jump - 1) // 2 + nf + k * jump) % nf
    x2 = (-np.pi + L / nf * col) - x[i]
    y2 = y[i] + (x2 - L * np.trunc(x2 / np.pi)) / dx[i] * dy[i]
    row = 1 + np.trunc(gi * (y2 - L * np.trunc(y2 / np.pi) + np.pi)).astype(np.int64)
    keep = (row >= 1) & (row < nf)
    cell = np.bincount(col[keep] * nf + row[keep], weights=np.sign(dx[i])[keep],
                       minlength=nf * nf)
    f = qjump * (np.cumsum(cell.reshape(nf, nf), axis=1) + bottom[:, None])
    f = _average(_average(f))
    return f - f.mean()


def _exact_dropin(case, seed):
    ng, kd = case["ng"], case["kd"]
    x, y, nxt, qjump = _rings(case, seed)
    qc = _contour_field(ng, x, y, nxt, qjump)
    qs = _half_complex(_half_complex(qc.T).T).T
    half = ng // 2
    k = np.arange(ng)
    kk = np.where(k <= half, k, ng - k).astype(np.float64)
    k2 = kk[:, None] ** 2 + kk[None, :] ** 2 + kd * kd
    green = np.zeros((ng, ng))
    green.flat[1:] = -1.0 / k2.flat[1:]
    damp = np.where(k == half, 0.0, kk * np.exp(-36.0 * (kk / half) ** 36))
    dk = np.where(k < half, damp, -damp)
    psi = np.fft.fft2(qc) * green  # green is symmetric in k <-> ng-k
    vv = np.fft.ifft2(1j * dk[:, None] * psi).real
    uu = -np.fft.ifft2(1j * dk[None, :] * psi).real
    xx, yy = ng / L * (x + np.pi), ng / L * (y + np.pi)
    i0, j0 = np.trunc(xx).astype(np.int64), np.trunc(yy).astype(np.int64)
    px, py = xx - i0, yy - j0
    i1, j1 = (i0 + 1) % ng, (j0 + 1) % ng
    uq, vq = ((1 - py) * ((1 - px) * f[i0, j0] + px * f[i1, j0])
              + py * ((1 - px) * f[i0, j1] + px * f[i1, j1]) for f in (uu, vv))
    return dict(qc=qc, qs=qs, uu=uu, vv=vv, pp=green * qs, uq=uq, vq=vq)


def _exact_train(case, seed):
    n, m = case["ng"], case["nodes"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    w0 = torch.from_numpy(_weights(seed)).to(dev, torch.float64).requires_grad_(True)
    in3, xn, yn, tu, tv = (torch.from_numpy(a).to(dev, torch.float64)
                           for a in _snapshot(case, seed))
    a = torch.cat([in3.reshape(n, n, 3), torch.zeros(n, n, 1, device=dev,
                                                     dtype=torch.float64)], dim=-1)
    at = 0
    for i, (ci, co) in enumerate(CNN_CHANNELS):
        w = w0[at:at + co * ci * 9].reshape(co, ci, 9)
        at += co * ci * 9
        z = w0[at:at + co]
        at += co
        for tap in range(9):
            shifted = torch.roll(a, (1 - tap // 3, 1 - tap % 3), dims=(0, 1))
            z = z + (shifted.reshape(n * n, ci) @ w[:, :, tap].T.contiguous()).reshape(n, n, co)
        a = torch.nn.functional.gelu(z) if i < 3 else z
    xx, yy = n / L * (xn + math.pi), n / L * (yn + math.pi)
    i0, j0 = xx.long(), yy.long()
    px, py = (xx - i0)[:, None], (yy - j0)[:, None]
    i0, j0, i1, j1 = i0 % n, j0 % n, (i0 + 1) % n, (j0 + 1) % n
    out = ((1 - py) * ((1 - px) * a[i0, j0] + px * a[i1, j0])
           + py * ((1 - px) * a[i0, j1] + px * a[i1, j1]))
    loss = ((out - torch.stack([tu, tv], dim=-1)) ** 2).sum() / m
    loss.backward()
    g = w0.grad
    # Adam's first step: both moments are the gradient's own
    w1 = w0.detach() - 1e-3 * g / (g.abs() + 1e-8)
    return dict(weights=w1.cpu().numpy(), loss=float(loss))
