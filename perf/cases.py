"""What is timed: the work that programs have this framework do, through its
Python entry points (0buf_amd), over the range of sizes, forms and options.

A case is a dict of plain values.  `kind` says what one pass is:

  run    `steps` calls of the time step (Pic.run, as the reference's main loop
         runs between two of its diagnostics), then the six E and H arrays
         read back for the diagnostic, and in the FP64 form the cell counts
  grad   one gradient of the differentiable form: back to the initial state,
         the forward run with checkpoints, the reverse sweep, the adjoint of
         the initial state in host arrays that the program keeps
  diag   one time step and the diagnostics of the state after it: the per-cell
         moments of every sort, the Gauss-law residual, the global moments

`form` is the precision form (f64, f32).  The particles of small boxes are
drawn here and loaded from the host (`source` host, as a program that reads or
makes its own particles does); those of large ones are drawn by the device
initializer (`source` device).  Plasmas are those of the beam-plasma
workloads: ions, plasma electrons of a thermal spread, and an electron beam,
uniform or (profile 1) with a transverse Gaussian profile.
"""
import importlib
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

pic = importlib.import_module("0buf_amd")

H = 0.1                                   # cell size of every workload
PARTS = ("x", "y", "z", "px", "py", "pz")
FIELDS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")
OPS = ("density", "kinetic_energy", "velocity", "current")


def _case(name, kind, form, n, ppc, steps, *, tau=0.05, bx0=0.0, profile=0, source="device",
          ckpt=0):
    c = {"kind": kind, "form": form, "nx": n[0], "ny": n[1], "nz": n[2], "ions": ppc[0],
         "electrons": ppc[1], "beam": ppc[2], "steps": steps, "tau": tau, "bx0": bx0,
         "profile": profile, "source": source, "ckpt": ckpt}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest workload, particles from the host: latency and launches count
        _case("run_f64_32x8x8", "run", "f64", (32, 8, 8), (16, 16, 16), 100, source="host"),
        # a small box in the FP32 form, more steps between diagnostics
        _case("run_f32_64x16x16", "run", "f32", (64, 16, 16), (8, 16, 8), 200, source="host"),
        # a box that no tile divides, an uneven mix of species, a field along x
        _case("run_f64_45x27x19", "run", "f64", (45, 27, 19), (13, 27, 11), 40, tau=0.04,
              bx0=0.3, source="host"),
        # the production box of the plain form, and the same in the FP32 form
        _case("run_f64_256x64x64", "run", "f64", (256, 64, 64), (16, 32, 16), 20),
        _case("run_f32_256x64x64", "run", "f32", (256, 64, 64), (16, 32, 16), 40),
        # the FP32 form on a box that no tile divides
        _case("run_f32_101x50x37", "run", "f32", (101, 50, 37), (21, 21, 9), 40, tau=0.04),
        # the largest: the magnetised comparison workload's cross-section, half its length
        _case("run_f32_256x128x128", "run", "f32", (256, 128, 128), (24, 24, 24), 40, bx0=0.5),
        # gradients: a small box over a whole run, host particles
        _case("grad_f64_64x16x16", "grad", "f64", (64, 16, 16), (8, 16, 8), 200, source="host",
              ckpt=20),
        # ... and large ones in both forms with a narrow beam, whose cells on the
        # axis hold ten times the mean and send as much on (for these every pass
        # starts again from the initial state; a plain run would go on for
        # thousands of steps, past the collapse of such a beam)
        _case("grad_f64_beam_128x64x64", "grad", "f64", (128, 64, 64), (16, 16, 16), 20,
              profile=1, ckpt=10),
        _case("grad_f32_beam_256x64x64", "grad", "f32", (256, 64, 64), (16, 16, 16), 40,
              profile=1, ckpt=20),
        # diagnostics of a small plain-form box and of a production FP32 box
        _case("diag_f64_33x24x20", "diag", "f64", (33, 24, 20), (12, 24, 12), 1, tau=0.04,
              source="host"),
        _case("diag_f32_256x64x64", "diag", "f32", (256, 64, 64), (16, 32, 16), 1),
    ]


def _particles(c):
    return c["nx"] * c["ny"] * c["nz"] * (c["ions"] + c["electrons"] + c["beam"])


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("run", "run", "run", "grad", "diag"))
        form = rng.choice(("f64", "f32"))
        n = (_spread(rng, 8, 256), _spread(rng, 8, 128), _spread(rng, 8, 128))
        profile = 1 if kind == "grad" and min(n[1], n[2]) >= 24 and rng.random() < 0.5 else 0
        top = 8 if profile else 24         # a profiled beam's axis holds ten times its mean
        a, b = rng.randint(4, top), rng.randint(4, top)
        ppc = (a, rng.choice((a, 2 * a)), b)
        steps = 1 if kind == "diag" else _spread(rng, 10, 200)
        c = _case("", kind, form, n, ppc, steps, tau=rng.choice((0.04, 0.03)),
                  bx0=rng.choice((0.0, 0.0, 0.5)), profile=profile,
                  ckpt=rng.choice((5, 10, 20)) if kind == "grad" else 0)
        P = _particles(c)
        c["source"] = "host" if P <= 1_000_000 and not profile else "device"
        # no more than the largest listed cases, within what a host checks quickly
        most = {"run": 40e6, "diag": 40e6, "grad": 12e6}[kind] / (2 if profile else 1)
        if P <= most and P * steps <= {"run": 1.5e9, "diag": 1e9, "grad": 2e8}[kind]:
            return c


# ---------------------------------------------------------------------------
# what a program has in hand before the call
# ---------------------------------------------------------------------------

def _weights(c):
    """(sort, particles per cell, charge weight, q/m, drift, thermal spread)"""
    nb = 0.05 if c["profile"] else 0.01
    return [(pic.ION, c["ions"], (1.0 + nb) / c["ions"], 1.0 / 1836.0, 0.0, 0.0),
            (pic.PLASMA_ELECTRON, c["electrons"], -1.0 / c["electrons"], -1.0, 0.0, 0.02),
            (pic.BEAM_ELECTRON, c["beam"], -nb / c["beam"], -1.0, 0.3, 0.005)]


def _host_species(c, seed):
    """Particles drawn uniformly in every cell: (sort, x..pz, m, q_m) each."""
    n = (c["nx"], c["ny"], c["nz"])
    rng = np.random.default_rng(seed)
    grid = np.stack(np.meshgrid(*[np.arange(k, dtype=np.float64) for k in n], indexing="ij"))
    cells = grid.reshape(3, -1)
    out = []
    for sort, ppc, m, q_m, drift, vth in _weights(c):
        at = np.repeat(cells, ppc, axis=1)
        x = (at + rng.uniform(1e-9, 1.0 - 1e-9, at.shape)) * H
        u = rng.normal(0.0, 1.0, at.shape) * vth
        u[0] += drift
        p = u / np.sqrt(1.0 - (u * u).sum(0))
        out.append((sort, *x, *p, m, q_m))
    return out


def _device_species(c):
    """The same plasma for the device initializer, the ions' mean charge that
    of the electrons for the profiled beam too."""
    nb = nb_mean = 0.05 if c["profile"] else 0.01
    if c["profile"]:
        y = np.arange(c["ny"]) + 0.5 - 0.5 * c["ny"]
        z = np.arange(c["nz"]) + 0.5 - 0.5 * c["nz"]
        nb_mean = nb * float(np.exp(-(y[:, None] ** 2 + z[None, :] ** 2) / 128.0).mean())
    return [pic.species_spec(pic.ION, c["ions"], 1.0 + nb_mean, 1.0, 1.0 / 1836.0),
            pic.species_spec(pic.PLASMA_ELECTRON, c["electrons"], 1.0, -1.0, -1.0,
                             vth=(0.02, 0.02, 0.02)),
            pic.species_spec(pic.BEAM_ELECTRON, c["beam"], nb, -1.0, -1.0, drift=(0.3, 0.0, 0.0),
                             vth=(0.005, 0.005, 0.005), profile=c["profile"], sigma_cells=8.0)]


def prepare(case, seed):
    c = case
    n = (c["nx"], c["ny"], c["nz"])
    grad = c["kind"] == "grad"
    params = pic.make_params(n, tuple(k * H for k in n), c["tau"],
                             precision=pic.FP32 if c["form"] == "f32" else pic.FP64,
                             departure_cap=0,   # runs go past the reference's storage limit
                             differentiable=1 if grad else 0, ghost_mode=1 if grad else 0)
    g = pic.Pic(params)
    if c["source"] == "host":
        for sort, x, y, z, px, py, pz, m, q_m in _host_species(c, seed):
            g.load_particles(sort, x, y, z, px, py, pz, m, q_m)
    else:
        g.generate_device(_device_species(c), seed=seed + 1)
    if c["bx0"]:
        g.load_field(pic.HX, np.full(g.G, c["bx0"]))
    g.cell_counts()
    state = {"case": c, "g": g, "nt": 1, "again": False}
    if grad:
        # the energies of the last quarter of the run make the loss; the
        # gradient lands in pinned arrays that the program keeps
        w = np.zeros(c["steps"])
        w[-max(1, c["steps"] // 4):] = 1.0
        state["weights"] = w
        ids = g.id_count()
        state["out"] = {k: torch.empty(s, dtype=torch.float64, pin_memory=True).numpy()
                        for names, s in ((PARTS, ids), (FIELDS, g.G)) for k in names}
    return state


def run(state):
    c, g = state["case"], state["g"]
    if c["kind"] == "grad":
        if state["again"]:
            g.rewind()
        state["again"] = True
        W = g.forward_record(c["steps"], c["ckpt"])
        return {"energy": W, "grad": g.adjoint(weights=state["weights"], out=state["out"])}
    W = g.run(state["nt"], c["steps"])
    state["nt"] += c["steps"]
    if c["kind"] == "run":
        out = {"energy": W, "fields": [g.get_field(k) for k in range(6)]}
        if c["form"] == "f64":
            out["counts"] = g.cell_counts()
        return out
    return {"energy": W,
            "cells": {"%s%d" % (op, s): g.cell_moments(s, op) for s in range(3) for op in OPS},
            "gauss": g.gauss_residual(want_array=True)[1],
            "moments": g.moments()}


def work(case):
    """Bytes: every step reads and writes each particle's position and momentum
    and each field once (E and H read and written; the current is made and used
    in a step); the results are written once.  The reverse sweep reads the
    particles and the fields of each step and reads and writes their adjoints
    (FP64), besides a forward run; the diagnostics read each particle and E once.
    Operations: about 300 a particle and step (gather 120, push 80, deposit 100),
    twice that in the reverse sweep."""
    c = case
    w = 8 if c["form"] == "f64" else 4
    P, N = _particles(c), c["nx"] * c["ny"] * c["nz"]
    step_b, step_f = P * 12 * w + N * 12 * w, P * 300 + N * 60
    b, f = c["steps"] * step_b, c["steps"] * step_f
    if c["kind"] == "run":
        b += N * 6 * 8
    elif c["kind"] == "grad":
        b += c["steps"] * (P * (6 * w + 96) + N * (6 * w + 96)) + (6 * P + 6 * N) * 8
        f += c["steps"] * (P * 600 + N * 100)
    else:
        b += P * 6 * w + N * 3 * w + N * 25 * 8
        f += P * 150
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch: the step of the reference on a periodic
# box (Yee leapfrog with its ghost nodes, trilinear gather, Boris push,
# charge-conserving current of the straight path, split at the faces of the
# cells around the grid nodes)
# ---------------------------------------------------------------------------

def _pad(a, shape):
    """a with zeros behind it up to shape"""
    p = []
    for have, want in zip(reversed(a.shape), reversed(shape)):
        p += [0, want - have]
    return torch.nn.functional.pad(a, p)


def _curl_h(E, c1, shape):
    Ex, Ey, Ez = E
    qx = 0.5 * (c1[2] * (Ey[:, :-1, 1:] - Ey[:, :-1, :-1]) - c1[1] * (Ez[:, 1:, :-1] - Ez[:, :-1, :-1]))
    qy = 0.5 * (c1[0] * (Ez[1:, :, :-1] - Ez[:-1, :, :-1]) - c1[2] * (Ex[:-1, :, 1:] - Ex[:-1, :, :-1]))
    qz = 0.5 * (c1[1] * (Ex[:-1, 1:] - Ex[:-1, :-1]) - c1[0] * (Ey[1:, :-1] - Ey[:-1, :-1]))
    return [_pad(q, shape) for q in (qx, qy, qz)]


class _Box:
    """Constants of a case, and its step on plain tensors."""

    def __init__(self, c, m, qm, dev):
        self.c, self.m, self.qm = c, m, qm
        self.n = (c["nx"], c["ny"], c["nz"])
        self.shape = tuple(k + 2 for k in self.n)
        self.L = [k * H for k in self.n]
        self.h = [a / k for a, k in zip(self.L, self.n)]
        self.tau = c["tau"]
        self.c1 = [self.tau / a for a in self.h]
        self.stride = (self.shape[1] * self.shape[2], self.shape[2], 1)
        self.ghosts = 1 if c["kind"] == "grad" else 0
        self.dev = dev

    def cells(self, X):
        return [torch.clamp((x.detach() / h).floor(), 0, k - 1) for x, h, k in zip(X, self.h, self.n)]

    def gather(self, F, cell, o, rd, centre):
        """F at the particles; centre[d]: its values lie at the cells' centres along d"""
        base, far = 0, []
        for d in range(3):
            base = base + (cell[d] + rd[d] if centre[d] else cell[d]).long() * self.stride[d]
            far.append(o[d] + 0.5 - rd[d] if centre[d] else o[d])
        F, total = F.reshape(-1), 0.0
        for k in range(8):
            at, w = base, 1.0
            for d in range(3):
                one = (k >> d) & 1
                at = at + one * self.stride[d]
                w = w * (far[d] if one else 1.0 - far[d])
            total = total + w * F[at]
        return total

    def segment(self, J, cell, r, a, b):
        """adds the current of the straight path a -> b inside the dual cell r"""
        base = sum((cell[d] + r[d]).long() * self.stride[d] for d in range(3))
        D = [y - x for x, y in zip(a, b)]
        mid = [0.5 * (x + y) - (k - 0.5) for x, y, k in zip(a, b, r)]
        for d in range(3):
            e, f = [q for q in range(3) if q != d]
            q = self.m * self.h[d] / self.tau * D[d]
            s = D[e] * D[f] / 12.0
            for i in range(2):
                for j in range(2):
                    w = (mid[e] if i else 1.0 - mid[e]) * (mid[f] if j else 1.0 - mid[f])
                    w = w + s if i == j else w - s
                    J[d] = J[d].index_add(0, base + i * self.stride[e] + j * self.stride[f], q * w)

    def fold(self, J):
        J = [j.reshape(self.shape).clone() for j in J]
        for axis in range(3):
            for d in range(3):
                a = J[d].movedim(axis, 0)
                last = a.shape[0] - 1
                if axis != d:
                    a[1] = a[1] + a[last]
                if axis != 1 or d != 1:
                    a[last] = a[1]
                a[0] = a[0] + a[last - 1]
                a[last - 1] = a[0]
        return J

    def step(self, X, P, E, Hf):
        tau, h = self.tau, self.h
        Q = _curl_h(E, self.c1, self.shape)
        Hf = [a + q for a, q in zip(Hf, Q)]
        cell = self.cells(X)
        o = [x / a - k for x, a, k in zip(X, h, cell)]
        rd = [(q.detach() >= 0.5).to(q.dtype) for q in o]
        at = [self.gather(F, cell, o, rd, k) for F, k in
              zip(E + Hf, ((0, 1, 1), (1, 0, 1), (1, 1, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)))]
        t1 = self.qm * tau * 0.5
        p = [a + t1 * e for a, e in zip(P, at[:3])]
        ps = t1 / torch.sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2] + 1.0)
        b = [ps * a for a in at[3:]]
        s = [p[0] + p[1] * b[2] - p[2] * b[1], p[1] + p[2] * b[0] - p[0] * b[2],
             p[2] + p[0] * b[1] - p[1] * b[0]]
        bs = b[0] * s[0] + b[1] * s[1] + b[2] * s[2]
        sb = [s[1] * b[2] - s[2] * b[1], s[2] * b[0] - s[0] * b[2], s[0] * b[1] - s[1] * b[0]]
        den = 1.0 + b[0] * b[0] + b[1] * b[1] + b[2] * b[2]
        P = [(s[d] + bs * b[d] + sb[d]) / den + t1 * at[d] for d in range(3)]
        gi = 1.0 / torch.sqrt(P[0] * P[0] + P[1] * P[1] + P[2] * P[2] + 1.0)
        dX = [tau * gi * q for q in P]
        du = [a / k for a, k in zip(dX, h)]
        o1 = [a + k for a, k in zip(o, du)]
        # the current: one straight piece, or two that meet on the crossed faces
        r1 = [(a.detach() + 0.5).floor() for a in o1]
        cr = [(a != k) for a, k in zip(rd, r1)]
        many = sum(k.long() for k in cr)
        on = (many > 0) & (many < 3)
        zero = torch.zeros_like(o[0])
        num = sum(torch.where(cr[d], (0.5 - o[d]) * du[d] * h[d] ** 2, zero) for d in range(3))
        den = sum(torch.where(cr[d], du[d] * du[d] * h[d] ** 2, zero) for d in range(3))
        sr = torch.where(on, num, zero) / torch.where(on, den, torch.ones_like(zero))
        meet = [torch.where(cr[d], torch.full_like(zero, 0.5), o[d] + du[d] * sr) for d in range(3)]
        split = many > 0
        J = [torch.zeros(self.shape, dtype=zero.dtype, device=self.dev).reshape(-1) for _ in range(3)]
        self.segment(J, cell, rd, o, [torch.where(split, a, k) for a, k in zip(meet, o1)])
        self.segment(J, cell, r1, [torch.where(split, a, k) for a, k in zip(meet, o1)], o1)
        J = self.fold(J)
        X1 = [x + a for x, a in zip(X, dX)]
        X = [torch.where(x > a, x - a, torch.where(x < 0, x + a, x)) for x, a in zip(X1, self.L)]
        # fields
        Hf = [a + q for a, q in zip(Hf, Q)]
        c1 = self.c1
        E = [e.clone() for e in E]
        Hx, Hy, Hz = Hf
        N = [k + 1 for k in self.n]
        E[0][:N[0], 1:N[1], 1:N[2]] += (
            c1[1] * (Hz[:N[0], 1:N[1], 1:N[2]] - Hz[:N[0], :N[1] - 1, 1:N[2]]) -
            c1[2] * (Hy[:N[0], 1:N[1], 1:N[2]] - Hy[:N[0], 1:N[1], :N[2] - 1]) -
            tau * J[0][:N[0], 1:N[1], 1:N[2]])
        E[1][1:N[0], :N[1], 1:N[2]] += (
            c1[2] * (Hx[1:N[0], :N[1], 1:N[2]] - Hx[1:N[0], :N[1], :N[2] - 1]) -
            c1[0] * (Hz[1:N[0], :N[1], 1:N[2]] - Hz[:N[0] - 1, :N[1], 1:N[2]]) -
            tau * J[1][1:N[0], :N[1], 1:N[2]])
        E[2][1:N[0], 1:N[1], :N[2]] += (
            c1[0] * (Hy[1:N[0], 1:N[1], :N[2]] - Hy[:N[0] - 1, 1:N[1], :N[2]]) -
            c1[1] * (Hx[1:N[0], 1:N[1], :N[2]] - Hx[1:N[0], :N[1] - 1, :N[2]]) -
            tau * J[2][1:N[0], 1:N[1], :N[2]])

        def wrap(a, axis):
            a = a.movedim(axis, 0)
            a[0] = a[a.shape[0] - 2]
            a[a.shape[0] - 1] = a[1]

        # the reference's ghost copies: y along x, z along x, x along z, y along z
        wrap(E[1][:, :N[1], 1:N[2]], 0)
        wrap(E[2][:, 1:N[1], :N[2]], 0)
        wrap(E[0][:N[0]], 2)
        wrap(E[1][:, :N[1]], 2)
        if self.ghosts:
            wrap(E[0], 1)
            wrap(E[2], 1)
        W = sum((e * e).sum() for e in E)
        return X, P, E, Hf, W


def _start(c, seed, dev):
    sp = _host_species(c, seed)
    cols = [torch.from_numpy(np.concatenate([s[1 + k] for s in sp])).to(dev) for k in range(6)]
    lens = [len(s[1]) for s in sp]
    m = torch.cat([torch.full((k,), s[7], dtype=torch.float64) for s, k in zip(sp, lens)]).to(dev)
    qm = torch.cat([torch.full((k,), s[8], dtype=torch.float64) for s, k in zip(sp, lens)]).to(dev)
    sort = torch.cat([torch.full((k,), s[0], dtype=torch.int64) for s, k in zip(sp, lens)]).to(dev)
    box = _Box(c, m, qm, dev)
    E = [torch.zeros(box.shape, dtype=torch.float64, device=dev) for _ in range(3)]
    Hf = [torch.zeros_like(e) for e in E]
    Hf[0] += c["bx0"]
    return box, sort, cols[:3], cols[3:], E, Hf


def _diagnostics(box, sort, X, P, E):
    NC = box.n[0] * box.n[1] * box.n[2]
    cell = box.cells(X)
    at = ((cell[0] * box.n[1] + cell[1]) * box.n[2] + cell[2]).long()
    gm = torch.sqrt(1.0 + P[0] ** 2 + P[1] ** 2 + P[2] ** 2)
    kin = box.m / box.qm * (P[0] ** 2 + P[1] ** 2 + P[2] ** 2) / (gm + 1.0)
    cells, moments = {}, []
    for s in range(3):
        k = sort == s

        def per_cell(v):
            return torch.zeros(NC, dtype=v.dtype, device=v.device).index_add(0, at[k], v[k])

        num = per_cell(torch.ones_like(gm))
        u = [p / gm for p in P]
        cells["density%d" % s] = per_cell(box.m)
        cells["kinetic_energy%d" % s] = per_cell(kin)
        cells["velocity%d" % s] = torch.stack([per_cell(a) / num.clamp(min=1) for a in u])
        cells["current%d" % s] = torch.stack([per_cell(box.m * a) for a in u])
        moments.append(torch.stack([k.sum().double()] + [a[k].sum() for a in (*X, *P)] +
                                   [kin[k].sum(), sum(p[k].abs().sum() for p in P)]))
    # charge on the lattice of the cells' centres, shared among the eight nearest
    rho = torch.zeros(NC, dtype=gm.dtype, device=gm.device)
    lo = [(x / h - 0.5).floor() for x, h in zip(X, box.h)]
    far = [x / h - 0.5 - k for x, h, k in zip(X, box.h, lo)]
    for q in range(8):
        w, idx = box.m, 0
        for d in range(3):
            one = (q >> d) & 1
            w = w * (far[d] if one else 1.0 - far[d])
            idx = idx * box.n[d] + torch.remainder(lo[d] + one, box.n[d])
        rho = rho.index_add(0, idx.long(), w)
    div = sum((e[1:-1, 1:-1, 1:-1] - e.roll(1, d)[1:-1, 1:-1, 1:-1]) / box.h[d]
              for d, e in enumerate(E))
    return cells, div.reshape(-1) - rho, torch.stack(moments)


def exact(case, seed):
    c = case
    if c["source"] != "host" or _particles(c) * c["steps"] > 1.2e8:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    box, sort, X, P, E, Hf = _start(c, seed, dev)
    if c["kind"] != "grad":
        W = []
        with torch.no_grad():
            for _ in range(c["steps"]):
                X, P, E, Hf, w = box.step(X, P, E, Hf)
                W.append(w)
            W = torch.stack(W)
            if c["kind"] == "run":
                out = {"energy": W, "fields": [f.reshape(-1) for f in E + Hf]}
                if c["form"] == "f64":
                    out["counts"] = None
                return out
            cells, gauss, moments = _diagnostics(box, sort, X, P, E)
            return {"energy": W, "cells": cells, "gauss": gauss, "moments": moments}
    leaves = [a.requires_grad_() for a in X + P + E + Hf]
    state, W = list(leaves), []
    for _ in range(c["steps"]):
        def one(*a):
            X, P, E, Hf, w = box.step(list(a[:3]), list(a[3:6]), list(a[6:9]), list(a[9:]))
            return (*X, *P, *E, *Hf, w)
        *state, w = checkpoint(one, *state, use_reentrant=False)
        W.append(w)
    W = torch.stack(W)
    W[-max(1, c["steps"] // 4):].sum().backward()
    grads = {k: a.grad.reshape(-1) for k, a in zip(PARTS + FIELDS, leaves)}
    return {"energy": W.detach(), "grad": grads}
