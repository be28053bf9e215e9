"""Performance cases of the phase-field framework: what its users run, through
the host classes and the C ABI.

A case is a dict of plain values. `listed()` names the fixed ones, `draw(rng)`
gives another of the same ranges; `prepare` builds what a program holds before
the call, `run` makes one pass, `work` is the traffic and arithmetic the pass
cannot do without, `exact` is the same pass in 64-bit torch.

The 2D and 3D steps are specified bit for bit (binary32 fields in a fixed
operation order, Q5.27 integer aggregates, fixed-order fp64 reductions), so
their tolerance is "exact". The learned surrogate computes in bfloat16 with
binary32 sums; its tolerances are four times the difference seen between the
kernels and the same network with unrounded activations.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = Path(__file__).resolve().parent.parent / "phase-field-gh200_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

from pfh import abi, ensemble, params, params3d, sim2d, sim3d  # noqa: E402
from pfh import surrogate as su  # noqa: E402

DEV = "cuda:0"
TILE = 288
CROP = su.CROP
# active window (width, height, tile column, tile row) of each shape class
CLASSES = ((144, 144, 64, 64), (176, 144, 32, 64), (144, 176, 64, 32),
           (160, 160, 32, 32), (224, 224, 32, 32), (286, 286, 1, 1))


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a handful of cells, single launches: latency of one step
        {"name": "step2d_few", "kind": "step2d", "N": 16, "L": 384, "R": 20.0, "steps": 1,
         "graph": False, "observe": 0},
        # the headline 2D monolayer, one six-step graph replay
        {"name": "step2d_monolayer", "kind": "step2d", "N": 1024, "L": 2048, "R": 20.0,
         "steps": 6, "graph": True, "observe": 0},
        # the default population of large cells at 90% packing (odd side)
        {"name": "step2d_large_cells", "kind": "step2d", "N": 288, "L": 1554, "R": 49.0,
         "steps": 6, "graph": True, "observe": 0},
        # a step sampled by the spatial velocity observer
        {"name": "step2d_observed", "kind": "step2d", "N": 256, "L": 1024, "R": 20.0,
         "steps": 1, "graph": False, "observe": 2},
        # a batch of independent replicas advanced by one launch
        {"name": "ensemble", "kind": "ensemble", "replicas": 64, "steps": 1},
        # few small 3D cells: latency of the three launches of a step
        {"name": "step3d_few", "kind": "step3d", "N": 8, "L": 96, "R": 8.0, "lam": 3.5,
         "B": 48, "steps": 1, "graph": False},
        # the headline 3D population, one two-step graph replay
        {"name": "step3d_population", "kind": "step3d", "N": 128, "L": 256, "R": 12.0,
         "lam": 3.5, "B": 56, "steps": 2, "graph": True},
        # more cells in the largest bricks on an odd side
        {"name": "step3d_large_bricks", "kind": "step3d", "N": 224, "L": 331, "R": 13.0,
         "lam": 3.5, "B": 64, "steps": 1, "graph": False},
        # the network alone on every cell of the monolayer (forward)
        {"name": "surrogate_infer", "kind": "infer", "N": 1024, "L": 2048, "R": 20.0},
        # one checked 8-step surrogate block of the monolayer
        {"name": "surrogate_block", "kind": "block", "N": 1024, "L": 2048, "R": 20.0},
        # one training step on a minibatch: forward, backward, Adam
        {"name": "surrogate_train", "kind": "train", "batch": 128},
        # a fresh population: fields, moments, aggregate, queue order, records
        {"name": "setup2d", "kind": "setup2d", "N": 1024, "L": 2048, "R": 20.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side2d(rng, N, R):
    rho = rng.uniform(0.3, 0.9)
    return max(287, math.ceil(math.sqrt(N * math.pi * R * R / rho)))


def draw(rng):
    kind = rng.choice(["step2d", "step2d", "step2d", "ensemble", "step3d", "step3d", "step3d",
                       "infer", "block", "train", "setup2d"])
    if kind == "step2d":
        observe = rng.choice([0, 0, 0, 1, 2])
        N = _log_int(rng, 5, 1024)
        R = round(rng.uniform(14.0, 49.0), 1)
        graph = observe == 0 and rng.random() < 0.7
        return {"kind": kind, "N": N, "L": _side2d(rng, N, R), "R": R,
                "steps": 6 if graph else 1, "graph": graph, "observe": observe}
    if kind == "ensemble":
        return {"kind": kind, "replicas": _log_int(rng, 3, 60), "steps": 1}
    if kind == "step3d":
        N = _log_int(rng, 3, 200)
        R = round(rng.uniform(8.0, 13.0), 1)
        # the automatic edge has no slack for the relaxing tail: at least 8 more
        B = min(64, 8 * math.ceil((2.0 * R + 24.0) / 8.0) + rng.choice([8, 16]))
        rho = rng.uniform(0.03, 0.08)
        L = max(B + 17, math.ceil((N * 4.0 / 3.0 * math.pi * R ** 3 / rho) ** (1.0 / 3.0)))
        graph = rng.random() < 0.6
        return {"kind": kind, "N": N, "L": L, "R": R, "lam": 3.5, "B": B,
                "steps": 2 if graph else 1, "graph": graph}
    if kind == "train":
        return {"kind": kind, "batch": _log_int(rng, 9, 128)}
    N = _log_int(rng, 40, 1024)
    R = round(rng.uniform(16.0, 24.0), 1)
    return {"kind": kind, "N": N, "L": _side2d(rng, N, R), "R": R}


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
def _monolayer(N, L, R, seed):
    g = math.ceil(math.sqrt(N))
    return params.monolayer(N, L, R, g, 0.0625 * L / g, seed % (1 << 31))


def _sim2d(case, seed, warm, graph=True):
    """A relaxed monolayer: the initial profiles after `warm` plain steps."""
    sim = sim2d.Sim2D(_monolayer(case["N"], case["L"], case["R"], seed), device=DEV)
    if graph:
        sim.capture_graph()
    sim.run(warm)
    return sim


def _replicas(case, seed):
    """The benchmark ensemble's sides and populations, with the seed's
    placements and Philox streams."""
    return [params.ensemble_replica(wl.params.Nx, wl.params.num_cells, seed % (1 << 30) + r)
            for r, wl in enumerate(params.ensemble_c4(replicas=case["replicas"]))]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step2d":
        sim = _sim2d(case, seed, 60, case["graph"])
        if case["observe"] == 2:
            sim.attach_moments()
        return {"kind": kind, "sim": sim, "steps": case["steps"], "observe": case["observe"]}
    if kind == "ensemble":
        sim = ensemble.Ensemble2D(_replicas(case, seed), device=DEV)
        sim.run(24)
        return {"kind": kind, "sim": sim, "steps": case["steps"]}
    if kind == "step3d":
        wl = params3d.workload("population", case["N"], case["R"], case["lam"], case["L"],
                               seed=seed % (1 << 31), brick_edge_override=case["B"])
        sim = sim3d.Sim3D(wl, device=DEV)
        if case["graph"]:
            sim.capture_graph()
        sim.run(60)
        return {"kind": kind, "sim": sim, "steps": case["steps"]}
    if kind == "infer":
        sim = _sim2d(case, seed, 60)
        net = su.Net.load(device=DEV)
        w4, b4 = su.deploy_weights(net)
        return {"kind": kind, "sim": sim, "net": net, "w4": w4, "b4": b4,
                "ws": su.Workspace(sim.N, sim.dev, hidden=False)}
    if kind == "block":
        sim = _sim2d(case, seed, 300)
        runner = su.SurrogateRunner(sim, su.Net.load(device=DEV))
        runner.prepare()
        return {"kind": kind, "sim": sim, "runner": runner}
    if kind == "train":
        n = case["batch"]
        sim = _sim2d({"N": n, "L": max(287, 64 * math.ceil(math.sqrt(n))), "R": 20.0}, seed, 300)
        net = su.Net.load(device=DEV)
        ws = su.Workspace(n, sim.dev, train=True)
        su.crop_sim(sim, ws)
        after = torch.zeros_like(ws.phic)
        sim.run(net.K)
        su.recrop_sim(sim, ws.origin, after)
        return {"kind": kind, "net": net, "ws": ws, "n": n,
                "target": (after - ws.phic) / net.scale}
    # setup2d
    wl = _monolayer(case["N"], case["L"], case["R"], seed)
    sim = sim2d.Sim2D(wl, device=DEV)
    cells = torch.from_numpy(sim.host_cells().view(np.uint8).reshape(-1).copy()).to(DEV)
    sim.cell.copy_(cells)
    return {"kind": kind, "sim": sim, "wl": wl,
            "cx": torch.from_numpy(wl.cx).to(DEV), "cy": torch.from_numpy(wl.cy).to(DEV),
            "traj": torch.zeros(sim.N * abi.TRAJ_DTYPE.itemsize, dtype=torch.uint8, device=DEV)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _fields2d(sim):
    return {"phi": sim.phi[sim.steps_done % 2], "S": sim.S_slot(sim.steps_done % 3),
            "cells": sim.cell, "classes": sim.cls, "flags": sim.flags}


def run(state):
    kind = state["kind"]
    if kind == "step2d":
        sim = state["sim"]
        if state["observe"]:
            sim.step(state["steps"], state["observe"])
        else:
            sim.run(state["steps"])
        out = _fields2d(sim)
        if state["observe"] == 2:
            out["moments"] = sim.moments
        return out
    if kind == "ensemble":
        sim = state["sim"]
        sim.run(state["steps"])
        s = sim.steps_done % 3
        return {"phi": sim.phi[sim.steps_done % 2],
                "S": sim.S[s * sim.words:(s + 1) * sim.words], "cells": sim.cell,
                "classes": sim.cls, "flags": sim.flags}
    if kind == "step3d":
        sim = state["sim"]
        sim.run(state["steps"])
        s = sim.steps_done % 2
        return {"phi": sim.phi[s], "S": sim.S[s], "cells": sim.cell, "flags": sim.flags}
    if kind == "infer":
        ws = state["ws"]
        su.infer_cells(state["net"], state["sim"], ws, W4=state["w4"], b4=state["b4"])
        return {"dphi": ws.dphi, "pred": ws.pred, "origin": ws.origin}
    if kind == "block":
        state["runner"].run(state["runner"].K)
        return dict(_fields2d(state["sim"]), pred=state["runner"].ws.pred)
    if kind == "train":
        net, ws, n = state["net"], state["ws"], state["n"]
        su.forward(net, ws, n, pred=False)
        loss = su.backward(net, ws, n, state["target"])
        su.adam_step(net, 1e-3)
        return {"dphi": ws.dphi, "loss": loss, "grad": net.g, "weights": net.w}
    # setup2d
    sim, p = state["sim"], state["wl"].params
    lib, sp = sim.lib, sim._sp()
    phi0, phi1 = sim.phi[0].data_ptr(), sim.phi[1].data_ptr()
    cell, cls, perm = sim.cell.data_ptr(), sim.cls.data_ptr(), sim.perm.data_ptr()
    S, flags, N, L, P = sim.S.data_ptr(), sim.flags.data_ptr(), sim.N, sim.L, sim.P
    abi.check(lib.pfh2d_zero_u32(S, sim.words, sp), "pfh2d_zero_u32")
    abi.check(lib.pfh2d_init_tiles(phi0, phi1, cell, cls, N, L, state["cx"].data_ptr(),
                                   state["cy"].data_ptr(), ctypes.c_float(p.init_radius()).value,
                                   ctypes.c_float(p.interface_k()).value, sp),
              "pfh2d_init_tiles")
    abi.check(lib.pfh2d_init_moments(cell, cls, phi0, N, sp), "pfh2d_init_moments")
    abi.check(lib.pfh2d_scatter_all(phi0, cell, cls, S, N, L, P, flags, sp), "pfh2d_scatter_all")
    abi.check(lib.pfh2d_morton_sort(cell, perm, N, 1 << (N - 1).bit_length(), L, sp),
              "pfh2d_morton_sort")
    abi.check(lib.pfh2d_pack_traj(cell, cls, state["traj"].data_ptr(), N, L, sp),
              "pfh2d_pack_traj")
    return {"phi": sim.phi[0], "other": sim.phi[1], "S": sim.S_slot(0), "cells": sim.cell,
            "perm": sim.perm, "traj": state["traj"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
_W0 = 144 * 144            # window of the round class


def _q2(R):
    """Pixels of a 2D cell with a nonzero quantised square (lambda = 7)."""
    return min(_W0, math.pi * (R + 13.7) ** 2)


def _step2d_bytes(N, L, R):
    P = 32 * math.ceil(L / 32)
    return N * (12.0 * _W0 + 8.0 * _q2(R)) + 4.0 * P * L


# multiply-adds of the three 3x3 hidden layers and the output layer per pixel
_NET_MAC = 9 * (4 * 32 + 32 * 32 + 32 * 32 + 32)


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        b = f = 0.0
        for wl in _replicas(case, 100):
            b += _step2d_bytes(wl.params.num_cells, wl.params.Nx, 20.0)
            f += 60.0 * _W0 * wl.params.num_cells
        return {"bytes": case["steps"] * b, "flops": case["steps"] * f}
    if kind == "step3d":
        vox = case["N"] * float(case["B"]) ** 3
        q3 = case["N"] * min(float(case["B"]) ** 3, 4.0 / 3.0 * math.pi * (case["R"] + 6.9) ** 3)
        L = case["L"]
        per = 16.0 * vox + 8.0 * q3 + 4.0 * 32 * math.ceil(L / 32) * L * L
        return {"bytes": case["steps"] * per, "flops": case["steps"] * 110.0 * vox}
    if kind == "train":
        n, pix = case["batch"], CROP * CROP
        # forward, data gradient and weight gradient of each layer
        return {"bytes": n * pix * (2.0 * 8 + 4.0 + 4.0) + 4.0 * 8 * su.NPARAM,
                "flops": 2.0 * n * pix * (3 * _NET_MAC - 9 * 4 * 32)}
    N, L, R = case["N"], case["L"], case["R"]
    if kind == "step2d":
        return {"bytes": case["steps"] * _step2d_bytes(N, L, R),
                "flops": case["steps"] * 60.0 * _W0 * N}
    infer = {"bytes": N * 4.0 * (_W0 + CROP * CROP) + 4.0 * L * L,
             "flops": 2.0 * N * CROP * CROP * _NET_MAC}
    if kind == "infer":
        return {"bytes": infer["bytes"] + N * 4.0 * CROP * CROP, "flops": infer["flops"]}
    if kind == "block":
        return {"bytes": infer["bytes"] + _step2d_bytes(N, L, R),
                "flops": infer["flops"] + 60.0 * _W0 * N}
    # setup2d: both tiles and the aggregate written, the window read back
    return {"bytes": N * (8.0 * TILE * TILE + 4.0 * _W0 + 8.0 * _q2(R)) + 4.0 * L * L,
            "flops": 60.0 * _W0 * N}


def tolerance(case):
    kind = case["kind"]
    if kind == "infer":
        return {"rel": 2e-2, "max": 0.5}
    if kind == "block":
        # cells whose check error lies at a threshold may change sides
        return {"rel": 1e-4, "max": 0.1, "differ": 0.01}
    if kind == "train":
        return {"rel": 2e-2, "max": 0.5}
    return "exact"


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 on numpy arrays of counters."""
    c = [np.asarray(v, np.uint64) & np.uint64(0xFFFFFFFF) for v in
         np.broadcast_arrays(c0, c1, c2, c3)]
    k0, k1 = key & 0xFFFFFFFF, (key >> 32) & 0xFFFFFFFF
    m = np.uint64(0xFFFFFFFF)
    for rnd in range(10):
        if rnd:
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m]
    return c


def _u53(a, b):
    return (((a << np.uint64(32)) | b) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _containing(ex, ey, slack):
    best, area = -1, 0
    for c, (wx, wy, _, _) in enumerate(CLASSES):
        if ex + slack <= wx and ey + slack <= wy and (best < 0 or wx * wy < area):
            best, area = c, wx * wy
    return best


class _Mono64:
    """The 2D population in 64 bits: a state taken from the device buffers,
    then plain steps in torch double."""

    def __init__(self, p, phi, S, cells, step, offset=0):
        f = lambda k: torch.from_numpy(cells[k].astype(np.float64)).to(DEV)  # noqa: E731
        self.p, self.L, self.N, self.step_no = p, p.Nx, len(cells), step
        self.phi = phi.view(-1, TILE, TILE)[offset:offset + self.N].double()
        P = S.numel() // self.L
        self.S = (S.view(self.L, P)[:, :self.L].long() & 0xFFFFFFFF).double() * 2.0 ** -27
        self.gx, self.gy = cells["gx0"].astype(np.int64), cells["gy0"].astype(np.int64)
        self.cls = cells["cls"].astype(np.int64)
        self.gid = cells["global_id"].astype(np.uint64)
        self.theta = cells["theta"].astype(np.float64)
        self.V, self.Cx, self.Cy = (cells[k].astype(np.float64) for k in ("V", "Cx", "Cy"))
        self.box = np.stack([cells[k].astype(np.int64) for k in
                             ("bb_lo_x", "bb_hi_x", "bb_lo_y", "bb_hi_y")], 1)
        self.pctr = cells["promote_ctr"].astype(np.int64)
        self.gamma, self.vA, self.M = f("gamma"), cells["v_A"].astype(np.float64), f("M_pf")
        self.t = torch.arange(TILE, device=DEV)

    def _geom(self, cls):
        g = np.array(CLASSES)[cls]
        wx, wy, tx, ty = (torch.from_numpy(g[:, i].copy()).to(DEV)[:, None] for i in range(4))
        inx = (self.t >= tx) & (self.t < tx + wx)
        iny = (self.t >= ty) & (self.t < ty + wy)
        return tx, ty, inx, iny

    def _world(self, cls):
        """World column and row index of every tile column and row."""
        tx, ty, inx, iny = self._geom(cls)
        gx, gy = (torch.from_numpy(v).to(DEV)[:, None] for v in (self.gx, self.gy))
        return (self.t - tx + gx) % self.L, (self.t - ty + gy) % self.L, inx, iny

    def _plan(self, cls):
        """Class and shift of the step (hysteresis, recentring)."""
        dcls, sx, sy = cls.copy(), np.zeros(self.N, np.int64), np.zeros(self.N, np.int64)
        for n in range(self.N):
            wx, wy = CLASSES[cls[n]][:2]
            lo_x, hi_x, lo_y, hi_y = self.box[n]
            ex, ey = hi_x - lo_x + 1, hi_y - lo_y + 1
            if ex > 0:
                if ex + 8 > wx or ey + 8 > wy:
                    g = _containing(ex, ey, 8)
                    if g >= 0 and max(CLASSES[g][:2]) < self.L:
                        dcls[n] = g
                    self.pctr[n] = 0
                else:
                    s = _containing(ex, ey, 20)
                    if s >= 0 and s != cls[n] and CLASSES[s][0] * CLASSES[s][1] < wx * wy:
                        self.pctr[n] += 1
                        if self.pctr[n] >= 200:
                            dcls[n], self.pctr[n] = s, 0
                    else:
                        self.pctr[n] = 0
            dwx, dwy = CLASSES[dcls[n]][:2]
            sx[n] = round(self.Cx[n] / self.V[n] - 0.5 * (dwx - 1))
            sy[n] = round(self.Cy[n] / self.V[n] - 0.5 * (dwy - 1))
            lx, ly = (4, 4) if dcls[n] == cls[n] else (wx, wy)
            sx[n], sy[n] = max(-lx, min(lx, sx[n])), max(-ly, min(ly, sy[n]))
        return dcls, sx, sy

    def step(self, dt=None, scatter=True):
        p, N = self.p, self.N
        dt = float(np.float32(p.dt if dt is None else dt))
        cls = self.cls
        r = _philox(self.step_no & 0xFFFFFFFF, self.step_no >> 32, self.gid, 0xA5A5A5A5,
                    p.polarity_stream())
        tum = _u53(r[0], r[1]) < p.p_tumble()
        theta = np.where(tum, np.float32(2.0 * math.pi * _u53(r[2], r[3])), self.theta)
        dcls, sx, sy = self._plan(cls)
        X, Y, inx, iny = self._world(cls)
        bulk, rep = float(np.float32(p.bulk())), float(np.float32(p.interaction()))
        mot = float(np.float32(p.motility()))
        vol = torch.from_numpy(p.volume() * (p.area0() - self.V)).to(DEV)
        new = torch.zeros_like(self.phi)
        for a in range(0, N, 128):
            b = min(N, a + 128)
            pad = torch.nn.functional.pad(self.phi[a:b], (1, 1, 1, 1))
            c = pad[:, 1:-1, 1:-1]
            e, w, n, s = pad[:, 1:-1, 2:], pad[:, 1:-1, :-2], pad[:, 2:, 1:-1], pad[:, :-2, 1:-1]
            lap = (4.0 * (n + s + e + w) + pad[:, 2:, 2:] + pad[:, 2:, :-2] + pad[:, :-2, 2:]
                   + pad[:, :-2, :-2] - 20.0 * c) / 6.0
            other = (self.S[Y[a:b, :, None], X[a:b, None, :]] - c * c).clamp_(min=0.0)
            mask = inx[a:b, None, :] & iny[a:b, :, None]
            gx, gy = 0.5 * (e - w), 0.5 * (n - s)
            co = c * other * mask
            Ix, Iy = (co * gx).sum((1, 2)), (co * gy).sum((1, 2))
            th = torch.from_numpy(theta[a:b].astype(np.float64)).to(DEV)
            vA = torch.from_numpy(self.vA[a:b]).to(DEV)
            vx = (vA * torch.cos(th) + mot * Ix)[:, None, None]
            vy = (vA * torch.sin(th) + mot * Iy)[:, None, None]
            gam = self.gamma[a:b, None, None]
            rhs = (gam * lap - bulk * gam * (c * (1.0 - c) * (1.0 - 2.0 * c))
                   + vol[a:b, None, None] * c - rep * c * other)
            mrel = (self.M[a:b] / 0.5)[:, None, None]
            new[a:b] = (c + dt * (mrel * rhs - (vx * gx + vy * gy))) * mask
        # the shift: source window pixel (x, y) goes to (x - sx, y - sy)
        tab = np.array(CLASSES)
        ddx = tab[dcls, 2] - tab[cls, 2] - sx
        ddy = tab[dcls, 3] - tab[cls, 3] - sy
        for n in np.nonzero((ddx != 0) | (ddy != 0))[0]:
            moved = torch.zeros_like(new[n])
            dx, dy = int(ddx[n]), int(ddy[n])
            src = new[n, max(0, -dy):TILE - max(0, dy), max(0, -dx):TILE - max(0, dx)]
            moved[max(0, dy):TILE + min(0, dy), max(0, dx):TILE + min(0, dx)] = src
            new[n] = moved
        self.gx, self.gy = (self.gx + sx) % self.L, (self.gy + sy) % self.L
        self.cls, self.theta = dcls, theta
        self.step_no += 1
        self._commit(new, scatter)

    def _commit(self, new, scatter):
        """Window zeros, moments, support and the aggregate of the new field."""
        tx, ty, inx, iny = self._geom(self.cls)
        X, Y, _, _ = self._world(self.cls)
        new *= inx[:, None, :] & iny[:, :, None]
        self.phi = new
        if not scatter:
            return
        S = torch.zeros(self.L * self.L, dtype=torch.float64, device=DEV)
        box = np.empty_like(self.box)
        for a in range(0, self.N, 128):
            b = min(self.N, a + 128)
            sq = new[a:b] ** 2
            col = (self.t - tx[a:b]).double()
            row = (self.t - ty[a:b]).double()
            cs, rs = sq.sum(1), sq.sum(2)
            self.V[a:b] = cs.sum(1).cpu().numpy()
            self.Cx[a:b] = (cs * col).sum(1).cpu().numpy()
            self.Cy[a:b] = (rs * row).sum(1).cpu().numpy()
            sup = new[a:b] > 1e-5
            for k, (hit, org) in enumerate(((sup.any(1), tx[a:b]), (sup.any(2), ty[a:b]))):
                i = hit.long()
                box[a:b, 2 * k] = (i.argmax(1) - org[:, 0]).cpu().numpy()
                box[a:b, 2 * k + 1] = (TILE - 1 - i.flip(1).argmax(1) - org[:, 0]).cpu().numpy()
            idx = (Y[a:b, :, None] * self.L + X[a:b, None, :]).reshape(-1)
            S.index_add_(0, idx, sq.reshape(-1))
        self.box, self.S = box, S.view(self.L, self.L)


def _cells(sim):
    return sim.cell.cpu().numpy().view(abi.CELL_DTYPE).copy()


def _mono64(sim):
    s = sim.steps_done
    return _Mono64(sim.p, sim.phi[s % 2], sim.S_slot(s % 3), _cells(sim), s)


def _crops64(m):
    """Inputs of the network (phi, S_other, cos, sin) and the crop origins
    relative to the tile, of a _Mono64 state."""
    tx, ty, _, _ = m._geom(m.cls)
    ox = np.rint(m.gx + m.Cx / m.V).astype(np.int64) - CROP // 2
    oy = np.rint(m.gy + m.Cy / m.V).astype(np.int64) - CROP // 2
    t = torch.arange(CROP, device=DEV)
    tox = torch.from_numpy(ox - m.gx).to(DEV)[:, None] + tx + t      # tile column
    toy = torch.from_numpy(oy - m.gy).to(DEV)[:, None] + ty + t
    n = torch.arange(m.N, device=DEV)[:, None, None]
    phi = m.phi[n, toy[:, :, None], tox[:, None, :]]
    wx = (torch.from_numpy(ox).to(DEV)[:, None] + t) % m.L
    wy = (torch.from_numpy(oy).to(DEV)[:, None] + t) % m.L
    other = (m.S[wy[:, :, None], wx[:, None, :]] - phi * phi).clamp(min=0.0)
    th = torch.from_numpy(m.theta).to(DEV)[:, None, None]
    x = torch.stack([phi, other, torch.cos(th).expand_as(phi), torch.sin(th).expand_as(phi)], 1)
    return x, phi, tox, toy


def _conv64(x, w, b):
    """3x3 convolution with zero padding, w [out][9][in]."""
    n, cin = x.shape[:2]
    u = torch.nn.functional.unfold(x, 3, padding=1).view(n, cin, 9, -1)
    wt = w.view(w.shape[0], 9, cin).permute(0, 2, 1).reshape(w.shape[0], cin * 9)
    y = torch.matmul(wt, u.reshape(n, cin * 9, -1))
    return (y + b[:, None]).view(n, -1, CROP, CROP)


def _net_weights(net):
    """bf16 values of the hidden layers (real channels), binary32 of the rest."""
    v = {k: t.detach().double() for k, t in net.views.items()}
    for k in ("W1", "W2", "W3"):
        v[k] = net.views[k].to(torch.bfloat16).double()
    v["W1"] = v["W1"].view(32, 9, 8)[:, :, :4].reshape(-1)
    return v


def _forward64(x, v):
    h = torch.relu(_conv64(x, v["W1"].view(32, 9, 4), v["b1"]))
    h = torch.relu(_conv64(h, v["W2"].view(32, 9, 32), v["b2"]))
    h = torch.relu(_conv64(h, v["W3"].view(32, 9, 32), v["b3"]))
    return _conv64(h, v["W4"].view(1, 9, 32), v["b4"])[:, 0]


def _infer64(x, v):
    return torch.cat([_forward64(x[a:a + 32], v) for a in range(0, len(x), 32)])


def _exact_block(state):
    """The checked block: the prediction, the explicit step of K dt, the
    per-cell rule."""
    runner, sim = state["runner"], state["sim"]
    m = _mono64(sim)
    x, phi_c, tox, toy = _crops64(m)
    pred = phi_c + _infer64(x, _net_weights(runner.net)) * runner.net.scale
    del x
    now, cls0, gx0, gy0 = m.phi, m.cls.copy(), m.gx.copy(), m.gy.copy()
    m.step(dt=sim.p.dt * runner.K, scatter=False)
    out = now.clone()
    tab = np.array(CLASSES)
    n = torch.arange(m.N, device=DEV)[:, None, None]
    full = torch.zeros_like(now)
    full[n, toy[:, :, None], tox[:, None, :]] = pred
    # the check field in the frame of the current window
    chk = m.phi.clone()
    fx = tab[cls0, 2] + (m.gx - gx0 + m.L // 2) % m.L - m.L // 2 - tab[m.cls, 2]
    fy = tab[cls0, 3] + (m.gy - gy0 + m.L // 2) % m.L - m.L // 2 - tab[m.cls, 3]
    for i in np.nonzero((fx != 0) | (fy != 0))[0]:
        chk[i] = torch.roll(m.phi[i], (int(fy[i]), int(fx[i])), (0, 1))
    norm = lambda t: t.flatten(1).norm(dim=1)  # noqa: E731
    e = norm(full - chk) / norm(chk)
    chk_c = chk[n, toy[:, :, None], tox[:, None, :]]
    inc = norm(full - chk) / norm(chk_c - phi_c)
    take = (e <= runner.tol) & (inc <= runner.tol_inc) & \
        (runner.acc.double() + e <= runner.budget)
    _, _, inx, iny = m._geom(cls0)
    out = torch.where(take[:, None, None], full * (inx[:, None, :] & iny[:, :, None]), m.phi)
    return {"phi": out.reshape(-1), "S": None, "cells": None, "classes": None, "flags": None,
            "pred": pred.reshape(-1)}


def _exact_train(state):
    net, ws, n = state["net"], state["ws"], state["n"]
    x = ws.X0.view(torch.bfloat16).view(n, CROP, CROP, 8)[..., :4].permute(0, 3, 1, 2).double()
    tgt = state["target"].view(n, CROP, CROP).double()
    v = {k: t.requires_grad_(True) for k, t in _net_weights(net).items()}
    dphi, loss = [], 0.0
    for a in range(0, n, 8):
        y = _forward64(x[a:a + 8], v)
        part = ((y - tgt[a:a + 8]) ** 2).sum() / (n * CROP * CROP)
        part.backward()
        loss += float(part)
        dphi.append(y.detach())
    g = {k: t.grad for k, t in v.items()}
    w1 = torch.zeros(32, 9, 8, dtype=torch.float64, device=DEV)
    w1[:, :, :4] = g["W1"].view(32, 9, 4)
    g["W1"] = w1
    grad = torch.cat([g[k].reshape(-1) for k in su.ORDER])
    w = net.w.double() - 1e-3 * grad / (grad.abs() + 1e-8)     # Adam's first step
    return {"dphi": torch.cat(dphi).reshape(-1), "loss": loss, "grad": grad, "weights": w}


def _exact_step3d(state):
    sim = state["sim"]
    p, N, B, L = sim.p, sim.N, sim.B, sim.L
    s = sim.steps_done % 2
    phi = sim.phi[s].view(N, B, B, B).double()
    S = (sim.S[s].view(L, L, sim.P)[:, :, :L].long() & 0xFFFFFFFF).double() * 2.0 ** -27
    cells = sim.cells()
    org = np.stack([cells[k] for k in ("origin_z", "origin_y", "origin_x")], 1)
    pol = np.stack([cells[k] for k in ("polarity_z", "polarity_y", "polarity_x")], 1)
    pol = pol.astype(np.float64)
    gid, key = cells["global_id"].astype(np.uint64), p.polarity_stream()
    t = torch.arange(B, device=DEV)
    ic, mot = float(np.float32(p.interaction())), float(np.float32(p.motility()))
    gam = torch.from_numpy(cells["gamma"].astype(np.float64)).to(DEV)[:, None, None, None]
    vA = cells["v_A"].astype(np.float64)[:, None]
    dt, bulk = float(np.float32(p.dt)), float(np.float32(p.bulk()))
    step = int(sim.counters[0].item())
    for k in range(state["steps"]):
        st = step + k
        ev = _philox(st & 0xFFFFFFFF, st >> 32, gid, (gid >> np.uint64(32)) ^
                     np.uint64(0x54554D45), key)
        ve = _philox(st & 0xFFFFFFFF, st >> 32, gid, (gid >> np.uint64(32)) ^
                     np.uint64(0x54554D56), key)
        tum = _u53(ev[0], ev[1]) < p.p_tumble()
        z = 2.0 * _u53(ev[2], ev[3]) - 1.0
        az = 2.0 * math.pi * _u53(ve[0], ve[1])
        rad = np.sqrt(np.maximum(0.0, 1.0 - z * z))
        draw_ = np.stack([z, rad * np.sin(az), rad * np.cos(az)], 1)
        pol = np.where(tum[:, None], draw_, pol)
        new = torch.zeros_like(phi)
        Snew = torch.zeros(L * L * L, dtype=torch.float64, device=DEV)
        for n in range(N):
            f = torch.nn.functional.pad(phi[n:n + 1], (1,) * 6)[0]
            c = f[1:-1, 1:-1, 1:-1]
            iz, iy, ix = ((t + int(org[n, a])) % L for a in range(3))
            other = (S[iz[:, None, None], iy[None, :, None], ix[None, None, :]]
                     - c * c).clamp(min=0.0)
            g = [0.5 * (f[2:, 1:-1, 1:-1] - f[:-2, 1:-1, 1:-1]),
                 0.5 * (f[1:-1, 2:, 1:-1] - f[1:-1, :-2, 1:-1]),
                 0.5 * (f[1:-1, 1:-1, 2:] - f[1:-1, 1:-1, :-2])]
            sq = c * c
            V = float(sq.sum())
            hit = c.abs() > 1e-5
            co = c * other
            sh, vel = [], []
            for a in range(3):
                dims = tuple(d for d in range(3) if d != a)
                prof = sq.sum(dims)
                cen = float((prof * t).sum()) / V - 0.5 * (B - 1)
                on = torch.nonzero(hit.any(dims[1]).any(dims[0]))
                q = max(-4, min(4, round(cen)))
                if len(on):
                    q = max(min(q, int(on[0])), int(on[-1]) - (B - 1))
                sh.append(q)
                vel.append(float(vA[n, 0] * pol[n, a] + mot * float((co * g[a]).sum())))
            lap = torch.zeros_like(c)
            for dz in range(3):
                for dy in range(3):
                    for dx in range(3):
                        wgt = (-128.0, 14.0, 3.0, 1.0)[(dz != 1) + (dy != 1) + (dx != 1)]
                        lap += wgt * f[dz:dz + B, dy:dy + B, dx:dx + B]
            ga = float(gam[n])
            rhs = (ga * lap / 30.0 - bulk * ga * c * (1.0 - c) * (1.0 - 2.0 * c)
                   + p.volume() * (p.volume0() - V) * c - ic * c * other
                   - (vel[0] * g[0] + vel[1] * g[1] + vel[2] * g[2]))
            nx = c + dt * rhs
            lo = [max(0, q) for q in sh]
            hi = [B + min(0, q) for q in sh]
            new[n, lo[0] - sh[0]:hi[0] - sh[0], lo[1] - sh[1]:hi[1] - sh[1],
                lo[2] - sh[2]:hi[2] - sh[2]] = nx[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]]
            org[n] += np.array(sh)
            iz, iy, ix = ((t + int(org[n, a])) % L for a in range(3))
            idx = (iz[:, None, None] * L + iy[None, :, None]) * L + ix[None, None, :]
            Snew.index_add_(0, idx.reshape(-1), (new[n] ** 2).reshape(-1))
        phi, S = new, Snew.view(L, L, L)
    return {"phi": phi.reshape(-1), "S": None, "cells": None, "flags": None}


def _exact_setup(case, state):
    wl, L = state["wl"], case["L"]
    p = wl.params
    wx, wy, tx, ty = CLASSES[0]
    cx, cy = (torch.from_numpy(v.astype(np.float64)).to(DEV)[:, None] for v in (wl.cx, wl.cy))
    t = torch.arange(wx, device=DEV).double()
    d = []
    for c in (cx, cy):
        o = torch.round((c - 0.5 * (wx - 1)).float()).double() % L
        v = o + t - c
        v = torch.where(v > 0.5 * L, v - L, v)
        d.append(torch.where(v < -0.5 * L, v + L, v))
    r = torch.sqrt(d[0][:, None, :] ** 2 + d[1][:, :, None] ** 2)
    k, r0 = float(np.float32(p.interface_k())), float(np.float32(p.init_radius()))
    phi = torch.zeros(case["N"], TILE, TILE, dtype=torch.float64, device=DEV)
    phi[:, ty:ty + wy, tx:tx + wx] = 0.5 * (1.0 - torch.tanh(k * (r - r0)))
    return {"phi": phi.reshape(-1), "other": torch.zeros_like(phi).reshape(-1), "S": None,
            "cells": None, "perm": None, "traj": None}


def exact(case, seed):
    kind = case["kind"]
    state = prepare(case, seed)
    if kind == "step2d":
        m = _mono64(state["sim"])
        for _ in range(state["steps"]):
            m.step()
        out = {"phi": m.phi.reshape(-1), "S": None, "cells": None, "classes": None,
               "flags": None}
        return dict(out, moments=None) if case["observe"] == 2 else out
    if kind == "ensemble":
        sim = state["sim"]
        s = sim.steps_done
        out = torch.empty(sim.N, TILE, TILE, dtype=torch.float64, device=DEV)
        arena = sim.S[(s % 3) * sim.words:(s % 3 + 1) * sim.words]
        cells = _cells(sim)
        for r, wl in enumerate(sim.wls):
            o, n, so = int(sim.cell_off[r]), sim.Ns[r], int(sim.s_off[r])
            m = _Mono64(wl.params, sim.phi[s % 2], arena[so:so + sim.Ps[r] * sim.Ls[r]],
                        cells[o:o + n], s, offset=o)
            for _ in range(state["steps"]):
                m.step()
            out[o:o + n] = m.phi
        return {"phi": out.reshape(-1), "S": None, "cells": None, "classes": None, "flags": None}
    if kind == "step3d":
        return _exact_step3d(state)
    if kind == "infer":
        net = state["net"]
        x, phi, _, _ = _crops64(_mono64(state["sim"]))
        dphi = _infer64(x, _net_weights(net)) * net.scale
        return {"dphi": dphi.reshape(-1), "pred": (phi + dphi).reshape(-1), "origin": None}
    if kind == "block":
        return _exact_block(state)
    if kind == "train":
        return _exact_train(state)
    return _exact_setup(case, state)
