"""The work this framework is used for, as cases that can be timed and checked.

A case is a plain dict. ``prepare(case, seed)`` sets up what a program holds
before the call, ``run(state)`` is one pass through the public entry points,
``work(case)`` what that pass cannot do without, and ``exact(case, seed)`` the
same outputs in FP64 from plain torch, with no code of this repository.

Kinds of pass:

``step``      ``step_n``: time steps of one cluster (``Simulator``) or of a batch
              (``BatchSimulator``); outputs are the state buffers bound at set-up.
``residual``  ``BatchSimulator.residual_window``: a window of steps and the init
              residual of every cluster (the loop of the warm-started init phase).
``loop``      ``BatchSimulator.run_loop``: steps with sampled steps, whose
              observables and series each cluster stores on the host.
``phase``     ``Simulator.run_sim_core``: a whole phase of one cluster.
``predict``   ``WarmStartGNN.forward``: the init state of a batch of clusters.
``train``     forward, loss, backward and Adam of the warm-start network.

Physics: ``plain`` Na/K/Cl/P/M at 1 ms; ``channels`` adds Ca, the Ca pump and
Nav/Kv channels at 0.1 ms; ``full`` adds Cav and the reaction network.
"""

import functools
import math
import random

import numpy as np
import torch

from betse_amd.batch import BatchSimulator, batched_worlds
from betse_amd.cells import Cells
from betse_amd.channels import draw_channel_state
from betse_amd.gnn import WarmStartGNN, init_params_np
from betse_amd.parameters import Parameters
from betse_amd.sim import SimPhase, SimPhaseKind, Simulator

PRESET = {"plain": "small", "channels": "large", "full": "full"}
# membranes, cells and grid squares of a single cluster follow from its radius and grid
HEX_CELL = math.sqrt(3.0) / 2.0 * 1.0e-10          # area of a cell of the 10 um lattice, m^2
FEATURES, TARGETS, HIDDEN, LAYERS = 13, 4, 64, 6   # the warm-start network


def listed():
    return [
        # one step per call on the smallest cluster: a program that changes an
        # event (applied voltage, block) before every step
        dict(name="one_step_tiny", kind="step", physics="plain", radius_um=30.0, grid=16, flux="fp64", steps=1),
        # a 362-cell cluster, the size most simulations of a tissue patch have
        dict(name="step_small", kind="step", physics="plain", radius_um=100.0, grid=50, flux="fp64", steps=100),
        # a ragged mid-size cluster with channels on the mixed-precision path,
        # an odd number of steps
        dict(name="step_mid_channels_f32", kind="step", physics="channels", radius_um=370.0, grid=117, flux="fp32",
             steps=75),
        # 23k cells with Ca and Nav/Kv: steps between two sampled steps
        dict(name="step_large_channels", kind="step", physics="channels", radius_um=800.0, grid=256, flux="fp64",
             steps=100),
        # 105k cells, channels and the reaction network
        dict(name="step_full", kind="step", physics="full", radius_um=1700.0, grid=512, flux="fp64", steps=100),
        # the batched workload: 256 independent clusters, 500k cells
        dict(name="step_batch256", kind="step", physics="plain", clusters=256, cells_lo=100, cells_hi=5000, grid_lo=32,
             grid_hi=128, flux="fp64", steps=50),
        # a window of the init phase of the warm start's clusters
        dict(name="residual_batch48_f32", kind="residual", physics="plain", clusters=48, cells_lo=500, cells_hi=2000,
             grid_lo=48, grid_hi=88, flux="fp32", steps=50),
        # a batch through two sampled steps, observables and series included
        dict(name="loop_batch12", kind="loop", physics="plain", clusters=12, cells_lo=100, cells_hi=5000, grid_lo=32,
             grid_hi=128, flux="fp64", steps=120, every=50),
        # the whole init phase of the small cluster: set-up, 1,000 steps, 9 sampled steps
        dict(name="phase_small", kind="phase", physics="plain", radius_um=100.0, grid=50, flux="fp64", steps=1000,
             every=100),
        # the network on a batch to be warm-started
        dict(name="predict_128", kind="predict", clusters=128, cells_lo=500, cells_hi=2000),
        # one training step on a minibatch of 32 clusters, as training runs it
        dict(name="train_32", kind="train", clusters=32, cells_lo=500, cells_hi=2000),
        # and on a few small clusters
        dict(name="train_small", kind="train", clusters=6, cells_lo=60, cells_hi=200),
    ]


def draw(rng: random.Random):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "step", "step", "batch", "residual", "loop", "phase", "predict", "train"])
    flux = rng.choice(["fp64", "fp32"])
    if kind in ("step", "phase"):
        physics = rng.choice(["plain", "channels", "full"])
        radius = math.exp(rng.uniform(math.log(30.0), math.log(900.0 if kind == "step" else 200.0)))
        # squares of about half a cell spacing to two spacings, at least the 1.25 x radius world
        grid = max(16, min(300, int(2.5 * radius / 10.0 * rng.uniform(0.7, 1.6))))
        case = dict(kind=kind, physics=physics, radius_um=round(radius, 1), grid=grid, flux=flux,
                    steps=log_int(1, 120) if kind == "step" else log_int(150, 600))
        if kind == "phase":
            case["every"] = log_int(40, 100)
        return case
    lo = log_int(60, 900)
    hi = int(lo * rng.uniform(1.5, 6.0))
    if kind in ("predict", "train"):
        return dict(kind=kind, clusters=log_int(2, 64), cells_lo=lo, cells_hi=min(hi, 2500))
    case = dict(kind="step" if kind == "batch" else kind, physics=rng.choice(["plain", "channels", "plain"]),
                clusters=log_int(2, 16 if kind == "loop" else 64), cells_lo=lo, cells_hi=min(hi, 4000),
                grid_lo=rng.randint(40, 52), grid_hi=rng.randint(88, 130), flux=flux, steps=log_int(10, 100))
    if kind == "loop":
        case["steps"], case["every"] = log_int(60, 150), rng.randint(25, 50)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _world(radius_um, grid):
    p = Parameters.preset("small")
    p.cluster_radius, p.grid_size = radius_um * 1.0e-6, grid
    return Cells.make_world(p)


@functools.lru_cache(maxsize=3)
def _clusters(n, lo, hi, g_lo, g_hi):
    """(radius, grid, geometry) of each cluster of a batch."""
    return [(p.cluster_radius, p.grid_size, c) for p, c in
            batched_worlds(n, cells_range=(lo, hi), grid_range=(g_lo, g_hi), seed=7)]


def _vary(p, rng):
    """Membrane diffusivities and pump rate log-uniform over a decade."""
    p.mem_perms = dict(p.mem_perms)
    for ion in ("Na", "K", "Cl"):
        p.mem_perms[ion] *= 10.0 ** rng.uniform(-0.5, 0.5)
    p.alpha_NaK *= 10.0 ** rng.uniform(-0.5, 0.5)
    return p


def _problem(case, seed):
    """[(Parameters, Cells)] of the case: geometry by its sizes, everything else from the seed."""
    rng = np.random.RandomState(seed)
    out = []
    if "clusters" in case:
        geo = _clusters(case["clusters"], case["cells_lo"], case["cells_hi"], case["grid_lo"], case["grid_hi"])
    else:
        geo = [(case["radius_um"] * 1.0e-6, case["grid"], _world(case["radius_um"], case["grid"]))]
    for radius, grid, cells in geo:
        p = Parameters.preset(PRESET[case["physics"]])
        p.cluster_radius, p.grid_size = radius, grid
        _vary(p, rng)
        if "every" in case:
            p.init_time_total = p.init_time_step * (case["steps"] + 0.5)
            p.init_time_sampling = p.init_time_step * case["every"]
        p.set_phase_time("init")
        if p.channels:
            p.channel_seed = int(rng.randint(1 << 30))
            draw_channel_state(p, cells.n_cells, cells.n_mems)
        out.append((p, cells))
    return out


def _start(p, cells, seed):
    """Cell concentrations of a single cluster away from its default profile:
    every cell's Na, K, Cl a few percent off and M such that its charge gives
    a Vmem between -60 and -20 mV, as a loaded or warm-started state has."""
    rng = np.random.RandomState(seed + 1)
    names = p.ion_names()
    cc = np.repeat(np.array([p.cell_concs[n] for n in names])[:, None], cells.n_cells, axis=1)
    z = np.array([float(p.ion_charge[n]) for n in names])
    for n in ("Na", "K", "Cl"):
        cc[names.index(n)] *= 1.0 + 0.05 * rng.uniform(-1.0, 1.0, cells.n_cells)
    vm = rng.uniform(-0.06, -0.02, cells.n_cells)
    m = names.index("M")
    cc[m] = 0.0
    cc[m] = (vm * p.cm / (p.F * cells.diviterm) - z @ cc) / z[m]
    return cc


@functools.lru_cache(maxsize=2)
def _graph(n, lo, hi):
    """Neighbour CSR of a batch's cells (int32)."""
    ptr, idx, off, eoff = [np.zeros(1, np.int64)], [], 0, 0
    for _, _, c in _clusters(n, lo, hi, 48, 88):
        ptr.append(c.cell_nn_ptr[1:] + eoff)
        idx.append(c.cell_nn_idx + off)
        eoff += int(c.cell_nn_ptr[-1])
        off += c.n_cells
    return np.concatenate(ptr).astype(np.int32), np.concatenate(idx).astype(np.int32)


def _net_inputs(case, seed):
    ptr, idx = _graph(case["clusters"], case["cells_lo"], case["cells_hi"])
    rng = np.random.RandomState(seed)
    n = len(ptr) - 1
    X = rng.standard_normal((n, FEATURES)).astype(np.float32)
    T = (0.5 * rng.standard_normal((n, TARGETS))).astype(np.float32)
    weights = {k: np.asarray(v, dtype=np.float32)
               for k, v in init_params_np(FEATURES, TARGETS, HIDDEN, LAYERS, seed % (1 << 31)).items()}
    for k in weights:
        if k.startswith("b"):
            weights[k] = (0.1 * rng.standard_normal(weights[k].shape)).astype(np.float32)
    return X, T, ptr, idx, weights


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("predict", "train"):
        X, T, ptr, idx, weights = _net_inputs(case, seed)
        net = WarmStartGNN(FEATURES, TARGETS, HIDDEN, LAYERS, params=weights)
        X, T, ptr, idx = (torch.from_numpy(a).to(net.device) for a in (X, T, ptr, idx))
        return dict(kind=kind, net=net, X=X, T=T, ptr=ptr, idx=idx, mask=torch.ones_like(T))
    worlds = _problem(case, seed)
    state = dict(kind=kind, steps=case["steps"])
    if "clusters" in case:
        sim = BatchSimulator(worlds, flux_mode=case["flux"])
        sim.init("init")
        if kind == "loop":
            sim.prepare_sampling()
    else:
        p, cells = worlds[0]
        sim = Simulator(p, flux_mode=case["flux"])
        phase = SimPhase(SimPhaseKind.INIT, p, cells, sim)
        sim.init_core(phase)
        sim.cc_cells = _start(p, cells, seed)
        sim.c_lag = sim.cc_cells.copy()
        state["phase"] = phase
        if kind != "phase":
            sim.prepare(phase)
    state["sim"] = sim
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
STATE = ("c_cell", "vm_cell", "c_env", "E_x", "E_y", "v_env", "gates", "c_net")


def _buffers(sim, names):
    """The state buffers the program bound to the context, on the device."""
    d = sim._dev
    return {k: d[k] for k in names if k in d and d[k].numel() > 2}


def run(state):
    kind = state["kind"]
    if kind == "predict":
        return state["net"].forward(state["X"], state["ptr"], state["idx"], keep=False)
    if kind == "train":
        net = state["net"]
        y = net.forward(state["X"], state["ptr"], state["idx"])
        loss, dY = net.loss(y, state["T"], state["mask"], float(y.numel()))
        grads = net.backward(dY, state["ptr"], state["idx"])
        net.adam(grads, lr=2.0e-3)
        return {"loss": loss, "y": y, "grads": grads, "weights": net.params}
    sim = state["sim"]
    if kind == "step":
        sim.step_n(state["steps"])
        return _buffers(sim, STATE)
    if kind == "residual":
        return {"residual": sim.residual_window(state["steps"]), **_buffers(sim, ("c_cell", "vm_cell", "c_env"))}
    if kind == "loop":
        sim.run_loop(state["steps"])
        return {"state": _buffers(sim, STATE),
                "series": [(st.vm_time[-1], st.I_mem_time[-1], st.I_tot_x_time[-1]) for st in sim.states]}
    sim.run_sim_core(state["phase"])
    return {"cc_cells": sim.cc_cells, "vm_cell": sim.vm_cell, "cc_env": sim.cc_env, "E_x": sim.E_env_x,
            "v_env": sim.v_env, "vm_time": np.stack(sim.vm_time), "I_mem_time": np.stack(sim.I_mem_time),
            "I_tot_x_time": np.stack(sim.I_tot_x_time)}


# ---------------------------------------------------------------------------
# compulsory work
# ---------------------------------------------------------------------------
def _sizes(case):
    """(cells, membranes, squares) from the case's own numbers."""
    if "clusters" in case:
        r_lo, r_hi = math.sqrt(case["cells_lo"] / math.pi), math.sqrt(case["cells_hi"] / math.pi)
        cells = case["clusters"] * math.pi * (r_lo * r_lo + r_lo * r_hi + r_hi * r_hi) / 3.0
        g_lo, g_hi = case.get("grid_lo", 0), case.get("grid_hi", 0)
        squares = case["clusters"] * (g_lo * g_lo + g_lo * g_hi + g_hi * g_hi) / 3.0
    else:
        cells = math.pi * (case["radius_um"] * 1.0e-6) ** 2 / HEX_CELL
        squares = case["grid"] ** 2
    return cells, 6.0 * cells, squares


def work(case):
    """Bytes: per step, every array element of one ideal fused pass read once
    and written once (indices, surface areas, state, diffusivities of the
    squares' grid as constants of the cluster); network: inputs, weights and
    outputs, and for training each layer's activations once in each direction.
    Operations: the flux laws, stencils and sums; the network's products."""
    C, M, S = _sizes(case)
    if case["kind"] in ("predict", "train"):
        per_node = 2.0 * (FEATURES * HIDDEN + LAYERS * 2 * HIDDEN * HIDDEN + HIDDEN * TARGETS)
        if case["kind"] == "predict":
            return {"bytes": C * 4.0 * (FEATURES + TARGETS + 7), "flops": C * per_node}
        return {"bytes": C * 4.0 * (FEATURES + 3 * TARGETS + 14 + 2 * 3 * LAYERS * HIDDEN), "flops": 3 * C * per_node}
    ions = 5 if case["physics"] == "plain" else 6
    chan = {"plain": 0, "channels": 2, "full": 3}[case["physics"]]
    species = 8 if case["physics"] == "full" else 0
    step_bytes = (M * (16 + 32 * chan) + C * (32 * ions + 36 + 8 * chan + 16 * species) + S * (16 * ions + 24))
    step_flops = M * (60.0 * ions + 60.0 + 50.0 * chan) + C * 100.0 * chan + S * (60.0 + 30.0 * ions)
    n = case["steps"]
    samples = max(0, (n - 1) // case["every"]) if "every" in case else 0
    return {"bytes": n * step_bytes + samples * 8.0 * (M * (6 + 2 * ions) + C * (3 + ions) + S * (9 + 3 * ions)),
            "flops": n * step_flops}


# ---------------------------------------------------------------------------
# the same in plain FP64 torch
# ---------------------------------------------------------------------------
def _ghk(cA, cB, D, d, z, v, F_RT):
    a = z * (v + 1.0e-25) * F_RT
    e = torch.expm1(-a)
    return (D * a / d) * (cB - cA * (1.0 + e)) / e


def _grad(f, h, axis):
    """Central differences, one-sided at the ends."""
    f = f.transpose(0, axis)
    g = torch.cat([(f[1:2] - f[:1]) / h, (f[2:] - f[:-2]) / (2.0 * h), (f[-1:] - f[-2:-1]) / h])
    return g.transpose(0, axis)


def _div(fx, fy, h):
    """Divergence as the finite-volume update takes it: the one-sided ends carry the opposite sign."""
    gx, gy = _grad(fx, h, 1).clone(), _grad(fy, h, 0).clone()
    for g, ax in ((gx, 1), (gy, 0)):
        g.select(ax, 0).neg_()
        g.select(ax, -1).neg_()
    return gx + gy


def _rates(kind, V):
    exp = torch.exp
    if kind == "Nav1p2":
        a = V - 10.0

        def ratio(k, x, s):
            return k * x / (-torch.expm1(-x / s))

        al, be = ratio(0.182, a + 35.0, 9.0), ratio(0.124, -a - 35.0, 9.0)
        return (al / (al + be), 1.0 / (al + be), 1.0 / (1.0 + exp((V + 55.0) / 6.2)),
                1.0 / (ratio(0.024, a + 50.0, 5.0) + ratio(0.0091, -a - 75.000123, 5.0)))
    if kind == "Kv1p1":
        return (1.0 / (1.0 + exp((V + 30.5) / -11.3943)), 30.0 / (1.0 + exp((V + 76.56) / 26.1479)),
                1.0 / (1.0 + exp((V + 30.0) / 27.3943)), 15000.0 / (1.0 + exp((V + 160.56) / -100.0)))
    W = V - 10.0
    return (1.0 / (1.0 + exp((W + 30.0) / -6.0)), 5.0 + 20.0 / (1.0 + exp((W + 25.0) / 5.0)),
            1.0 / (1.0 + exp((W + 80.0) / 6.4)), 20.0 + 50.0 / (1.0 + exp((W + 40.0) / 7.0)))


class _Exact:
    """One cluster in FP64 torch."""

    def __init__(self, p, cells, cc0=None):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.p, self.dev = p, dev

        def t(a, dtype=torch.float64):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=dev)

        self.t = t
        self.names = n = p.ion_names()
        self.z = [float(p.ion_charge[i]) for i in n]
        self.shape = cells.X.shape
        G = cells.X.size
        self.cell, self.nn = t(cells.mem_to_cells, torch.int64), t(cells.nn_i, torch.int64)
        self.sq, self.sa = t(cells.map_mem2ecm, torch.int64), t(cells.mem_sa)
        self.inner = (self.nn != torch.arange(len(self.nn), device=dev)).double()
        self.vol, self.csa, self.nm = t(cells.cell_vol), t(cells.cell_sa), t(cells.num_mems)
        self.div, self.h = t(cells.diviterm), float(cells.delta)
        self.gj_len = float(cells.gj_len)
        self.nx, self.ny = t(cells.mem_vects_flat[:, 2]), t(cells.mem_vects_flat[:, 3])
        C = cells.n_cells
        cc = cc0 if cc0 is not None else np.repeat(np.array([p.cell_concs[i] for i in n])[:, None], C, axis=1)
        self.c, self.lag = t(cc), t(cc)
        self.ce = torch.stack([torch.full(self.shape, p.env_concs[i], dtype=torch.float64, device=dev) for i in n])
        self.D = torch.full((len(n), G), 0.0, dtype=torch.float64, device=dev)
        for i, name in enumerate(n):
            self.D[i] = p.free_diff[name]
        z2 = np.array(self.z) ** 2
        ko = np.sqrt(sum(p.NAv * p.q ** 2 * z2[i] / (p.er * p.eo * p.kb * p.T) * p.env_concs[x] for i, x in enumerate(n)))
        self.has = torch.zeros(G, dtype=torch.float64, device=dev).index_add_(0, self.sq, torch.ones_like(self.sa)) > 0
        sq_sa = torch.zeros(G, dtype=torch.float64, device=dev).index_add_(0, self.sq, self.sa)
        self.volume = p.cell_height * self.h ** 2
        self.u_scale = self.volume / float(sq_sa[self.sq].mean()) / (ko * p.eo * p.er)
        self.screen = 2.0 / (ko * self.h) * (p.cell_radius / p.true_cell_size)
        x = np.arange(-4, 5)
        w = np.exp(-0.5 * x ** 2)
        self.w = t(w / w.sum())
        self.gates = [[t(g[0]), t(g[1])] for g in p.channel_gates0] if p.channels else []
        self.mult = [t(m) for m in p.channel_cell_mult] if p.channels else []
        self.cn = t(np.repeat(np.asarray(p.network.c0)[:, None], C, axis=1)) if p.network is not None else None
        self.volt()
        self.field()

    def per_cell(self, x):
        return torch.zeros_like(self.vol).index_add_(0, self.cell, x)

    def per_sq(self, x):
        return torch.zeros(self.has.shape, dtype=torch.float64, device=self.dev).index_add_(0, self.sq, x)

    def volt(self):
        rho = sum(z * self.p.F * self.c[i] for i, z in enumerate(self.z))
        self.v = rho * self.div / self.p.cm

    def field(self):
        rho = sum(z * self.p.F * self.ce[i] for i, z in enumerate(self.z)).reshape(-1)
        u = torch.where(self.has, rho * self.u_scale, torch.zeros_like(rho)).reshape(self.shape)
        for ax in (0, 1):
            u = torch.nn.functional.pad(u, (0, 0, 4, 4) if ax == 0 else (4, 4, 0, 0))
            n = self.shape[ax]
            u = sum(self.w[k] * u.narrow(ax, k, n) for k in range(9))
        self.venv = u
        s = self.screen * u
        self.Ex, self.Ey = -_grad(s, self.h, 1), -_grad(s, self.h, 0)

    def step(self):
        p, F_RT, RT = self.p, self.p.F / (self.p.R * self.p.T), self.p.R * self.p.T
        names, N = self.names, len(self.names)
        env = self.ce.reshape(N, -1)
        v, lag, cell, sq = self.v[self.cell], self.lag, self.cell, self.sq
        vn, other = v[self.nn], cell[self.nn]
        iNa, iK = names.index("Na"), names.index("K")
        # Na/K pump
        nai, nao, ki, ko = lag[iNa][cell], env[iNa][sq], lag[iK][cell], env[iK][sq]
        Q = (p.cADP * 1e-3 * p.cPi * 1e-3 * (nao * 1e-3) ** 3 * (ki * 1e-3) ** 2) / (
            p.cATP * 1e-3 * (nai * 1e-3) ** 3 * (ko * 1e-3) ** 2)
        keq = torch.exp(-(p.deltaGATP / RT - p.F * v / RT))
        na, kk, atp = (nai / p.KmNK_Na) ** 3, (ko / p.KmNK_K) ** 2, p.cATP / p.KmNK_ATP
        pump = -3.0 * p.NaKATP_block * p.alpha_NaK * (na * kk * atp) / ((1 + na) * (1 + kk) * (1 + atp)) * (1 - Q / keq)
        fm, fg = [], []
        for i, name in enumerate(names):
            f = _ghk(env[i][sq], lag[i][cell], p.mem_perms[name], p.tm, self.z[i], v, F_RT)
            f = f + (pump if i == iNa else -(2.0 / 3.0) * pump if i == iK else 0.0)
            fm.append(f)
            fg.append(self.inner * _ghk(lag[i][cell], lag[i][other], p.free_diff[name] * p.gj_surface, self.gj_len,
                                        self.z[i], vn - v, F_RT))
        # the environment
        mid, self.fx, self.fy = [], [], []
        for i, name in enumerate(names):
            c = self.ce[i].clone()
            for edge in (c[0], c[-1], c[:, 0], c[:, -1]):
                edge.fill_(p.env_concs[name])
            D = self.D[i].reshape(self.shape)
            al = D * self.z[i] * p.q / (p.kb * p.T)
            fx = -D * _grad(c, self.h, 1) + al * self.Ex * c
            fy = -D * _grad(c, self.h, 0) + al * self.Ey * c
            mid.append(c + _div(-fx, -fy, self.h) * p.dt)
            self.fx.append(fx)
            self.fy.append(fy)
        mid = torch.stack(mid).reshape(N, -1)
        if "Ca" in names and p.alpha_Ca > 0.0:
            i = names.index("Ca")
            ci, co = self.c[i][cell].clamp(min=0.0), mid[i][sq].clamp(min=0.0)
            Q = p.cADP * p.cPi * co / (p.cATP * ci)
            keq = torch.exp(-(p.deltaGATP / RT - 2.0 * p.F * v / RT))
            atp = p.cATP / p.KmCa_ATP
            fm[i] = fm[i] - p.alpha_Ca * (ci / p.KmCa_Ca * atp) / ((1 + ci / p.KmCa_Ca) * (1 + atp)) * (1 - Q / keq)
        fch = {}
        for k, spec in enumerate(p.channels):
            i = {"Nav1p2": iNa, "Kv1p1": iK}.get(spec.kind, names.index("Ca") if "Ca" in names else 0)
            mi, mt, hi, ht = (r[cell] for r in _rates(spec.kind, self.v * 1000.0))
            m, h = self.gates[k]
            dt = p.dt * 1000.0
            m, h = (mt * m + dt * mi) / (mt + dt), (ht * h + dt * hi) / (ht + dt)
            self.gates[k] = [m, h]
            P = {"Nav1p2": m ** 3 * h, "Kv1p1": m * h ** 2}.get(spec.kind, m ** 2 * h)
            fch[i] = _ghk(mid[i][sq], self.c[i][cell], P * spec.max_dm * self.mult[k][cell], p.tm, self.z[i], v, F_RT)
        c, lag, ce = [], [], []
        for i in range(N):
            base, e = self.c[i], mid[i]
            if i in fch:
                base = base + self.per_cell(fch[i] * self.sa) / self.vol * p.dt
                e = e - self.per_sq(fch[i] * self.sa) / self.volume * p.dt
            c1 = base + self.per_cell(fm[i] * self.sa) / self.vol * p.dt
            lag.append(c1)
            c.append((c1 - self.per_cell(fg[i] * self.sa) / self.vol * p.dt).clamp(min=0.0))
            ce.append(e - self.per_sq(fm[i] * self.sa) / self.volume * p.dt)
        self.fm, self.fg, self.fch = fm, fg, fch
        self.c, self.lag, self.ce = torch.stack(c), torch.stack(lag), torch.stack(ce).reshape(self.ce.shape)
        if self.cn is not None:
            self.network()
        self.volt()
        self.field()

    def network(self):
        p, net, c = self.p, self.p.network, self.cn

        def alpha(x):
            a = torch.ones_like(c[0])
            for s in x.activators:
                y = (c[s.species] / s.km) ** s.n
                a = a * y / (1 + y)
            for s in x.inhibitors:
                a = a / (1 + (c[s.species] / s.km) ** s.n)
            return a

        d = torch.zeros_like(c)
        for g in net.growth:
            x = c[g.species] / g.gad_scale
            d[g.species] += g.time_factor * (g.r_production * alpha(g) - g.r_decay * x - g.decay_max * x)
        for r in net.reactions:
            rate = r.vmax * alpha(r)
            if r.delta_Go is not None:
                Q = torch.ones_like(c[0])
                for s, k, _ in r.products:
                    Q = Q * (1e-3 * c[s] ** k)
                for s, k, _ in r.reactants:
                    Q = Q / (1e-3 * c[s] ** k)
                rate = rate * (1 - Q / math.exp(-r.delta_Go / (p.R * p.T)))
            else:
                for s, k, km in r.reactants:
                    x = (c[s] / km) ** k
                    rate = rate * x / (1 + x)
            for s, k, _ in r.reactants:
                d[s] -= k * rate
            for s, k, _ in r.products:
                d[s] += k * rate
        self.cn = (c + d * p.dt).clamp(min=0.0)

    # what a sampled step stores: Vmem and transmembrane current per membrane,
    # and the divergence-free part of the environment's current along x
    def sample(self):
        p, N = self.p, len(self.names)
        zF = [z * p.F for z in self.z]
        j = sum(zF[i] * (self.fg[i] - self.fm[i]) for i in range(N)) - sum(zF[i] * f for i, f in self.fch.items())
        ave = self.per_cell(j * self.sa) / self.csa
        w = p.smooth_cells * self.nm
        jn = ((w - 1) / w)[self.cell] * j + (ave / w)[self.cell]
        jx, jy = (sum(zF[i] * f[i] for i in range(N)) for f in (self.fx, self.fy))
        n1, n2 = self.shape[0] - 2, self.shape[1] - 2
        rhs = (_grad(jy, self.h, 1) - _grad(jx, self.h, 0))[1:-1, 1:-1]        # -div(-jy, jx)

        def dst(n):
            k = torch.arange(1, n + 1, dtype=torch.float64, device=self.dev)
            return torch.sin(math.pi * k[:, None] * k / (n + 1)), 2.0 * torch.cos(math.pi * k / (n + 1)) - 2.0

        (S1, l1), (S2, l2) = dst(n1), dst(n2)
        A = S1 @ ((S1 @ rhs @ S2) * self.h ** 2 * 4.0 / ((n1 + 1) * (n2 + 1)) / (l1[:, None] + l2)) @ S2
        A = torch.nn.functional.pad(A, (1, 1, 1, 1))
        return self.v[self.cell], -jn * self.sa, -_grad(A, self.h, 0)

    def state(self):
        out = {"c_cell": self.c, "vm_cell": self.v, "c_env": self.ce.reshape(len(self.names), -1),
               "E_x": self.Ex.reshape(-1), "E_y": self.Ey.reshape(-1), "v_env": self.venv.reshape(-1)}
        if self.gates:
            out["gates"] = torch.stack([torch.stack(g) for g in self.gates])
        if self.cn is not None:
            out["c_net"] = self.cn
        return out


def _exact_net(case, seed):
    X, T, ptr, idx, weights = _net_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    X, T = (torch.as_tensor(a, dtype=torch.float64, device=dev) for a in (X, T))
    W = {k: torch.as_tensor(v, dtype=torch.float64, device=dev).requires_grad_(case["kind"] == "train")
         for k, v in weights.items()}
    deg = np.diff(ptr)
    src = torch.as_tensor(np.repeat(np.arange(len(deg)), deg), device=dev)
    dst = torch.as_tensor(idx.astype(np.int64), device=dev)
    deg = torch.as_tensor(np.maximum(deg, 1), dtype=torch.float64, device=dev)[:, None]
    h = torch.nn.functional.silu(X @ W["W_in"] + W["b_in"])
    for k in range(LAYERS):
        nbr = torch.zeros_like(h).index_add(0, src, h[dst]) / deg
        h = h + torch.nn.functional.silu(torch.cat([h, nbr], 1) @ W["W%d" % k] + W["b%d" % k])
    y = h @ W["W_out"] + W["b_out"]
    if case["kind"] == "predict":
        return y
    loss = ((y - T) ** 2).mean()
    loss.backward()
    # the first Adam step is the sign of each gradient nearly everywhere, so the weights have no error to speak of
    return {"loss": float(loss), "y": y.detach(), "grads": {k: v.grad for k, v in W.items()}, "weights": None}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("predict", "train"):
        return _exact_net(case, seed)
    worlds = _problem(case, seed)
    if len(worlds) * case["steps"] > 3000:
        return None                                   # over 20 seconds
    names = ("c_cell", "vm_cell", "c_env") if kind == "residual" else STATE
    parts, series, rs = [], [], []
    for p, cells in worlds:
        e = _Exact(p, cells, None if "clusters" in case else _start(p, cells, seed))
        at, samples = (int(case["every"]) if "every" in case else 0), []
        c0 = e.c
        for s in range(case["steps"]):
            e.step()
            if at and s == at and s < case["steps"]:
                samples.append(e.sample())
                at = at + int(case["every"]) if at < case["steps"] - case["every"] else 0
        rs.append(float(((e.c - c0).abs() / e.c.abs()).max()) / case["steps"])
        parts.append(e.state())
        series.append(samples)
    dims = {"gates": 2}
    whole = {k: torch.cat([x[k] for x in parts], dim=dims.get(k, -1)) for k in names if k in parts[0]}
    if kind == "step":
        return whole
    if kind == "residual":
        # the change over a window against the value: FP64 state, so its own
        # rounding shows where a cluster hardly moves
        return {"residual": np.array(rs), **whole}
    if kind == "loop":
        return {"state": whole, "series": [tuple(x.cpu().numpy() for x in s[-1]) for s in series]}
    vm, im, it = (np.stack([x[k].cpu().numpy() for x in series[0]]) for k in range(3))
    return {"cc_cells": whole["c_cell"], "vm_cell": whole["vm_cell"], "cc_env": whole["c_env"],
            "E_x": whole["E_x"].reshape(worlds[0][1].X.shape), "v_env": whole["v_env"], "vm_time": vm,
            "I_mem_time": im, "I_tot_x_time": it}
