"""Performance cases: what a program that uses this framework has it do.

Every case is one call (or the few calls that belong together) of the public
Python entry points on a lattice handle that the program keeps:

  md           Landau-Lifshitz dynamics of one spin configuration
  dopri5       the response to one pulse with the adaptive Dormand-Prince
               stepper, observed on a grid
  pump_probe   a 2DCS delay scan: M0, M1(tau) and M01(tau) of every delay
  ensemble     undriven trajectories of many start states (pyrochlore samples)
  dssf         dynamical structure factor S(q, w) of such an ensemble
  adjoint      loss and gradient of Kitaev couplings fitted to a measured M(t)
  mixed        the delay scan of the SU(2) + SU(3) (Fe/Tm) lattice
  mixed_grad   loss and derivative with respect to the Fe-Tm coupling scale

listed() gives the sizes that are looked at one by one, draw() more of the
same ranges, prepare() the handle and the inputs, run() one pass, work() the
bytes and operations it cannot do without, tolerance() how far two correct
FP64 implementations may differ and exact() the same results from plain torch
operations in FP64.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch
import torch.utils.checkpoint

from classical_mcmc_spin_amd import GPULattice, adjoint, gpu, gpu_mixed, mixed_model, model, seeding

KITAEV = dict(K=-1.0, Gamma=0.25, Gammap=-0.02)
AMP, WIDTH = 0.5, 0.5
T0_PULSE = -1.0


def listed():
    return [
        # a quick look at a small cluster: one short trajectory, where the
        # call itself counts as much as the arithmetic
        {"name": "md_6x6", "kind": "md", "L1": 6, "L2": 6, "steps": 100},
        # plain dynamics of the 24x24 honeycomb from a random state
        {"name": "md_24x24", "kind": "md", "L1": 24, "L2": 24, "steps": 1000},
        # one pulse on the same lattice with the adaptive integrator
        {"name": "dopri5_24x24", "kind": "dopri5", "L1": 24, "L2": 24, "steps": 80},
        # a coarse delay scan of an odd-sized cluster (convergence in size)
        {"name": "pump_probe_15x13", "kind": "pump_probe", "L1": 15, "L2": 13, "n_tau": 12, "steps": 500},
        # the production 2DCS scan: 256 delays, 513 trajectories; 20 units of
        # time, over which two orders of summation still agree to 12 digits
        {"name": "pump_probe_36x36", "kind": "pump_probe", "L1": 36, "L2": 36, "n_tau": 256, "steps": 2048},
        # structure factor of a small pyrochlore ensemble
        {"name": "dssf_pyrochlore_4", "kind": "dssf", "L": 4, "samples": 8, "steps": 256, "every": 8},
        # pyrochlore samples that do not fit one compute unit
        {"name": "ensemble_pyrochlore_16", "kind": "ensemble", "L": 16, "samples": 32, "steps": 256},
        # one fit iteration from a few starts on a small lattice
        {"name": "adjoint_12x12", "kind": "adjoint", "L1": 12, "L2": 12, "starts": 4, "steps": 250},
        # the fit of the 24x24 lattice from 32 starts
        {"name": "adjoint_24x24", "kind": "adjoint", "L1": 24, "L2": 24, "starts": 32, "steps": 2000},
        # a coarse mixed-lattice scan
        {"name": "mixed_4x4x4", "kind": "mixed", "L": 4, "n_tau": 16, "steps": 200},
        # the production mixed-lattice scan (128 delays, 257 trajectories)
        {"name": "mixed_8x8x8", "kind": "mixed", "L": 8, "n_tau": 128, "steps": 512},
        # one iteration of a coupling fit on the mixed lattice
        {"name": "mixed_grad_4x4x4", "kind": "mixed_grad", "L": 4, "n_tau": 8, "steps": 128},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["md", "md", "dopri5", "pump_probe", "pump_probe", "dssf", "ensemble", "ensemble", "adjoint",
                       "adjoint", "mixed", "mixed", "mixed_grad"])
    if kind == "md":
        return {"kind": kind, "L1": rng.randint(4, 36), "L2": rng.randint(4, 36), "steps": log_int(100, 1500)}
    if kind == "dopri5":
        return {"kind": kind, "L1": rng.randint(4, 24), "L2": rng.randint(4, 24), "steps": rng.randint(20, 100)}
    if kind == "pump_probe":
        return {"kind": kind, "L1": rng.randint(6, 36), "L2": rng.randint(6, 36), "n_tau": log_int(4, 256),
                "steps": log_int(200, 2000)}
    if kind == "dssf":
        return {"kind": kind, "L": rng.randint(2, 6), "samples": log_int(1, 16), "steps": log_int(64, 256),
                "every": rng.randint(4, 16)}
    if kind == "ensemble":
        return {"kind": kind, "L": rng.randint(2, 16), "samples": log_int(4, 32), "steps": log_int(64, 256)}
    if kind == "adjoint":
        return {"kind": kind, "L1": rng.randint(6, 24), "L2": rng.randint(6, 24), "starts": log_int(1, 64),
                "steps": log_int(100, 1000)}
    if kind == "mixed":
        return {"kind": kind, "L": rng.randint(2, 8), "n_tau": log_int(4, 128), "steps": log_int(64, 512)}
    return {"kind": kind, "L": rng.randint(2, 6), "n_tau": log_int(2, 32), "steps": log_int(32, 128)}


# ------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=4)
def _kitaev(L1, L2, h):
    uc = model.build_kitaev_honeycomb(field_strength=h, field_direction=np.ones(3) / math.sqrt(3.0), **KITAEV)
    return model.Lattice(uc, L1, L2, 1)


@functools.lru_cache(maxsize=2)
def _pyrochlore(L):
    return model.Lattice(model.build_pyrochlore_conventional(Jzz=1.0, Jpm=0.05, Jpmpm=0.02, Jzpm=-0.01), L, L, L)


@functools.lru_cache(maxsize=2)
def _mixed(L):
    return mixed_model.MixedLattice(mixed_model.build_tmfeo3_mixed(), L, L, L)


def _ground(lat, seed, sweeps=40):
    """A relaxed state with small thermal tilts."""
    s = seeding.quench(lat, seeding.random_spins(lat.lattice_size, seed), sweeps=sweeps)
    return seeding.tilt(s, 0.01, seed=seed + 1)


def _pyro_samples(lat, n, seed):
    sigma = 0.05 + 0.45 * seeding.uniform01(n, seed, stream=11)
    aiao = model.all_in_all_out(lat)
    return np.stack([seeding.tilt(aiao, float(s), seed=seed + 1000 * (b + 1)) for b, s in enumerate(sigma)])


def _measured(n, dt, seed):
    """M(t) as a measurement gives it: a few damped lines on each component."""
    t = dt * np.arange(n)[:, None]
    u = seeding.uniform01(4 * 9, seed, stream=3).reshape(4, 9)
    return 0.1 * (u[0] - 0.5) + 0.05 * u[1] * np.exp(-0.1 * u[2] * t) * np.cos((0.3 + 2.0 * u[3]) * t)


def _mixed_state(ml, seed):
    """Fe: the antiferromagnetic G pattern with tilts; Tm: near its
    crystal-field ground state."""
    fe = np.zeros((ml.N2, 3))
    fe[:, 2] = np.array([1.0, -1.0, 1.0, -1.0])[np.arange(ml.N2) % 4]
    fe = seeding.tilt(fe, 0.1, seed=seed)
    tm = ml.su3.field / np.linalg.norm(ml.su3.field, axis=1, keepdims=True)
    return ml.flat_state(fe, seeding.tilt(tm, 0.1, seed=seed + 1))


def _t_end(t0, steps, dt):
    return t0 + (steps + 0.5) * dt


DT = {"md": 0.01, "dopri5": 0.05, "pump_probe": 0.01, "ensemble": 0.02, "dssf": 0.02, "adjoint": 0.01,
      "mixed": 0.005, "mixed_grad": 0.005}


def _pulse_dirs(n_atoms):
    f = np.zeros((n_atoms, 3))
    f[:, 0] = 1.0
    return f


def _mixed_fields():
    f2, f3 = np.zeros((4, 3)), np.zeros((4, 8))
    f2[:, 0] = 1.0
    f3[:, 1] = 1.0
    return f2, f3


def _scan(n_tau, step):
    """(t_pulse [B, 2], scale [B, 2]) of M0, M1(tau), M01(tau)."""
    taus = step * np.arange(n_tau)
    tp, sc = np.zeros((1 + 2 * n_tau, 2)), np.zeros((1 + 2 * n_tau, 2))
    sc[0, 0] = 1.0
    tp[1:1 + n_tau, 0] = taus
    sc[1:1 + n_tau, 0] = 1.0
    tp[1 + n_tau:, 1] = taus
    sc[1 + n_tau:] = 1.0
    return tp, sc


def _tau_step(c):
    # delays over three quarters of the observed time
    span = c["steps"] * DT[c["kind"]] + T0_PULSE
    return round(max(0.75 * span / max(c["n_tau"] - 1, 1), 1e-3), 4)


def _inputs(case, seed):
    kind = case["kind"]
    if kind == "md":
        lat = _kitaev(case["L1"], case["L2"], 0.0)
        return {"lat": lat, "spins": seeding.random_spins(lat.lattice_size, seed)}
    if kind in ("pump_probe", "dopri5"):
        lat = _kitaev(case["L1"], case["L2"], 0.1)
        return {"lat": lat, "ground": _ground(lat, seed), "field": _pulse_dirs(2)}
    if kind in ("ensemble", "dssf"):
        lat = _pyrochlore(case["L"])
        return {"lat": lat, "init": _pyro_samples(lat, case["samples"], seed)}
    if kind == "adjoint":
        lat = _kitaev(case["L1"], case["L2"], 0.0)
        u = seeding.uniform01(5 * case["starts"], seed, stream=5).reshape(-1, 5)
        return {"lat": lat, "init": seeding.tilt(_ground(lat, seed, 30), 0.05, seed=seed + 2),
                "theta": np.array([-1.0, 0.25, -0.02, 0.01, 0.05]) * (0.9 + 0.2 * u),
                "target": _measured(case["steps"] + 1, DT[kind], seed)}
    ml = _mixed(case["L"])
    d = {"ml": ml, "ground": _mixed_state(ml, seed)}
    if kind == "mixed_grad":
        m = _measured(case["steps"] + 1, DT[kind], seed)
        d["target"] = np.zeros((case["steps"] + 1, 34))
        d["target"][:, :33] = np.tile(m, 4)[:, :33]
        d["weights"] = np.r_[np.ones(33), 0.0]
    return d


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case, s.kind, s.dt = case, case["kind"], DT[case["kind"]]
    s.__dict__.update(_inputs(case, seed))
    if s.kind in ("mixed", "mixed_grad"):
        s.gm = gpu_mixed.GPUMixedLattice(s.ml)
        if s.kind == "mixed_grad":
            f2, f3 = _mixed_fields()
            for sp, f in ((2, f2), (3, f3)):
                d = s.gm.drive_dirs(sp, f)
                s.gm.set_pulse(sp, np.stack([d, d]), AMP, WIDTH, 0.0, 0.0, 0.0)
            s.tp, s.sc = _scan(case["n_tau"], _tau_step(case))
    elif s.kind == "adjoint":
        s.fit = adjoint.KitaevFit(case["L1"], case["L2"], s.init, s.target, 0.0, _t_end(0.0, case["steps"], s.dt),
                                  s.dt, pulse=(AMP, WIDTH, 0.0, 1.0), alpha=0.02)
    else:
        s.gl = GPULattice(s.lat)
        if s.kind == "dssf":
            s.pos = s.lat.unit_cell.lattice_pos
    return s


def run(s):
    c = s.case
    if s.kind == "md":
        r = gpu.molecular_dynamics(s.gl, s.spins, 0.0, _t_end(0.0, c["steps"], s.dt), s.dt)
        return {"times": r["times"], "mags": r["mags"], "energy": r["energy"], "spins": s.gl.get_spins()}
    if s.kind == "dopri5":
        times, mags = gpu.single_pulse_drive(s.gl, s.ground, s.field, 0.0, AMP, WIDTH, 0.0, T0_PULSE,
                                             _t_end(T0_PULSE, c["steps"], s.dt), s.dt, method="dopri5")
        return {"times": times, "mags": mags}
    if s.kind == "pump_probe":
        d = _tau_step(c)
        r = gpu.pump_probe_spectroscopy(s.gl, s.ground, s.field, AMP, WIDTH, 0.0, 0.0, d * (c["n_tau"] - 0.5), d,
                                        T0_PULSE, _t_end(T0_PULSE, c["steps"], s.dt), s.dt)
        return {k: r[k] for k in ("times", "tau", "M0", "M1", "M01")}
    if s.kind == "ensemble":
        B = c["samples"]
        r = s.gl.integrate_batched(s.init, np.zeros((B, 2)), np.zeros((B, 2)), 0.0, _t_end(0.0, c["steps"], s.dt),
                                   s.dt, tgrid="boost", want_final=True)
        return {k: r[k] for k in ("times", "mags", "energy", "final")}
    if s.kind == "dssf":
        r = s.gl.structure_factor(s.init, 0.0, _t_end(0.0, c["steps"], s.dt), s.dt, c["every"], (c["L"],) * 3,
                                  s.pos, want_mags=True)
        return {"sqw": r["sqw"], "mags": r["mags"]}
    if s.kind == "adjoint":
        loss, grad = s.fit(s.theta)
        return {"loss": loss, "grad": grad}
    f2, f3 = _mixed_fields()
    if s.kind == "mixed":
        d = _tau_step(c)
        r = gpu_mixed.pump_probe_spectroscopy(s.gm, s.ground, f2, f3, AMP, WIDTH, 0.0, AMP, WIDTH, 0.0, 0.0,
                                              d * (c["n_tau"] - 0.5), d, T0_PULSE,
                                              _t_end(T0_PULSE, c["steps"], s.dt), s.dt)
        return {k: r[k] for k in ("times", "tau", "M0", "M1", "M01")}
    r = s.gm.scale_gradient(s.ground, s.tp, s.target, s.weights, s.sc, T0_PULSE,
                            _t_end(T0_PULSE, c["steps"], s.dt), s.dt, want_records=True)
    return {k: r[k] for k in ("loss", "grad", "records", "trecords")}


# --------------------------------------------------------------- what it needs

def work(case):
    kind = case["kind"]
    if kind in ("md", "dopri5", "pump_probe", "adjoint"):
        N = 2 * case["L1"] * case["L2"]
    else:
        N = (16 if kind in ("ensemble", "dssf") else 4) * case["L"] ** 3
    # FP64 operations per site and RK stage: bond products 18 z, cross product
    # 9, updates 12, field 3
    if kind == "md":
        n, B, per = case["steps"], 1, 4 * (18 * 3 + 24) + 13
        out = (n + 1) * 11 + N * 3
    elif kind == "dopri5":
        n, B, per = case["steps"], 1, 6 * (18 * 3 + 12) + 3 * 60   # one accepted step an interval
        out = n * 10 + N * 3
    elif kind == "pump_probe":
        n, B, per = case["steps"], 1 + 2 * case["n_tau"], 4 * (18 * 3 + 24) + 48 + 7
        out = (n + 1) * (B * 9 + 1)
    elif kind in ("ensemble", "dssf"):
        n, B, per = case["steps"], case["samples"], 4 * (18 * 6 + 24) + 13
        out = (n + 1) * B * 10 + B * N * 6
        if kind == "dssf":
            nt = n // case["every"]
            per += 5 * 2 * math.log2(max(N, 2)) / case["every"]
            out += case["L"] ** 3 * nt - B * N * 3 - (n + 1) * B
    elif kind == "adjoint":
        # a forward and a transposed step, five parameter derivatives
        n, B, per = case["steps"], case["starts"], 465 + 2119
        out = (n + 1) * 9 + N * 3 + B * 11
    else:
        n, B = case["steps"], 1 + 2 * case["n_tau"]
        per = 4 * (543 + 556) * (2 if kind == "mixed_grad" else 1)  # one Fe and one Tm site
        out = (n + 1) * B * 34 * (2 if kind == "mixed_grad" else 1) + N * 11
    return {"bytes": 8.0 * out, "flops": float(per) * N * B * n}


def tolerance(case):
    # FP64 throughout; the rounding by which two orders of summation differ at
    # a step grows along the trajectory (some times what was measured with
    # inputs changed in their last bit, at the longest runs of the ranges)
    return {"rel": {"md": 1e-11, "dopri5": 1e-11, "pump_probe": 1e-11, "ensemble": 1e-12, "dssf": 1e-12,
                    "adjoint": 1e-11, "mixed": 1e-13, "mixed_grad": 1e-12}[case["kind"]]}


# -------------------------------------------------------------------- exact

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


class _Su2:
    """H = -B + 2 A S + sum_k J_k S_nb(k) of lattices whose sites all have
    the same number of bonds."""

    def __init__(self, lat):
        N = lat.lattice_size
        z = int(lat.bi_offset[1] - lat.bi_offset[0])
        assert np.all(np.diff(lat.bi_offset.astype(np.int64)) == z)
        self.N, self.z, self.A = N, z, lat.N_atoms
        self.nb = torch.as_tensor(lat.bi_partner.astype(np.int64).reshape(N, z), device=_dev())
        self.J = _t(lat.bi_J.reshape(N, z, 3, 3))
        self.B = _t(lat.field)
        self.A2 = _t(2.0 * lat.onsite) if np.any(lat.onsite) else None
        self.R = _t(lat.frames)
        self.sg = _t(lat.afm_signs)
        self.atom = torch.arange(N, device=_dev()) % self.A

    def field(self, S, J=None, B=None):
        """S [..., N, 3]; J, B: tables with a leading batch dimension."""
        J = self.J if J is None else J
        H = -(self.B if B is None else B)
        if self.A2 is not None:
            H = H + (self.A2 * S[..., None, :]).sum(-1)
        for k in range(self.z):
            H = H + (J[..., k, :, :] * S[..., self.nb[:, k], :][..., None, :]).sum(-1)
        return H

    def records(self, S):
        """[..., 3, 3]: staggered, local and global magnetisation."""
        per_atom = S.reshape(S.shape[:-2] + (self.N // self.A, self.A, 3)).sum(-3)
        g = (self.R * per_atom[..., None, :]).sum(-1)
        return torch.stack([(self.sg[:, None] * g).sum(-2), per_atom.sum(-2), g.sum(-2)], -2) / self.N

    def energy(self, S, H):
        return 0.5 * (S * (H - self.B)).sum((-1, -2)) / self.N


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=-1)


def _pulse(t, tp, amp):
    return amp * torch.exp(-((t - tp) / (2.0 * WIDTH)) ** 2)


def _rk4(f, x, t, dt):
    k1 = f(x, t)
    k2 = f([a + 0.5 * dt * k for a, k in zip(x, k1)], t + 0.5 * dt)
    k3 = f([a + 0.5 * dt * k for a, k in zip(x, k2)], t + 0.5 * dt)
    k4 = f([a + dt * k for a, k in zip(x, k3)], t + dt)
    return [a + dt / 6.0 * p + dt / 3.0 * q + dt / 3.0 * r + dt / 6.0 * s
            for a, p, q, r, s in zip(x, k1, k2, k3, k4)]


def _host(v):
    return v.detach().cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    n = case.get("steps", 0)
    d, dt = _inputs(case, seed), DT[kind]
    return {"md": _exact_md, "dopri5": _exact_dopri5, "pump_probe": _exact_pump_probe, "ensemble": _exact_ensemble,
            "dssf": _exact_dssf, "adjoint": _exact_adjoint, "mixed": _exact_mixed,
            "mixed_grad": _exact_mixed_grad}[kind](case, d, n, dt)


def _undriven(su, S, n, dt, energy=True, at=None):
    """(records [n+1, ...], energies, S) of n undriven RK4 steps."""
    recs, en = [], []
    f = lambda x, t: [_cross(su.field(x[0]), x[0])]
    for i in range(n + 1):
        recs.append(su.records(S))
        if energy:
            en.append(su.energy(S, su.field(S)))
        if at is not None:
            at(i, S)
        if i < n:
            S = _rk4(f, [S], i * dt, dt)[0]
    return torch.stack(recs), (torch.stack(en) if energy else None), S


def _exact_md(case, d, n, dt):
    su = _Su2(d["lat"])
    m, e, S = _undriven(su, _t(d["spins"]), n, dt)
    return {"times": dt * np.arange(n + 1), "mags": _host(m), "energy": _host(e), "spins": _host(S)}


def _exact_ensemble(case, d, n, dt):
    su = _Su2(d["lat"])
    m, e, S = _undriven(su, _t(d["init"]), n, dt)
    return {"times": dt * np.arange(n + 1), "mags": _host(m), "energy": _host(e), "final": _host(S)}


def _exact_dssf(case, d, n, dt):
    lat = d["lat"]
    su, every, L = _Su2(lat), case["every"], case["L"]
    nt = n // every
    pos = _t(lat.unit_cell.lattice_pos)
    q = 2.0 * math.pi / L * torch.arange(L, device=_dev(), dtype=torch.float64)
    qg = torch.stack(torch.meshgrid(q, q, q, indexing="ij"), -1)
    ph = torch.exp(-1j * (qg[..., None, :] * pos).sum(-1))       # [L, L, L, A]
    St = []

    def at(i, S):
        if i % every == 0 and i // every < nt:
            g = S.reshape(S.shape[0], L, L, L, su.A, 3).to(torch.complex128)
            St.append((torch.fft.fftn(g, dim=(1, 2, 3)) * ph[..., None]).sum(-2))
    m, _, _ = _undriven(su, _t(d["init"]), n, dt, False, at)
    sw = torch.fft.fft(torch.stack(St), dim=0)                   # [nt, B, L, L, L, 3]
    B = sw.shape[1]
    p = (sw.abs() ** 2).sum((1, 5)) / (B * su.N * nt)
    return {"sqw": _host(p.reshape(nt, -1).T.contiguous()), "mags": _host(m)}


def _exact_pump_probe(case, d, n, dt):
    su = _Su2(d["lat"])
    tp, sc = _scan(case["n_tau"], _tau_step(case))
    tp, amp = _t(tp), AMP * _t(sc)
    drive = (su.R * _t(d["field"])[:, None, :]).sum(-1)[su.atom]   # [N, 3]

    def f(x, t):
        g = _pulse(t, tp, amp).sum(-1)[:, None, None]
        return [_cross(su.field(x[0]) - g * drive, x[0])]
    S = _t(d["ground"]).expand(tp.shape[0], -1, -1)
    recs = []
    for i in range(n):
        S = _rk4(f, [S], T0_PULSE + i * dt, dt)[0]
        recs.append(su.records(S))                                 # the start is not observed
    m, k = _host(torch.stack(recs, 1)), case["n_tau"]
    return {"times": T0_PULSE + dt * np.arange(1, n + 1), "tau": _tau_step(case) * np.arange(k), "M0": m[0],
            "M1": m[1:1 + k], "M01": m[1 + k:]}


def _exact_dopri5(case, d, n, dt, tol=1e-8):
    su = _Su2(d["lat"])
    drive = (su.R * _t(d["field"])[:, None, :]).sum(-1)[su.atom]
    f = lambda x, t: _cross(su.field(x) - AMP * math.exp(-(t / (2.0 * WIDTH)) ** 2) * drive, x)
    c = [0.0, 1 / 5, 3 / 10, 4 / 5, 8 / 9, 1.0, 1.0]
    a = [[], [1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
         [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
         [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
         [35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
    e = [35 / 384 - 5179 / 57600, 0.0, 500 / 1113 - 7571 / 16695, 125 / 192 - 393 / 640,
         -2187 / 6784 + 92097 / 339200, 11 / 84 - 187 / 2100, -1 / 40]
    comb = lambda w, k: sum(q * v for q, v in zip(w, k) if q)
    eps = 2.220446049250313e-16
    S, h, m = _t(d["ground"]), dt, []
    for i in range(n):
        t = T0_PULSE + i * dt
        end = t + dt
        while end - t > eps:
            if t + h - end > eps:      # the last step lands on the interval's end
                h = end - t
            k = [f(S, t)]
            for row, ci in zip(a[1:], c[1:]):
                y = S + h * comb(row, k)
                k.append(f(y, t + ci * h))
            err = float(((h * comb(e, k)).abs() / (tol + tol * (S.abs() + h * k[0].abs()))).max())
            if err > 1.0:
                h *= max(0.9 * err ** (-1.0 / 3.0), 0.2)
                continue
            t, S = t + h, y
            if err < 0.5:
                h *= 0.9 * max(err, 5.0 ** -5) ** (-1.0 / 5.0)
        m.append(su.records(S))
    return {"times": T0_PULSE + dt * np.arange(1, n + 1), "mags": _host(torch.stack(m))}


def _exact_adjoint(case, d, n, dt, alpha=0.02):
    lat = d["lat"]
    su = _Su2(lat)
    dJ, dB = [], []
    for p in range(5):
        one = np.eye(5)[p]
        uc = model.build_kitaev_honeycomb(K=one[0], Gamma=one[1], Gammap=one[2], J=one[3], field_strength=one[4],
                                          field_direction=(1.0, 1.0, 1.0))
        lp = model.Lattice(uc, case["L1"], case["L2"], 1)
        dJ.append(_t(lp.bi_J.reshape(su.N, su.z, 3, 3)))
        dB.append(_t(lp.field))
    dJ, dB = torch.stack(dJ), torch.stack(dB)
    theta = _t(d["theta"]).requires_grad_(True)
    target = _t(d["target"]).reshape(-1, 3, 3)[:, 2]
    drive = (su.R * _t(_pulse_dirs(2))[:, None, :]).sum(-1)[su.atom]

    def steps(S, J, B, i0, i1):
        def f(x, t):
            H = su.field(x[0], J, B) - AMP * math.exp(-((t - 1.0) / (2.0 * WIDTH)) ** 2) * drive
            v = _cross(H, x[0])
            return [v - alpha * _cross(x[0], v) / x[0].norm(dim=-1, keepdim=True)]
        loss = 0.0
        for i in range(i0, i1):
            loss = loss + ((su.records(S)[:, 2] - target[i]) ** 2).sum(-1)
            S = _rk4(f, [S], i * dt, dt)[0]
        return S, loss

    J = torch.tensordot(theta, dJ, 1)
    B = torch.tensordot(theta, dB, 1)
    S = _t(d["init"]).expand(case["starts"], -1, -1)
    loss = 0.0
    for i in range(0, n, 25):
        S, part = torch.utils.checkpoint.checkpoint(steps, S, J, B, i, min(i + 25, n), use_reentrant=False)
        loss = loss + part
    loss = loss + ((su.records(S)[:, 2] - target[n]) ** 2).sum(-1)
    loss.sum().backward()
    return {"loss": _host(loss), "grad": _host(theta.grad)}


class _Mixed:
    """Fields of the Fe (3 components) and Tm (8 components) sites."""

    def __init__(self, ml):
        self.fe = _Su2(ml.su2)
        self.N = ml.N2
        assert ml.N3 == ml.N2 and len(ml.su3.bi_partner) == 0 and not np.any(ml.su3.onsite)
        z = int(ml.m2_offset[1])
        assert np.all(np.diff(ml.m2_offset.astype(np.int64)) == z) and np.all(np.diff(ml.m3_offset.astype(np.int64)) == z)
        idx = lambda p: torch.as_tensor(p.astype(np.int64).reshape(-1, z), device=_dev())
        self.z, self.p2, self.p3 = z, idx(ml.m2_partner), idx(ml.m3_partner)
        self.J2, self.J3 = _t(ml.m2_J.reshape(-1, z, 3, 8)), _t(ml.m3_J.reshape(-1, z, 8, 3))
        self.B3 = _t(ml.su3.field)
        self.R3 = _t(ml.su3.frames)
        g = torch.as_tensor(mixed_model.gell_mann(), dtype=torch.complex128, device=_dev())
        c = torch.einsum("aij,bjk->abik", g, g)
        self.f = (torch.einsum("abij,cji->abc", c - c.transpose(0, 1), g) / 4j).real.contiguous()
        self.atom = torch.arange(self.N, device=_dev()) % 4
        f2, f3 = _mixed_fields()
        # the drive enters in the storage frame: F^T b
        self.d2 = (self.fe.R.transpose(1, 2) * _t(f2)[:, None, :]).sum(-1)[self.atom]
        self.d3 = (self.R3.transpose(1, 2) * _t(f3)[:, None, :]).sum(-1)[self.atom]

    def fields(self, S, L, scale=1.0):
        H2, H3 = self.fe.field(S), -self.B3
        for k in range(self.z):
            H2 = H2 + scale * (self.J2[:, k] * L[..., self.p2[:, k], :][..., None, :]).sum(-1)
            H3 = H3 + scale * (self.J3[:, k] * S[..., self.p3[:, k], :][..., None, :]).sum(-1)
        return H2, H3

    def rhs(self, x, g, scale=1.0):
        H2, H3 = self.fields(x[0], x[1], scale)
        H2, H3 = H2 - g * self.d2, H3 - g * self.d3
        # f_abc H_b l_c
        dl = [sum(float(self.fh[a, b, c]) * H3[..., b] * x[1][..., c] for b, c in self.nz[a]) for a in range(8)]
        return [_cross(H2, x[0]), torch.stack(dl, -1)]

    def prepare_f(self):
        self.fh = self.f.cpu().numpy()
        self.nz = [[(b, c) for b in range(8) for c in range(8) if abs(self.fh[a, b, c]) > 1e-12] for a in range(8)]

    def records(self, S, L, energy=True):
        m2 = self.fe.records(S)
        atoms = L.reshape(L.shape[:-2] + (self.N // 4, 4, 8)).sum(-3)
        sg = torch.tensor([1.0, -1.0, 1.0, -1.0], dtype=torch.float64, device=_dev())
        g = (self.R3 * atoms[..., None, :]).sum(-1)
        m3 = torch.stack([(sg[:, None] * atoms).sum(-2), atoms.sum(-2), g.sum(-2)], -2) / self.N
        H2, H3 = self.fields(S, L)
        e = 0.5 * ((S * (H2 - self.fe.B)).sum((-1, -2)) + (L * (H3 - self.B3)).sum((-1, -2))) / (2 * self.N)
        return torch.cat([m2.flatten(-2), m3.flatten(-2), e[..., None]], -1)


def _mixed_run(case, d, n, dt, on_record, tangent=False):
    mx = _Mixed(d["ml"])
    mx.prepare_f()
    tp, sc = _scan(case["n_tau"], _tau_step(case))
    tp, amp = _t(tp), AMP * _t(sc)
    drv = lambda t: _pulse(t, tp, amp).sum(-1)[:, None, None]
    s2, s3 = d["ml"].split_state(d["ground"])
    x = [_t(v).repeat(tp.shape[0], 1, 1) for v in (s2, s3)]
    if not tangent:
        f = lambda x, t: mx.rhs(x, drv(t))
    else:
        x = x + [torch.zeros_like(x[0]), torch.zeros_like(x[1])]

        def f(x, t):
            g, z = drv(t), torch.ones((), dtype=torch.float64, device=_dev())
            v, dv = torch.func.jvp(lambda a, b, s: tuple(mx.rhs([a, b], g, s)), (x[0], x[1], z), (x[2], x[3], z))
            return list(v) + list(dv)
    for i in range(n + 1):
        on_record(i, mx, x)
        if i < n:
            x = _rk4(f, x, T0_PULSE + i * dt, dt)


def _split(m):
    return {"M2": m[..., :9].reshape(m.shape[:-1] + (3, 3)), "M3": m[..., 9:33].reshape(m.shape[:-1] + (3, 8)),
            "energy": m[..., 33]}


def _exact_mixed(case, d, n, dt):
    recs = []
    _mixed_run(case, d, n, dt, lambda i, mx, x: recs.append(mx.records(x[0], x[1])) if i else None)
    m, k = _host(torch.stack(recs, 1)), case["n_tau"]
    return {"times": T0_PULSE + dt * np.arange(1, n + 1), "tau": _tau_step(case) * np.arange(k),
            "M0": _split(m[0]), "M1": _split(m[1:1 + k]), "M01": _split(m[1 + k:])}


def _exact_mixed_grad(case, d, n, dt):
    recs, tan = [], []

    def rec(i, mx, x):
        r, dr = torch.func.jvp(lambda a, b: mx.records(a, b), (x[0], x[1]), (x[2], x[3]))
        recs.append(r)
        tan.append(dr)
    _mixed_run(case, d, n, dt, rec, True)
    m, tm, w, tg = torch.stack(recs), torch.stack(tan), _t(d["weights"]), _t(d["target"])[:, None]
    diff = w * (m - tg)
    return {"loss": _host((diff * (m - tg)).sum((0, 2))), "grad": _host(2.0 * (diff * tm).sum((0, 2))),
            "records": _host(m), "trecords": None}
