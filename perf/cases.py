"""The calls that programs make of this library, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" says which call it stands for:

  wave, box, sedov, disc, sod, hcp   steps of a simulation (GpuSolver.evolve_once) from a kept
                                     state, put back before them as in a replay or a parameter
                                     scan, and the read-out of the fields on the device
  plummer                            a density and force pass on a clustered set
  gradient                           a differentiable rollout, forward and backward
  phases                             the single-phase C entries on the caller's own arrays
  sort                               the key sort alone

`listed()` holds the named cases, `draw(rng)` gives more of the same ranges, `prepare` makes what a
program holds before the call (inputs from the seed alone), `run` is one pass, `work` what a pass
cannot do without, and `exact` the values of a pass in plain 64-bit torch, by direct sums over all
pairs, for the sets that are small enough.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from shamrock_amd import setups
from shamrock_amd._lib import KERNEL_IDS, check, lib
from shamrock_amd.adjoint import rollout_state
from shamrock_amd.math import get_ideal_hcp_box
from shamrock_amd.setups import KERNEL_HFACT, KERNEL_RKERN
from shamrock_amd.solver import GpuSolver

KERNELS = ("M4", "M6", "M8", "C2", "C4", "C6")
FIELDS = ("x", "y", "z", "vx", "vy", "vz", "ax", "ay", "az", "h", "u", "du")
WARM = 3  # steps of a run before its state is kept: the first has dt = 0 and settles h
EXACT_MAX = 40_000  # particles: direct sums over all pairs stay within seconds


def listed():
    return [
        # the smallest step anyone runs (the size of the smoke test): host reads and launches
        dict(name="wave_12", kind="wave", side=12, kernel="M4", mixed=False, steps=4),
        # the sound wave at its usual size, the first thing a user tries
        dict(name="wave_32", kind="wave", side=32, kernel="M4", mixed=False, steps=4),
        # a disordered set, wide kernel, mixed precision
        dict(name="box_34_m8_mixed", kind="box", side=34, kernel="M8", mixed=True, periodic=True,
             steps=4),
        # the Sod tube of the regression suite: varying viscosity, 646 such steps per run
        dict(name="sod_128", kind="sod", resol=128, steps=4),
        # fitting initial conditions through the solver, one optimiser iteration
        dict(name="gradient_kh_40", kind="gradient", side=40, steps=3, checkpoint=2,
             fp32=False),
        # the blast wave in mixed precision, an odd lattice side
        dict(name="sedov_101_mixed", kind="sedov", side=101, kernel="M6", mixed=True, steps=3),
        # the headline step: blast wave, 2.1 M particles, FP64
        dict(name="sedov_128", kind="sedov", side=128, kernel="M6", mixed=False, steps=3),
        # a protoplanetary disc with its central sink, free boundaries, h over a factor of 20
        dict(name="disc_1M_mixed", kind="disc", n=1_000_003, mixed=True, steps=3),
        # the homogeneous benchmark: HCP lattice, varying viscosity
        dict(name="hcp_cd10", kind="hcp", target=1 << 20, steps=3),
        # a strongly clustered set, leaves of hundreds of particles
        dict(name="plummer_4M", kind="plummer", n=4_194_304, mixed=False),
        # a program with its own time loop that calls the phases one by one
        dict(name="phases_33", kind="phases", side=33, kernel="M4"),
        # the key sort of a large set
        dict(name="sort_16M", kind="sort", n=16_777_216, bits=30),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("wave", "box", "sedov", "disc", "sod", "hcp", "plummer", "gradient",
                       "phases", "sort"))
    if kind == "wave":
        return dict(kind=kind, side=rng.randint(11, 48), kernel=rng.choice(("M4", "M6")),
                    mixed=rng.random() < 0.5, steps=rng.randint(2, 4))
    if kind == "box":
        return dict(kind=kind, side=rng.randint(16, 64), kernel=rng.choice(KERNELS),
                    mixed=rng.random() < 0.5, periodic=rng.random() < 0.7,
                    steps=rng.randint(1, 4))
    if kind == "sedov":
        return dict(kind=kind, side=_log_int(rng, 16, 127), kernel=rng.choice(("M4", "M6")),
                    mixed=rng.random() < 0.5, steps=rng.randint(1, 3))
    if kind == "disc":
        return dict(kind=kind, n=_log_int(rng, 20_000, 1_000_000), mixed=rng.random() < 0.5,
                    steps=rng.randint(1, 3))
    if kind == "sod":
        return dict(kind=kind, resol=rng.randint(32, 127), steps=rng.randint(1, 4))
    if kind == "hcp":
        return dict(kind=kind, target=_log_int(rng, 30_000, 1_000_000),
                    steps=rng.randint(1, 3))
    if kind == "plummer":
        return dict(kind=kind, n=_log_int(rng, 50_000, 4_000_000), mixed=rng.random() < 0.5)
    if kind == "gradient":
        return dict(kind=kind, side=rng.randint(12, 40), steps=rng.randint(2, 3),
                    checkpoint=rng.randint(1, 2), fp32=rng.random() < 0.5)
    if kind == "phases":
        return dict(kind=kind, side=rng.randint(10, 60), kernel=rng.choice(KERNELS))
    return dict(kind=kind, n=_log_int(rng, 1_000, 16_000_000), bits=rng.choice((30, 30, 32, 16)))


# ------------------------------------------------------------------------------- setups
def _disorder(cfg, f, seed, dr, pos=0.05, u=0.02, v=1e-3):
    """The lattice setups with the disorder a set has after some steps, from the seed."""
    rng = np.random.default_rng(seed)
    lo, hi = np.asarray(cfg["box_min"]), np.asarray(cfg["box_max"])
    for i, k in enumerate(("x", "y", "z")):
        p = f[k] + rng.uniform(-pos, pos, f[k].size) * dr
        if cfg["periodic"]:
            size = hi[i] - lo[i]
            p = lo[i] + np.mod(p - lo[i], size)
            p[p >= hi[i]] = lo[i]
        f[k] = p
    f["u"] = f["u"] * (1 + rng.uniform(-u, u, f["u"].size))
    for k in ("vx", "vy", "vz"):
        f[k] = f[k] + v * rng.standard_normal(f[k].size)
    return cfg, f


def _setup(case, seed):
    """(cfg, fields) of a step, phases or gradient case."""
    kind = case["kind"]
    if kind == "wave":
        cfg, f = setups.sound_wave(case["side"], case["kernel"])
        cfg, f = _disorder(cfg, f, seed, 1.0 / case["side"])
    elif kind == "box":
        cfg, f = setups.random_box(case["side"] ** 3, seed, case["kernel"], case["periodic"])
    elif kind == "phases":
        cfg, f = setups.random_box(case["side"] ** 3, seed, case["kernel"], False)
    elif kind == "sedov":
        cfg, f = setups.sedov(case["side"], case["kernel"])
        cfg, f = _disorder(cfg, f, seed, 1.0 / case["side"])
    elif kind == "disc":
        cfg, f = setups.disc(case["n"], seed)
    elif kind == "sod":
        cfg, f = setups.sod_tube(case["resol"])
        cfg, f = _disorder(cfg, f, seed, float(f["h"].min()), pos=0.02)
    elif kind == "hcp":
        # the box, lattice spacing and injected energy of the homogeneous benchmark
        dr = (0.74 * 1.2**3 / case["target"] / (4.0 / 3.0 * 3.1416)) ** (1.0 / 3.0)
        lo, hi = get_ideal_hcp_box(dr, (-0.6, -0.6, -0.6), (0.6, 0.6, 0.6))
        pos = setups.hcp_lattice(dr, lo, hi)
        vol = float(np.prod(np.subtract(hi, lo)))
        u = setups.kernel_W("M4", np.sqrt((pos**2).sum(1)), 16 * dr)
        cfg = setups.base_config("M4", lo, hi, gpart_mass=vol / len(pos), cfl_cour=0.1,
                                 cfl_force=0.1, av_kind=1)
        cfg, f = _disorder(cfg, setups.fields_from(pos, dr, u + 1e-3), seed, dr, pos=0.02)
    elif kind == "gradient":
        cfg, f = setups.kelvin_helmholtz(case["side"], seed=seed)
        cfg = dict(cfg, epsilon_h=1e-12, cfl_cour=0.1, cfl_force=0.1,
                   adjoint_fp32=int(case["fp32"]))
        rng = np.random.default_rng(seed)
        for k in ("vx", "vy", "vz"):
            f[k] = f[k] + 1e-3 * rng.standard_normal(f[k].size)
        f["u"] = f["u"] * (1 + 0.05 * rng.standard_normal(f["u"].size))
    cfg["mixed_precision"] = int(case.get("mixed", False))
    return cfg, f


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda()


class _Context:
    """The context handle of the single-phase entries."""

    def __init__(self):
        self.h = C.c_void_p()
        check(lib().shamx_ctx_create(C.byref(self.h)))

    def __del__(self):
        lib().shamx_ctx_destroy(self.h)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "sort":
        g = torch.Generator(device="cuda").manual_seed(seed)
        st["keys"] = torch.randint(-(1 << 31), 1 << 31, (case["n"],), generator=g, device="cuda",
                                   dtype=torch.int64).to(torch.int32)
        if case["bits"] < 32:
            st["keys"] &= (1 << case["bits"]) - 1
        st["work"] = torch.empty_like(st["keys"])
        st["perm"] = torch.empty_like(st["keys"])
        st["ctx"] = _Context()
    elif kind == "phases":
        st["cfg"], f = _setup(case, seed)
        st["f"] = {k: _dev(v) for k, v in f.items()}
        # the neighbour list keeps its room from build to build
        n, nn = _count(case)
        st["ids"] = torch.zeros(int(2 * n * nn), dtype=torch.int32, device="cuda")
        st["ctx"] = _Context()
    elif kind == "plummer":
        cfg, f = setups.plummer(case["n"], seed, r_max=30.0)
        cfg["mixed_precision"] = int(case["mixed"])
        st["solver"] = GpuSolver(cfg, f)
        st["h0"] = _dev(f["h"])
        st["out"] = {k: torch.empty_like(st["h0"]) for k in ("h", "ax", "ay", "az", "du")}
    elif kind == "gradient":
        st["cfg"], st["f"] = _setup(case, seed)
        f = st["f"]
        st["v0"] = _dev(np.stack([f["vx"], f["vy"], f["vz"]], 1))
        st["u0"] = _dev(f["u"])
    else:
        cfg, f = _setup(case, seed)
        s = GpuSolver(cfg, f)
        for _ in range(WARM):
            s.evolve_once()
        st["solver"], st["start"] = s, s.snapshot()
        st["out"] = {k: torch.empty(s.n, dtype=torch.float64, device="cuda") for k in FIELDS}
    return st


# ------------------------------------------------------------------------------- passes
def _read(st, log):
    out = {k: st["solver"].get_device(k, out=v) for k, v in st["out"].items()}
    out["next_dt"] = log["next_dt"]
    out["pairs"] = log["n_interacting"]
    return out


def _run_phases(st):
    f, cfg, L = st["f"], st["cfg"], lib()
    n, k = f["x"].numel(), KERNEL_IDS[cfg["kernel"]]
    R = KERNEL_RKERN[cfg["kernel"]]
    m, ctx, s = cfg["gpart_mass"], st["ctx"].h, C.c_void_p(torch.cuda.current_stream().cuda_stream)
    new = lambda: torch.empty(n, dtype=torch.float64, device="cuda")  # noqa: E731
    x, y, z, h = (f[c].data_ptr() for c in "xyzh")
    check(L.shamx_tree_build(ctx, s, n, x, y, z, h, cfg["tree_reduction_level"], 1.1))
    check(L.shamx_neigh_build(ctx, s, n, x, y, z, h, 1.1, R))
    sz = (C.c_uint32 * 4)()
    check(L.shamx_neigh_sizes(ctx, sz))
    cnt = torch.empty(n, dtype=torch.int32, device="cuda")
    off, ids = torch.empty_like(cnt), st["ids"]
    if sz[1] > ids.numel():
        raise RuntimeError("more neighbours than the list has room for")
    order = torch.empty_like(cnt)
    check(L.shamx_neigh_get(ctx, s, cnt.data_ptr(), off.data_ptr(), ids.data_ptr(), None, None,
                            None, None))
    check(L.shamx_tree_get(ctx, s, None, order.data_ptr(), *[None] * 9))
    csr = (cnt.data_ptr(), off.data_ptr(), ids.data_ptr())
    hn, eps = f["h"].clone(), torch.full_like(f["h"], 100.0)
    mm = (C.c_double * 2)()
    check(L.shamx_h_iterate(s, k, n, *csr, x, y, z, h, hn.data_ptr(), eps.data_ptr(), m, 1.1, 1.1,
                            0, mm))
    o = {c: new() for c in ("omega", "P", "cs", "ax_old", "ay_old", "az_old", "du_old", "vsig",
                            "dt")}
    acc = {c: f[c].clone() for c in ("ax", "ay", "az", "du")}
    p = {c: v.data_ptr() for c, v in {**o, **acc}.items()}
    hp, u = hn.data_ptr(), f["u"].data_ptr()
    check(L.shamx_omega(s, k, n, *csr, x, y, z, hp, p["omega"], m))
    check(L.shamx_eos(s, k, n, cfg["eos_kind"], cfg["gamma"], cfg["eos_cs"], cfg["eos_cs0"],
                      cfg["eos_q"], cfg["eos_r0"], hp, u, x, y, z, p["P"], p["cs"], m))
    dt = (C.c_double * 1)()
    check(L.shamx_force(s, k, n, *csr, x, y, z, *(f[c].data_ptr() for c in ("vx", "vy", "vz")), hp,
                        p["omega"], u, p["P"], p["cs"], p["ax"], p["ay"], p["az"], p["du"],
                        p["ax_old"], p["ay_old"], p["az_old"], p["du_old"], p["vsig"], p["dt"], m,
                        cfg["alpha_u"], cfg["alpha_AV"], cfg["beta_AV"], cfg["cfl_cour"],
                        cfg["cfl_force"], 0, dt))
    return dict(order=order, cnt=cnt, ids=ids, h=hn, omega=o["omega"], P=o["P"], cs=o["cs"],
                vsig=o["vsig"], dt=o["dt"], **acc)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "sort":
        st["work"].copy_(st["keys"])
        s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        check(lib().shamx_sort(st["ctx"].h, s, case["n"], case["bits"], st["work"].data_ptr(),
                               st["perm"].data_ptr()))
        return dict(keys=st["work"], perm=st["perm"])
    if kind == "phases":
        return _run_phases(st)
    if kind == "plummer":
        st["solver"].set_device("h", st["h0"])  # every pass starts from the same h
        return _read(st, st["solver"].density_force())
    if kind == "gradient":
        v0 = st["v0"].clone().requires_grad_(True)
        u0 = st["u0"].clone().requires_grad_(True)
        rho, u = rollout_state(st["cfg"], st["f"], v0, u0, case["steps"],
                               checkpoint_every=case["checkpoint"])
        (rho.square().mean() + u.square().mean()).backward()
        return dict(rho=rho.detach(), u=u.detach(), v_grad=v0.grad, u_grad=u0.grad)
    st["solver"].restore(st["start"])
    for _ in range(case["steps"]):
        log = st["solver"].evolve_once()
    return _read(st, log)


# ------------------------------------------------------------------------------- work
def _count(case):
    """Particles and mean neighbours inside the kernel support of a case."""
    kind = case["kind"]
    kernel = case.get("kernel", "M6" if kind == "sod" else "M4")
    nn = 4.0 / 3.0 * math.pi * (KERNEL_HFACT[kernel] * KERNEL_RKERN[kernel]) ** 3
    if kind in ("wave", "box", "sedov", "phases"):
        n = case["side"] ** 3
    elif kind == "gradient":
        n = case["side"] ** 3
    elif kind == "sod":
        n = case["resol"] * 648
    elif kind == "hcp":
        n = case["target"]
    else:
        n = case["n"]
    return n, nn


def work(case):
    n, nn = _count(case)
    kind = case["kind"]
    if kind == "sort":
        return dict(bytes=12 * n, flops=0)  # keys in, keys and permutation out
    # per pair of neighbours: one density sweep (40), the grad-h sum (40) and the forces (120)
    pair = 200
    if kind in ("sod", "hcp"):
        pair += 170  # div v, curl v, d(div v)/dt
    passes = case.get("steps", 1)
    if kind == "gradient":
        pair *= 3  # the reverse pass evaluates each pair function and its derivative
    # the twelve fields read and written once per step
    return dict(bytes=passes * n * 2 * 12 * 8, flops=passes * n * nn * pair)


# ------------------------------------------------------------------------------- exact values
def _poly(kernel, q):
    """f(q), f'(q) of the kernel: W = norm f(r / h) / h^3."""
    z = torch.zeros_like(q)
    if kernel in ("M4", "M6", "M8"):
        p, R, c = {"M4": (3, 2, (0.25, -1.0)), "M6": (5, 3, (1.0, -6.0, 15.0)),
                   "M8": (7, 4, (1.0, -8.0, 28.0, -56.0))}[kernel]
        f, df = z.clone(), z.clone()
        for i, ci in enumerate(c):
            t = (R - i - q).clamp_min(0)
            f += ci * t**p
            df -= ci * p * t ** (p - 1)
        return f, df
    t = (1 - q / 2).clamp_min(0)
    if kernel == "C2":
        return t**4 * (1 + 2 * q), torch.where(q < 2, 2 * (t**4 - t**3 * (1 + 2 * q)), z)
    if kernel == "C4":
        s = (q - 2).clamp_max(0)
        return t**6 * (1 + 3 * q + 35 / 12 * q * q), 7 / 96 * s**5 * q * (2 + 5 * q)
    s = (q - 2).clamp_max(0)
    return (t**8 * (1 + 4 * q + 25 / 4 * q * q + 4 * q**3),
            11 / 512 * s**7 * q * (2 + 7 * q + 8 * q * q))


_NORM = {"M4": 1 / math.pi, "M6": 1 / (120 * math.pi), "M8": 1 / (6720 * math.pi),
         "C2": 21 / (16 * math.pi), "C4": 495 / (256 * math.pi), "C6": 1365 / (512 * math.pi)}


class _Exact:
    """A set of particles evaluated by direct sums over all pairs (nearest image)."""

    def __init__(self, cfg, f):
        self.cfg, self.k = cfg, cfg["kernel"]
        self.m, self.R, self.hf = cfg["gpart_mass"], KERNEL_RKERN[self.k], KERNEL_HFACT[self.k]
        self.norm = _NORM[self.k]
        self.p = torch.stack([_dev(f[c]) for c in "xyz"], 1)
        self.v = torch.stack([_dev(f["v" + c]) for c in "xyz"], 1)
        self.a = torch.stack([_dev(f["a" + c]) for c in "xyz"], 1)
        self.h, self.u, self.du = (_dev(f[c]) for c in ("h", "u", "du"))
        self.lo = torch.tensor(cfg["box_min"], dtype=torch.float64, device="cuda")
        self.size = torch.tensor(cfg["box_max"], dtype=torch.float64, device="cuda") - self.lo
        self.n, self.t, self.dt, self.cfl = self.p.shape[0], 0.0, 0.0, 1e-2
        self.rows = max(1, 16_000_000 // self.n)

    def pairs(self, idx):
        """r_a - r_b and |r_ab| of the particles idx against all, in chunks of rows."""
        for i in range(0, idx.numel(), self.rows):
            a = idx[i:i + self.rows]
            d = self.p[a][:, None, :] - self.p[None, :, :]
            if self.cfg["periodic"]:
                d = d - self.size * torch.round(d / self.size)
            yield a, d, d.square().sum(-1).sqrt()

    def rho(self, h):
        return self.m * (self.hf / h) ** 3

    def newton(self, idx, h_old, h, up_all, up_iter):
        """One Newton sweep of the density equation: (h, eps) of the particles idx."""
        hn, en = h.clone(), torch.empty(idx.numel(), dtype=torch.float64, device="cuda")
        at = 0
        for a, _, r in self.pairs(idx):
            ha = h[a]
            fq, dq = _poly(self.k, r / ha[:, None])
            s = self.m * self.norm * fq.sum(1) / ha**3
            ds = -self.m * self.norm * (3 * fq + r / ha[:, None] * dq).sum(1) / ha**4
            rh = self.rho(ha)
            new = ha - (s - rh) / (ds + 3 * rh / ha)
            new = torch.minimum(torch.maximum(new, ha / up_iter), ha * up_iter)
            ok = new < h_old[a] * up_all
            en[at:at + a.numel()] = torch.where(ok, (new - ha).abs() / h_old[a],
                                                torch.full_like(ha, -1.0))
            hn[a] = torch.where(ok, new, h_old[a] * up_all)
            at += a.numel()
        return hn, en

    def solve_h(self):
        c = self.cfg
        for _ in range(c["h_max_subcycles"]):
            h_old = self.h.clone()
            eps = torch.full_like(self.h, 100.0)
            for _ in range(c["h_iter_per_subcycles"]):
                idx = (eps > 1e-6).nonzero().flatten()
                self.h, eps[idx] = self.newton(idx, h_old, self.h, c["htol_up_coarse"],
                                               c["htol_up_fine"])
                if float(eps.max()) < c["epsilon_h"]:
                    break
            if float(eps.max()) < c["epsilon_h"] and not float(eps.min()) < 0:
                return
        raise RuntimeError("h does not converge")

    def omega(self):
        om = torch.empty_like(self.h)
        for a, _, r in self.pairs(torch.arange(self.n, device="cuda")):
            ha = self.h[a]
            fq, dq = _poly(self.k, r / ha[:, None])
            s = -self.m * self.norm * (3 * fq + r / ha[:, None] * dq).sum(1) / ha**4
            om[a] = 1 + ha / (3 * self.rho(ha)) * s
        return om

    def eos(self):
        rho = self.rho(self.h)
        if self.cfg["eos_kind"] == 0:
            P = (self.cfg["gamma"] - 1) * rho * self.u
            return P, (self.cfg["gamma"] * P / rho).sqrt()
        return self.cfg["eos_cs"] ** 2 * rho, torch.full_like(rho, self.cfg["eos_cs"])

    def force(self, om, P, cs):
        """a, du/dt, signal speed and the number of interacting pairs (constant viscosity)."""
        c, m = self.cfg, self.m
        al, be = c["alpha_AV"], c["beta_AV"]
        rho, h = self.rho(self.h), self.h
        a_, du, vs, count = (torch.empty_like(self.p), torch.empty_like(h), torch.empty_like(h), 0)
        for a, d, r in self.pairs(torch.arange(self.n, device="cuda")):
            ha, hb = h[a][:, None], h[None, :]
            near = r <= torch.maximum(ha, hb) * self.R
            inv = torch.where(r >= 1e-9, 1 / r, 0.0)
            ru = d * inv[..., None]
            dv = self.v[a][:, None, :] - self.v[None, :, :]
            vr = (dv * ru).sum(-1)
            Fa = self.norm * _poly(self.k, r / ha)[1] / ha**4
            Fb = self.norm * _poly(self.k, r / hb)[1] / hb**4
            ra, rb = rho[a][:, None], rho[None, :]
            ca, cb = cs[a][:, None], cs[None, :]
            Pa = P[a][:, None] + (-0.5 * ra * (al * ca + be * vr.abs()) * vr).clamp_min(0)
            Pb = P[None, :] + (-0.5 * rb * (al * cb + be * vr.abs()) * vr).clamp_min(0)
            oa, ob = om[a][:, None], om[None, :]
            t = -m * (Pa / (ra * ra * oa) * Fa + Pb / (rb * rb * ob) * Fb)
            a_[a] = torch.where(near[..., None], t[..., None] * ru, 0.0).sum(1)
            vu = ((P[a][:, None] - P[None, :]).abs() / (0.5 * (ra + rb))).sqrt()
            w = Pa / (oa * ra * ra) * m * vr * Fa + m * c["alpha_u"] * vu * 0.5 * (
                self.u[a][:, None] - self.u[None, :]) * (Fa / (oa * ra) + Fb / (rb * ob))
            du[a] = torch.where(near, w, 0.0).sum(1)
            vs[a] = torch.where(near, ca + 2 * vr.abs(), 0.0).amax(1)
            count += int(near.sum())
        return a_, du, vs, count

    def step(self):
        c, dt = self.cfg, self.dt
        half = self.v + dt / 2 * self.a
        self.p = self.p + dt * half
        self.v = half + dt / 2 * self.a
        self.u = self.u + dt / 2 * self.du + dt / 2 * self.du
        if c["periodic"]:
            self.p = self.lo + torch.remainder(self.p - self.lo, self.size)
        self.solve_h()
        om = self.omega()
        while True:
            a0, du0 = self.a, self.du
            self.a, self.du, vs, self.count = self.force(om, *self.eos())
            lim = torch.minimum(c["cfl_cour"] * self.cfl * self.h / vs, c["cfl_force"] * self.cfl *
                                (self.h / self.a.square().sum(1).sqrt()).sqrt())
            dv = dt / 2 * (self.a - a0)
            self.v = self.v + dv
            self.u = self.u + dt / 2 * (self.du - du0)
            vmean = float(self.v.square().sum() / self.n) ** 0.5
            ev = float(dv.square().sum(1).max()) ** 0.5 / vmean if vmean > 0 else 0.0
            if ev <= 1e-2:
                break
            self.cfl /= 2
        self.dt, self.t = float(lim.min()), self.t + dt
        s = c["cfl_multiplier_stiffness"]
        self.cfl = (self.cfl * s + 1) / (s + 1)


def exact(case, seed):
    if case["kind"] not in ("wave", "box", "phases") or _count(case)[0] > EXACT_MAX:
        return None
    cfg, f = _setup(case, seed)
    e = _Exact(cfg, f)
    if case["kind"] == "phases":
        e.h, _ = e.newton(torch.arange(e.n, device="cuda"), e.h, e.h, 1.1, 1.1)
        om = e.omega()
        P, cs = e.eos()
        a, du, vs, _ = e.force(om, P, cs)
        dt = torch.minimum(cfg["cfl_cour"] * e.h / vs,
                           cfg["cfl_force"] * (e.h / a.square().sum(1).sqrt()).sqrt())
        return dict(order=None, cnt=None, ids=None, h=e.h, omega=om, P=P, cs=cs, vsig=vs, dt=dt,
                    ax=a[:, 0], ay=a[:, 1], az=a[:, 2], du=du)
    for _ in range(WARM + case["steps"]):
        e.step()
    out = {k + c: t[:, i] for k, t in (("", e.p), ("v", e.v), ("a", e.a))
           for i, c in enumerate("xyz")}
    return dict(out, h=e.h, u=e.u, du=e.du, next_dt=e.dt, pairs=None)
