"""The mixed loops (h sweep, force) that fetch a particle's records by its four lanes together,
against the one-lane loops (SHAMX_PAIR_LANES=1), where each lane gathers its own records: row lengths
of every remainder modulo a turn's 8 and 16 entries, rows that hold only the particle itself, waves
with rows of very unequal length, partial waves.  One dropped or doubled entry is a term of the sum.

Bounds (u = 2^-24): the pair terms are the same FP32 operations on the same records in both, but for
Omega, a sum of FP32 terms in another order, which enters a term as a divisor (so it changes a term
by as much as the two runs' Omegas differ).  The sums are Kahan sums kept with their compensation,
2 u of the sum of magnitudes each; so accelerations and du/dt may differ by 16 u of the sum of their
terms' magnitudes, and by those relative differences of Omega, per particle.  h by 64 u: the density
sum's 4 u over the slope of Newton's step, which is at least rho / (8 h) here."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from shamrock_amd import setups  # noqa: E402
from shamrock_amd.solver import GpuSolver  # noqa: E402

U = 2.0**-24


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _case(case):
    if case == "plummer":
        cfg, f = setups.plummer(2_501, seed=3, r_max=30.0)
        f["vx"] = np.random.default_rng(1).normal(0, 0.1, f["x"].size)
    else:
        cfg, f = setups.random_box(int(case.split("_")[0])**3, seed=5, periodic=False)
        if case.endswith("lonely"):
            f["h"] = f["h"] * 1e-3
        if case.endswith("coincident"):
            for k in ("x", "y", "z"):
                f[k][1::2] = f[k][0:-1:2]
        if case.endswith("unequal"):
            f["h"][::29] *= 4
    return dict(cfg, mixed_precision=1), f


def _both(cfg, f, monkeypatch):
    out = []
    for lanes in ("4", "1"):
        monkeypatch.setenv("SHAMX_PAIR_LANES", lanes)
        g = GpuSolver(cfg, f)
        log = g.density_force()
        out.append((log, {k: g.get(k) for k in ("ax", "ay", "az", "du", "h")}, g.transient()))
        g.close()
    return out


def _bounds(cfg, f, h, t, t2):
    """Per particle, the bounds of the acceleration and of du/dt: their pair terms' magnitudes (M4)
    times 16 u and the relative difference of the Omega that divides the term."""
    n, m = h.size, cfg["gpart_mass"]
    pos = np.stack([f["x"], f["y"], f["z"]], 1)
    v = np.stack([np.broadcast_to(f[k], n) for k in ("vx", "vy", "vz")], 1)
    u = np.broadcast_to(f["u"], n)
    rho, P, cs = m * (1.2 / h)**3, t["P"][:n], t["cs"][:n]
    om = np.abs(t["omega"])
    w = 16 * U + np.abs(t["omega"] - t2["omega"]) / om
    df = lambda q: np.where(q < 1, -3 * q + 9 / 4 * q * q,
                            np.where(q < 2, -3 + 3 * q - 3 / 4 * q * q, 0))
    A, D = np.zeros(n), np.zeros(n)
    for a in range(n):
        d = pos[a] - pos
        r = np.sqrt((d * d).sum(1))
        on = r <= 2 * np.maximum(h[a], h)
        d, r, b = d[on], r[on], np.flatnonzero(on)
        vr = ((v[a] - v[b]) * d).sum(1) / np.maximum(r, 1e-300)
        Fa, Fb = (np.abs(df(r / x)) / (np.pi * x**4) for x in (h[a], h[b]))
        q = [np.maximum(-0.5 * rho[i] * (cfg["alpha_AV"] * cs[i] + cfg["beta_AV"] * np.abs(vr)) *
                        vr, 0) for i in (a, b)]
        ta = w[a] * (P[a] + q[0]) * Fa / (rho[a]**2 * om[a])
        A[a] = m * (ta + w[b] * (P[b] + q[1]) * Fb / (rho[b]**2 * om[b])).sum()
        vu = np.sqrt(np.abs(P[a] - P[b]) / ((rho[a] + rho[b]) / 2))
        D[a] = m * (ta * np.abs(vr) + cfg["alpha_u"] * vu * np.abs(u[a] - u[b]) / 2 *
                    (w[a] * Fa / (rho[a] * om[a]) + w[b] * Fb / (rho[b] * om[b]))).sum()
    return A, D


@pytest.mark.parametrize("case", ["2", "5", "7", "9", "7_lonely", "7_coincident", "9_unequal",
                                  "plummer"])
def test_force(case, monkeypatch):
    print(f"[mixed_rows] force {case}", flush=True)
    cfg, f = _case(case)
    cfg["h_iter_per_subcycles"] = 0  # the same h in both
    (la, a, ta), (lb, b, tb) = _both(cfg, f, monkeypatch)
    assert la["n_interacting"] == lb["n_interacting"]
    np.testing.assert_array_equal(a["h"], b["h"])
    if case == "7_lonely":
        assert la["n_interacting"] == a["h"].size
    A, D = _bounds(cfg, f, b["h"], tb, ta)
    for k, s in (("ax", A), ("ay", A), ("az", A), ("du", D)):
        assert (np.abs(a[k] - b[k]) <= s).all(), k
    np.testing.assert_allclose(ta["vsig"], tb["vsig"], rtol=4 * U)


@pytest.mark.parametrize("case", ["5", "7", "9", "16", "plummer"])
def test_sweeps(case, monkeypatch):
    print(f"[mixed_rows] sweeps {case}", flush=True)
    cfg, f = _case(case)
    (la, a, _), (lb, b, _) = _both(cfg, f, monkeypatch)
    np.testing.assert_allclose(a["h"], b["h"], rtol=64 * U)
