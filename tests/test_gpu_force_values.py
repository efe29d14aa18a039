"""The force loop over the solver's rows against the general loop (SHAMX_PAIR_LANES=2) at values
where an operation of its own could round or propagate otherwise.  The two have the same operations
in the same order, so every output must keep its bits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from shamrock_amd import setups  # noqa: E402
from shamrock_amd.solver import GpuSolver  # noqa: E402

OUT = ("ax", "ay", "az", "du", "h")


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _pass(cfg, f, monkeypatch, lanes):
    with monkeypatch.context() as m:
        if lanes:
            m.setenv("SHAMX_PAIR_LANES", lanes)
        g = GpuSolver(cfg, f)
        log = g.density_force()
        out = {k: g.get(k) for k in OUT} | {"vsig": g.get_f64(12, g.n), "cs": g.transient()["cs"]}
        g.close()
    return log, out


def _same(cfg, f, monkeypatch):
    (la, a), (lb, b) = (_pass(cfg, f, monkeypatch, v) for v in (None, "2"))
    for k in ("n_interacting", "next_dt"):
        assert la[k] == lb[k], k
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    return a


@pytest.mark.parametrize("kernel", ["M4", "M6"])
def test_sound_speed_that_is_no_number(kernel, monkeypatch):
    """A negative internal energy gives a negative pressure and a NaN sound speed; such a particle
    has no signal speed above the maximum's start, 0 (the maximum passes over a NaN)."""
    print(f"[force_values] nan cs {kernel}", flush=True)
    cfg, f = setups.random_box(9**3, seed=4, kernel=kernel)
    f["u"][::13] *= -1
    out = _same(cfg, f, monkeypatch)
    assert np.isnan(out["cs"]).any() and (out["vsig"][::13] == 0).all()


@pytest.mark.parametrize("kernel", ["M4", "C2"])
@pytest.mark.parametrize("k", [0, -1, 5, -20])
def test_distances_of_all_ones(k, kernel, monkeypatch):
    """Two square layers at the distance 2^k (1 - 2^-53), whose significand is all ones: the one
    divisor that Newton's correction of a reciprocal leaves one ulp off (Markstein, 1990)."""
    print(f"[force_values] all ones 2^{k} {kernel}", flush=True)
    s, m = 2.0**k, 24
    i, j, l = np.meshgrid([0.0, 1 - 2.0**-53], np.arange(m), np.arange(m), indexing="ij")
    n = i.size
    rng = np.random.default_rng(k + 100)
    cfg, _ = setups.random_box(8, kernel=kernel, periodic=False)
    cfg = dict(cfg, gpart_mass=s**3)
    f = {"x": s * i.ravel(), "y": s * 1.25 * j.ravel(), "z": s * 1.5 * l.ravel(),
         "h": np.full(n, 1.2 * s), "u": 1 + rng.random(n)}
    f |= {c: rng.normal(0, 0.5, n) for c in ("vx", "vy", "vz")}
    assert np.sqrt(f["x"].max() ** 2) == s * (1 - 2.0**-53)
    _same(cfg, f, monkeypatch)


@pytest.mark.parametrize("kernel,side,av", [("M4", 5, 0), ("M4", 16, 1), ("M6", 17, 0),
                                            ("M8", 11, 0), ("C2", 12, 0), ("C4", 13, 0),
                                            ("C6", 13, 0)])
def test_wide_offsets(kernel, side, av, monkeypatch):
    """The force rows' 64-bit record offsets (sets of more than 29.8 M merged particles by
    themselves) against the 32-bit ones: whole steps, every kernel, same bits."""
    print(f"[force_values] wide {kernel} {side} av={av}", flush=True)
    cfg, f = setups.random_box(side**3, seed=side, kernel=kernel)
    cfg = dict(cfg, av_kind=av)
    out = []
    for wide in ("0", "1"):
        monkeypatch.setenv("SHAMX_WIDE_OFFSETS", wide)
        g = GpuSolver(cfg, f)
        logs = [g.evolve_once() for _ in range(2)]
        out.append(({k: g.get(k) for k in (*OUT, "x", "vx", "u")},
                    [(m["n_interacting"], m["next_dt"], m["energy"]) for m in logs]))
        g.close()
    assert out[0][1] == out[1][1]
    for k in out[0][0]:
        np.testing.assert_array_equal(out[0][0][k], out[1][0][k], err_msg=k)
