"""The force loop over the solver's rows (records fetched by four lanes together) against the
general loop on the same step: SHAMX_PAIR_LANES=2 takes the general one, whose sums have the same
order, so every field must keep its bits.  Row lengths of every remainder modulo four, rows empty
of neighbours, rows past a wave's shortest by far (clustered set), partial waves and blocks,
varying viscosity, every kernel, and particles whose h is far outside the reciprocal path."""
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from shamrock_amd import setups  # noqa: E402
from shamrock_amd.solver import GpuSolver  # noqa: E402

OUT = ("x", "vx", "ax", "ay", "az", "h", "u", "du", "alpha_AV")


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _two(cfg, f, run, monkeypatch, lanes):
    out = []
    for v in (None, lanes):
        with monkeypatch.context() as m:
            if v:
                m.setenv("SHAMX_PAIR_LANES", v)
            g = GpuSolver(cfg, f)
            logs = [run(g) for _ in range(2)]
            out.append((logs, {k: g.get(k) for k in OUT}, g.get_f64(12, g.n)))
            g.close()
    (la, fa, va), (lb, fb, vb) = out
    for p, q in zip(la, lb):
        for k in ("n_interacting", "next_dt", "energy", "corrector_iterations"):
            assert p[k] == q[k], k
    for k in OUT:
        np.testing.assert_array_equal(fa[k], fb[k], err_msg=k)
    np.testing.assert_array_equal(va, vb)


@pytest.mark.parametrize("kernel,side,av", [("M4", 5, 0), ("M4", 16, 1), ("M6", 9, 0), ("M6", 17, 1),
                                            ("M8", 11, 0), ("C2", 12, 0), ("C4", 13, 0),
                                            ("C6", 13, 0)])
def test_steps_keep_their_bits(kernel, side, av, monkeypatch):
    print(f"[force_rows] {kernel} {side} av={av}", flush=True)
    sys.stdout.flush()
    cfg, f = setups.random_box(side**3, seed=side, kernel=kernel)
    _two(dict(cfg, av_kind=av), f, lambda g: g.evolve_once(), monkeypatch, "2")


@pytest.mark.parametrize("case", ["plummer", "lonely", "tiny", "coincident"])
def test_passes_keep_their_bits(case, monkeypatch):
    """Density and force passes (no step need converge): a clustered set; particles too far apart
    to have neighbours; lengths of 1e-60, where h^4 leaves the reciprocal range and the plain
    divisions run; particles at the same point."""
    print(f"[force_rows] {case}", flush=True)
    if case == "plummer":
        cfg, f = setups.plummer(9_001, seed=3, r_max=30.0)
    else:
        cfg, f = setups.random_box(7**3, seed=5, periodic=False)
        if case == "lonely":
            f["h"] = f["h"] * 1e-3
        if case == "tiny":
            for k in ("x", "y", "z", "h"):
                f[k] = f[k] * 1e-60
            cfg = dict(cfg, gpart_mass=cfg["gpart_mass"] * 1e-180)
        if case == "coincident":
            for k in ("x", "y", "z"):
                f[k][1::2] = f[k][0:-1:2]
    _two(cfg, f, lambda g: g.density_force(), monkeypatch, "2")
