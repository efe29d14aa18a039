"""The smoothing-length loop and the pass reductions on the GPU against the oracle: sweep counts and
h at the edges of the active-row compaction (4096 rows per tile), a convergence limit that no sweep
reaches (all rows drop out long before the last sweep, which must still be counted), loops shorter
and longer than the one before, and dt, energy and pair count past the one-block reduction (8192
block partials, reached at 524,289 particles).  h within the parity contract's 1e-10, counts equal."""
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

import oracle_lib as orc  # noqa: E402
from shamrock_amd import setups  # noqa: E402
from shamrock_amd.solver import GpuSolver  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _close(a, b, tol):
    scale = np.maximum(np.abs(b), np.abs(b).max() * 1e-3)
    return np.max(np.abs(a - b) / scale) <= tol


@pytest.mark.parametrize("side,epsilon_h", [(9, 1e-6), (15, 1e-12), (16, 1e-6), (17, 1e-12),
                                            (26, 1e-3), (26, 1e-6), (26, 1e-12)])
def test_sweeps_match_the_oracle(side, epsilon_h):
    print(f"[h_loop] side={side} epsilon_h={epsilon_h}", flush=True)
    sys.stdout.flush()
    cfg, f = setups.random_box(side**3, seed=side)
    cfg = dict(cfg, epsilon_h=epsilon_h, h_max_subcycles=100 if epsilon_h > 1e-9 else 1)
    g, o = GpuSolver(cfg, f), orc.Solver(cfg, f)
    for _ in range(3):
        if epsilon_h > 1e-9:
            lg, lo = g.evolve_once(), o.evolve_once()
            assert lg["h_iterations"] == lo["h_iterations"]
            assert lg["subcycles"] == lo["subcycles"]
        else:  # no step converges: the single-subcycle pass
            lg, lo = g.density_force(), o.density_force()
            assert lg["h_iterations"] == lo["h_iterations"] == cfg["h_iter_per_subcycles"]
        assert _close(g.get("h"), o.get("h"), 1e-10)
    g.close()


@pytest.mark.parametrize("side", [80, 81])
def test_pass_reductions(side, monkeypatch):
    """Below and above the one-block reduction.  One lane per particle takes a quarter of the
    blocks (always one-block here), so its counts and minima must be the same."""
    print(f"[pass_reductions] side={side}", flush=True)
    cfg, f = setups.sound_wave(side)
    g, o, one = GpuSolver(cfg, f), orc.Solver(cfg, f), GpuSolver(cfg, f)
    for _ in range(2):
        lg, lo = g.evolve_once(), o.evolve_once()
        with monkeypatch.context() as m:
            m.setenv("SHAMX_PAIR_LANES", "1")
            l1 = one.evolve_once()
        for k in ("n_interacting", "next_dt", "energy", "eps_v"):
            assert lg[k] == l1[k], k
        assert abs(lg["next_dt"] - lo["next_dt"]) <= 1e-10 * lo["next_dt"]
        e = cfg["gpart_mass"] * float(np.sum(
            g.get("u") + 0.5 * (g.get("vx")**2 + g.get("vy")**2 + g.get("vz")**2)))
        assert abs(lg["energy"] - e) <= 1e-12 * e
    g.close()
    one.close()
