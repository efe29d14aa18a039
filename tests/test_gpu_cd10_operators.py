"""The varying-viscosity operators on the GPU (div v, curl v, d(div v)/dt and the alpha they give)
against the oracle over whole steps, for every kernel, on disordered sets whose rows have every
length modulo the four lanes of a particle and whose particle counts are no multiple of the 64
particles of a block.  Both sides evaluate the same IEEE operations in the same order, so the
tolerance is the parity contract's 1e-10 relative."""
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


@pytest.mark.parametrize("kernel,side", [("M4", 6), ("M4", 7), ("C2", 7), ("M6", 8), ("C4", 9),
                                         ("M8", 11), ("C6", 11)])
def test_operators_match_the_oracle(kernel, side):
    print(f"[cd10_operators] {kernel} {side}", flush=True)
    sys.stdout.flush()
    cfg, f = setups.random_box(side**3, seed=side, kernel=kernel)
    cfg = dict(cfg, av_kind=1, alpha_min=0.0, alpha_max=1.0, sigma_decay=0.1)
    g, o = GpuSolver(cfg, f), orc.Solver(cfg, f)
    for _ in range(3):
        lg, lo = g.evolve_once(), o.evolve_once()
        assert lg["n_interacting"] > 0 and lg["n_pairs"] == lo["n_pairs"]
    for k in ("divv", "curlx", "curly", "curlz", "dtdivv", "alpha_AV", "ax", "du"):
        a, b = g.get(k), o.get(k)
        assert np.all(np.isfinite(b)) and np.any(b != 0), k
        scale = np.maximum(np.abs(b), np.abs(b).max() * 1e-3)
        assert np.max(np.abs(a - b) / scale) <= 1e-10, k
    g.close()
