"""The neighbour build's bookkeeping of local rows (their sorted positions, the permutation of the
next storage reorder) and the batched field gathers of that reorder, against the oracle over whole
steps at the edges of the compaction's tiles: merged sets of one tile (1024 entries) and of several,
with images and without (then every position is local).  Neighbour lists must agree exactly and
fields within the parity contract's 1e-10; the storage order must be a permutation that a second
solver started in it continues from bit for bit."""
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

import oracle_lib as orc  # noqa: E402
from shamrock_amd import setups  # noqa: E402
from shamrock_amd.solver import FIELDS, GpuSolver  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("side,periodic", [(5, True), (6, True), (9, True), (12, True), (10, False),
                                           (11, False)])
def test_rows_and_reorder(side, periodic):
    print(f"[storage_rows] side={side} periodic={periodic}", flush=True)
    sys.stdout.flush()
    cfg, f = setups.random_box(side**3, seed=side, periodic=periodic)
    rng = np.random.default_rng(side)
    order = rng.permutation(f["x"].size)  # the storage starts far from any sorted order
    f = {k: v[order] for k, v in f.items()}
    g, o = GpuSolver(cfg, f), orc.Solver(cfg, f)
    for _ in range(3):
        lg, lo = g.evolve_once(), o.evolve_once()
        assert lg["n_pairs"] == lo["n_pairs"] and lg["n_merged"] == lo["n_merged"]
        a, b = g.transient(), o.transient()
        np.testing.assert_array_equal(a["part_cnt"], b["part_cnt"])
        np.testing.assert_array_equal(a["owner"], b["owner"])
        for k in ("x", "vx", "ax", "h", "u", "du"):
            p, q = g.get(k), o.get(k)
            scale = np.maximum(np.abs(q), np.abs(q).max() * 1e-3)
            assert np.max(np.abs(p - q) / scale) <= 1e-10, k
    so = g.storage_order()
    assert np.array_equal(np.sort(so), np.arange(g.n))
    twin = GpuSolver(cfg, {k: g.get(k) for k in FIELDS})
    twin.set_storage_order(so)
    tm = g.time()
    twin.set_time(tm["t"], tm["dt"], tm["cfl_mult"])
    assert g.evolve_once()["energy"] == twin.evolve_once()["energy"]
    for k in FIELDS:
        assert np.array_equal(g.get(k), twin.get(k)), k
    g.close()
    twin.close()


@pytest.mark.parametrize("side,periodic", [(5, True), (6, True), (9, True), (12, True), (10, False),
                                           (11, False)])
def test_row_contents(side, periodic):
    """The ids of the solver's own rows (fixed capacity, sorted positions, given back as particle
    ids) against the oracle's, over two steps of the sets above: the same ids in the same order
    where no two particles share a code, else the same ids (equal codes may sort either way)."""
    print(f"[storage_rows] contents side={side} periodic={periodic}", flush=True)
    cfg, f = setups.random_box(side**3, seed=side, periodic=periodic)
    order = np.random.default_rng(side).permutation(f["x"].size)
    f = {k: v[order] for k, v in f.items()}
    g, o = GpuSolver(cfg, f), orc.Solver(cfg, f)
    for _ in range(2):
        g.evolve_once(), o.evolve_once()
        a, b = g.transient(), o.transient()
        np.testing.assert_array_equal(a["part_cnt"], b["part_cnt"])
        np.testing.assert_array_equal(a["part_offset"], b["part_offset"])
        unique = np.unique(b["sorted_codes"]).size == b["sorted_codes"].size
        for i in range(g.n):
            k = slice(b["part_offset"][i], b["part_offset"][i] + b["part_cnt"][i])
            p, q = a["part_ids"][k], b["part_ids"][k]
            np.testing.assert_array_equal(*((p, q) if unique else (np.sort(p), np.sort(q))))
    g.close()
