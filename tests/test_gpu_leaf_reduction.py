"""Leaf reduction on the GPU (the two-launch compaction per iteration) against the oracle's tree at
the edges of its tiles: 1024 list entries per tile (4096 past 2^23 positions), one launch for a
single tile, 64 entries per ballot, runs of equal codes across tile boundaries, reduction levels 0 to 4.  Index products, so
exactly equal."""
import ctypes as C
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

import oracle_lib as orc  # noqa: E402
from shamrock_amd._lib import check, lib  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("runs", [False, True])
@pytest.mark.parametrize("n,level", [(1, 3), (63, 3), (64, 1), (65, 4), (1023, 3), (1024, 3),
                                     (1025, 3), (8193, 0), (70_001, 3), (70_001, 2)])
def test_reduction_matches_the_oracle(n, level, runs):
    print(f"[leaf_reduction] n={n} level={level} runs={runs}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(n + level)
    pos = rng.uniform(-1, 1, (n, 3))
    if runs:  # long runs of equal codes: points copied thousands of times
        pos = pos[rng.integers(0, max(1, n // 3000), n)]
        pos[0], pos[-1] = (-1, -1, -1), (1, 1, 1)
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (*pos.T, np.full(n, 0.1))]
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    s = torch.cuda.current_stream().cuda_stream
    check(lib().shamx_tree_build(ctx, s, n, *[a.data_ptr() for a in t], level, 1.1))
    sz = (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    L, I = sz[1], sz[2]
    g = dict(sorted=n, reduc_map=L + 2, lchild=I, rchild=I, endrange=I)
    g = {k: torch.zeros(max(m, 1), dtype=torch.int32, device="cuda") for k, m in g.items()}
    check(lib().shamx_tree_get(ctx, s, g["sorted"].data_ptr(), None, g["reduc_map"].data_ptr(),
                               g["lchild"].data_ptr(), g["rchild"].data_ptr(), None, None,
                               g["endrange"].data_ptr(), None, None, None))
    torch.cuda.synchronize()
    lib().shamx_ctx_destroy(ctx)
    o = orc.Tree(pos, orc.bbox(pos), level, bits=32)
    assert L == o.L and I == o.I
    got = {k: v.cpu().numpy().view(np.uint32) for k, v in g.items()}
    np.testing.assert_array_equal(got["sorted"], o.sorted_codes[:n])
    np.testing.assert_array_equal(got["reduc_map"], o.reduc_map)
    for k in ("lchild", "rchild", "endrange"):
        np.testing.assert_array_equal(got[k][:I], getattr(o, k), err_msg=k)


def _delta(m, i, j):
    """Common leading bits of the codes at i and j, -1 outside the array (math.hpp:825-828)."""
    n = m.size
    ok = (i >= 0) & (i < n) & (j >= 0) & (j < n)
    x = m[np.clip(i, 0, n - 1)] ^ m[np.clip(j, 0, n - 1)]
    return np.where(ok, 32 - np.frexp(x.astype(np.float64))[1], -1)


def test_reduction_large_tiles():
    """The large tiles against the iteration (reduction_alg.cpp:196-244) in numpy."""
    n, level = (1 << 23) + 5, 3
    print(f"[leaf_reduction] n={n} level={level}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    t = [torch.rand(n, generator=g, device="cuda", dtype=torch.float64) for _ in range(3)]
    h = torch.full_like(t[0], 0.1)
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    s = torch.cuda.current_stream().cuda_stream
    check(lib().shamx_tree_build(ctx, s, n, *[a.data_ptr() for a in (*t, h)], level, 1.1))
    sz = (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    L = sz[1]
    codes = torch.zeros(n, dtype=torch.int32, device="cuda")
    rmap = torch.zeros(L + 2, dtype=torch.int32, device="cuda")
    check(lib().shamx_tree_get(ctx, s, codes.data_ptr(), None, rmap.data_ptr(), *[None] * 8))
    torch.cuda.synchronize()
    lib().shamx_ctx_destroy(ctx)
    m = codes.cpu().numpy().view(np.uint32)
    F = np.flatnonzero(np.r_[True, m[1:] != m[:-1]])
    for _ in range(level):
        b1, b2, nx = np.r_[-1, F[:-1]], np.r_[-2, -1, F[:-2]], np.r_[F[1:], n]
        d0, dm, dmm = _delta(m, F, nx), _delta(m, F, b1), _delta(m, b1, b2)
        F = F[~((d0 < dm) & (dmm < dm))]
    assert L == F.size
    np.testing.assert_array_equal(rmap.cpu().numpy().view(np.uint32)[:L], F)
