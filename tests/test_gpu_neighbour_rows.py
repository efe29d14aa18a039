"""Stage 2 of the neighbour cache on the GPU against the pair test written out in numpy: the row of
a particle is, over the leaf list of its owner leaf and the sorted range of each of those leaves,
every particle for which not both cut radii are smaller than the distance (NeighbourCache.cpp:
454-536), in that order.  The same IEEE operations on the same doubles, so the rows must be equal
exactly.  The sizes are the edges of the kernel's 64-wide pieces: members of a leaf below, at and
over 64, candidates below, at and over a full queue, near ones that are all or few of them."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from shamrock_amd._lib import check, lib  # noqa: E402

HTOL, R = 1.1, 2.0


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("shape", ["even", "clumps", "two_scales"])
@pytest.mark.parametrize("n,n_local,level", [(1, 1, 0), (63, 63, 6), (64, 64, 6), (65, 65, 6),
                                             (129, 100, 8), (640, 639, 2), (4000, 3001, 0),
                                             (4000, 4000, 3), (20_000, 15_000, 7)])
def test_rows(n, n_local, level, shape):
    """level: 2^level codes at least share a leaf; clumps: runs of 200 particles at one point's
    surroundings (leaves of several member batches); two_scales: radii that differ by a factor
    of 6, so pairs are kept by either side's radius."""
    print(f"[rows] n={n} n_local={n_local} level={level} {shape}", flush=True)
    rng = np.random.default_rng(n + level)
    pos = rng.uniform(0, 1, (n, 3))
    h = rng.uniform(0.8, 1.2, n) * 0.6 * n ** (-1 / 3)
    if shape == "clumps":
        pos = pos[np.arange(n) // 200 * 200] + 1e-3 * rng.normal(size=(n, 3))
        h = rng.uniform(0.5, 1.5, n) * 5e-4
    elif shape == "two_scales":
        h[pos[:, 0] > 0.5] *= 6 if n < 10_000 else 3
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (*pos.T, h)]
    p = [a.data_ptr() for a in t]
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    s = torch.cuda.current_stream().cuda_stream
    check(lib().shamx_tree_build(ctx, s, n, *p, level, HTOL))
    check(lib().shamx_neigh_build(ctx, s, n_local, *p, HTOL, R))
    sz, ns = (C.c_uint32 * 4)(), (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    check(lib().shamx_neigh_sizes(ctx, ns))
    L, I, P, PL = sz[1], sz[2], ns[1] + (ns[2] << 32), ns[3]
    ints = lambda k: torch.zeros(max(k, 1), dtype=torch.int32, device="cuda")
    order, first = ints(n), ints(L + 2)
    check(lib().shamx_tree_get(ctx, s, None, order.data_ptr(), first.data_ptr(), *[None] * 8))
    out = [ints(k) for k in (n_local, n_local, P, n_local, L, L, PL)]
    check(lib().shamx_neigh_get(ctx, s, *[a.data_ptr() for a in out]))
    torch.cuda.synchronize()
    lib().shamx_ctx_destroy(ctx)
    order, first, cnt, off, ids, own, lcnt, loff, lids = (
        a.cpu().numpy().view(np.uint32) for a in (order, first, *out))
    ra = h * HTOL
    cut = ra * ra * (R * R)
    assert int(cnt.sum()) == P
    for a in range(0, n_local, max(1, n_local // 500)):
        leaves = lids[loff[own[a]]:loff[own[a]] + lcnt[own[a]]] - I
        c = np.concatenate([order[first[k]:first[k + 1]] for k in leaves])
        d = pos[a] - pos[c]
        d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        want = c[~((d2 > cut[a]) & (d2 > cut[c]))]
        np.testing.assert_array_equal(ids[off[a]:off[a] + cnt[a]], want, err_msg=str(a))
