"""The neighbour build on positions other than those that the tree's boxes were made from (a caller
who moves particles between shamx_tree_build and shamx_neigh_build).  The owner of a particle is the
last leaf whose box contains the position it is passed with (NeighbourCache.cpp:406-451), wherever
the tree keeps the particle; one inside no box is refused.  Comparisons of the same doubles: owners
and the moved particles' rows must be equal exactly to numpy's."""
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


def _dev(pos, h):
    return [torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda() for a in (*pos.T, h)]


def _build(ctx, n, level, t, moved):
    s = torch.cuda.current_stream().cuda_stream
    check(lib().shamx_tree_build(ctx, s, n, *[a.data_ptr() for a in t], level, HTOL))
    check(lib().shamx_neigh_build(ctx, s, n, *[a.data_ptr() for a in moved], HTOL, R))


def _read(ctx, n):
    s = torch.cuda.current_stream().cuda_stream
    sz, ns = (C.c_uint32 * 4)(), (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    check(lib().shamx_neigh_sizes(ctx, ns))
    L, I, P, PL = sz[1], sz[2], ns[1] + (ns[2] << 32), ns[3]
    ints = lambda k: torch.zeros(max(k, 1), dtype=torch.int32, device="cuda")
    box = [torch.zeros(3 * (I + L), dtype=torch.float64, device="cuda") for _ in range(2)]
    order, first = ints(n), ints(L + 2)
    check(lib().shamx_tree_get(ctx, s, None, order.data_ptr(), first.data_ptr(), *[None] * 5,
                               *[b.data_ptr() for b in box], None))
    out = [ints(k) for k in (n, n, P, n, L, L, PL)]
    check(lib().shamx_neigh_get(ctx, s, *[a.data_ptr() for a in out]))
    torch.cuda.synchronize()
    lo, hi = (b.cpu().numpy().reshape(-1, 3)[I:] for b in box)
    return (I, lo, hi, *(a.cpu().numpy().view(np.uint32) for a in (order, first, *out)))


@pytest.mark.parametrize("n,level", [(40, 0), (70, 1), (600, 0), (600, 4), (5000, 2), (40_000, 1)])
def test_moved_particles(n, level):
    """One particle in 37 moves to another one's place: mostly into boxes that no other leaf's box
    meets, before and after its own leaf."""
    print(f"[owner_leaves] n={n} level={level}", flush=True)
    rng = np.random.default_rng(n + level)
    pos = rng.uniform(0, 1, (n, 3))
    h = rng.uniform(0.8, 1.2, n) * 0.6 * n ** (-1 / 3)
    who = np.arange(0, n, 37)
    new = pos.copy()
    new[who] = pos[rng.integers(0, n, who.size)]
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    _build(ctx, n, level, _dev(pos, h), _dev(new, h))
    I, lo, hi, order, first, cnt, off, ids, own, lcnt, loff, lids = _read(ctx, n)
    lib().shamx_ctx_destroy(ctx)
    cut = (h * HTOL) * (h * HTOL) * (R * R)
    mine = np.empty(n, np.int64)  # the leaf that keeps each particle
    for l in range(lo.shape[0]):
        mine[order[first[l]:first[l + 1]]] = l
    elsewhere = 0
    for a in np.unique(np.r_[who, np.arange(0, n, max(1, n // 1000))]):
        inside = np.flatnonzero(np.all((lo <= new[a]) & (new[a] <= hi), axis=1))
        assert own[a] == inside[-1], a
        if own[a] == mine[a]:
            continue
        elsewhere += 1
        leaves = lids[loff[own[a]]:loff[own[a]] + lcnt[own[a]]] - I
        c = np.concatenate([order[first[k]:first[k + 1]] for k in leaves])
        d = new[a] - new[c]
        d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        want = c[~((d2 > cut[a]) & (d2 > cut[c]))]
        np.testing.assert_array_equal(ids[off[a]:off[a] + cnt[a]], want, err_msg=str(a))
    assert elsewhere >= who.size // 2
    assert int(cnt[:n].sum()) == ids.size


@pytest.mark.parametrize("n,level", [(1, 0), (64, 1), (65, 0), (5000, 2)])
def test_outside_every_box_is_refused(n, level):
    print(f"[owner_leaves] outside n={n}", flush=True)
    pos = np.random.default_rng(n).uniform(0, 1, (n, 3))
    new = pos.copy()
    new[n // 2, 1] = 1.5
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    t, m = _dev(pos, np.full(n, 0.3 * n ** (-1 / 3))), _dev(new, np.full(n, 0.3 * n ** (-1 / 3)))
    with pytest.raises(RuntimeError, match="outside every leaf box"):
        _build(ctx, n, level, t, m)
    _build(ctx, n, level, t, t)  # the context is usable afterwards
    lib().shamx_ctx_destroy(ctx)


@pytest.mark.parametrize("size", [0.1, 0.3, 0.6, 1.0])
@pytest.mark.parametrize("n,level", [(64, 0), (600, 1), (5000, 2), (5000, 4)])
def test_reach_below_zero(n, level, size):
    """Negative smoothing lengths shrink a leaf's box by its reach, to nothing where the reach is
    more than half an edge: such a box meets none (BBAA::cella_neigh_b, geometry_utils.hpp:125-135).
    Owners don't depend on the reach."""
    print(f"[owner_leaves] reach n={n} level={level} size={size}", flush=True)
    rng = np.random.default_rng(n)
    pos = rng.uniform(0, 1, (n, 3))
    h = rng.uniform(0.8, 1.2, n) * 0.5 * n ** (-1 / 3)
    h[pos[:, 0] > 0.3] *= -size
    t = _dev(pos, h)
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    _build(ctx, n, level, t, t)
    I, lo, hi, order, first, cnt, off, ids, own, lcnt, loff, lids = _read(ctx, n)
    lib().shamx_ctx_destroy(ctx)
    r = np.array([h[order[a:b]].max() for a, b in zip(first[:lo.shape[0]], first[1:])])[:, None]
    r = r * HTOL * R
    meet = lambda p, q, u, v: np.all(np.maximum(p, u) <= np.minimum(q, v), axis=-1)
    for g in range(0, lo.shape[0], max(1, lo.shape[0] // 400)):
        want = np.flatnonzero(meet(lo[g], hi[g], lo - r, hi + r) |
                              meet(lo[g] - r[g], hi[g] + r[g], lo, hi))
        np.testing.assert_array_equal(lids[loff[g]:loff[g] + lcnt[g]], I + want, err_msg=str(g))
    for a in range(0, n, max(1, n // 1000)):
        assert own[a] == np.flatnonzero(np.all((lo <= pos[a]) & (pos[a] <= hi), axis=1))[-1]


@pytest.mark.parametrize("n", [2, 65, 600])
def test_cells_without_a_length(n):
    """Lengths that are all NaN: the largest of a leaf starts at the type's lowest value, which
    htol > 1 takes to -inf, and so it stays for every cell above."""
    print(f"[owner_leaves] nan h n={n}", flush=True)
    pos = np.random.default_rng(n).uniform(0, 1, (n, 3))
    t = _dev(pos, np.full(n, np.nan))
    ctx = C.c_void_p()
    s = torch.cuda.current_stream().cuda_stream
    check(lib().shamx_ctx_create(C.byref(ctx)))
    check(lib().shamx_tree_build(ctx, s, n, *[a.data_ptr() for a in t], 0, HTOL))
    sz = (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    r = torch.zeros(sz[1] + sz[2], dtype=torch.float64, device="cuda")
    check(lib().shamx_tree_get(ctx, s, *[None] * 10, r.data_ptr()))
    torch.cuda.synchronize()
    lib().shamx_ctx_destroy(ctx)
    np.testing.assert_array_equal(r.cpu().numpy(), -np.inf)
