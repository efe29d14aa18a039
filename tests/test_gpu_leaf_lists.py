"""Stage 1 of the neighbour cache on the GPU (leaf lists and owner leaves) against the criterion
written out in numpy on the tree's own leaf boxes: leaf n is in leaf g's list when g's box meets
n's box widened by n's reach, or g's widened box meets n's box (NeighbourCache.cpp:276-404), in
index order; the owner of a particle is the last leaf whose box contains it (:406-451).  Both are
comparisons of the same doubles, so they must agree exactly.  The leaf counts are the edges of the
8-ary tiers and of the waves (8 leaves per wave, 64 cells per step)."""
import ctypes as C
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from shamrock_amd._lib import check, lib  # noqa: E402

R = 2.0


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module", autouse=True)
def gpu_ready():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda()


def meet(alo, ahi, blo, bhi):
    return np.all(np.maximum(alo, blo) <= np.minimum(ahi, bhi), axis=-1)


@pytest.mark.parametrize("outliers", [False, True])
@pytest.mark.parametrize("n,level", [(1, 0), (2, 0), (8, 0), (9, 0), (64, 0), (65, 0), (512, 0),
                                     (513, 0), (4097, 0), (33_000, 0), (20_000, 3)])
def test_leaf_lists_and_owners(n, level, outliers):
    """level 0: one leaf per distinct code, so (nearly) n leaves; outliers: one particle in
    97 with 20 times the smoothing length (lists of thousands, queues that wrap)."""
    say(f"[leaf_lists] n={n} level={level} outliers={outliers}")
    rng = np.random.default_rng(n + outliers)
    pos = rng.uniform(0, 1, (n, 3))
    if level:
        pos[:, 2] *= 0.02  # long runs of codes give leaf boxes that meet
    h = rng.uniform(0.8, 1.2, n) * 0.5 * n ** (-1 / 3)
    if outliers:
        h[::97] *= 20
    x, y, z, hh = (dev(a) for a in (*pos.T, h))
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    s = torch.cuda.current_stream().cuda_stream
    p = [t.data_ptr() for t in (x, y, z, hh)]
    check(lib().shamx_tree_build(ctx, s, n, *p, level, 1.1))
    check(lib().shamx_neigh_build(ctx, s, n, *p, 1.1, R))
    sz, ns = (C.c_uint32 * 4)(), (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    check(lib().shamx_neigh_sizes(ctx, ns))
    L, I, PL = sz[1], sz[2], ns[3]
    box = [torch.zeros(3 * (I + L), dtype=torch.float64, device="cuda") for _ in range(2)]
    rint = torch.zeros(I + L, dtype=torch.float64, device="cuda")
    check(lib().shamx_tree_get(ctx, s, *[None] * 8, box[0].data_ptr(), box[1].data_ptr(),
                               rint.data_ptr()))
    own, cnt, off, ids = (torch.zeros(max(k, 1), dtype=torch.int32, device="cuda")
                          for k in (n, L, L, PL))
    check(lib().shamx_neigh_get(ctx, s, None, None, None, own.data_ptr(), cnt.data_ptr(),
                                off.data_ptr(), ids.data_ptr()))
    torch.cuda.synchronize()
    lib().shamx_ctx_destroy(ctx)
    lo, hi = (b.cpu().numpy().reshape(-1, 3)[I:] for b in box)
    r = rint.cpu().numpy()[I:, None] * R
    cnt, off, ids, own = (t.cpu().numpy().view(np.uint32) for t in (cnt, off, ids, own))
    np.testing.assert_array_equal(off[:L], np.r_[0, np.cumsum(cnt[:L])[:-1]])
    assert int(cnt[:L].sum()) == PL
    step = max(1, L // 600)
    for g in [*range(0, L, step), L - 1]:
        want = np.flatnonzero(meet(lo[g], hi[g], lo - r, hi + r) |
                              meet(lo[g] - r[g], hi[g] + r[g], lo, hi))
        np.testing.assert_array_equal(ids[off[g]:off[g] + cnt[g]], I + want)
    for a in range(0, n, max(1, n // 2000)):
        inside = np.flatnonzero(np.all((lo <= pos[a]) & (pos[a] <= hi), axis=1))
        assert own[a] == inside[-1]


@pytest.mark.parametrize("n,level", [(2, 0), (8, 0), (9, 0), (64, 0), (65, 0), (512, 0), (513, 0),
                                     (4097, 0), (4608, 0), (33_000, 0), (20_000, 3)])
def test_internal_boxes(n, level):
    """Box and largest rint of every internal cell against the leaves of its range (from its
    index to endrange): min and max, so exactly equal."""
    say(f"[internal_boxes] n={n} level={level}")
    rng = np.random.default_rng(n)
    pos = rng.normal(0, 1, (n, 3))
    h = rng.uniform(0.01, 0.1, n)
    t = [dev(a) for a in (*pos.T, h)]
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    s = torch.cuda.current_stream().cuda_stream
    check(lib().shamx_tree_build(ctx, s, n, *[a.data_ptr() for a in t], level, 1.1))
    sz = (C.c_uint32 * 4)()
    check(lib().shamx_tree_sizes(ctx, sz))
    L, I = sz[1], sz[2]
    end = torch.zeros(max(I, 1), dtype=torch.int32, device="cuda")
    box = [torch.zeros(3 * (I + L), dtype=torch.float64, device="cuda") for _ in range(2)]
    rint = torch.zeros(I + L, dtype=torch.float64, device="cuda")
    check(lib().shamx_tree_get(ctx, s, *[None] * 7, end.data_ptr(), box[0].data_ptr(),
                               box[1].data_ptr(), rint.data_ptr()))
    torch.cuda.synchronize()
    lib().shamx_ctx_destroy(ctx)
    lo, hi = (b.cpu().numpy().reshape(-1, 3) for b in box)
    r, end = rint.cpu().numpy(), end.cpu().numpy()
    assert r[0] == h.max() * 1.1
    for i in range(I):
        a, b = min(i, end[i]), max(i, end[i]) + 1
        assert np.array_equal(lo[i], lo[I + a:I + b].min(0)), i
        assert np.array_equal(hi[i], hi[I + a:I + b].max(0)), i
        assert r[i] == r[I + a:I + b].max(), i


def test_nan_position_is_refused():
    """A particle with a NaN coordinate lies in no leaf box: the build raises, as the reference's
    search finds no owner for it."""
    say("[leaf_lists] nan")
    n = 100
    pos = np.random.default_rng(0).uniform(0, 1, (n, 3))
    pos[17, 1] = np.nan
    t = [dev(a) for a in (*pos.T, np.full(n, 0.1))]
    ctx = C.c_void_p()
    check(lib().shamx_ctx_create(C.byref(ctx)))
    s = torch.cuda.current_stream().cuda_stream
    p = [a.data_ptr() for a in t]
    check(lib().shamx_tree_build(ctx, s, n, *p, 3, 1.1))
    with pytest.raises(RuntimeError, match="outside every leaf box"):
        check(lib().shamx_neigh_build(ctx, s, n, *p, 1.1, R))
    lib().shamx_ctx_destroy(ctx)
