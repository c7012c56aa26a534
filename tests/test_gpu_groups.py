"""The walks that give a query a group of lanes, at the sizes where a group, a wave or the
k-best list is only partly filled; results against the brute-force oracle, bit for bit."""
import ctypes
import gc

import numpy as np
import pytest

from test_gpu_parity import A, eq, random_gaussians, random_tris  # noqa: F401

pytestmark = pytest.mark.gpu


def scene(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == 0:
        return random_tris(rng, n)
    if kind == 1:
        p = rng.uniform(-30, 30, (n, 3)).astype(np.float32)
        p[n // 2:] = p[: n - n // 2]  # equal distances: ordered by index
        return p
    return random_gaussians(rng, n)


@pytest.mark.parametrize("mode", [3, 5, 6])  # 64, 16 and 32 lanes per query
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_group_walk_edges(A, orc, kind, mode):  # noqa: F811
    A.lib().qr_set_traversal_mode(mode)
    try:
        # (primitives, queries, k): fewer primitives than k, one query, the last group of a
        # wave and the last wave of a workgroup partly filled, every capacity of the list
        for n, nq, k in ((2, 1, 1), (5, 3, 32), (17, 5, 16), (300, 63, 2), (1000, 65, 4), (1000, 17, 5),
                         (3000, 129, 8), (3000, 250, 15), (3000, 33, 17), (3000, 7, 32)):
            print(f"kind={kind} mode={mode} n={n} nq={nq} k={k}", flush=True)
            items = scene(kind, n, n + nq)
            q = np.random.default_rng(k).uniform(-40, 40, (nq, 3)).astype(np.float32)
            b = A.Bvh(kind, items)
            b.build_wide()
            want = orc.knn_brute(kind, items, q, k, threads=8)
            assert eq(b.knn(q, k, order=A.ORDER_MORTON, wide=True)[0], want), (n, nq, k)
            want = orc.knn_brute(kind, items, q, 0, threads=8)
            assert eq(b.closest(q, order=A.ORDER_INPUT, wide=True)[0], want), (n, nq)
    finally:
        A.lib().qr_set_traversal_mode(0)


@pytest.mark.parametrize("mode", [3, 5, 6])
def test_group_walk_unusual_queries(A, orc, mode):  # noqa: F811
    """NaN queries have no answer (index -1) and leave the others of their wave alone;
    infinite ones are infinitely far from everything: the lowest indices."""
    items = scene(1, 500, 3)
    q = np.random.default_rng(4).uniform(-40, 40, (40, 3)).astype(np.float32)
    bad, far = [3, 17, 18], [5, 30]
    q[bad, 1] = np.nan
    q[far, 0] = np.inf
    rest = np.setdiff1d(np.arange(40), bad + far)
    b = A.Bvh(1, items)
    b.build_wide()
    A.lib().qr_set_traversal_mode(mode)
    try:
        for k in (0, 4):
            got = b.knn(q, k, order=A.ORDER_INPUT, wide=True)[0] if k else b.closest(q, order=A.ORDER_INPUT, wide=True)[0]
            want = orc.knn_brute(1, items, q[rest], k, threads=8)
            assert eq(got[rest], want)
            assert np.all(got[bad, :, 1].view(np.int32) == -1)
            assert np.all(got[far, :, 0].view(np.float32) == np.inf)
            assert eq(got[far, :, 1], np.tile(np.arange(max(k, 1), dtype=np.uint32), (len(far), 1)))
    finally:
        A.lib().qr_set_traversal_mode(0)


# 64, 32 and 16 lanes per query (points change at 3,072 and 12,288 queries), on workgroups of
# 256 and 64 lanes; k above 16 needs at least 32 lanes
@pytest.mark.parametrize("variant", ["wide_lds256", "wide_lds64"])
@pytest.mark.parametrize("nq,k", [(1, 0), (3071, 9), (3073, 0), (12287, 16), (12289, 0), (12290, 3), (12291, 20)])
def test_batch_groups(A, orc, variant, nq, k):  # noqa: F811
    print(f"variant={variant} nq={nq} k={k}", flush=True)
    rng = np.random.default_rng(nq + k)
    sizes = [2, 3, 700, 64, 5, 1500]
    items = np.concatenate([scene(1, n, n) for n in sizes])
    poff = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    cuts = np.sort(rng.integers(0, nq + 1, len(sizes) - 1))
    qoff = np.concatenate([[0], cuts, [nq]]).astype(np.int32)
    qoff[1] = 0  # a scene without queries
    q = rng.uniform(-40, 40, (nq, 3)).astype(np.float32)
    batch = A.Batch(1, items, poff)
    plan = A.BatchPlan(batch, q, qoff, k, tune=(A.BATCH_VARIANTS.index(variant), bool(nq % 2)))
    plan.run()
    got = plan.read()
    for s in range(len(sizes)):
        a, b = qoff[s], qoff[s + 1]
        if b > a:
            want = orc.knn_brute(1, items[poff[s]:poff[s + 1]], q[a:b], k, threads=8)
            assert eq(got[a:b], want), s


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_binary_group_walk(A, orc, kind):  # noqa: F811
    """Binary nodes (wide=False) at every group width, a leaf directly below the root included."""
    for n, nq, k in ((2, 1, 1), (3, 5, 4), (300, 63, 7), (2000, 3073, 16), (2000, 12289, 0), (700, 65537, 2),
                     (700, 33, 32)):
        print(f"kind={kind} n={n} nq={nq} k={k}", flush=True)
        items = scene(kind, n, n + nq)
        q = np.random.default_rng(k).uniform(-40, 40, (nq, 3)).astype(np.float32)
        for builder in (0, 1):
            b = A.Bvh(kind, items, builder)
            got = (b.knn(q, k, order=A.ORDER_INPUT) if k else b.closest(q, order=A.ORDER_MORTON))[0]
            assert eq(got, orc.knn_brute(kind, items, q, k, threads=16)), (n, nq, k, builder)


def unusual_rays(rng, items, n):
    """Rays from everywhere to everywhere: some along the axes, some from inside with a
    negative tMin, some with a short tMax."""
    o = rng.uniform(-40, 40, (n, 3))
    d = items.reshape(-1, 9)[rng.integers(0, items.shape[0], n), 0:3] - o + rng.normal(0, 1, (n, 3))
    axis = rng.integers(0, 9, n)
    for a in range(3):
        d[axis == a] = 0.0
        d[axis == a, a] = rng.choice([-1.0, 1.0], (axis == a).sum())
    r = np.concatenate([o, d, np.full((n, 1), 1e-6), np.full((n, 1), np.inf)], 1).astype(np.float32)
    r[::7, 6] = -50.0
    r[::5, 7] = 1.0
    return r


# the counts at which the lanes per ray change, and one ray
@pytest.mark.parametrize("count", [1, 3071, 3072, 12289, 49153, 393217])
def test_ray_group_edges(A, orc, count):  # noqa: F811
    print(f"rays={count}", flush=True)
    rng = np.random.default_rng(count)
    items = random_tris(rng, 400, size=8.0)
    rays = unusual_rays(rng, items, count)
    want = orc.ray_brute(items, rays, threads=16)
    L = A.lib()
    dr, res, hit = A.DeviceArray(rays), A.DeviceArray.empty(count, np.uint64), A.DeviceArray.empty(count, np.int32)
    prims, ms = [], ctypes.c_double()
    for builder in (0, 1):
        b = A.Bvh(0, items, builder)
        b.build_wide()
        for wide in (0, 1):
            assert eq(b.raycast(rays, order=A.ORDER_MORTON, wide=bool(wide))[0], want), (builder, wide)
            A.check(L.qr_raycast_save_device(b.h, dr.ptr, count, res.ptr, hit.ptr, A.ORDER_INPUT, wide, ctypes.byref(ms)))
            assert eq(res.download(), want), (builder, wide)
            prims.append(hit.download())
    assert all(eq(p, prims[0]) for p in prims)
    assert eq(prims[0] >= 0, (want >> np.uint64(32)) != 0)


def test_deep_tree(A, orc):  # noqa: F811
    """Exponentially spaced points: a SAH tree twice as deep as a balanced one."""
    x = np.exp2(np.linspace(-120, 0, 30000))
    items = np.zeros((x.size, 3), np.float32)
    items[:, 0] = x
    b = A.Bvh(1, items, A.BUILDER_SAH)
    b.build_wide()
    print("depth", b.info().depth, flush=True)
    assert 2 * 15 <= b.info().depth <= 64  # (15 if balanced; the walks' stacks are proven for 64)
    q = np.zeros((100, 3), np.float32)
    q[:, 0] = np.exp2(np.linspace(-100, 1, 100))
    for k in (0, 5):
        want = orc.knn_brute(1, items, q, k, threads=8)
        for wide in (False, True):
            got = (b.knn(q, k, wide=wide) if k else b.closest(q, wide=wide))[0]
            assert eq(got, want), (k, wide)


# one workgroup orders a scene of up to 16,384 queries, the general order takes more; above
# 4,096 scenes the keys need a fourth digit; scenes without queries are passed over
@pytest.mark.parametrize("counts", [[16384, 0, 5], [16385, 5, 0], [0, 1, 3] * 1500])
def test_batch_query_order(A, orc, counts):  # noqa: F811
    print(f"scenes={len(counts)} most={max(counts)}", flush=True)
    rng = np.random.default_rng(len(counts))
    S = len(counts)
    items = rng.uniform(-30, 30, (S, 3, 3)).astype(np.float32)
    qoff = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    q = rng.uniform(-40, 40, (int(qoff[-1]), 3)).astype(np.float32)
    batch = A.Batch(1, items.reshape(-1, 3), np.arange(0, 3 * S + 1, 3, dtype=np.int32))
    got = []
    for variant in ("lds64", "wide_lds64"):
        plan = A.BatchPlan(batch, q, qoff, 2, tune=(A.BATCH_VARIANTS.index(variant), True))
        for graph in (True, False, True):
            plan.run(graph=graph)
            got.append(plan.read())
    assert all(eq(g, got[0]) for g in got)
    for s in range(0, S, max(1, S // 40)):
        a, b = qoff[s], qoff[s + 1]
        if b > a:
            assert eq(got[0][a:b], orc.knn_brute(1, items[s], q[a:b], 2, threads=8)), s


# lanes per query change at 16,384 and 40,960 queries, the one-workgroup offsets end at 32,768
@pytest.mark.parametrize("nq", [1, 14, 16384, 32768, 32769, 40961])
def test_radius_segment_lengths(A, orc, nq):  # noqa: F811
    """Segments at the edges of every way of sorting them: registers (64), the workgroup's
    network (2,048), the capture's room (2,048 for few queries), none at all."""
    sizes = [0, 1, 2, 63, 64, 65, 127, 128, 129, 1024, 1025, 2047, 2048, 2049]
    print(f"nq={nq}", flush=True)
    rng = np.random.default_rng(nq)
    centers = np.zeros((len(sizes), 3), np.float32)
    centers[:, 0] = 10.0 * np.arange(len(sizes))
    parts = [c + rng.uniform(-0.3, 0.3, (m, 3)) for c, m in zip(centers, sizes)]
    items = np.concatenate(parts).astype(np.float32)[rng.permutation(sum(sizes))]
    q = centers[np.arange(nq) % len(sizes)].copy()
    if nq > 14:  # mostly short segments: the rest of the queries near nothing or few points
        q[14:] = rng.uniform(-5, 25, (nq - 14, 3)) * np.float32([1, 0.02, 0.02])
    want = orc.radius_brute(1, items, q, 1.0, threads=16)
    for builder in (0, 1):
        b = A.Bvh(1, items, builder)
        for wide in (False, True):
            for order in (A.ORDER_INPUT, A.ORDER_MORTON):
                offs, keys, _, _ = b.radius(q, 1.0, order=order, wide=wide) if not wide else (
                    b.build_wide(), b.radius(q, 1.0, order=order, wide=True))[1]
                assert eq(offs, want[0]), (builder, wide, order)
                assert eq(keys, want[1]), (builder, wide, order)
        pb = A.PointBuffer(q)
        for _ in range(2):  # the second call moves the hits before the host knows their number
            _, offs, keys = pb.radius(b, 1.0, keep=True)
            assert eq(offs, want[0]) and eq(keys, want[1])


# one mask word, its edges, one and two blocks of 1,024 internal nodes, and more words than the
# one-workgroup scan takes (32,768)
@pytest.mark.parametrize("n", [2, 3, 64, 65, 66, 1025, 1026, 5000, (1 << 21) + 70])
@pytest.mark.parametrize("builder", [0, 1])
def test_wide_nodes_are_the_even_depth_nodes(A, n, builder):  # noqa: F811
    print(f"n={n} builder={builder}", flush=True)
    items = np.random.default_rng(n).uniform(-9, 9, (n, 3)).astype(np.float32)
    b = A.Bvh(1, items, builder)
    b.build_wide()
    raw, _ = b.read()
    nodes = raw.view(np.int32).reshape(-1, 8)
    kids = nodes[: n - 1, 6:8]
    depth = np.full(n - 1, -1)
    level, d = np.array([0]), 0
    while level.size:
        depth[level] = d
        level = kids[level].reshape(-1)
        level, d = level[level < n - 1], d + 1
    even = np.nonzero(depth % 2 == 0)[0]
    index = np.full(n - 1, -1)
    index[even] = np.arange(even.size)
    info = b.info()
    assert info.wide_count == even.size
    wide = np.zeros((even.size, 4, 8), np.int32)
    A.check(A.lib().qr_dev_download(A.ptr(wide), info.d_wide_nodes, wide.nbytes))
    # a child that is a leaf stands for itself, an interior one for its two children, in order
    src = np.full((even.size, 4), -1)
    at = np.zeros(even.size, int)
    rows = np.arange(even.size)
    for side in (0, 1):
        c = kids[even, side]
        leaf = c >= n - 1
        pair = kids[np.where(leaf, 0, c)]
        src[rows, at] = np.where(leaf, c, pair[:, 0])
        two = ~leaf
        src[rows[two], at[two] + 1] = pair[two, 1]
        at += np.where(leaf, 1, 2)
    used = src >= 0
    assert eq(wide[used][:, :6], nodes[src[used], :6])
    want = np.where(src[used] >= n - 1, nodes[src[used], 6], index[np.minimum(src[used], n - 2)])
    assert eq(wide[used][:, 6], want)
    assert np.all(wide[~used][:, 6] == np.iinfo(np.int32).min)


# both sides of every count from which a requested order is made
@pytest.mark.parametrize("count", [12287, 12288, 24576, 65535, 65536, 98304, 131072])
def test_order_is_made_or_not(A, orc, count):  # noqa: F811
    print(f"count={count}", flush=True)
    rng = np.random.default_rng(count)
    tris, pts = random_tris(rng, 300), scene(1, 300, 5)
    q = rng.uniform(-40, 40, (count, 3)).astype(np.float32)
    rays = unusual_rays(rng, tris, count)
    for kind, items in ((0, tris), (1, pts)):
        b = A.Bvh(kind, items)
        b.build_wide()
        for wide in (False, True):
            assert eq(b.closest(q, order=A.ORDER_MORTON, wide=wide)[0], orc.knn_brute(kind, items, q, 0, threads=16))
            assert eq(b.knn(q, 3, order=A.ORDER_MORTON, wide=wide)[0], orc.knn_brute(kind, items, q, 3, threads=16))
            o, k, _, _ = b.radius(q, 2.0, order=A.ORDER_MORTON, wide=wide)
            wo, wk = orc.radius_brute(kind, items, q, 2.0, threads=16)
            assert eq(o, wo) and eq(k, wk)
            if kind == 0:
                want = orc.ray_brute(tris, rays, threads=16)
                for order in (A.ORDER_MORTON, A.ORDER_MORTON_DIRECTION):
                    assert eq(b.raycast(rays, order=order, wide=wide)[0], want)


@pytest.mark.parametrize("mode", [0, 1, 2, 3, 5, 6])
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_nan_queries_are_not_walked(A, orc, kind, mode):  # noqa: F811
    """A NaN coordinate makes every distance NaN: no answer, in any shape, and no walk of the
    whole tree (a NaN's box distance is 0 and never bounded by a k-th distance)."""
    items = scene(kind, 3000, 3)
    q = np.random.default_rng(4).uniform(-40, 40, (130, 3)).astype(np.float32)
    nan = q.copy()
    nan[np.arange(130), np.arange(130) % 3] = np.nan
    some = q.copy()
    some[::3] = nan[::3]
    b = A.Bvh(kind, items)
    b.build_wide()
    A.lib().qr_set_traversal_mode(mode)
    try:
        for k in (0, 5):
            want = orc.knn_brute(kind, items, q, k, threads=8)
            want[::3] = (0, 0xffffffff)
            for wide in (False, True):
                def run(p):
                    return b.knn(p, k, wide=wide, stats=True) if k else b.closest(p, wide=wide, stats=True)
                got, _, st = run(nan)
                assert st.nodes_opened <= 130, (k, wide)  # (groups of lanes: the root)
                assert np.all(got == np.array([0, 0xffffffff], np.uint32)), (k, wide)
                assert eq(run(some)[0], want), (k, wide)
    finally:
        A.lib().qr_set_traversal_mode(0)


def test_nan_queries_of_a_batch(A, orc):  # noqa: F811
    items = scene(1, 600, 3)
    q = np.random.default_rng(4).uniform(-40, 40, (100, 3)).astype(np.float32)
    want = np.concatenate([orc.knn_brute(1, items[a:b], q[c:d], 3, threads=8)
                           for a, b, c, d in ((0, 200, 0, 50), (200, 600, 50, 100))])
    q[::7, 2] = np.nan
    want[::7] = (0, 0xffffffff)
    batch = A.Batch(1, items, np.array([0, 200, 600], np.int32))
    for v, name in enumerate(A.BATCH_VARIANTS):
        plan = A.BatchPlan(batch, q, np.array([0, 50, 100], np.int32), 3, tune=(v, True))
        plan.run()
        assert eq(plan.read(), want), name


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_lane_mode_on_binary_nodes(A, orc, kind):  # noqa: F811
    """Mode 1 walks binary nodes one lane per query too.  That walk counts a test per opened
    node; the groups count the entries that pass."""
    items = scene(kind, 3000, 3)
    q = np.random.default_rng(4).uniform(-40, 40, (500, 3)).astype(np.float32)
    b = A.Bvh(kind, items)
    for k in (0, 5):
        want = orc.knn_brute(kind, items, q, k, threads=8)
        for mode in (0, 1):
            A.lib().qr_set_traversal_mode(mode)
            try:
                got, _, st = b.knn(q, k, stats=True) if k else b.closest(q, stats=True)
            finally:
                A.lib().qr_set_traversal_mode(0)
            assert eq(got, want)
            assert (st.node_tests == st.nodes_opened) == (mode == 1), (k, mode)


def test_timed_shapes_belong_to_one_tree(A, orc):  # noqa: F811
    """The next tree in the memory of a destroyed, rebuilt or edited one is timed again: in its
    second call (the first too, where no like call has been timed)."""
    def kept():
        n = ctypes.c_int()
        A.check(A.lib().qr_kept_shapes(ctypes.byref(n)))
        return n.value

    items = scene(1, 3000, 3)
    q = np.random.default_rng(4).uniform(-40, 40, (65536, 3)).astype(np.float32)
    want = orc.knn_brute(1, items, q, 0, threads=16)
    gc.collect()  # (trees of other tests)
    before = kept()
    for _ in range(2):  # the second tree gets the first one's memory
        b = A.Bvh(1, items)
        b.build_wide()
        for _ in range(2):
            assert eq(b.closest(q, wide=True)[0], want)
        assert kept() == before + 1
        b.build_wide()  # the same topology: nothing to time again
        b.closest(q, wide=True)
        assert kept() == before + 1
        for _ in range(2):
            b.knn(q, 3, wide=True)
        assert kept() == before + 2
        b.update(items[:2000], deleted=np.arange(2000, 3000))
        assert kept() == before
        b.build_wide()
        for _ in range(2):
            assert eq(b.closest(q, wide=True)[0], orc.knn_brute(1, items[:2000], q, 0, threads=16))
        assert kept() == before + 1
        b.close()
        assert kept() == before
    b = A.Bvh(1, items)  # called once, as a mesh that moves is: a like call's shape, no timing
    b.build_wide()
    assert eq(b.closest(q, wide=True)[0], want)
    assert kept() == before


# every visit belongs to one part, whole runs of 256 or a piece of one at the end: below, at
# and above the count from which the timed shapes share the queries
@pytest.mark.parametrize("count", [65536, 196607, 196608, 196609, 197631, 200000])
def test_timed_calls_answer_every_query(A, orc, count):  # noqa: F811
    print(f"count={count}", flush=True)
    items = scene(1, 700, 3)
    q = np.random.default_rng(count).uniform(-40, 40, (count, 3)).astype(np.float32)
    for k in (0, 3, 17):  # three shapes to time, and two
        want = orc.knn_brute(1, items, q, k, threads=16)
        for order in (A.ORDER_INPUT, A.ORDER_MORTON):
            b = A.Bvh(1, items)
            b.build_wide()
            for _ in range(3):  # one of the first two times
                got = (b.knn(q, k, order=order, wide=True) if k else b.closest(q, order=order, wide=True))[0]
                assert eq(got, want), (k, order)
            b.close()


@pytest.mark.parametrize("count", [100, 70000])  # by query count, and timed
def test_deepest_lbvh(A, orc, count):  # noqa: F811
    """One point per leading bit of the Morton code and 20,000 in one place, told apart by their
    index: 30 + 15 levels, every 4-wide level with something to come back to."""
    corner = np.zeros((31, 3), np.float32)
    for bit in range(30):  # bit 3 i + a of the code is bit i of axis a's 10
        corner[bit, bit % 3] = 2.0 ** (bit // 3)
    corner[30] = 1023.0
    items = np.concatenate([corner, np.zeros((20000, 3), np.float32)])
    b = A.Bvh(1, items)
    b.build_wide()
    print("depth", b.info().depth, flush=True)
    assert 40 < b.info().depth <= 64
    q = np.random.default_rng(1).uniform(-1, 1, (count, 3)).astype(np.float32)
    q *= np.exp2(np.random.default_rng(2).uniform(-2, 10, (count, 1))).astype(np.float32)
    for mode in (0, 1):
        A.lib().qr_set_traversal_mode(mode)
        try:
            for k in (0, 5):
                for wide in (False, True):
                    got = (b.knn(q, k, wide=wide) if k else b.closest(q, wide=wide))[0]
                    assert eq(got[:100], orc.knn_brute(1, items, q[:100], k, threads=8)), (mode, k, wide)
            o, keys, _, _ = b.radius(q[:100], 3.0, wide=True)
            wo, wk = orc.radius_brute(1, items, q[:100], 3.0, threads=8)
            assert eq(o, wo) and eq(keys, wk), mode
        finally:
            A.lib().qr_set_traversal_mode(0)
