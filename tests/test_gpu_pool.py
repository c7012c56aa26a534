"""The cache of freed device memory behind every buffer: blocks come back only when nothing
uses them, also with several threads and streams, and are given back."""
import ctypes
import threading
import time

import numpy as np
import pytest
import torch  # (before the library loads: both then use one HIP runtime)

from test_gpu_parity import A, eq, random_tris  # noqa: F401

pytestmark = pytest.mark.gpu


def used(torch_free_before):
    return torch_free_before - torch.cuda.mem_get_info()[0]


def alloc(A, n):  # noqa: F811
    p = ctypes.c_void_p()
    A.check(A.lib().qr_dev_alloc(n, ctypes.byref(p)))
    return p


def side_stream_work(stream, ms=300):
    """Queues about that much work on the stream: products of one size, timed once."""
    with torch.cuda.stream(stream):
        m = torch.ones((4096, 4096), device="cuda")
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        out = torch.mm(m, m)
        a.record()
        torch.mm(m, m, out=out)
        b.record()
        b.synchronize()
        for _ in range(int(ms / max(a.elapsed_time(b), 0.05)) + 1):
            torch.mm(m, m, out=out)
        done = torch.cuda.Event()
        done.record()
    return done


def test_alloc_free_trim(A):  # noqa: F811
    L = A.lib()
    held = []
    for n in (1, 511, 513, 4096, 1 << 20, (1 << 20) + 1, 3 << 20):
        for _ in range(3):
            p = ctypes.c_void_p()
            A.check(L.qr_dev_alloc(n, ctypes.byref(p)))
            assert p.value and p.value % 256 == 0
            held.append((p, n))
    spans = sorted((p.value, n) for p, n in held)
    assert all(a + n <= b for (a, n), (b, _) in zip(spans, spans[1:]))  # no two overlap
    for p, n in held:
        x = np.arange(n, dtype=np.uint8)
        A.check(L.qr_dev_upload(p, A.ptr(x), n))
    for p, n in held:
        back = np.zeros(n, np.uint8)
        A.check(L.qr_dev_download(A.ptr(back), p, n))
        assert eq(back, np.arange(n, dtype=np.uint8))
        A.check(L.qr_dev_free(p))
        assert L.qr_dev_free(p) != A.QR_OK  # freed already
    A.check(L.qr_dev_trim())
    A.check(L.qr_dev_free(None))


def test_free_waits_for_queued_work(A, orc):  # noqa: F811
    """A buffer and a tree freed while kernels that read them are still queued on a
    non-blocking stream: their memory must not reach the next owner before those end."""
    L = A.lib()
    rng = np.random.default_rng(2)
    items = random_tris(rng, 20000)
    q = rng.uniform(-30, 30, (60000, 3)).astype(np.float32)
    n = q.shape[0]
    stream = torch.cuda.Stream()
    want = None
    for late in (False, True):
        b = A.Bvh(0, items)
        ones = A.DeviceArray(np.ones(n, np.float32))
        res, aux = A.DeviceArray.empty((n, 2), np.uint32), A.DeviceArray.empty(n, np.int32)
        pts = alloc(A, q.nbytes)
        A.check(L.qr_dev_upload(pts, A.ptr(q), q.nbytes))
        ms = ctypes.c_double()
        A.check(L.qr_closest_device(b.h, pts, n, res.ptr, A.ORDER_MORTON, 0, ctypes.byref(ms)))
        A.check(L.qr_closest_save_aux(b.h, pts, n, res.ptr, aux.ptr))
        g = A.DeviceArray.empty((n, 3), np.float32)
        A.check(L.qr_dev_trim())
        A.check(L.qr_set_stream(ctypes.c_void_p(stream.cuda_stream)))
        try:
            done = side_stream_work(stream) if late else None
            A.check(L.qr_adjoint_closest(b.h, pts, n, res.ptr, aux.ptr, ones.ptr, g.ptr, None))
        finally:
            A.check(L.qr_set_stream(None))
        if late:
            assert not done.query()  # the adjoint has not begun
            A.check(L.qr_dev_free(pts))
            other = alloc(A, q.nbytes)
            assert other.value == pts.value
            A.check(L.qr_dev_upload(other, A.ptr(np.zeros_like(q)), q.nbytes))
            b.close()
            A.Bvh(0, items[::-1].copy()).close()
        torch.cuda.synchronize()
        got = g.download()
        want = got if want is None else want
        assert eq(got, want), late
        A.check(L.qr_dev_free(pts))  # (late: the block's second owner)


def test_destroying_a_tree_waits_for_queued_work(A, orc):  # noqa: F811
    L = A.lib()
    rng = np.random.default_rng(2)
    items = random_tris(rng, 20000)
    q = rng.uniform(-30, 30, (60000, 3)).astype(np.float32)
    n = q.shape[0]
    dq, ones = A.DeviceArray(q), A.DeviceArray(np.ones(n, np.float32))
    res, aux = A.DeviceArray.empty((n, 2), np.uint32), A.DeviceArray.empty(n, np.int32)
    stream = torch.cuda.Stream()
    want = None
    for late in (False, True):
        b = A.Bvh(0, items)
        ms = ctypes.c_double()
        A.check(L.qr_closest_device(b.h, dq.ptr, n, res.ptr, A.ORDER_MORTON, 0, ctypes.byref(ms)))
        A.check(L.qr_closest_save_aux(b.h, dq.ptr, n, res.ptr, aux.ptr))
        g = A.DeviceArray.empty((n, 3), np.float32)
        A.check(L.qr_set_stream(ctypes.c_void_p(stream.cuda_stream)))
        try:
            done = side_stream_work(stream) if late else None
            A.check(L.qr_adjoint_closest(b.h, dq.ptr, n, res.ptr, aux.ptr, ones.ptr, g.ptr, None))
        finally:
            A.check(L.qr_set_stream(None))
        was = {b.info().d_nodes, b.info().d_items, b.info().d_prim_ids}
        assert not late or not done.query()
        b.close()
        c = A.Bvh(0, items[::-1].copy())
        assert not late or c.info().d_items in was  # the same memory, other contents
        torch.cuda.synchronize()
        got = g.download()
        want = got if want is None else want
        assert eq(got, want), late
        c.close()


def test_threads_and_streams(A, orc):  # noqa: F811
    rng = np.random.default_rng(3)
    work = [(random_tris(rng, n), rng.uniform(-30, 30, (m, 3)).astype(np.float32))
            for n, m in ((3000, 500), (3100, 700), (2900, 90), (3050, 2000))]
    want = [orc.knn_brute(0, t, q, 4, threads=8) for t, q in work]
    wrong = []

    def run(i):
        try:
            stream = torch.cuda.Stream() if i % 2 else torch.cuda.default_stream()
            A.check(A.lib().qr_set_stream(ctypes.c_void_p(stream.cuda_stream)))
            for _ in range(10):
                t, q = work[i]
                b = A.Bvh(0, t, i % 2)
                b.build_wide()
                if not eq(b.knn(q, 4, order=A.ORDER_MORTON, wide=True)[0], want[i]):
                    wrong.append(i)
                b.close()
        except Exception as e:  # noqa: BLE001
            wrong.append((i, repr(e)))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong


def test_radius_results_do_not_wait_for_other_streams(A, orc):  # noqa: F811
    """A radius result whose device pointers nobody asked for has no reader left once the call
    returned: neither destroying it nor a grown key buffer inside the call waits for the work
    of other streams."""
    L = A.lib()
    rng = np.random.default_rng(5)
    items = rng.uniform(-10, 10, (20000, 3)).astype(np.float32)
    q = rng.uniform(-10, 10, (500, 3)).astype(np.float32)
    b = A.Bvh(1, items)
    pb = A.PointBuffer(q)
    want = {r: orc.radius_brute(1, items, q, r, threads=8) for r in (0.5, 1.5)}
    pb.radius(b, 1.5, wide=False)  # (the call's own buffers have grown)
    pb.radius(b, 0.5, wide=False)  # (and its guess of the number of hits is small)
    stream = torch.cuda.Stream()
    done = side_stream_work(stream)
    for r in (0.5, 1.5, 1.5, 0.5):
        _, offs, keys = pb.radius(b, r, wide=False, keep=True)
        assert eq(offs, want[r][0]) and eq(keys, want[r][1])
    assert not done.query()
    done.synchronize()

    done = side_stream_work(stream)  # asked for, they may have readers on any stream
    csr, ms, offs, keys = (ctypes.c_void_p(), ctypes.c_double(), ctypes.c_void_p(), ctypes.c_void_p())
    A.check(L.qr_radius(b.h, pb.h, 0.5, 0, A.ORDER_INPUT, 0, ctypes.byref(csr), ctypes.byref(ms)))
    A.check(L.qr_radius_device_ptrs(csr, ctypes.byref(offs), ctypes.byref(keys)))
    assert not done.query()
    A.check(L.qr_radius_destroy(csr))
    assert done.query()


def test_cached_blocks_are_bounded_and_given_back(A):  # noqa: F811
    """Freed blocks are kept (the same address comes back), at most 4 GiB of them, none past
    10 s once another buffer is allocated, and trim returns them to the runtime."""
    L = A.lib()
    A.check(L.qr_dev_trim())
    p = alloc(A, 64 << 20)
    A.check(L.qr_dev_free(p))
    q = alloc(A, 64 << 20)
    assert p.value == q.value
    A.check(L.qr_dev_free(q))
    A.check(L.qr_dev_trim())
    free0 = torch.cuda.mem_get_info()[0]

    held = [alloc(A, 1 << 30) for _ in range(6)]
    slack = 64 << 20  # other allocations on the card
    assert used(free0) >= (6 << 30) - slack
    for h in held:
        A.check(L.qr_dev_free(h))
    assert (3 << 30) - slack <= used(free0) <= (4 << 30) + slack
    A.check(L.qr_dev_trim())
    assert used(free0) <= slack

    A.check(L.qr_dev_free(alloc(A, 1 << 30)))
    assert used(free0) >= (1 << 30) - slack
    print("idle", flush=True)
    time.sleep(10.5)
    small = alloc(A, 4096)  # nothing is freed here: allocating is enough
    assert used(free0) <= slack
    A.check(L.qr_dev_free(small))


# from 4 KiB on a block is at most an eighth larger than asked for
@pytest.mark.parametrize("n", [4097, 131073, (1 << 20) + 1, (9 << 20) + 1])
def test_rounding(A, n):  # noqa: F811
    L = A.lib()
    A.check(L.qr_dev_trim())
    p = alloc(A, n)
    A.check(L.qr_dev_free(p))
    q = alloc(A, n + n // 8 + 512)  # more than the block can hold: another one
    assert q.value != p.value
    A.check(L.qr_dev_free(q))
