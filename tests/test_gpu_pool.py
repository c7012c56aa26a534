"""The cache of freed device memory behind every buffer: blocks come back only when nothing
uses them, also with several threads and streams, and are given back."""
import ctypes
import threading

import numpy as np
import pytest
import torch  # (before the library loads: both then use one HIP runtime)

from test_gpu_parity import A, eq, random_tris  # noqa: F401

pytestmark = pytest.mark.gpu


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
    """The adjoint call returns before its kernel ends; the tree destroyed right after it
    must not give its arrays to the next build early."""
    rng = np.random.default_rng(2)
    items = random_tris(rng, 20000)
    q = rng.uniform(-30, 30, (60000, 3)).astype(np.float32)
    dq, ones = A.DeviceArray(q), A.DeviceArray(np.ones(q.shape[0], np.float32))
    res, aux = A.DeviceArray.empty((q.shape[0], 2), np.uint32), A.DeviceArray.empty(q.shape[0], np.int32)
    want = None
    for _ in range(5):
        b = A.Bvh(0, items)
        b.build_wide()
        ms = ctypes.c_double()
        A.check(A.lib().qr_closest_device(b.h, dq.ptr, q.shape[0], res.ptr, A.ORDER_MORTON, 1, ctypes.byref(ms)))
        A.check(A.lib().qr_closest_save_aux(b.h, dq.ptr, q.shape[0], res.ptr, aux.ptr))
        g = A.DeviceArray.empty((q.shape[0], 3), np.float32)
        A.check(A.lib().qr_adjoint_closest(b.h, dq.ptr, q.shape[0], res.ptr, aux.ptr, ones.ptr, g.ptr, None))
        b.close()
        A.Bvh(0, items[::-1].copy()).close()
        got = g.download()
        want = got if want is None else want
        assert eq(got, want)


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
