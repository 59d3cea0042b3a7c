"""The grouped calls' route weights follow the stream: weights that a queued
download still has to bring into page-locked memory are the ones used, whether
the call is made before or after they arrive; weights in pageable memory are
read before the call returns."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_grouped_tables import GS, _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [3, 4])
def test_weights_follow_the_stream(be, bits):
    rng = np.random.default_rng(31)
    B, K, H, I = 2, 3, 256, 128
    n = B * K
    mats = [[_matrix(rng, bits, r, c) for r, c in ((I, H), (I, H), (H, I))] for _ in range(n)]
    dev = [[(be.upload(q), be.upload(s)) for q, s, _ in m] for m in mats]
    tables = []
    for k in range(3):
        for part in range(2):
            tables.append((C.c_void_p * n)(*(dev[e][k][part].p.value for e in range(n))))
    x = rng.standard_normal((B, H)).astype(np.float16)
    dx, dy = be.upload(x), be.alloc(B * H * 4)
    fn = be.lib.coli_cuda_grouped_q4_mlp_batch_f16 if bits == 4 else be.lib.coli_cuda_grouped_q3_mlp_batch_f16

    def call(w):
        be.check(fn(be.ctx, dy.p, dx.p, *tables, w, B, K, H, I, GS, H // GS * GS * bits // 8, H // GS,
                    I // GS * GS * bits // 8, I // GS), "grouped")

    w = [rng.uniform(0.05, 0.5, n).astype(np.float32) for _ in range(3)]
    want = []
    for v in w:
        pageable = v.copy()
        call(pageable.ctypes.data_as(C.c_void_p))
        pageable[:] = 9.0  # read before the call returned
        want.append(be.download(dy, (B, H), np.float32))

    pinned = C.c_void_p()
    be.check(be.lib.coli_cuda_malloc_host(be.ctx, C.byref(pinned), 4 * n), "malloc_host")
    try:
        C.memmove(pinned, w[0].ctypes.data, 4 * n)
        call(pinned)
        assert np.array_equal(be.download(dy, (B, H), np.float32), want[0])
        big = [be.alloc(1 << 28) for _ in range(2)]
        for v, y in zip(w[1:], want[1:]):
            dw = be.upload(v)
            be.sync()
            for _ in range(20):  # milliseconds of queued copies ahead of the download
                be.check(be.lib.coli_cuda_copy(be.ctx, big[0].p, big[1].p, 1 << 28), "copy")
            be.check(be.lib.coli_cuda_download(be.ctx, pinned, dw.p, 4 * n), "download")
            call(pinned)
            assert np.array_equal(be.download(dy, (B, H), np.float32), y)
    finally:
        be.sync()
        be.lib.coli_cuda_free_host(be.ctx, pinned)
