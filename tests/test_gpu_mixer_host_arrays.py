"""The mixer calls on host arrays: the same rows as the device forms, bit for
bit, whatever memory holds the arrays (pageable, page-locked, some of each),
below and above the size that is staged; page-locked inputs that a queued
download still has to bring are the ones used; and a call of two tokens does not
wait for a blocking copy per array."""
import ctypes as C
import time

import numpy as np
import pytest

from test_gpu_mixers import _dev_attn, _dev_gdn

pytestmark = pytest.mark.gpu


class _Pinned:
    def __init__(self, be, a):
        self.be, self.p = be, C.c_void_p()
        a = np.ascontiguousarray(a, np.float32)
        be.check(be.lib.coli_cuda_malloc_host(be.ctx, C.byref(self.p), a.nbytes), "malloc_host")
        self.a = np.ctypeslib.as_array(C.cast(self.p, C.POINTER(C.c_float)), (a.size,)).reshape(a.shape)
        self.a[:] = a

    def free(self):
        self.be.sync()
        self.be.lib.coli_cuda_free_host(self.be.ctx, self.p)


def _p(a):
    return C.c_void_p(a.ctypes.data)


def _gdn_slots(be, dev, y, x, a, b, slot, pos):
    be.check(be.lib.coli_cuda_gdn_slots_q4_f16(be.ctx, _p(y), _p(x), _p(a), _p(b), x.shape[0], _p(slot), _p(pos),
                                               *dev._weights(), dev.slots, *dev._dims()), "gdn slots")


@pytest.mark.parametrize("B", [1, 2, 5, 16])
@pytest.mark.parametrize("H", [256, 288])  # 288: outside whole 128-column groups
def test_gdn_arrays_of_any_memory(be, B, H):
    from oracle import pyoracle as po
    g = po.HostGdn(131, H, 1, 4, 64, 32)
    rng = np.random.default_rng(132)
    X, A, Bv = (rng.standard_normal((B, n)).astype(np.float32) for n in (H, 4, 4))
    slot, pos = np.arange(B, dtype=np.int32), np.arange(B, dtype=np.int32)
    dev = _dev_gdn(be, g, slots=B)
    want = dev.slots_step(X, A, Bv, list(slot), list(pos), device_io=True)
    cs, st = dev.read_state()
    for kinds in (0, 1, 2, 7, 8, 15):  # bits: x, a, b, y in page-locked memory
        pins = [_Pinned(be, v) if kinds >> i & 1 else None for i, v in enumerate((X, A, Bv, np.zeros((B, H))))]
        x, a, b, y = (p.a if p else v for p, v in zip(pins, (X, A, Bv, np.zeros((B, H), np.float32))))
        dev.reset()
        _gdn_slots(be, dev, y, x, a, b, slot, pos)
        assert np.array_equal(y, want), kinds
        dcs, dst = dev.read_state()
        assert np.array_equal(dcs, cs) and np.array_equal(dst, st), kinds
        for p in pins:
            if p:
                p.free()


@pytest.mark.parametrize("rows", [1, 4, 17, 127, 128, 129])  # 128 rows of 1,024: 512 KB
@pytest.mark.parametrize("pinned", ["none", "x", "y", "both"])
def test_attention_arrays_of_any_memory(be, rows, pinned):
    from oracle import pyoracle as po
    at = po.HostAttn(133, 1024, 4, 2, 64, 32, o_fmt=1)
    dev = _dev_attn(be, at, rows)
    X = np.random.default_rng(134).standard_normal((rows, 1024)).astype(np.float32)
    plain = dev.prefill(X, 0)
    if rows <= 4:  # the device form's rows
        again = _dev_attn(be, at, rows)
        for r in range(rows):
            got = again.slots_step(X[r:r + 1], [0], [r], device_io=True)
            assert np.abs(got[0] - plain[r]).max() <= 1e-4 * np.sqrt(np.mean(plain ** 2))
    px = _Pinned(be, X) if pinned in ("x", "both") else None
    py = _Pinned(be, np.zeros((rows, 1024))) if pinned in ("y", "both") else None
    x, y = px.a if px else X, py.a if py else np.zeros((rows, 1024), np.float32)
    be.check(be.lib.coli_cuda_gqa_prefill_q4_f16(be.ctx, _p(y), _p(x), rows, 0, *dev._weights(), rows, *dev._tail()),
             "prefill")
    assert np.array_equal(y, plain)
    for p in (px, py):
        if p:
            p.free()


def test_page_locked_inputs_follow_the_stream(be):
    from oracle import pyoracle as po
    at = po.HostAttn(135, 256, 4, 2, 64, 32, o_fmt=4)
    rng = np.random.default_rng(136)
    X = [rng.standard_normal((2, 256)).astype(np.float32) for _ in range(2)]
    want = _dev_attn(be, at, 2).prefill(X[1], 0)
    dev, px, dx = _dev_attn(be, at, 2), _Pinned(be, X[0]), be.upload(X[1])
    big = [be.alloc(1 << 28) for _ in range(2)]
    be.sync()
    for _ in range(20):  # milliseconds of queued copies ahead of the download
        be.check(be.lib.coli_cuda_copy(be.ctx, big[0].p, big[1].p, 1 << 28), "copy")
    be.check(be.lib.coli_cuda_download(be.ctx, px.p, dx.p, X[1].nbytes), "download")
    y = np.zeros((2, 256), np.float32)
    be.check(be.lib.coli_cuda_gqa_prefill_q4_f16(be.ctx, _p(y), px.p, 2, 0, *dev._weights(), 2, *dev._tail()), "prefill")
    assert np.array_equal(y, want)
    px.free()


def test_two_tokens_wait_for_no_copy_each(be):
    """Two S35 Gated DeltaNet tokens on host arrays, against the same tokens on
    the device among others: 51 and 27 us; 77 with a copy for each array."""
    from oracle import pyoracle as po
    g = po.HostGdn(137, 2048, 16, 32, 128, 128)
    dev = _dev_gdn(be, g, slots=2)
    rng = np.random.default_rng(138)
    X, A, Bv = (rng.standard_normal((2, n)).astype(np.float32) for n in (2048, 32, 32))
    y, slot, pos = np.zeros((2, 2048), np.float32), np.arange(2, dtype=np.int32), np.zeros(2, np.int32)
    dx, da, db, dy = be.upload(X), be.upload(A), be.upload(Bv), be.alloc(y.nbytes)

    def device():
        be.check(be.lib.coli_cuda_gdn_slots_q4_f16_device(be.ctx, dy.p, dx.p, da.p, db.p, 2, _p(slot), _p(pos),
                                                          *dev._weights(), 2, *dev._dims()), "gdn slots")

    us = []
    for call in (device, lambda: _gdn_slots(be, dev, y, X, A, Bv, slot, pos)):
        best = np.inf
        for _ in range(10):
            be.sync()
            t = time.perf_counter()
            for _ in range(40):
                call()
            be.sync()
            best = min(best, (time.perf_counter() - t) / 40 * 1e6)
        us.append(best)
    print(f"[host arrays] two tokens: device {us[0]:.1f}, host {us[1]:.1f} us", flush=True)
    assert us[1] < 2.6 * us[0]
