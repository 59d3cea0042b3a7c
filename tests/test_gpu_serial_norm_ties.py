"""rmsnorm_zero on rows whose squares tie often (bf16 and fp16 values, integers,
rows made of ties) or change binade often: the same bits as the serial chain
(c/qwen.c:1780-1784), in steps that switch between runs of integer adds and
single adds, and no longer than a small multiple of a row without ties."""
import time

import numpy as np
import pytest

from test_gpu_output_head import _run

pytestmark = pytest.mark.gpu


def _bf16(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def _rows(rng, n):
    x = rng.standard_normal(n).astype(np.float32)
    yield "bf16", _bf16(x)
    yield "fp16", x.astype(np.float16)
    i = np.arange(n)
    yield "bf16 from the middle on", np.where(i < n // 2, x, _bf16(x))
    yield "bf16 up to the middle", np.where(i < n // 2, _bf16(x), x)
    yield "bf16 in every other step", np.where(i // 512 % 2, x, _bf16(x))
    yield "bf16 at the ends of steps", np.where(i % 512 < 300, x, _bf16(x))
    yield "integers", rng.integers(-7, 8, n)
    ties = np.full(n, 0.5)
    ties[0] = 2560.0
    yield "ties", ties
    yield "growing", 1.02 ** (i % 3000)
    yield "growing slowly", 1.003 ** (i % 9000) * np.abs(x)


@pytest.mark.parametrize("n", [512, 520, 576, 1000, 1024, 1536, 2048, 4096, 4100, 8192, 9001])
def test_ties_equal_the_chain(be, oracle, n):
    rng = np.random.default_rng(n)
    names, rows = zip(*_rows(rng, n))
    X = np.ascontiguousarray(np.stack([np.asarray(r, np.float32) for r in rows]))
    w = (rng.standard_normal(n) * 0.1).astype(np.float32)
    dx, dw, dy = be.upload(X), be.upload(w), be.alloc(X.nbytes)
    print(f"[norm ties] n={n}", flush=True)
    be.check(be.lib.coli_cuda_rmsnorm_zero_batch(be.ctx, dy.p, dx.p, dw.p, len(names), n, np.float32(1e-6)), "rmsnorm")
    got = be.download(dy, X.shape, np.float32)
    for b, name in enumerate(names):
        want = oracle.rmsnorm_zero(X[b], w, 1e-6)
        assert np.array_equal(got[b].view(np.uint32), want.view(np.uint32)), f"{name}, n={n}"


@pytest.mark.parametrize("n", [576, 1000, 4096])
def test_ties_equal_the_chain_in_the_output_head(be, oracle, n):
    """The head's norm bounds its runs at other counts."""
    rng = np.random.default_rng(n + 1)
    names, rows = zip(*_rows(rng, n))
    X = np.ascontiguousarray(np.stack([np.asarray(r, np.float32) for r in rows]))
    w = (rng.standard_normal(n) * 0.1).astype(np.float32)
    pad = (n + 15) // 16 * 16
    q = rng.integers(-127, 128, (64, pad)).astype(np.int8)
    hid, _ = _run(be, q, np.full(64, 1e-3, np.float32), X, w, 64, n, pad)
    for b, name in enumerate(names):
        want = oracle.rmsnorm_zero(X[b], w, 1e-6)
        assert np.array_equal(hid[b].view(np.uint32), want.view(np.uint32)), f"{name}, n={n}"


@pytest.mark.parametrize("n", [2048, 4096])
def test_ties_take_no_longer_than_single_adds(be, n):
    """A row without ties takes about half of what single adds take; rows of
    ties took 5 to 25 times as long before their runs were bounded."""
    rng = np.random.default_rng(7)
    dw, dy = be.upload(np.zeros(n, np.float32)), be.alloc(4 * n)

    def us(row):
        dx = be.upload(np.asarray(row, np.float32))
        best = np.inf
        for _ in range(8):
            be.sync()
            t = time.perf_counter()
            for _ in range(40):
                be.check(be.lib.coli_cuda_rmsnorm_zero(be.ctx, dy.p, dx.p, dw.p, n, np.float32(1e-6)), "rmsnorm")
            be.sync()
            best = min(best, (time.perf_counter() - t) / 40 * 1e6)
        return best

    plain = us(rng.standard_normal(n))
    for name, row in _rows(rng, n):
        t = us(row)
        print(f"[norm ties] n={n} {name}: {t:.1f} us, no ties {plain:.1f}", flush=True)
        assert t < 2.5 * plain, name
