"""rmsnorm_zero's serial fp32 sum of squares (c/qwen.c:1780-1784) is taken as
runs of integer adds within one binade on the device; rows made to hit every
way a run ends must still equal the serial chain bit for bit: ties (squares
that lie halfway between two values of the running sum), many binade steps,
terms larger than the sum, zeros, sums below and above the exactly scaled
range, infinities and NaN, and lengths around the 64-term start, the 512-term
step and the 4,096-term chunk."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(rng, n):
    i = np.arange(n, dtype=np.float32)
    yield "normal", rng.standard_normal(n)
    yield "ones", np.ones(n)  # exact, no event but binade steps
    yield "small integers", rng.integers(0, 8, n) * 1.0
    # squares of few bits against a sum that starts at 2^23 or 2^24: ties all along
    for top in (2.0**12, 2.0**12 * 1.4142135, 4097.0):
        x = np.sqrt(rng.integers(0, 64, n) * 0.5).astype(np.float32)
        x = np.round(x * 4) / 4
        x[0] = top
        yield f"ties behind {top}", x
    yield "halves", np.where(rng.random(n) < 0.5, 0.5, 2.0**11)
    yield "growing", 1.02 ** (i % 2000)
    yield "falling", 1e6 / (i + 1)
    yield "spikes", np.where(rng.random(n) < 0.01, 1e5, 1e-3) * rng.standard_normal(n)
    z = np.zeros(n)
    z[n // 2:] = rng.standard_normal(n - n // 2)
    yield "zeros first", z
    yield "all zero", np.zeros(n)
    yield "tiny", rng.standard_normal(n) * 1e-19  # squares around the smallest normals
    yield "tiny to normal", np.exp(np.linspace(-45, 0, n))
    yield "overflow", rng.standard_normal(n) * 3e18
    y = rng.standard_normal(n)
    y[n // 3] = np.inf
    yield "infinity", y
    y = rng.standard_normal(n)
    y[-1] = np.nan
    yield "nan", y


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 2048, 4095, 4096, 4097, 9000])
def test_serial_sum_of_squares(be, oracle, n):
    rng = np.random.default_rng(n)
    names, rows = zip(*_rows(rng, n))
    X = np.ascontiguousarray(np.stack([np.asarray(r, np.float32) for r in rows]))
    w = (rng.standard_normal(n) * 0.1).astype(np.float32)
    B = len(names)
    dx, dw, dy = be.upload(X), be.upload(w), be.alloc(X.nbytes)
    print(f"[serial norm] n={n}", flush=True)
    be.check(be.lib.coli_cuda_rmsnorm_zero_batch(be.ctx, dy.p, dx.p, dw.p, B, n, np.float32(1e-6)), "rmsnorm")
    got = be.download(dy, X.shape, np.float32)
    with np.errstate(all="ignore"):
        for b in range(B):
            want = oracle.rmsnorm_zero(X[b], w, 1e-6)
            same = (got[b].view(np.uint32) == want.view(np.uint32)) | (np.isnan(got[b]) & np.isnan(want))
            assert same.all(), f"{names[b]}, n={n}: {int((~same).sum())} values differ"
