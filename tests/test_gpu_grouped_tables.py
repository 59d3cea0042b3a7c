"""The pointer-table grouped MLP calls (c/backend_cuda.h:87-110) at the edges
of their route table, against float64 sums of the dequantised rows: one route
and the full 64, tokens with one expert, rows that do not fill a workgroup of
four, widths that leave a partial group, a partial 8-code unit or an unaligned
second activation row, activations that start off a 16-byte boundary."""
import ctypes as C

import numpy as np
import pytest

from conftest import assert_close_rms

pytestmark = pytest.mark.gpu
GS = 128


def _matrix(rng, bits, rows, cols):
    ng = (cols + GS - 1) // GS
    q = rng.integers(0, 256, (rows, ng * GS * bits // 8), dtype=np.uint8)
    s = (rng.uniform(0.5, 1.5, (rows, ng)) / (4.0 * np.sqrt(cols))).astype(np.float32)
    if bits == 4:
        codes = np.stack([q & 15, q >> 4], -1).reshape(rows, -1).astype(np.int64) - 8
    else:
        b = q.reshape(rows, -1, 3).astype(np.int64)
        word = b[..., 0] | (b[..., 1] << 8) | (b[..., 2] << 16)
        codes = np.stack([(word >> (3 * j)) & 7 for j in range(8)], -1).reshape(rows, -1) - 4
    return q, s, codes[:, :cols] * np.repeat(s.astype(np.float64), GS, 1)[:, :cols]


@pytest.mark.parametrize("bits", [3, 4])
@pytest.mark.parametrize("B,K,H,I,shift", [(1, 1, 128, 128, 0), (8, 8, 256, 130, 0), (8, 1, 520, 257, 0),
                                           (3, 5, 260, 72, 0), (2, 7, 384, 200, 1), (4, 8, 2048, 512, 0)])
def test_grouped_batch_edges(be, bits, B, K, H, I, shift):
    rng = np.random.default_rng(bits * 1000 + B * K + H)
    n = min(B * K, 11)
    mats = [[_matrix(rng, bits, r, c) for r, c in ((I, H), (I, H), (H, I))] for _ in range(n)]
    pick = rng.integers(0, n, B * K)
    x = rng.standard_normal((B, H)).astype(np.float16)
    w = rng.uniform(0.05, 0.5, B * K).astype(np.float32)
    dev = [[(be.upload(q), be.upload(s)) for q, s, _ in m] for m in mats]
    tables = []
    for k in range(3):
        for part in range(2):
            t = (C.c_void_p * (B * K))()
            for j, e in enumerate(pick):
                t[j] = dev[e][k][part].p
            tables.append(t)
    dx, dy = be.upload(np.concatenate([np.zeros(shift, np.float16), x.ravel()])), be.alloc(B * H * 4)
    fn = be.lib.coli_cuda_grouped_q4_mlp_batch_f16 if bits == 4 else be.lib.coli_cuda_grouped_q3_mlp_batch_f16
    ngh, ngi = (H + GS - 1) // GS, (I + GS - 1) // GS
    print(f"[grouped tables] int{bits} {B} x {K} routes, H={H} I={I} shift={shift}", flush=True)
    be.check(fn(be.ctx, dy.p, C.c_void_p(C.cast(dx.p, C.c_void_p).value + 2 * shift), *tables, w.ctypes.data_as(C.c_void_p),
                B, K, H, I, GS, ngh * GS * bits // 8, ngh, ngi * GS * bits // 8, ngi), "grouped")
    got = be.download(dy, (B, H), np.float32)
    want = np.zeros((B, H))
    for r, e in enumerate(pick):
        g, u, d = (m[2] for m in mats[e])
        v = x[r // K].astype(np.float64)
        a = g @ v
        want[r // K] += w[r] * (d @ (a / (1.0 + np.exp(-a)) * (u @ v)))
    # a dot is a chain of at most cols / 64 + 14 fp32 roundings (40 here, 2.4e-6 of
    # the terms' magnitudes, whose sum is up to 36 times the dot's RMS), three dots deep
    assert_close_rms(got, want, 3e-4, "grouped")


@pytest.mark.parametrize("routes", [0, 65])
def test_grouped_batch_refuses(be, routes):
    """No route, and more than the call's 64."""
    d = be.alloc(1 << 16)
    t = (C.c_void_p * 72)(*([d.p] * 72))
    w = np.ones(72, np.float32)
    assert be.lib.coli_cuda_grouped_q4_mlp_batch_f16(be.ctx, d.p, d.p, t, t, t, t, t, t, w.ctypes.data_as(C.c_void_p), 1,
                                                     routes, 128, 128, GS, 64, 1, 64, 1) == -1
