"""The mixer projections on the int8 matrix cores (calls of two and more tokens
over 128-column groups) at the edges of their tiles: row counts that are not
multiples of 16, 1 to 64 groups a row, token counts around the 16-token tile,
convolutions of 2 to 4 taps whose tokens share or own their slots, int4 and
int8 output rows; against the oracle (or_gdn_forward / or_attn_forward).

Tolerance: a projection of n <= 8192 products in fp32 is within n 2^-24
sum|p| / RMS = 2^-24 n^1.5 of another order at worst and sqrt(n) of that in
practice; with n = 512 here, and the layer's norms passing it on, 1e-4 x RMS
leaves a factor of ten over the worst observed.  A wrong row, token or group
shows at it, and a lost one of the two upper digits (up to 1 and 2^-7 of a
group's largest value); the lower ones are test_gpu_mixer_precision.py's, which
judges single projections against 64 bits."""
import numpy as np
import pytest

from conftest import assert_close_rms
from test_gpu_mixers import _dev_attn, _dev_gdn, _x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,kh,vh,dk,dv,K,slots,pos", [
    (128, 1, 4, 24, 32, 4, [0, 1], [0, 5]),                                   # one group a row, 176 + 128 rows
    (256, 1, 2, 40, 64, 3, [0, 1, 0, 0, 2], [0, 7, 1, 2, 0]),                 # three taps, repeated slots
    (384, 2, 4, 20, 32, 2, [3, 1, 0, 2, 4, 6, 5, 7, 9, 8, 10, 11, 12, 13, 14], list(range(15))),
    (2176, 1, 4, 16, 32, 4, [0] * 16, list(range(16))),                       # 17 groups, one sequence
    (4224, 1, 4, 16, 32, 4, [0, 1, 1], [2, 0, 1]),                            # 33 groups
], ids=["1group", "3taps", "15tok", "17groups", "33groups"])
def test_gdn_projection_edges(be, oracle, H, kh, vh, dk, dv, K, slots, pos):
    from oracle import pyoracle as po
    g = po.HostGdn(51, H, kh, vh, dk, dv, K=K)
    ns = max(slots) + 1
    dev = _dev_gdn(be, g, slots=ns)
    CS, ST = g.new_state(ns)
    rng = np.random.default_rng(52)
    for turn in range(2):  # the second continues the states and rings of the first
        p = [q + turn * len(slots) for q in pos]
        X = _x(rng, len(slots), H)
        X[0, : H // 2] *= 1e-3  # groups of very different magnitude
        X[-1] = 0.0
        AB = [po.oracle_gdn_gates(oracle, g, X[r]) for r in range(len(slots))]
        A, Bv = np.stack([a for a, _ in AB]), np.stack([b for _, b in AB])
        want = np.stack([po.oracle_gdn_step(oracle, g, X[r], A[r], Bv[r], p[r], CS[s], ST[s])
                         for r, s in enumerate(slots)])
        print(f"[gdn edges] H={H} K={K} tokens {len(slots)} turn {turn}", flush=True)
        got = dev.slots_step(X, A, Bv, slots, p, device_io=bool(turn))
        assert_close_rms(got, want, 1e-4, "output")
    dcs, dst = dev.read_state()
    for s in range(ns):
        assert_close_rms(dcs[s].ravel(), CS[s].ravel(), 1e-4, f"ring {s}")
        assert_close_rms(dst[s].ravel(), ST[s].ravel(), 1e-4, f"state {s}")


@pytest.mark.parametrize("H,nh,nkv,o_fmt,rows", [(128, 2, 2, 4, 2), (128, 2, 1, 1, 15), (256, 4, 2, 4, 17),
                                                 (2304, 32, 2, 1, 33), (2304, 66, 6, 4, 16),
                                                 # q, k, v in 128 x 128 blocks of one and two groups, both ragged;
                                                 # o of 80 and 72 groups, which the vector kernels take
                                                 (256, 160, 10, 4, 401), (128, 144, 9, 1, 1025)])
def test_gqa_projection_edges(be, oracle, H, nh, nkv, o_fmt, rows):
    from oracle import pyoracle as po
    at = po.HostAttn(61, H, nh, nkv, 64, 32, o_fmt=o_fmt)
    dev = _dev_attn(be, at, rows + 1)
    kc, vc = (c[0] for c in at.new_cache(rows + 1))
    rng = np.random.default_rng(62)
    X = _x(rng, rows, H)
    print(f"[gqa edges] H={H} heads {nh} rows {rows} o_fmt {o_fmt}", flush=True)
    got = dev.prefill(X, 0)
    # every token of a small call; from 64 on the first, the last and some between
    some = range(rows) if rows <= 64 else [0, 15, 16, 127, 128, rows - 2, rows - 1]
    if rows > 64:  # the keys and values of the others are the device's own, checked at the rows below
        dk, dv = dev.read_cache()
        kc[:], vc[:] = dk[0], dv[0]
    want = np.stack([po.oracle_attn_step(oracle, at, X[r], r, kc, vc) for r in some])
    got = got[list(some)]
    assert_close_rms(got, want, 1e-4, "output")
    dk, dvv = dev.read_cache()
    assert_close_rms(dk[0][:rows].ravel(), kc[:rows].ravel(), 1e-4, "k cache")
    assert_close_rms(dvv[0][:rows].ravel(), vc[:rows].ravel(), 1e-4, "v cache")


def test_projection_non_finite_rows(be, oracle):
    """An infinity or NaN in one token reaches that token's outputs only."""
    from oracle import pyoracle as po
    at = po.HostAttn(71, 256, 2, 2, 64, 32, o_fmt=4)
    dev = _dev_attn(be, at, 2, slots=4)
    X = _x(np.random.default_rng(72), 4, 256)
    clean = dev.slots_step(X, [0, 1, 2, 3], [0, 0, 0, 0])
    X[1, 130], X[3, 7] = np.inf, np.nan
    got = dev.slots_step(X, [0, 1, 2, 3], [0, 0, 0, 0])
    assert np.array_equal(got[[0, 2]], clean[[0, 2]])
    assert not np.isfinite(got[[1, 3]]).any()


@pytest.mark.parametrize("pos", [[0, 900, 31, 63, 64, 500], [300, 300], [5, 0, 15, 16]], ids=["mixed", "equal", "short"])
def test_gqa_slots_of_different_lengths(be, oracle, pos):
    """Key splits of one length for all rows: rows of one to several splits in
    one call, and calls whose rows have one split each (no merge)."""
    from oracle import pyoracle as po
    at = po.HostAttn(81, 256, 4, 2, 64, 32, o_fmt=4)
    n, seq = len(pos), max(pos) + 1
    dev = _dev_attn(be, at, seq, slots=n)
    kc, vc = at.new_cache(seq, n)
    rng = np.random.default_rng(82)
    import ctypes as C
    for host, buf in ((kc, dev.k_cache), (vc, dev.v_cache)):
        host[:] = rng.standard_normal(host.shape)
        be.check(be.lib.coli_cuda_upload(be.ctx, buf.p, C.c_void_p(host.ctypes.data), host.nbytes), "upload")
    be.sync()
    X = _x(rng, n, 256)
    print(f"[gqa slots] positions {pos}", flush=True)
    want = np.stack([po.oracle_attn_step(oracle, at, X[r], pos[r], kc[r], vc[r]) for r in range(n)])
    got = dev.slots_step(X, list(range(n)), pos, device_io=True)
    assert_close_rms(got, want, 1e-4, "output")
