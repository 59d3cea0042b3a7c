"""Routing with many routes a token (K up to the 32 a layer may have): a token
that the bounds leave uncertain needs K and a few exact chains.  Indices equal
router_topk's on the reference's fp32 logits (c/qwen.c:3421-3426), weights within
1e-5, for steps with a few uncertain tokens and with more of them than the
launch holds at once; and a step's uncertain tokens take one round of chains."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _route(be, L, dx, T, K):
    di, dw = be.alloc(T * K * 4), be.alloc(T * K * 4)
    L.route(dx, T, di, dw)
    return be.download(di, (T, K), np.int32), be.download(dw, (T, K), np.float32)


@pytest.mark.parametrize("H,E,K,T", [(1024, 128, 1, 40), (2048, 256, 17, 40), (4096, 512, 24, 8), (4096, 512, 25, 8),
                                     (4096, 512, 32, 8), (1024, 128, 32, 700)])
def test_many_routes_equal_router_topk(be, oracle, H, E, K, T):
    from shiftwing_amd import MoeLayer
    L = MoeLayer(be, H, E, K, 16, 64, 4)
    L.synthesize(95, 0)
    x = np.random.default_rng(9).standard_normal((T, H)).astype(np.float32)
    before = L.route_stats_full()
    idx, w = _route(be, L, be.upload(x), T, K)
    after = L.route_stats_full()
    print(f"[many routes] H={H} E={E} K={K} T={T}: {after[1] - before[1]} uncertain tokens", flush=True)
    hl = oracle.host_layer(95, 0, H, E, K, 16, 64, 4)
    some = range(T) if T <= 40 else range(0, T, 35)
    for t in some:
        logits = np.array([oracle.dot(x[t], hl.router_w[e]) for e in range(E)], np.float32)
        want, ww = oracle.router_topk(logits, K)
        assert np.array_equal(idx[t], want), f"token {t}"
        assert np.abs(w[t] - ww).max() <= 1e-5, f"token {t}"
    L.close()


def test_uncertain_tokens_take_one_round(be):
    """Eight tokens, three of them uncertain at K 24: the step takes one chain of
    4,096 adds (26 us) longer than a certified one, not two."""
    from shiftwing_amd import MoeLayer
    H, E, T = 4096, 512, 8
    dx = be.upload(np.random.default_rng(9).standard_normal((T, H)).astype(np.float32))
    us = {}
    for K in (8, 24):
        L = MoeLayer(be, H, E, K, 16, 64, 4)
        L.synthesize(95, 0)
        di, dw = be.alloc(T * K * 4), be.alloc(T * K * 4)
        L.route(dx, T, di, dw)
        us[K] = np.inf
        for _ in range(10):
            be.sync()
            t = time.perf_counter()
            for _ in range(40):
                L.route(dx, T, di, dw)
            be.sync()
            us[K] = min(us[K], (time.perf_counter() - t) / 40 * 1e6)
        tokens, uncertain, _ = L.route_stats_full()
        print(f"[many routes] K={K}: {us[K]:.1f} us, {uncertain} of {tokens} tokens uncertain", flush=True)
        assert (uncertain > 0) == (K == 24)
        L.close()
    assert us[24] < 2.7 * us[8]  # 55 against 24; two rounds took 73 to 79
