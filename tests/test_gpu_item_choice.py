"""The automatic choice between expert items of 64 and of 16 tokens is the
faster one or within a few percent of it: many tokens an expert on few experts
or short rows (items of 16, however many tokens), and on experts that fill the
device (items of 64)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,K,I,fmt,T,best", [
    (2048, 16, 4, 512, 4, 216, 16), (4096, 8, 2, 1024, 3, 216, 16), (1024, 64, 6, 512, 4, 427, 16),
    (2048, 256, 8, 512, 4, 480, 16), (2048, 256, 8, 512, 3, 1280, 64), (4096, 32, 4, 2048, 3, 800, 64)])
def test_automatic_items_are_the_faster(be, H, E, K, I, fmt, T, best):
    from shiftwing_amd import MoeLayer
    L = MoeLayer(be, H, E, K, I, 512, fmt)
    L.synthesize(5, 0)
    x = np.random.default_rng(9).standard_normal((T, H)).astype(np.float32)
    dx, dy, di, dw = be.upload(x), be.alloc(x.nbytes), be.alloc(T * K * 4), be.alloc(T * K * 4)
    us = {16: np.inf, 64: np.inf, 0: np.inf}
    try:
        for _ in range(6):
            for items in us:
                be.check(be.lib.coli_cuda_moe_set_item_tokens(be.ctx, items))
                for n in (2, 10):
                    be.sync()
                    t = time.perf_counter()
                    for _ in range(n):
                        be.check(be.lib.coli_cuda_moe_forward(be.ctx, L.h, dy.p, dx.p, T, di.p, dw.p))
                    be.sync()
                    t = (time.perf_counter() - t) / n * 1e6
                us[items] = min(us[items], t)
    finally:
        be.check(be.lib.coli_cuda_moe_set_item_tokens(be.ctx, 0))
    print(f"[item choice] H={H} E={E} I={I} T={T}: 16 {us[16]:.1f}, 64 {us[64]:.1f}, automatic {us[0]:.1f} us", flush=True)
    # the other choice is 7% to 25% slower here
    assert us[0] <= 1.05 * us[best]
    L.close()
