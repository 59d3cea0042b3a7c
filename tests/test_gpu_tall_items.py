"""Steps in items of 64 tokens (forced: the automatic choice is another test's)
against the same step in items of 16: the same arithmetic per (row, token) in the same order, so equal
bits; and against the oracle.  Shapes at the edges: row tiles of I and H that
do not fill a workgroup, partial 128-column groups, one group, experts with 0,
1, 16, 17, 64, 65 and more tokens, int3, int4 and int2."""
import numpy as np
import pytest

from conftest import assert_close_rms

pytestmark = pytest.mark.gpu


def _layer(be, seed, H, E, K, I, Ish, fmt):
    from shiftwing_amd import MoeLayer
    L = MoeLayer(be, H, E, K, I, Ish, fmt)
    L.synthesize(seed, 0)
    return L


def _forward(be, L, x, items):
    be.check(be.lib.coli_cuda_moe_set_item_tokens(be.ctx, items), "set_item_tokens")
    try:
        return L.forward_host(x)
    finally:
        be.check(be.lib.coli_cuda_moe_set_item_tokens(be.ctx, 0), "set_item_tokens")


@pytest.mark.parametrize("H,E,K,I,Ish,fmt,T", [
    (128, 4, 2, 128, 64, 3, 40),       # one group each way
    (192, 4, 2, 144, 80, 4, 70),       # 12 and 9 row tiles, a partial group
    (576, 8, 3, 400, 128, 3, 129),     # 36 row tiles of H: a second chunk of 4; 25 of I
    (1088, 6, 1, 272, 64, 4, 300),     # 68 row tiles: two chunks and a bit; one route a token
    (256, 3, 3, 128, 64, 2, 65),       # every token on every expert: 65 each
    (2048, 16, 4, 512, 512, 4, 200),
    (4096, 8, 2, 1024, 1024, 3, 100),
])
def test_tall_items_equal_wide_items(be, oracle, H, E, K, I, Ish, fmt, T):
    L = _layer(be, 91, H, E, K, I, Ish, fmt)
    x = np.random.default_rng(92).standard_normal((T, H)).astype(np.float32)
    print(f"[tall items] H={H} E={E} K={K} I={I} fmt={fmt} T={T}", flush=True)
    y0, i0, w0 = _forward(be, L, x, 16)
    y1, i1, w1 = _forward(be, L, x, 64)
    assert np.array_equal(i0, i1) and np.array_equal(w0, w1)
    assert np.array_equal(y0.view(np.uint32), y1.view(np.uint32))
    hl = oracle.host_layer(91, 0, H, E, K, I, Ish, fmt)
    for t in (0, T // 2, T - 1):
        want, _ = oracle.moe_forward(hl, x[t], trace=True)
        assert_close_rms(y1[t], want, 1e-3, f"token {t}")
    L.close()


def test_tall_items_uneven_experts(be):
    """Token counts per expert of 0, 1, 16, 17, 64, 65 and the rest: a router
    that reads one feature per expert, tokens that set one of them."""
    import ctypes as C
    H, E, I = 256, 7, 128
    counts = [0, 1, 16, 17, 64, 65, 40]
    L = _layer(be, 93, H, E, 1, I, 64, 3)
    router = np.zeros((E, H), np.float32)
    router[np.arange(E), np.arange(E)] = 1.0
    be.check(be.lib.coli_cuda_upload(be.ctx, C.c_void_p(L.router_ptr()), C.c_void_p(router.ctypes.data), router.nbytes))
    be.sync()
    rng = np.random.default_rng(94)
    which = rng.permutation(np.repeat(np.arange(E), counts))
    x = rng.standard_normal((which.size, H)).astype(np.float32)
    x[:, :E] = 0.0
    x[np.arange(which.size), which] = 8.0
    y0, i0, _ = _forward(be, L, x, 16)
    y1, i1, _ = _forward(be, L, x, 64)
    assert np.array_equal(i1[:, 0], which) and np.array_equal(i0, i1)
    assert np.array_equal(y0.view(np.uint32), y1.view(np.uint32))
    L.close()
