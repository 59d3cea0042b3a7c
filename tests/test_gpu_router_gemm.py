"""Routing of steps large enough for the 32 x 32 blocks of the fp64 logit GEMM,
with token and expert counts that leave partial tiles, against the same tokens
routed in steps of 63 (the bounds kernels): router_topk's indices either way,
so equal; weights from fp64 logits of another summation order, 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,K,T", [(64, 500, 7, 803), (192, 1009, 3, 401), (512, 384, 10, 1025)])
def test_route_many_tokens_equals_small_steps(be, H, E, K, T):
    from shiftwing_amd import MoeLayer
    L = MoeLayer(be, H, E, K, 16, 64, 4)
    L.synthesize(95, 0)
    x = np.random.default_rng(96).standard_normal((T, H)).astype(np.float32)
    print(f"[router gemm] H={H} E={E} T={T}", flush=True)

    def route(rows):
        dx, di, dw = be.upload(rows), be.alloc(rows.shape[0] * K * 4), be.alloc(rows.shape[0] * K * 4)
        L.route(dx, rows.shape[0], di, dw)
        return (be.download(di, (rows.shape[0], K), np.int32), be.download(dw, (rows.shape[0], K), np.float32))

    idx, w = route(x)
    small = [route(np.ascontiguousarray(x[t:t + 63])) for t in range(0, T, 63)]
    assert np.array_equal(idx, np.concatenate([s[0] for s in small]))
    assert np.abs(w - np.concatenate([s[1] for s in small])).max() <= 1e-6
    L.close()
