"""Attention over long contexts at the lines of the key splits: one row either
side of one and two workgroups a compute unit (24,576 keys of two kv heads) and
of the 256 splits a row may have, a short prompt chunk and rows of very
different length, against the oracle (c/qwen.c:3094-3137)."""
import ctypes as C

import numpy as np
import pytest

from conftest import assert_close_rms
from test_gpu_mixers import _dev_attn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pos", [[8191], [8192], [24559], [24560], [24576], [70001], [8200, 8201, 8202], [24000, 24001],
                                 [3, 30000], [16383, 0, 24577]], ids=lambda p: "-".join(map(str, p)))
@pytest.mark.parametrize("chunk", [False, True], ids=["slots", "chunk"])
def test_long_context(be, oracle, pos, chunk):
    from oracle import pyoracle as po
    if chunk and pos != list(range(pos[0], pos[0] + len(pos))):
        pytest.skip("a chunk's rows are consecutive")
    at = po.HostAttn(121, 256, 4, 2, 64, 32, o_fmt=4)
    n, seq, slots = len(pos), max(pos) + 1, 1 if chunk else len(pos)
    dev = _dev_attn(be, at, seq, slots=slots)
    kc, vc = at.new_cache(seq, slots)
    rng = np.random.default_rng(122)
    for host, buf in ((kc, dev.k_cache), (vc, dev.v_cache)):
        host[:] = rng.standard_normal(host.shape, dtype=np.float32)
        be.check(be.lib.coli_cuda_upload(be.ctx, buf.p, C.c_void_p(host.ctypes.data), host.nbytes), "upload")
    be.sync()
    X = rng.standard_normal((n, 256)).astype(np.float32)
    print(f"[long context] positions {pos}, chunk {chunk}", flush=True)
    want = np.stack([po.oracle_attn_step(oracle, at, X[r], pos[r], kc[0 if chunk else r], vc[0 if chunk else r])
                     for r in range(n)])
    got = dev.prefill(X, pos[0]) if chunk else dev.slots_step(X, list(range(n)), pos, device_io=True)
    # softmax over n keys of N(0, 1) scores: sums of n terms in fp32, n^1/2 2^-24 of their size
    assert_close_rms(got, want, 1e-4, "output")
