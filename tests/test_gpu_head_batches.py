"""The output head of several tokens (k_head_mfma) bit for bit against the CPU
path (c/qwen.c:4505-4516): a vocabulary that does not fill a 16-row tile, fewer
tiles than waves and more than the waves of one pass, hidden sizes of one
64-column step, a partial 512-column chunk, an odd number of chunks and the
largest that the aligned rows take, one to three passes of 16 tokens, padded
rows, a last pass of one token."""
import numpy as np
import pytest

from test_gpu_output_head import _case, _run, _want

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,cols,rb,batch", [
    (1, 64, 64, 2), (17, 576, 576, 16), (130, 1536, 1552, 17), (5003, 2048, 2048, 2), (65539, 192, 192, 33),
    (3001, 4096, 4096, 4), (257, 4160, 4160, 16), (300, 8192, 8192, 5)])
def test_head_batches_bitexact(be, oracle, vocab, cols, rb, batch):
    rng = np.random.default_rng(vocab + cols + batch)
    q, s, x, w = _case(rng, vocab, cols, rb, batch)
    print(f"[head batches] vocab {vocab} hidden {cols} rows {batch}", flush=True)
    hid, lg = _run(be, q, s, x, w, vocab, cols, rb)
    n, want = _want(oracle, q, s, x, w, cols)
    assert np.array_equal(hid.view(np.uint32), n.view(np.uint32))
    bad = np.argwhere(lg.view(np.uint32) != want.view(np.uint32))
    assert bad.size == 0, f"{len(bad)} logits differ, first {bad[:4].tolist()}"
