"""How exactly the mixer projections of several tokens hold their activations:
single projections of an attention layer against float64 sums of the
dequantised codes, for int4 and int8 rows, a few tokens and prompt chunks.

The V rows of the cache are a projection of x and nothing else.  The output
rows are a projection of V / 2, exactly: the gate's codes are zero (sigmoid 1/2)
and a row attends to itself alone (queries and keys from the same matrix, their
norms so large that every other weight underflows).

Tolerances.  A fp32 sum of n products in any order is off by at most
depth 2^-24 sum|w x| per output, depth the most roundings that one term passes
through; that bound follows each row's own terms, so a row whose code is zero
for an outlier is judged by the rest.  Depth here: the group sum's conversions
and FMA, the scale and at most one add per group and wave.  Over one 128-column
group there are four roundings, each of at most 2^-24 (RMS 2^-24 / sqrt 12), 3.5e-8 of
the RMS together; a lost or misplaced lowest digit (2^-22 of the group's largest
value) gives 1.9e-7."""
import numpy as np
import pytest

from test_gpu_mixers import _dev_attn, _dev_gdn

pytestmark = pytest.mark.gpu
CUS = 256


def _codes(m):
    """[rows x cols] codes and scales of a quantised matrix, in 64 bits."""
    if m.fmt == 1:
        return m.q.astype(np.int64), np.repeat(m.s.astype(np.float64)[:, None], m.I, 1)
    c = np.stack([m.q & 15, m.q >> 4], -1).reshape(m.O, -1)[:, :m.I].astype(np.int64) - 8
    return c, np.repeat(m.s.astype(np.float64), m.gs, 1)[:, :m.I]


def _attn(seed, H, nh, nkv, hd, o_fmt):
    from oracle import pyoracle as po
    at = po.HostAttn(seed, H, nh, nkv, hd, 32, o_fmt=o_fmt)
    rows = np.arange(2 * nh * hd).reshape(nh, 2, hd)
    keys = np.arange(nkv * hd).reshape(nkv, hd)
    for h in range(nh):
        at.q.q[rows[h, 0]] = at.k.q[keys[h // (nh // nkv)]]
        at.q.s[rows[h, 0]] = at.k.s[keys[h // (nh // nkv)]]
    at.q.q[rows[:, 1].ravel()] = 0x88
    at.q_norm[:] = at.k_norm[:] = 30.0
    return at


def _check(got, m, x, what, depth, limit=None):
    c, s = _codes(m)
    w, x = c * s, x.astype(np.float64)
    want = x @ w.T
    bad = np.abs(got - want) - depth * 2.0**-24 * (np.abs(x) @ np.abs(w).T)
    t, r = np.unravel_index(np.argmax(bad), bad.shape)
    err = float(np.sqrt(np.mean((got - want) ** 2) / np.mean(want ** 2)))
    print(f"[precision] {what}: rms error {err:.2e}", flush=True)
    assert bad[t, r] <= 0, f"{what}: token {t} row {r}: {got[t, r]:.9g} for {want[t, r]:.9g}"
    if limit:
        assert err <= limit, f"{what}: rms error {err:.2e} > {limit:.1e}"


def _depth(cols):
    return cols // 128 + 24


def _takes_gemm(rows, mats):
    """The dispatch's line between 128 x 128 blocks and the weight streams."""
    nt, blocks = sum(-(-m.O // 16) for m in mats), sum(-(-m.O // 128) for m in mats)
    rounds = -(-blocks * -(-rows // 128) // CUS)
    return (32 if nt > CUS else 16) * rounds * CUS < -(-rows // 16) * nt


@pytest.mark.parametrize("o_fmt", [4, 1])
@pytest.mark.parametrize("H,nh,nkv,hd,rows", [(128, 2, 2, 64, 2), (128, 2, 1, 64, 16), (384, 6, 2, 64, 7),
                                              (2048, 16, 2, 256, 15)])
def test_few_tokens(be, H, nh, nkv, hd, rows, o_fmt):
    at = _attn(101, H, nh, nkv, hd, o_fmt)
    dev = _dev_attn(be, at, 1, slots=rows)
    X = np.random.default_rng(102).standard_normal((rows, H)).astype(np.float32)
    y = dev.slots_step(X, list(range(rows)), [0] * rows, device_io=True)
    v = dev.read_cache()[1][:, 0]
    _check(v, at.v, X, "v", _depth(H), 6e-8 if H == 128 else 4e-7)
    ctx = np.repeat(v.reshape(rows, nkv, hd), nh // nkv, 1).reshape(rows, -1) * 0.5
    _check(y, at.o, ctx, "o", _depth(nh * hd), 6e-8 if nh * hd == 128 else 4e-7)


@pytest.mark.parametrize("o_fmt", [4, 1])
@pytest.mark.parametrize("H,nh,nkv,hd,rows,qkv,o", [
    (128, 64, 16, 64, 1025, True, False),     # q, k, v of one group; o of 32
    (8192, 2, 2, 64, 1025, False, True),      # o of one group; q, k, v of 64
    (2048, 16, 2, 256, 529, True, True),      # 16 and 32 groups, a token tile of one
    (1088, 16, 2, 128, 1233, None, True),     # o rows that end inside a block; q, k, v outside whole groups
])
def test_prompt_chunk(be, H, nh, nkv, hd, rows, qkv, o, o_fmt):
    at = _attn(103, H, nh, nkv, hd, o_fmt)
    if qkv is not None:
        assert _takes_gemm(rows, [at.q, at.k, at.v]) == qkv
    assert _takes_gemm(rows, [at.o]) == o
    dev = _dev_attn(be, at, rows)
    X = np.random.default_rng(104).standard_normal((rows, H)).astype(np.float32)
    y = dev.prefill(X, 0)
    v = dev.read_cache()[1][0]
    _check(v, at.v, X, "v", _depth(H), 6e-8 if H == 128 else 4e-7)
    ctx = np.repeat(v.reshape(rows, nkv, hd), nh // nkv, 1).reshape(rows, -1) * 0.5
    _check(y, at.o, ctx, "o", _depth(nh * hd), 6e-8 if nh * hd == 128 else 4e-7)


def _wide(rng, kind, rows, H):
    """Rows whose 128-column groups hold values of very different size."""
    x = rng.standard_normal((rows, H))
    g = x.reshape(rows, H // 128, 128)
    if kind == "one outlier":
        for t in range(rows):
            g[t, :, rng.integers(128)] = 10.0 ** (t % 13)
    elif kind == "fifteen outliers":
        g[:, :, 40:55] *= 1e7
    elif kind == "most of it small":
        g[:, :, 24:] *= 1e-6
    elif kind == "every size":
        g *= 10.0 ** rng.uniform(-25, 10, g.shape)
    elif kind == "tiny":
        x *= 10.0 ** -np.linspace(25, 34, rows)[:, None]
    elif kind == "mostly zero":
        g[rng.random(g.shape) < 0.97] = 0.0
    return x.astype(np.float32)


KINDS = ["one outlier", "fifteen outliers", "most of it small", "every size", "tiny", "mostly zero"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,H", [(13, 256), (2, 2048), (16, 4224)])
def test_wide_groups_few_tokens(be, kind, rows, H):
    for o_fmt in (4, 1):
        at = _attn(105, H, 4, 2, 64, o_fmt)
        dev = _dev_attn(be, at, 1, slots=rows)
        X = _wide(np.random.default_rng(106), kind, rows, H)
        y = dev.slots_step(X, list(range(rows)), [0] * rows, device_io=True)
        v = dev.read_cache()[1][:, 0]
        _check(v, at.v, X, f"v, {kind}", _depth(H))
        ctx = np.repeat(v.reshape(rows, 2, 64), 2, 1).reshape(rows, -1) * 0.5
        _check(y, at.o, ctx, f"o{o_fmt}, {kind}", _depth(256))


@pytest.mark.parametrize("kind", KINDS)
def test_wide_groups_prompt_chunk(be, kind):
    at = _attn(107, 384, 16, 2, 256, 4)
    rows = 531
    assert _takes_gemm(rows, [at.q, at.k, at.v])
    dev = _dev_attn(be, at, rows)
    X = _wide(np.random.default_rng(108), kind, rows, 384)
    dev.prefill(X, 0)
    _check(dev.read_cache()[1][0], at.v, X, f"v, {kind}", _depth(384))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("H,slots,pos", [(256, [0, 1, 2], [0, 5, 2]), (2048, [0, 0, 0, 0, 1], [0, 1, 2, 3, 0]),
                                         (4224, list(range(16)), [7] * 16)])
def test_wide_groups_in_the_convolution_ring(be, kind, H, slots, pos):
    """The ring holds the qkv projection of each sequence's last tokens."""
    from oracle import pyoracle as po
    g = po.HostGdn(113, H, 1, 4, 32, 32)
    dev = _dev_gdn(be, g, slots=max(slots) + 1)
    X = _wide(np.random.default_rng(114), kind, len(slots), H)
    zero = np.zeros((len(slots), 4), np.float32)
    dev.slots_step(X, zero, zero, slots, pos, device_io=True)
    ring = dev.read_state()[0]
    raw = np.stack([ring[s, q % g.K] for s, q in zip(slots, pos)])
    _check(raw, g.qkv, X, f"qkv, {kind}", _depth(H))


def test_wide_groups_int8_prompt_chunk(be):
    """The int8 rows' operand: each kv head's V rows of one size, so that a
    128-column group of V / 2 holds heads of very different size."""
    at = _attn(109, 2048, 64, 64, 64, 1)
    at.v.s *= np.repeat(10.0 ** np.where(np.arange(64) % 2, -6.0, 0.0), 64)[:, None].astype(np.float32)
    rows = 531
    assert _takes_gemm(rows, [at.o])
    dev = _dev_attn(be, at, rows)
    X = np.random.default_rng(110).standard_normal((rows, 2048)).astype(np.float32)
    y = dev.prefill(X, 0)
    v = dev.read_cache()[1][0]
    _check(y, at.o, v * 0.5, "o", _depth(4096))


@pytest.mark.parametrize("rows", [2, 5, 531])
def test_infinities_are_signed(be, rows):
    """An infinity gives a signed infinity where its code is not zero, NaN where
    it is, as the sum of products does; a NaN gives NaN; other tokens keep their values."""
    at = _attn(111, 384, 16, 2, 256, 4)
    assert _takes_gemm(rows, [at.q, at.k, at.v]) == (rows > 500)
    dev = _dev_attn(be, at, rows)
    X = np.random.default_rng(112).standard_normal((rows, 384)).astype(np.float32)
    dev.prefill(X, 0)
    clean = dev.read_cache()[1][0].copy()
    X[1, 200] = -np.inf
    if rows > 2:
        X[3, 9], X[4, 70], X[4, 71] = np.inf, np.nan, np.inf
    dev.prefill(X, 0)
    v = dev.read_cache()[1][0]
    c = _codes(at.v)[0].astype(np.float64)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(v[1], c[:, 200] * -np.inf, equal_nan=True)
        if rows > 2:
            assert np.array_equal(v[3], c[:, 9] * np.inf, equal_nan=True)
            assert np.isnan(v[4]).all()
    keep = [t for t in range(rows) if t not in (1, 3, 4)]
    assert np.array_equal(v[keep], clean[keep])
