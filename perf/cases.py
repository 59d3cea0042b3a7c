"""Performance cases: what a program built on this framework calls while it serves a model.

The framework runs the layers of a hybrid decoder (Gated DeltaNet or gated GQA attention, then a
quantised mixture-of-experts block, and an int8 output head) behind one C ABI.  Each case is one call of
that ABI, or the few calls of one step, on tensors that are already where the caller has them: device
memory for the device forms, host arrays for the forms that take host activations.  Shapes are the two
that the repository's benchmark and tests use:

  s35    hidden 2048, 256 experts of 512 (top 8), shared expert 512, 16 / 32 DeltaNet heads, 16 query heads
  s397   hidden 4096, 512 experts of 1024 (top 10), shared expert 1024, 16 / 64 DeltaNet heads, 32 query heads

Weights are random codes with random group scales, scaled so that a projection of unit-variance input has
unit variance; activations are N(0, 1), as after a norm.  Skewed routing (`zipf`) holds one input feature at
1 and puts a rank bias into that router column, as the benchmark does.
"""
import ctypes
import math

import numpy as np
import torch

import shiftwing_amd as sw

SHAPES = {
    "s35": dict(H=2048, E=256, K=8, I=512, Ish=512, kh=16, vh=32, nh=16, zipf=0.424),
    "s397": dict(H=4096, E=512, K=10, I=1024, Ish=1024, kh=16, vh=64, nh=32, zipf=0.554),
}
DK = DV = 128          # Gated DeltaNet key and value dims
TAPS = 4               # causal convolution taps
HD, RD, NKV = 256, 64, 2  # attention head dim, rotary dim, kv heads
GS = 128               # quantisation group
THETA, EPS = 1e7, 1e-6
CODE_RMS = {2: math.sqrt(5.0), 3: 2.345, 4: 4.637}  # of uniform codes


def listed():
    return [
        # One token through consecutive MoE blocks: the inner loop of single-user decoding, the smallest call
        # of the path (latency and launches), with int4 experts and skewed routing.
        dict(name="decode-s35", kind="stack", model="s35", fmt=4, layers=8, tokens=1, zipf=True),
        # The same on the large model's int3 experts: the repository's headline workload, four layers of it.
        dict(name="decode-s397", kind="stack", model="s397", fmt=3, layers=4, tokens=1, zipf=False),
        # Continuous batching: one token of each of eight sequences through consecutive MoE blocks.
        dict(name="batch8-s397", kind="stack", model="s397", fmt=3, layers=2, tokens=8, zipf=True),
        # A prompt chunk through the MoE half of a decoder layer on the residual stream (norm, routing,
        # experts, residual add), its normalised rows and routes returned.
        dict(name="block512-s35", kind="block", model="s35", fmt=4, tokens=512, zipf=False),
        # A long, odd prompt chunk through one large MoE layer: the most arithmetic per byte of the MoE path.
        dict(name="prefill1999-s397", kind="moe", model="s397", fmt=3, tokens=1999, zipf=False),
        # Gated DeltaNet layer, one sequence's next token, activations on the device.
        dict(name="gdn1-s397", kind="gdn", model="s397", mode="slots", batch=1, pos=911),
        # The same for sixteen sequences in their own state slots (continuous batching at its limit).
        dict(name="gdn16-s397", kind="gdn", model="s397", mode="slots", batch=16, pos=911),
        # Attention layer, one sequence's next token at 4,096 cached positions.
        dict(name="gqa1-s397", kind="gqa", model="s397", batch=1, context=4097, o_fmt=4),
        # The same for thirteen sequences of different lengths (an odd batch), int8 output projection.
        dict(name="gqa13-s35", kind="gqa", model="s35", batch=13, context=6000, o_fmt=1),
        # A prompt chunk through an attention layer behind a 3,000-position prefix; host arrays in and out,
        # as that entry point takes them.
        dict(name="gqa-prefill-s397", kind="gqa_prefill", model="s397", rows=1000, base=3000, o_fmt=4),
        # Final norm and int8 output head for a batch of eight.
        dict(name="head8-s397", kind="head", model="s397", vocab=248320, batch=8),
        # The pointer-table call of hosts that keep their own expert cache: four tokens' routed experts.
        dict(name="grouped4-s35", kind="grouped", model="s35", fmt=4, batch=4, cached=32),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 0.02)))))


def draw(rng):
    kind = rng.choice(["stack", "stack", "moe", "block", "gdn", "gdn", "gqa", "gqa", "gqa_prefill", "head", "grouped"])
    model = rng.choice(sorted(SHAPES))
    fmt = rng.choice([2, 3, 4])
    zipf = rng.random() < 0.5
    if kind == "stack":
        return dict(kind=kind, model=model, fmt=fmt, layers=rng.randint(1, 8 if model == "s35" else 3),
                    tokens=_log_uniform(rng, 1, 64), zipf=zipf)
    if kind == "moe":
        return dict(kind=kind, model=model, fmt=fmt, tokens=_log_uniform(rng, 1, 1999), zipf=zipf)
    if kind == "block":
        return dict(kind=kind, model=model, fmt=fmt, tokens=_log_uniform(rng, 1, 1024), zipf=zipf)
    if kind == "gdn":
        mode = rng.choice(["slots", "block"])
        return dict(kind=kind, model=model, mode=mode, batch=rng.randint(1, 16 if mode == "slots" else 8),
                    pos=rng.choice([0, rng.randint(1, 100000)]))
    if kind == "gqa":
        return dict(kind=kind, model=model, batch=rng.randint(1, 16), context=_log_uniform(rng, 1, 8192),
                    o_fmt=rng.choice([1, 4]))
    if kind == "gqa_prefill":
        return dict(kind=kind, model=model, rows=_log_uniform(rng, 2, 1000), base=rng.choice([0, rng.randint(1, 3000)]),
                    o_fmt=rng.choice([1, 4]))
    if kind == "head":
        return dict(kind=kind, model=model, vocab=rng.choice([248320, _log_uniform(rng, 30000, 248320)]),
                    batch=rng.randint(1, 16))
    return dict(kind=kind, model=model, fmt=rng.choice([3, 4]), batch=rng.randint(1, 6),
                cached=_log_uniform(rng, 10, 100))


# ---- inputs -------------------------------------------------------------------------------------


class _Rand:
    """Values on the GPU from the case's seed, in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(1 + (int(seed) * 1000003) % (1 << 40))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(std)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)

    def codes(self, *shape):
        n = math.prod(shape)
        w = torch.randint(-(1 << 63), (1 << 63) - 1, ((n + 7) // 8,), generator=self.g, device="cuda",
                          dtype=torch.int64)
        return w.view(torch.uint8)[:n].view(*shape)


def _row_bytes(fmt, cols):
    return (cols + GS - 1) // GS * GS * fmt // 8


def _qmat(r, fmt, rows, cols, lead=()):
    """Random codes and group scales of a [rows x cols] matrix (or a stack of them) of unit gain."""
    s0 = 1.0 / (CODE_RMS[fmt] * math.sqrt(cols))
    return (r.codes(*lead, rows, _row_bytes(fmt, cols)),
            r.uniform(*lead, rows, (cols + GS - 1) // GS, lo=0.5 * s0, hi=1.5 * s0))


def _q8mat(r, rows, cols):
    s0 = 1.0 / (73.3 * math.sqrt(cols))
    q = r.codes(rows, cols).view(torch.int8)
    q.clamp_(min=-127)
    return q, r.uniform(rows, lo=0.5 * s0, hi=1.5 * s0)


def _moe_weights(r, case):
    """One MoE layer as a converted snapshot holds it."""
    m = SHAPES[case["model"]]
    H, E, I, Ish, fmt = m["H"], m["E"], m["I"], m["Ish"], case["fmt"]
    w = dict(fmt=fmt, router=r.normal(E, H, std=0.02), sgate=r.normal(H, std=0.02))
    if case["zipf"]:
        p = torch.arange(1, E + 1, device="cuda", dtype=torch.float64) ** -1.1
        order = torch.argsort(r.uniform(E))
        w["router"][order, H - 1] = (m["zipf"] * torch.log(p / p.sum())).float()
    w["shared"] = _q8mat(r, Ish, H) + _q8mat(r, Ish, H) + _q8mat(r, H, Ish)
    w["gate"], w["up"], w["down"] = _qmat(r, fmt, I, H, (E,)), _qmat(r, fmt, I, H, (E,)), _qmat(r, fmt, H, I, (E,))
    return w


def _moe_x(r, case, *lead):
    x = r.normal(*lead, SHAPES[case["model"]]["H"])
    if case["zipf"]:
        x[..., -1] = 1.0
    return x


def _gdn_inputs(r, case):
    m = SHAPES[case["model"]]
    H, kh, vh, B = m["H"], m["kh"], m["vh"], case["batch"]
    C, vd = 2 * kh * DK + vh * DV, vh * DV
    slots = B if case["mode"] == "slots" else 1
    w = dict(qkv=_qmat(r, 4, C, H), z=_qmat(r, 4, vd, H), out=_qmat(r, 4, H, vd),
             conv=r.normal(C, TAPS, std=0.5), a_log=r.normal(vh, std=0.5), dt_bias=r.normal(vh, std=0.5),
             norm=1.0 + r.normal(DV, std=0.1), ring=r.normal(slots, TAPS, C), state=r.normal(slots, vh, DK, DV, std=0.1),
             x=r.normal(B, H), a=r.normal(B, vh), b=r.normal(B, vh))
    if case["mode"] == "slots":  # sequences at different places
        w["pos"] = np.array([case["pos"] + 37 * i for i in range(B)], np.int32)
        w["slot"] = np.array([(5 * i + 3) % B if B % 5 else B - 1 - i for i in range(B)], np.int32)
    else:
        w["pos"] = np.arange(case["pos"], case["pos"] + B, dtype=np.int32)
        w["slot"] = np.zeros(B, np.int32)
    return w


def _gqa_inputs(r, case):
    m = SHAPES[case["model"]]
    H, nh = m["H"], m["nh"]
    if case["kind"] == "gqa":
        n, seq, slots = case["batch"], case["context"], case["batch"]
        # the longest sequence fills the context, the others stop at smaller, odd places
        pos = [max(0, (seq - 1) * (n - i) // n - (i % 3 if i else 0)) for i in range(n)]
        slot = [(i + 1) % n for i in range(n)]
    else:
        n, seq, slots = case["rows"], case["base"] + case["rows"], 1
        pos, slot = list(range(case["base"], seq)), [0] * n
    w = dict(q=_qmat(r, 4, 2 * nh * HD, H), k=_qmat(r, 4, NKV * HD, H), v=_qmat(r, 4, NKV * HD, H),
             o=_qmat(r, 4, H, nh * HD) if case["o_fmt"] == 4 else _q8mat(r, H, nh * HD),
             q_norm=r.normal(HD, std=0.1), k_norm=r.normal(HD, std=0.1),
             k_cache=r.normal(slots, seq, NKV * HD), v_cache=r.normal(slots, seq, NKV * HD), x=r.normal(n, H))
    w["pos"], w["slot"], w["seq"], w["slots"] = np.array(pos, np.int32), np.array(slot, np.int32), seq, slots
    return w


def _grouped_inputs(r, case):
    m = SHAPES[case["model"]]
    H, I, K, B, fmt = m["H"], m["I"], m["K"], case["batch"], case["fmt"]
    n = case["cached"]  # experts that the call's routes are taken from
    w = dict(gate=_qmat(r, fmt, I, H, (n,)), up=_qmat(r, fmt, I, H, (n,)), down=_qmat(r, fmt, H, I, (n,)),
             x=r.normal(B, H).half())
    w["expert"] = torch.stack([torch.argsort(r.uniform(n))[:K] for _ in range(B)]).cpu().numpy()
    p = torch.softmax(r.normal(B, K), 1)
    w["weight"] = np.ascontiguousarray(p.cpu().numpy(), np.float32)
    return w


def _head_inputs(r, case):
    H = SHAPES[case["model"]]["H"]
    q, s = _q8mat(r, case["vocab"], H)
    return dict(q=q, s=s, norm=r.normal(H, std=0.1), x=r.normal(case["batch"], H, std=2.0))


# ---- the calls ------------------------------------------------------------------------------------

_BACKEND = None


def _backend():
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = sw.Backend(0)
    return _BACKEND


class _Device:
    """Device memory of a tensor, as the framework's Python side takes it."""

    def __init__(self, t):
        self.t = t
        self.p = _ptr(t)


def _ptr(t):
    assert t.is_contiguous()
    return ctypes.c_void_p(t.data_ptr())


def _host(a):
    return ctypes.c_void_p(a.ctypes.data)


def _layer(be, case, w):
    m = SHAPES[case["model"]]
    L = sw.MoeLayer(be, m["H"], m["E"], m["K"], m["I"], m["Ish"], case["fmt"])
    torch.cuda.synchronize()
    L.set_router(_Device(w["router"]), _Device(w["sgate"]))
    L.set_shared_q8(*(_Device(t) for t in w["shared"]))
    mats = [t for k in ("gate", "up", "down") for t in w[k]]
    at, step = [t.data_ptr() for t in mats], [t.stride(0) * t.element_size() for t in mats]
    fn, arg = be.lib.coli_cuda_moe_layer_set_expert, ctypes.c_void_p
    for e in range(m["E"]):
        be.check(fn(be.ctx, L.h, e, *(arg(a + e * s) for a, s in zip(at, step))), "set_expert")
    be.sync()
    return L


def prepare(case, seed):
    be, r = _backend(), _Rand(seed)
    lib, ctx, kind = be.lib, be.ctx, case["kind"]
    m = SHAPES[case["model"]]
    H, K = m["H"], m["K"]
    if kind == "stack":
        n, T = case["layers"], case["tokens"]
        x = _moe_x(r, case, n, T)
        layers = [_layer(be, case, _moe_weights(r, case)) for _ in range(n)]
        y = torch.zeros(n, T, H, device="cuda")
        table = (ctypes.c_void_p * n)(*(L.h.value for L in layers))
        calls = [(lib.coli_cuda_moe_forward_layers, (ctx, table, n, _ptr(y), _ptr(x), T, T * H, T * H))]
        keep, out = (x, layers, table), {"y": y}
    elif kind in ("moe", "block"):
        T = case["tokens"]
        x = _moe_x(r, case, T)
        norm = r.normal(H, std=0.1)
        L = _layer(be, case, _moe_weights(r, case))
        y, idx = torch.zeros(T, H, device="cuda"), torch.zeros(T, K, device="cuda", dtype=torch.int32)
        weight = torch.zeros(T, K, device="cuda")
        out = {"y": y, "weight": weight, "idx": idx}
        if kind == "moe":
            calls = [(lib.coli_cuda_moe_forward, (ctx, L.h, _ptr(y), _ptr(x), T, _ptr(idx), _ptr(weight)))]
        else:  # the residual stream arrives in the previous layer's buffer
            out["hidden"] = torch.zeros(T, H, device="cuda")
            calls = [(lib.coli_cuda_copy, (ctx, _ptr(y), _ptr(x), T * H * 4)),
                     (lib.coli_cuda_moe_block_ex, (ctx, L.h, _ptr(y), _ptr(norm), ctypes.c_float(EPS), T,
                                                   _ptr(out["hidden"]), _ptr(idx), _ptr(weight)))]
        keep = (x, norm, L)
    elif kind == "gdn":
        w, B = _gdn_inputs(r, case), case["batch"]
        mats = [a for k in ("qkv", "z", "out") for a in (_ptr(w[k][0]), _ptr(w[k][1]), w[k][0].shape[1], w[k][1].shape[1])]
        mats += [_ptr(w[k]) for k in ("conv", "a_log", "dt_bias", "norm", "ring", "state")]
        dims = (H, m["kh"], m["vh"], DK, DV, TAPS, GS, ctypes.c_float(EPS))
        if case["mode"] == "slots":
            y = torch.zeros(B, H, device="cuda")
            calls = [(lib.coli_cuda_gdn_slots_q4_f16_device,
                      (ctx, _ptr(y), _ptr(w["x"]), _ptr(w["a"]), _ptr(w["b"]), B, _host(w["slot"]), _host(w["pos"]),
                       *mats, B, *dims))]
        else:
            y = np.zeros((B, H), np.float32)
            w.update({k: w[k].cpu().numpy() for k in ("x", "a", "b")})
            calls = [(lib.coli_cuda_gdn_block_q4_f16,
                      (ctx, _host(y), _host(w["x"]), _host(w["a"]), _host(w["b"]), B, *mats, int(w["pos"][0]), *dims))]
        keep, out = w, {"y": y, "ring": w["ring"], "state": w["state"]}
    elif kind in ("gqa", "gqa_prefill"):
        w = _gqa_inputs(r, case)
        n = w["x"].shape[0]
        mats = [a for k in ("q", "k", "v") for a in (_ptr(w[k][0]), _ptr(w[k][1]), w[k][0].shape[1], w[k][1].shape[1])]
        oq, os = w["o"]
        mats += [_ptr(oq), _ptr(os), case["o_fmt"], oq.shape[1], os.shape[1] if os.dim() == 2 else 0]
        mats += [_ptr(w[k]) for k in ("q_norm", "k_norm", "k_cache", "v_cache")]
        dims = (H, m["nh"], NKV, HD, RD, GS, ctypes.c_float(THETA), ctypes.c_float(EPS))
        if kind == "gqa":
            y = torch.zeros(n, H, device="cuda")
            calls = [(lib.coli_cuda_gqa_slots_q4_f16_device,
                      (ctx, _ptr(y), _ptr(w["x"]), n, _host(w["slot"]), _host(w["pos"]), *mats, w["slots"], w["seq"],
                       *dims))]
        else:
            y = np.zeros((n, H), np.float32)
            w["x"] = w["x"].cpu().numpy()
            calls = [(lib.coli_cuda_gqa_prefill_q4_f16,
                      (ctx, _host(y), _host(w["x"]), n, case["base"], *mats, w["seq"], *dims))]
        keep, out = w, {"y": y, "k": w["k_cache"], "v": w["v_cache"]}
    elif kind == "head":
        w, B = _head_inputs(r, case), case["batch"]
        V = case["vocab"]
        out = {"logits": torch.zeros(B, V, device="cuda"), "hidden": torch.zeros(B, H, device="cuda")}
        calls = [(lib.coli_cuda_output_head_q8,
                  (ctx, _ptr(out["logits"]), _ptr(out["hidden"]), _ptr(w["x"]), _ptr(w["norm"]), ctypes.c_float(EPS), B,
                   _ptr(w["q"]), _ptr(w["s"]), V, H, H))]
        keep = w
    else:
        w, B, fmt = _grouped_inputs(r, case), case["batch"], case["fmt"]
        tables = []
        for k in ("gate", "up", "down"):
            for t in w[k]:
                step = t.stride(0) * t.element_size()
                tables.append((ctypes.c_void_p * (B * K))(*(t.data_ptr() + int(e) * step for e in w["expert"].ravel())))
        y = torch.zeros(B, H, device="cuda")
        gq, gsc, uq, usc, dq, dsc = tables
        fn = lib.coli_cuda_grouped_q4_mlp_batch_f16 if fmt == 4 else lib.coli_cuda_grouped_q3_mlp_batch_f16
        calls = [(fn, (ctx, _ptr(y), _ptr(w["x"]), gq, gsc, uq, usc, dq, dsc, _host(w["weight"]), B, K, H, m["I"], GS,
                       _row_bytes(fmt, H), H // GS, _row_bytes(fmt, m["I"]), m["I"] // GS))]
        keep, out = (w, tables), {"y": y}
    torch.cuda.synchronize()
    return {"calls": calls, "out": out, "keep": keep}


def run(state):
    for fn, args in state["calls"]:
        if fn(*args) != 0:
            raise RuntimeError(_backend().last_error())
    return state["out"]


# ---- what a pass cannot do without ------------------------------------------------------------------


def _distinct_experts(case, T):
    """Experts that T tokens route to, by simulation of the router's logits."""
    m = SHAPES[case["model"]]
    E, K = m["E"], m["K"]
    rng = np.random.default_rng(T)
    logits = rng.standard_normal((T, E)) * 0.02 * math.sqrt(m["H"])
    if case["zipf"]:
        p = np.arange(1, E + 1) ** -1.1
        logits += m["zipf"] * np.log(p / p.sum())
    return len(np.unique(np.argpartition(-logits, K - 1, axis=1)[:, :K]))


def work(case):
    m, kind = SHAPES[case["model"]], case["kind"]
    H, E, K, I, Ish = m["H"], m["E"], m["K"], m["I"], m["Ish"]

    def q(fmt, rows, cols):
        return rows * (cols * fmt / 8 + cols / GS * 4)

    if kind in ("stack", "moe", "block"):
        T = case["tokens"]
        # an int2 expert is stored in two bits a weight
        expert = 2 * q(case["fmt"], I, H) + q(case["fmt"], H, I)
        layer = _distinct_experts(case, T) * expert + E * H * 4 + H * 4 + 3 * Ish * H + 8 * Ish + 4 * H + T * H * 8
        if kind != "stack":
            layer += T * K * 8
        if kind == "block":
            layer += T * H * 4 + H * 4
        n = case.get("layers", 1)
        return {"bytes": n * layer, "flops": n * T * (K * 6 * H * I + 6 * H * Ish + 2 * E * H)}
    if kind == "gdn":
        B, vh = case["batch"], m["vh"]
        C, vd, slots = 2 * m["kh"] * DK + vh * DV, vh * DV, B if case["mode"] == "slots" else 1
        b = q(4, C + vd, H) + q(4, H, vd) + slots * (2 * vh * DK * DV * 4 + 2 * TAPS * C * 4)
        b += C * TAPS * 4 + B * (2 * H * 4 + 2 * vh * 4)
        return {"bytes": b, "flops": B * (2 * (C + vd) * H + 2 * vd * H + 7 * vh * DK * DV + 2 * C * TAPS)}
    if kind in ("gqa", "gqa_prefill"):
        nh, kv = m["nh"], NKV * HD
        b = q(4, 2 * nh * HD + 2 * kv, H) + (q(4, H, nh * HD) if case["o_fmt"] == 4 else H * nh * HD + 4 * H)
        if kind == "gqa":
            n, seq = case["batch"], case["context"]
            keys = [max(0, (seq - 1) * (n - i) // n - (i % 3 if i else 0)) + 1 for i in range(n)]
            b += 2 * sum(keys) * kv * 4
        else:
            n, seq = case["rows"], case["base"] + case["rows"]
            keys = range(case["base"] + 1, seq + 1)
            b += 2 * seq * kv * 4
        b += n * 2 * H * 4
        return {"bytes": b, "flops": n * (2 * (2 * nh * HD + 2 * kv) * H + 2 * nh * HD * H) + 4 * nh * HD * sum(keys)}
    if kind == "head":
        B, V = case["batch"], case["vocab"]
        return {"bytes": V * H + V * 4 + H * 4 + B * (V * 4 + 2 * H * 4), "flops": 2 * B * V * H}
    B, fmt = case["batch"], case["fmt"]
    used = case["cached"] * (1 - (1 - K / case["cached"]) ** B)  # K per token
    return {"bytes": used * (2 * q(fmt, I, H) + q(fmt, H, I)) + B * H * 6, "flops": B * K * 6 * H * I}


def tolerance(case):
    kind = case["kind"]
    if kind == "head":
        return "exact"  # integer dots: the contract is the CPU path's result, bit for bit
    if kind in ("stack", "moe", "block"):
        return {"rel": 1.5e-4, "max": 5e-3}  # 16-bit activation digits: 2e-5 to 4e-5 off the 64-bit result
    return {"rel": 3e-6, "max": 2e-4}  # 32-bit sums: 2e-7 to 6e-7 off the 64-bit result


# ---- the same results in 64 bits ---------------------------------------------------------------------


def _values(fmt, codes, scales, cols):
    """The matrix that container bytes and group scales stand for, in 64 bits."""
    lead = codes.shape[:-1]
    if fmt == 3:
        b = codes.reshape(*lead, -1, 3).to(torch.int32)
        word = b[..., 0] | (b[..., 1] << 8) | (b[..., 2] << 16)
        v = torch.stack([(word >> (3 * j)) & 7 for j in range(8)], -1) - 4
    elif fmt == 4:
        b = codes.to(torch.int32)
        v = torch.stack([b & 15, b >> 4], -1) - 8
    else:
        b = codes.to(torch.int32)
        v = 2 * torch.stack([(b >> (2 * j)) & 3 for j in range(4)], -1) - 3
    v = v.reshape(*lead, -1)[..., :cols].double()
    return v * scales.double().repeat_interleave(GS, -1)[..., :cols]


def _norm_rows(x, w):
    """x / rms * (1 + w) as the CPU path forms it: fp32, the squares summed one after another.  What follows
    quantises these rows, so a rounding more or less would be another input."""
    x = x.cpu().numpy()
    ms = np.add.accumulate(x * x, axis=1, dtype=np.float32)[:, -1:]
    r = np.float32(1) / np.sqrt(ms / np.float32(x.shape[1]) + np.float32(EPS))
    return torch.from_numpy(x * r * (np.float32(1) + w.cpu().numpy())).cuda()


def _quantise_rows(x):
    """int8 rows and their scales (fp32 arithmetic: part of the result's definition)."""
    s = (x.abs().amax(1, keepdim=True) / 127.0).clamp_(min=1e-12)
    return torch.round(x * (1.0 / s)).double(), s


def _dot8(x, q, s):
    xq, sx = _quantise_rows(x)
    return (xq @ q.double().t()).float() * s * sx


def _silu(v):
    return v * torch.sigmoid(v)


def _exact_moe(case, w, x):
    K, T = SHAPES[case["model"]]["K"], x.shape[0]
    H, I, fmt = SHAPES[case["model"]]["H"], SHAPES[case["model"]]["I"], w["fmt"]
    xd = x.double()
    logits = xd @ w["router"].double().t()
    top, idx = torch.topk(logits, K, dim=1)
    weight = torch.softmax(top, 1)
    gq, gs, uq, us, dq, ds = w["shared"]
    h = _silu(_dot8(x, gq, gs).double()) * _dot8(x, uq, us).double()
    y = _dot8(h.float(), dq, ds).double() * torch.sigmoid(xd @ w["sgate"].double())[:, None]
    for e in idx.unique().tolist():
        t, k = torch.nonzero(idx == e, as_tuple=True)
        xe = xd[t]
        h = _silu(xe @ _values(fmt, w["gate"][0][e], w["gate"][1][e], H).t())
        h = h * (xe @ _values(fmt, w["up"][0][e], w["up"][1][e], H).t())
        y.index_add_(0, t, (h @ _values(fmt, w["down"][0][e], w["down"][1][e], I).t()) * weight[t, k][:, None])
    return y, weight


def _project(x, w, cols):
    return x @ _values(4, w[0], w[1], cols).t()


def _exact_gdn(case, w):
    m, B = SHAPES[case["model"]], case["batch"]
    H, kh, vh = m["H"], m["kh"], m["vh"]
    kd, vd = kh * DK, vh * DV
    x = w["x"].double()
    raw, z = _project(x, w["qkv"], H), _project(x, w["z"], H)
    ring, state, conv = w["ring"].double(), w["state"].double(), w["conv"].double()
    core = torch.zeros(B, vd, device="cuda", dtype=torch.float64)
    for t in range(B):
        s, pos = int(w["slot"][t]), int(w["pos"][t])
        ring[s, pos % TAPS] = raw[t]
        taps = [conv[:, k] * ring[s, (pos - (TAPS - 1 - k)) % TAPS] for k in range(TAPS) if pos - (TAPS - 1 - k) >= 0]
        mix = _silu(torch.stack(taps).sum(0))
        qv, kv, vv = mix[:kd].view(kh, DK), mix[kd:2 * kd].view(kh, DK), mix[2 * kd:].view(vh, DV)
        qv = qv / torch.sqrt((qv * qv).sum(1, keepdim=True) + 1e-6) / math.sqrt(DK)
        kv = kv / torch.sqrt((kv * kv).sum(1, keepdim=True) + 1e-6)
        qv, kv = qv.repeat_interleave(vh // kh, 0), kv.repeat_interleave(vh // kh, 0)
        beta = torch.sigmoid(w["b"][t].double())
        pre = w["a"][t].double() + w["dt_bias"].double()
        decay = torch.exp(-torch.exp(w["a_log"].double()) * torch.nn.functional.softplus(pre, threshold=700.0))
        S = state[s] * decay[:, None, None]
        delta = (vv - (S * kv[:, :, None]).sum(1)) * beta[:, None]
        S = S + kv[:, :, None] * delta[:, None, :]
        state[s] = S
        o = (S * qv[:, :, None]).sum(1)
        o = o / torch.sqrt((o * o).mean(1, keepdim=True) + EPS) * w["norm"].double()
        core[t] = (o * _silu(z[t].view(vh, DV))).reshape(-1)
    return {"y": _project(core, w["out"], vd), "ring": ring, "state": state}


def _rotate(v, pos):
    """Partial rotary embedding; the angles are fp32 by definition."""
    half = RD // 2
    e = np.float32(-2.0) * np.arange(half, dtype=np.float32) / np.float32(RD)
    angle = torch.from_numpy(pos.astype(np.float32)[:, None] * np.power(float(THETA), e.astype(np.float64)).astype(np.float32))
    co, si = angle.double().cos().cuda()[:, None], angle.double().sin().cuda()[:, None]
    a, b = v[..., :half], v[..., half:RD]
    return torch.cat([a * co - b * si, b * co + a * si, v[..., RD:]], -1)


def _exact_gqa(case, w):
    m = SHAPES[case["model"]]
    H, nh, n, G = m["H"], m["nh"], w["x"].shape[0], m["nh"] // NKV
    x = w["x"].double()

    def norm(v, g):
        return v / torch.sqrt((v * v).mean(-1, keepdim=True) + EPS) * (1.0 + g.double())

    qp = _project(x, w["q"], H).view(n, nh, 2, HD)
    q, gate = _rotate(norm(qp[:, :, 0], w["q_norm"]), w["pos"]), qp[:, :, 1]
    k = _rotate(norm(_project(x, w["k"], H).view(n, NKV, HD), w["k_norm"]), w["pos"]).reshape(n, -1)
    v = _project(x, w["v"], H)
    kc, vc = w["k_cache"].double(), w["v_cache"].double()
    slot, pos = torch.from_numpy(w["slot"]).long().cuda(), torch.from_numpy(w["pos"]).long().cuda()
    kc[slot, pos], vc[slot, pos] = k, v
    ctx = torch.zeros(n, nh, HD, device="cuda", dtype=torch.float64)
    if case["kind"] == "gqa":
        rows = [slice(i, i + 1) for i in range(n)]
    else:
        rows = [slice(i, min(n, i + 256)) for i in range(0, n, 256)]
    for rs in rows:
        top = int(pos[rs].max()) + 1
        hide = torch.arange(top, device="cuda")[None] > pos[rs][:, None]
        for h in range(nh):
            kvh = h // G * HD
            s = q[rs, h] @ kc[slot[rs][0], :top, kvh:kvh + HD].t() / math.sqrt(HD)
            p = torch.softmax(s.masked_fill(hide, -math.inf), 1)
            ctx[rs, h] = p @ vc[slot[rs][0], :top, kvh:kvh + HD]
    ctx = (ctx * torch.sigmoid(gate)).reshape(n, nh * HD)
    if case["o_fmt"] == 4:
        y = _project(ctx, w["o"], nh * HD)
    else:
        y = (ctx @ w["o"][0].double().t()) * w["o"][1].double()
    return {"y": y, "k": kc, "v": vc}


def exact(case, seed):
    r, kind = _Rand(seed), case["kind"]
    if kind == "stack":
        x = _moe_x(r, case, case["layers"], case["tokens"])
        return {"y": torch.stack([_exact_moe(case, _moe_weights(r, case), x[l])[0] for l in range(case["layers"])])}
    if kind in ("moe", "block"):
        x = _moe_x(r, case, case["tokens"])
        norm = r.normal(SHAPES[case["model"]]["H"], std=0.1)
        w = _moe_weights(r, case)
        n = _norm_rows(x, norm) if kind == "block" else x
        y, weight = _exact_moe(case, w, n)
        # near-equal probabilities may change places in idx: no 64-bit value
        out = {"y": y, "weight": weight, "idx": None}
        if kind == "block":
            out["y"], out["hidden"] = x.double() + y, n.double()
        return out
    if kind == "gdn":
        return _exact_gdn(case, _gdn_inputs(r, case))
    if kind in ("gqa", "gqa_prefill"):
        return _exact_gqa(case, _gqa_inputs(r, case))
    if kind == "head":
        w = _head_inputs(r, case)
        n = _norm_rows(w["x"], w["norm"])
        xq, sx = _quantise_rows(n)
        logits = torch.cat([xq @ q.double().t() * s.double() for q, s in zip(w["q"].split(32768), w["s"].split(32768))], 1)
        return {"logits": logits * sx.double(), "hidden": n.double()}
    w, B = _grouped_inputs(r, case), case["batch"]
    m = SHAPES[case["model"]]
    y = torch.zeros(B, m["H"], device="cuda", dtype=torch.float64)
    for t in range(B):
        xt = w["x"][t].double()
        for e, p in zip(w["expert"][t].tolist(), w["weight"][t].tolist()):
            h = _silu(_values(case["fmt"], w["gate"][0][e], w["gate"][1][e], m["H"]) @ xt)
            h = h * (_values(case["fmt"], w["up"][0][e], w["up"][1][e], m["H"]) @ xt)
            y[t] += p * (_values(case["fmt"], w["down"][0][e], w["down"][1][e], m["I"]) @ h)
    return {"y": y}
