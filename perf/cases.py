"""What a serving program asks of the INT4-G128 projections, as measurable cases.

Each case is one call (or one short sequence of calls) through
``xinfer_amd.ops`` with the weights, norms, workspaces and output buffers a
program holds between calls.  Sizes are the decode, verify and prefill shapes
that ``bench.py`` and the tests use (hidden 5120, intermediate 17408,
attention output 6144, vocabulary 151936), plus ragged ones.

Three regimes, by the number of activation rows M:

* decode, M = 1: one token;
* verify, M = 2..8: the tokens a speculative step proposes;
* prefill, M up to 512: one chunk of a prompt.  The last chunk of a prompt has
  whatever length is left, so every M from 1 to 512 is met.

The reference loads weights once per process and keeps its FP32-activation
overloads and the device dequantisation for cross-checks, so neither is here.
"""
import math

import torch
import torch.nn.functional as F

from xinfer_amd import ops

GROUP = 128
EPS = 1e-6
HIDDEN, INTER, ATTN, VOCAB = 5120, 17408, 6144, 151936

# Ranges that draw() covers (and the listed cases come from).
M_MAX, LM_HEAD_M_MAX = 512, 8
K_GROUPS = (4, 136)          # K = 512 .. 17408
N_RANGE = (48, 34816)        # output rows of one matrix
VOCAB_RANGE = (32000, 151936)
MOST_MACS = 2 * INTER * HIDDEN * M_MAX
MOST_WEIGHTS = VOCAB * HIDDEN


def listed():
    return [
        # The smallest call of a decode step: the attention output projection.
        {"name": "decode_o_proj", "op": "linear", "m": 1, "k": ATTN, "n": str(HIDDEN), "bias": False, "out": "f16"},
        # Decode: input norm and the three attention projections over one X.
        {"name": "decode_norm_qkv", "op": "norm_fused", "m": 1, "k": HIDDEN, "n": "12288,1024,1024"},
        # Decode: post-attention norm and the gated MLP's first half.
        {"name": "decode_norm_gate_up", "op": "norm_gate_up", "m": 1, "k": HIDDEN, "n": str(INTER)},
        # One decode step as it is issued: a layer's projections, the final
        # norm and the LM head, replayed from a captured graph.
        {"name": "decode_step_graph", "op": "step", "m": 1, "k": HIDDEN, "n": str(INTER), "vocab": VOCAB},
        # Verify: the MLP block of four proposed tokens.
        {"name": "verify_mlp_m4", "op": "mlp", "m": 4, "k": HIDDEN, "n": str(INTER)},
        # Verify: logits and greedy tokens of eight rows.
        {"name": "verify_lm_head_m8", "op": "lm_head", "m": 8, "k": HIDDEN, "n": str(VOCAB)},
        # Prefill, a full chunk: the four projections of a layer.
        {"name": "prefill_norm_qkv_m512", "op": "norm_fused", "m": 512, "k": HIDDEN, "n": "12288,1024,1024"},
        {"name": "prefill_norm_gate_up_m512", "op": "norm_gate_up", "m": 512, "k": HIDDEN, "n": str(INTER)},
        {"name": "prefill_down_m512", "op": "residual", "m": 512, "k": INTER, "n": str(HIDDEN)},
        # Prefill, the ragged end of a prompt: the linear-attention input
        # projections (two of them only 48 rows wide) of 77 tokens ...
        {"name": "prefill_norm_la_m77", "op": "norm_fused", "m": 77, "k": HIDDEN, "n": "10240,6144,48,48"},
        # ... and the MLP block of a short one.
        {"name": "prefill_mlp_m23", "op": "mlp", "m": 23, "k": HIDDEN, "n": str(INTER)},
        # Sizes that are no multiple of any tile, with bias and FP32 output
        # (per-token scores of a prompt): K = 27 groups, odd N.
        {"name": "ragged_bias_f32_m200", "op": "linear", "m": 200, "k": 3456, "n": "5003", "bias": True, "out": "f32"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    op = rng.choice(("linear", "linear", "residual", "norm_fused", "norm_fused", "norm_gate_up", "norm_gate_up", "mlp",
                     "lm_head"))
    while True:
        # widths of models: half of them multiples of 1024, the rest any
        # whole number of groups
        g = _log_int(rng, *K_GROUPS)
        k = GROUP * (max(8, 8 * round(g / 8)) if rng.random() < 0.5 else g)
        m = _log_int(rng, 1, LM_HEAD_M_MAX if op == "lm_head" else M_MAX)
        c = {"op": op, "m": m, "k": k}
        if op == "lm_head":
            c["n"] = str(_log_int(rng, *VOCAB_RANGE))
        elif op == "norm_fused":
            c["n"] = ",".join(str(_log_int(rng, N_RANGE[0], N_RANGE[1] // 2)) for _ in range(rng.randint(2, 4)))
        elif op in ("norm_gate_up", "mlp"):
            c["n"] = str(GROUP * _log_int(rng, K_GROUPS[0], K_GROUPS[1]))  # the width of the down projection's X
        else:
            c["n"] = str(_log_int(rng, *N_RANGE))
        if op == "linear":
            c["bias"] = rng.random() < 0.5
            c["out"] = rng.choice(("f16", "f16", "f32"))
        rows = sum(_rows(c)) * (2 if op == "mlp" else 1)
        if rows * k * m <= MOST_MACS and rows * k <= MOST_WEIGHTS:
            return c


def _rows(case):
    """Output rows of the matrices that read the case's X."""
    n = [int(v) for v in case["n"].split(",")]
    return n * 2 if case["op"] in ("norm_gate_up", "mlp", "step") else n


# ---- inputs -----------------------------------------------------------------

def _quantised(gen, n, k, row_gain=None):
    """Gaussian weights through the converter's symmetric group quantisation:
    packed nibbles [n][k/2] (low nibble first) and fp16 scales [n][k/128]."""
    w4 = torch.empty((n, k // 2), dtype=torch.uint8, device="cuda")
    s = torch.empty((n, k // GROUP), dtype=torch.float16, device="cuda")
    for r in range(0, n, 16384):
        w = torch.randn((min(16384, n - r), k // GROUP, GROUP), generator=gen, device="cuda") * 0.02
        if row_gain is not None:
            w *= row_gain[r:r + w.shape[0], None, None]
        sc = (w.abs().amax(-1) / 7).clamp_min(1e-6).half()
        q = (w / sc.float()[..., None]).round_().clamp_(-8, 7).to(torch.int8).view(w.shape[0], k)
        w4[r:r + w.shape[0]] = ((q[:, 0::2] & 15) | (q[:, 1::2] << 4)).view(torch.uint8)
        s[r:r + w.shape[0]] = sc
    return w4, s


def _f16(gen, m, k):
    return torch.randn((m, k), generator=gen, device="cuda").half()


def _norm_weight(gen, k):
    return 1.0 + 0.1 * torch.randn(k, generator=gen, device="cuda")


def _empty(m, n, dtype=torch.float16):
    return torch.empty((m, n), dtype=dtype, device="cuda")


def _norm_workspace(m, k):
    return torch.empty(max(16, ops.rmsnorm_projection_workspace_size(m, k)), dtype=torch.uint8, device="cuda")


def _lm_scratch(m, n, k):
    return torch.empty(max(16, ops.lm_head_argmax_scratch_size(m, n, k)), dtype=torch.uint8, device="cuda")


def _vocab_gain(gen, n):
    # rows of a vocabulary matrix differ in norm, which separates the top logits
    return torch.exp(0.3 * torch.randn(n, generator=gen, device="cuda"))


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    op, m, k = case["op"], case["m"], case["k"]
    n = [int(v) for v in case["n"].split(",")]
    st = {"op": op, "m": m, "k": k, "n": n[0]}
    if op == "linear":
        st["x"] = _f16(gen, m, k)
        st["w"], st["s"] = _quantised(gen, n[0], k)
        st["bias"] = torch.randn(n[0], generator=gen, device="cuda") if case["bias"] else None
        st["y"] = _empty(m, n[0], torch.float32 if case["out"] == "f32" else torch.float16)
    elif op == "residual":
        # the down projection's X is a gated product
        st["x"] = (F.silu(torch.randn((m, k), generator=gen, device="cuda")) *
                   torch.randn((m, k), generator=gen, device="cuda")).half()
        st["w"], st["s"] = _quantised(gen, n[0], k)
        st["hidden"] = _f16(gen, m, n[0])
        st["stream"] = _empty(m, n[0])
    elif op == "norm_fused":
        st["x"] = _f16(gen, m, k)
        st["norm"] = _norm_weight(gen, k)
        st["ws"] = _norm_workspace(m, k)
        st["descs"] = [ops.FusedProjectionDesc(_empty(m, r), *_quantised(gen, r, k), None, r) for r in n]
    elif op == "norm_gate_up":
        st["x"] = _f16(gen, m, k)
        st["norm"] = _norm_weight(gen, k)
        st["ws"] = _norm_workspace(m, k)
        st["gate"], st["up"] = _quantised(gen, n[0], k), _quantised(gen, n[0], k)
        st["y"] = _empty(m, n[0])
    elif op == "mlp":
        st["hidden"] = _f16(gen, m, k)
        st["stream"] = _empty(m, k)
        st["norm"] = _norm_weight(gen, k)
        st["ws"] = _norm_workspace(m, k)
        st["gate"], st["up"] = _quantised(gen, n[0], k), _quantised(gen, n[0], k)
        st["down"] = _quantised(gen, k, n[0])
        st["act"] = _empty(m, n[0])
    elif op == "lm_head":
        st["x"] = _f16(gen, m, k)
        st["w"], st["s"] = _quantised(gen, n[0], k, _vocab_gain(gen, n[0]))
        st["ids"] = torch.empty(m, dtype=torch.int32, device="cuda")
        st["logits"] = _empty(m, n[0], torch.float32)
        st["scratch"] = _lm_scratch(m, n[0], k)
    else:
        v = case["vocab"]
        st["hidden"], st["attn"] = _f16(gen, m, k), _f16(gen, m, ATTN)
        st["stream"], st["act"], st["last"] = _empty(m, k), _empty(m, n[0]), _empty(m, k)
        st["norms"] = [_norm_weight(gen, k) for _ in range(3)]
        st["ws"] = _norm_workspace(m, k)
        st["descs"] = [ops.FusedProjectionDesc(_empty(m, r), *_quantised(gen, r, k), None, r)
                       for r in (2 * ATTN, 1024, 1024)]
        st["o"] = _quantised(gen, k, ATTN)
        st["gate"], st["up"] = _quantised(gen, n[0], k), _quantised(gen, n[0], k)
        st["down"] = _quantised(gen, k, n[0])
        st["w"], st["s"] = _quantised(gen, v, k, _vocab_gain(gen, v))
        st["vocab"] = v
        st["ids"] = torch.empty(m, dtype=torch.int32, device="cuda")
        st["logits"] = _empty(m, v, torch.float32)
        st["scratch"] = _lm_scratch(m, v, k)
        _step(st)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            _step(st)
    return st


# ---- one pass ---------------------------------------------------------------

def _mlp(st, norm):
    m, k, n = st["m"], st["k"], st["n"]
    ops.rmsnorm_mlp_gate_up_swiglu_int4(st["act"], st["stream"], norm, EPS, *st["gate"], *st["up"], m, n, k,
                                        workspace=st["ws"])
    ops.linear_int4_residual(st["stream"], st["act"], *st["down"], None, m, k, n)


def _step(st):
    m, k = st["m"], st["k"]
    st["stream"].copy_(st["hidden"])
    ops.rmsnorm_linear_int4_fused(st["stream"], st["norms"][0], EPS, st["descs"], 3, m, k, workspace=st["ws"])
    ops.linear_int4_residual(st["stream"], st["attn"], *st["o"], None, m, k, ATTN)
    _mlp(st, st["norms"][1])
    ops.rmsnorm(st["last"], st["stream"], st["norms"][2], m, k, EPS)
    ops.lm_head_argmax_int4(st["ids"], st["logits"], st["last"], st["w"], st["s"], m, st["vocab"], k,
                            scratch=st["scratch"])


def run(st):
    op, m, k = st["op"], st["m"], st["k"]
    if op == "linear":
        ops.linear_int4(st["y"], st["x"], st["w"], st["s"], st["bias"], m, st["n"], k)
        return st["y"]
    if op == "residual":  # the residual stream is updated in place: it starts from this pass's hidden state
        st["stream"].copy_(st["hidden"])
        ops.linear_int4_residual(st["stream"], st["x"], st["w"], st["s"], None, m, st["n"], k)
        return st["stream"]
    if op == "norm_fused":
        ops.rmsnorm_linear_int4_fused(st["x"], st["norm"], EPS, st["descs"], len(st["descs"]), m, k,
                                      workspace=st["ws"])
        return [d.Y for d in st["descs"]]
    if op == "norm_gate_up":
        ops.rmsnorm_mlp_gate_up_swiglu_int4(st["y"], st["x"], st["norm"], EPS, *st["gate"], *st["up"], m, st["n"], k,
                                            workspace=st["ws"])
        return st["y"]
    if op == "mlp":
        st["stream"].copy_(st["hidden"])
        _mlp(st, st["norm"])
        return {"act": st["act"], "stream": st["stream"]}
    if op == "lm_head":
        ops.lm_head_argmax_int4(st["ids"], st["logits"], st["x"], st["w"], st["s"], m, st["n"], k,
                                scratch=st["scratch"])
        return {"ids": st["ids"], "logits": st["logits"]}
    st["graph"].replay()
    return {"ids": st["ids"], "logits": st["logits"], "qkv": [d.Y for d in st["descs"]], "stream": st["stream"]}


# ---- what a pass cannot do without -------------------------------------------

def _projection(m, n, k, out_bytes=2):
    """(bytes, flops) of one projection's weights, scales and output."""
    return n * k // 2 + n * (k // GROUP) * 2 + m * n * out_bytes, 2 * m * n * k


def work(case):
    op, m, k = case["op"], case["m"], case["k"]
    n = [int(v) for v in case["n"].split(",")]
    b, f = m * k * 2, 0  # X

    def add(rows, width, out_bytes=2, extra=0):
        nonlocal b, f
        pb, pf = _projection(m, rows, width, out_bytes)
        b, f = b + pb + extra, f + pf

    if op == "linear":
        add(n[0], k, 4 if case["out"] == "f32" else 2, 4 * n[0] if case["bias"] else 0)
    elif op == "residual":
        add(n[0], k, 2, 2 * m * n[0])
    elif op == "norm_fused":
        b += 4 * k
        for r in n:
            add(r, k)
    elif op == "norm_gate_up":
        b += 4 * k
        add(n[0], k, 0)
        add(n[0], k)
    elif op == "lm_head":
        add(n[0], k, 4, 4 * m)
    else:
        b += 4 * k
        add(n[0], k, 0)
        add(n[0], k)
        add(k, n[0])
        if op == "step":
            b += 8 * k + 2 * m * ATTN
            for r in (2 * ATTN, 1024, 1024):
                add(r, k)
            add(k, ATTN, 0)
            add(case["vocab"], k, 4, 4 * m)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # about four times the measured relative error against exact(): up to
    # 1.2e-5 (FP32 outputs), 4.4e-4 (one projection), 5.3e-4 (MLP block) and
    # 6.2e-4 (decode step)
    op, m, k = case["op"], case["m"], case["k"]
    if op == "lm_head" or (op == "linear" and case["out"] == "f32"):
        # FP32 sums of fp16 products, the order left open; an id may change
        # where two logits tie within that
        return {"rel": 5e-5, "max": 4e-4, "differ": 0.01}
    if op == "step":  # logits of a hidden state that was rounded to fp16 several times
        return {"rel": 2.5e-3, "max": 0.03, "differ": 0.01}
    if op == "mlp":  # the second projection reads rounded activations
        return {"rel": 2e-3, "max": 0.03}
    return {"rel": 1.7e-3, "max": 0.02}


# ---- the same in 64 bits ------------------------------------------------------

def _linear64(x, w4, s):
    """x [m][k] times the dequantised weights' transpose, in double."""
    m, k = x.shape
    y = torch.empty((m, w4.shape[0]), dtype=torch.float64, device="cuda")
    for r in range(0, w4.shape[0], 8192):
        p = w4[r:r + 8192]
        q = torch.stack(((p & 15).to(torch.int8), (p >> 4).to(torch.int8)), dim=-1).view(p.shape[0], k)
        q = torch.where(q > 7, q - 16, q).double().view(p.shape[0], k // GROUP, GROUP)
        w = (q * s[r:r + 8192].double()[..., None]).view(p.shape[0], k)
        y[:, r:r + 8192] = x @ w.t().contiguous()
    return y


def _norm64(x, weight):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * weight.double()


def _gate_up64(x, gate, up):
    g = _linear64(x, *gate)
    return g * torch.sigmoid(g) * _linear64(x, *up)


def exact(case, seed):
    st = prepare(case, seed)
    op = st["op"]
    if op == "linear":
        y = _linear64(st["x"].double(), st["w"], st["s"])
        return y if st["bias"] is None else y + st["bias"].double()
    if op == "residual":
        return st["hidden"].double() + _linear64(st["x"].double(), st["w"], st["s"])
    if op == "norm_fused":
        x = _norm64(st["x"].double(), st["norm"])
        return [_linear64(x, d.W_int4, d.scales) for d in st["descs"]]
    if op == "norm_gate_up":
        return _gate_up64(_norm64(st["x"].double(), st["norm"]), st["gate"], st["up"])
    if op == "lm_head":
        return {"ids": None, "logits": _linear64(st["x"].double(), st["w"], st["s"])}
    h = st["hidden"].double()
    if op == "mlp":
        act = _gate_up64(_norm64(h, st["norm"]), st["gate"], st["up"])
        return {"act": act, "stream": h + _linear64(act, *st["down"])}
    x = _norm64(h, st["norms"][0])
    qkv = [_linear64(x, d.W_int4, d.scales) for d in st["descs"]]
    h = h + _linear64(st["attn"].double(), *st["o"])
    act = _gate_up64(_norm64(h, st["norms"][1]), st["gate"], st["up"])
    h = h + _linear64(act, *st["down"])
    logits = _linear64(_norm64(h, st["norms"][2]), st["w"], st["s"])
    return {"ids": None, "logits": logits, "qkv": qkv, "stream": h}
