"""Measured cases of the MoE expert layer and its dense linears.

Two families, both through the public entry points a program calls:

* ``moe``: ``TP4MoE.forward_tensor`` at the DeepSeek-V4-Flash geometry (256
  routed experts + 1 shared, top-6, H=4096, I=2048), one call per pass.
  Weight formats: ``int4`` (int4-g128, the shared expert in the routed stack,
  router logits given by the caller, sigmoid scores), ``ckpt`` (the
  checkpoint's formats: MXFP4 routed experts and the FP8-block shared expert,
  the gate GEMM inside the call, sqrt-softplus scores with a selection bias)
  and ``w4a8`` (MXFP4 experts with e4m3 activations, the shared expert in the
  routed stack, the gate inside the call).
* ``linear``: the dense projections around the layer.  ``fp8``: W8A16 over
  the checkpoint's E4M3 weight as stored; ``int8``: W8A16 over int8 weights
  repacked at load time; ``w8a8``: block-FP8 activation quantisation and GEMM.
  ``graph`` cases replay one HIP graph of a decode step's projections, as a
  serving loop that captures its step does; the others call eagerly.

Weights are Gaussian (std 0.02) quantised in their own format, hidden states
N(0, 1) in bf16, router logits from the gate (or N(0, 1)).
"""

import importlib
import math

import torch

importlib.import_module("gaiban-lite_amd")

from gaiban_lite_amd import (  # noqa: E402
    ResidentFP8SharedExpert,
    ResidentGateWeights,
    ResidentInt4MoEWeights,
    ResidentMXFP4MoEWeights,
    TP4MoE,
    TP4MoEConfig,
    fp8_linear as F8,
    weight_only_linear as WL,
)

E, H, I, TOPK = 256, 4096, 2048, 6
ROUTE_SCALE, CLAMP = 1.5, 10.0
FP8 = torch.float8_e4m3fn
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _moe(name, fmt, tokens):
    return {"name": name, "kind": "moe", "fmt": fmt, "tokens": tokens}


def _linear(name, fmt, m, n, k=4096, graph=False):
    return {"name": name, "kind": "linear", "fmt": fmt, "m": m, "n": n, "k": k, "graph": graph}


def listed():
    return [
        # one user's decode step: latency and launches
        _moe("moe_int4_t1", "int4", 1),
        # a few concurrent users over the checkpoint as published
        _moe("moe_ckpt_t8", "ckpt", 8),
        # the decode batch the framework's headline is quoted on
        _moe("moe_int4_t64", "int4", 64),
        # a full serving batch (240 rows), fp8 activations
        _moe("moe_w4a8_t240", "w4a8", 240),
        # one chunk of a chunked prefill, ragged
        _moe("moe_ckpt_t1000", "ckpt", 1000),
        # a prompt of ordinary length, ragged, fp8 activations
        _moe("moe_w4a8_t3000", "w4a8", 3000),
        # the largest prefill batch
        _moe("moe_int4_t8192", "int4", 8192),
        # the projections of one decode step, captured: N = 1024, 4096 and 16384
        _linear("lin_fp8_m1_graph", "fp8", 1, "1024,4096,16384", graph=True),
        # the same for a ragged decode batch
        _linear("lin_fp8_m48_graph", "fp8", 48, "1024,4096,16384", graph=True),
        # a prefill chunk's output projection, int8 weights
        _linear("lin_int8_m512", "int8", 512, "4096"),
        # a prompt's wide projection, block-FP8 activations
        _linear("lin_w8a8_m2000", "w8a8", 2000, "16384"),
        # the largest prefill batch's projection over the checkpoint's bytes
        _linear("lin_fp8_m8192", "fp8", 8192, "4096"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    if rng.random() < 0.55:
        c = _moe("", rng.choice(("int4", "ckpt", "w4a8")), _log_int(rng, 1, 8192))
    else:
        fmt = rng.choice(("fp8", "int8", "w8a8"))
        m = _log_int(rng, 1, 8192)
        k = 128 * _log_int(rng, 8, 56)
        n = 16 * _log_int(rng, 32, 1024)
        graph = m <= 64 and rng.random() < 0.5
        c = _linear("", fmt, m, str(n), k, graph)
        if m > 1024 and m * n * k > 8192 * 16384 * 4096 // 2:
            c["m"] = 1024 + m % 1024
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------


def _gen(seed, what):
    return torch.Generator("cuda").manual_seed(seed * 1_000_003 + what)


def _randn(shape, seed, what):
    return torch.randn(shape, device="cuda", generator=_gen(seed, what))


def _int4_matrix(rows, k, seed, what):
    """(codes int8 [rows, k] in -8..7, bf16 scales [rows, k/128])."""

    w = _randn((rows, k // 128, 128), seed, what) * 0.02
    s = (w.abs().amax(-1) / 7.0).to(torch.bfloat16)
    q = torch.round(w / s.float()[..., None]).clamp_(-8, 7).to(torch.int8)
    return q.view(rows, k), s


def _mxfp4_matrix(rows, k, seed, what):
    """(E2M1 codes uint8 [rows, k], E8M0 bytes [rows, k/32])."""

    w = _randn((rows, k // 32, 32), seed, what) * 0.02
    e = torch.ceil(torch.log2(w.abs().amax(-1).clamp_min(1e-30) / 6.0)).clamp(-127, 127)
    v = w / torch.exp2(e)[..., None]
    mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda")
    code = torch.bucketize(v.abs(), mid).to(torch.uint8) | (v < 0).to(torch.uint8) << 3
    return code.view(rows, k), (e + 127).to(torch.uint8)


def _fp8_matrix(n, k, seed, what):
    """(E4M3 [n, k], E8M0 bytes [ceil(n/128), k/128])."""

    nb, kb = -(-n // 128), k // 128
    w = torch.zeros((nb * 128, k), device="cuda")
    w[:n] = _randn((n, k), seed, what) * 0.02
    w = w.view(nb, 128, kb, 128)
    e = torch.ceil(torch.log2(w.abs().amax((1, 3)).clamp_min(1e-30) / 448.0)).clamp(-127, 127)
    q = (w / torch.exp2(e)[:, None, :, None]).reshape(nb * 128, k)[:n].to(FP8)
    return q.contiguous(), (e + 127).to(torch.uint8).contiguous()


def _int8_matrix(n, k, seed, what):
    """(int8 [n, k], bf16 scales [n])."""

    w = _randn((n, k), seed, what) * 0.02
    s = (w.abs().amax(1) / 127.0).to(torch.bfloat16)
    return torch.round(w / s.float()[:, None]).clamp_(-127, 127).to(torch.int8), s


def _expert(fmt, e, seed):
    """Checkpoint codes and scales of expert e: (w13, s13, w2, s2)."""

    make = _int4_matrix if fmt == "int4" else _mxfp4_matrix
    return make(2 * I, H, seed, 10_000 + 2 * e) + make(H, I, seed, 10_001 + 2 * e)


def _shared_fp8(seed):
    return (_fp8_matrix(I, H, seed, 501) + _fp8_matrix(I, H, seed, 502) + _fp8_matrix(H, I, seed, 503))


def _hidden(tokens, seed):
    return _randn((tokens, H), seed, 1).to(torch.bfloat16)


def _gate(seed):
    return (_randn((E, H), seed, 2) * 0.03).to(torch.bfloat16), _randn((E,), seed, 3) * 0.1


def _nibbles(codes):
    c = codes.view(torch.uint8) & 15
    return c[:, 0::2] | c[:, 1::2] << 4


def _stack(fmt, seed, count):
    per = 128 if fmt == "int4" else 32
    sdt = torch.bfloat16 if fmt == "int4" else torch.uint8
    w13 = torch.empty((count, 2 * I, H // 2), dtype=torch.uint8, device="cuda")
    s13 = torch.empty((count, 2 * I, H // per), dtype=sdt, device="cuda")
    w2 = torch.empty((count, H, I // 2), dtype=torch.uint8, device="cuda")
    s2 = torch.empty((count, H, I // per), dtype=sdt, device="cuda")
    for e in range(count):
        q13, c13, q2, c2 = _expert(fmt, e, seed)
        w13[e], s13[e], w2[e], s2[e] = _nibbles(q13), c13, _nibbles(q2), c2
    return w13, s13, w2, s2


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------


def _prepare_moe(case, seed):
    fmt, tokens = case["fmt"], case["tokens"]
    grouped_shared = fmt != "ckpt"
    stack = _stack(fmt, seed, E + int(grouped_shared))
    adtype = FP8 if fmt == "w4a8" else None
    if fmt == "int4":
        res = ResidentInt4MoEWeights.from_checkpoint_layout(*stack, experts=E, has_shared=True)
        gate = ResidentGateWeights(weight=_gate(seed)[0])
    else:
        shared = None
        if fmt == "ckpt":
            shared = ResidentFP8SharedExpert.from_checkpoint(*_shared_fp8(seed))
        res = ResidentMXFP4MoEWeights.from_checkpoint_layout(*stack, experts=E, has_shared=grouped_shared,
                                                             shared_fp8=shared, marlin_input_dtype=adtype)
        wg, bias = _gate(seed)
        gate = ResidentGateWeights(weight=wg, bias=bias)
    del stack
    cfg = TP4MoEConfig(hidden_size=H, intermediate_size=I, experts=E, topk=TOPK, route_scale=ROUTE_SCALE,
                       clamp_limit=CLAMP, score_func="sigmoid" if fmt == "int4" else "sqrtsoftplus")
    layer = TP4MoE(config=cfg, resident=res, gate=gate, device=torch.device("cuda", torch.cuda.current_device()),
                   global_row_shapes=[tokens], marlin_input_dtype=adtype)
    state = {"layer": layer, "x": _hidden(tokens, seed).view(1, tokens, H), "logits": None}
    if fmt == "int4":
        state["logits"] = _randn((tokens, E), seed, 4)
    return state


def _projection(case, n, seed, what):
    """One projection's call on its own input, weight and buffers, and its outputs."""

    fmt, m, k = case["fmt"], case["m"], case["k"]
    x = _randn((m, k), seed, what).to(torch.bfloat16)
    out = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    if fmt == "w8a8":
        plan = F8.make_gemm_plan(m, n, k)
        quant = F8.make_quantization_plan(m, k)
        w, s = _fp8_matrix(n, k, seed, what + 1)
        s = s.view(torch.float8_e8m0fnu)
        q = torch.empty((m, k), dtype=FP8, device="cuda")
        qs = torch.empty((m, k // 128), dtype=torch.float8_e8m0fnu, device="cuda")
        ws = torch.empty(plan.workspace_shape, dtype=torch.float32, device="cuda")

        def call():
            F8.activation_quant_into(x, q, qs, plan=quant)
            F8.block_fp8_gemm_into(q, qs, w, s, out, ws, plan=plan)

        return call, (q.view(torch.uint8), qs.view(torch.uint8), out)
    plan = WL.make_gemm_plan(m, n, k)
    ws = WL.allocate_workspace(plan, x.device)
    if fmt == "int8":
        prepared = WL.prepare_int8_weight(*_int8_matrix(n, k, seed, what + 1))
        return lambda: WL.w8a16_prepared_gemm_into(x, prepared, out, ws, plan=plan), (out,)
    w, s = _fp8_matrix(n, k, seed, what + 1)
    s = s.view(torch.float8_e8m0fnu)
    return lambda: WL.w8a16_gemm_into(x, w, s, out, ws, plan=plan), (out,)


def _prepare_linear(case, seed):
    ns = [int(n) for n in case["n"].split(",")]
    calls = [_projection(case, n, seed, 100 + 10 * i) for i, n in enumerate(ns)]
    state = {"calls": [c for c, _ in calls], "outs": [o for _, outs in calls for o in outs], "graph": None}
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for call in state["calls"]:
                call()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for call in state["calls"]:
                call()
        state["graph"] = graph
    return state


def prepare(case, seed):
    return _prepare_moe(case, seed) if case["kind"] == "moe" else _prepare_linear(case, seed)


def run(state):
    if "layer" in state:
        return state["layer"].forward_tensor(state["x"], router_logits=state["logits"])
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        for call in state["calls"]:
            call()
    return state["outs"]


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------


def work(case):
    if case["kind"] == "moe":
        t, fmt = case["tokens"], case["fmt"]
        touched = E * (1.0 - (1.0 - TOPK / E) ** t)  # distinct experts of a uniform routing
        per_expert = 3 * H * I / 2 + (3 * H * I / 64 if fmt == "int4" else 3 * H * I / 32)
        shared = 3 * H * I * (1 + 1 / 16384) if fmt == "ckpt" else per_expert
        nbytes = touched * per_expert + shared + 2 * t * H * 2
        nbytes += t * E * 4 if fmt == "int4" else E * H * 2
        flops = 6.0 * t * (TOPK + 1) * H * I + (0.0 if fmt == "int4" else 2.0 * t * H * E)
        return {"bytes": nbytes, "flops": flops}
    m, k, fmt = case["m"], case["k"], case["fmt"]
    nbytes = flops = 0.0
    for n in (int(v) for v in case["n"].split(",")):
        scales = 2 * n if fmt == "int8" else -(-n // 128) * (k // 128)
        nbytes += n * k + scales + 2 * m * k + 2 * m * n
        if fmt == "w8a8":
            nbytes += m * k + m * (k // 128)
        flops += 2.0 * m * n * k
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # outputs are rounded once to bf16 (2^-9 relative), the expert layer's h
    # before the second product too; the w4a8 layer rounds h to e4m3, where a
    # last-bit difference of the first product moves some values by a code
    if case["kind"] == "moe":
        return {"rel": 2e-2 if case["fmt"] == "w4a8" else 1e-2}
    return {"rel": 1e-2}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------


def _route64(scores, bias):
    biased = scores if bias is None else scores + bias
    ids = biased.topk(TOPK, dim=-1).indices
    w = scores.gather(1, ids)
    return ids, w / w.sum(-1, keepdim=True) * ROUTE_SCALE


def _weight64(fmt, codes, scale):
    if fmt == "int4":
        return codes.double() * scale.double().repeat_interleave(128, 1)
    table = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device="cuda")
    return table[codes.int()] * torch.exp2(scale.double() - 127.0).repeat_interleave(32, 1)


def _fp8_64(codes, scale):
    n, k = codes.shape
    s = torch.exp2(scale.double() - 127.0).repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)
    return codes.double() * s


def _e4m3_rows(v):
    """Per-token e4m3 rounding (scale = largest magnitude / 448), dequantised."""

    f = v.float()
    s = f.abs().amax(-1, keepdim=True).clamp_min(1e-12) / 448.0
    return (f / s).clamp(-448.0, 448.0).to(FP8).double() * s.double()


def _ffn64(x, w13, w2, quantise):
    z = x @ w13.T
    g, u = z[:, :I].clamp(max=CLAMP), z[:, I:].clamp(-CLAMP, CLAMP)
    h = g * torch.sigmoid(g) * u
    return (_e4m3_rows(h.to(torch.bfloat16)) if quantise else h) @ w2.T


def exact(case, seed):
    if case["kind"] == "linear":
        outs = []
        for i, n in enumerate(int(v) for v in case["n"].split(",")):
            m, k, fmt, what = case["m"], case["k"], case["fmt"], 100 + 10 * i
            x = _randn((m, k), seed, what).to(torch.bfloat16)
            if fmt == "int8":
                q, s = _int8_matrix(n, k, seed, what + 1)
                outs.append(x.double() @ (q.double() * s.double()[:, None]).T)
                continue
            w = _fp8_64(*_fp8_matrix(n, k, seed, what + 1))
            if fmt == "fp8":
                outs.append(x.double() @ w.T)
                continue
            v = x.float().view(m, k // 128, 128)
            amax = v.abs().amax(-1).clamp_min(1e-4)
            e = torch.ceil(torch.log2(amax.double() * (1.0 / 448.0))).clamp(-126, 127)
            q = (v.double() / torch.exp2(e)[..., None]).clamp(-448, 448).float().to(FP8).double()
            outs += [None, None, (q * torch.exp2(e)[..., None]).view(m, k) @ w.T]
        return outs
    t, fmt = case["tokens"], case["fmt"]
    x = _hidden(t, seed).double()
    if fmt == "int4":
        ids, wts = _route64(torch.sigmoid(_randn((t, E), seed, 4).double()), None)
    else:
        wg, bias = _gate(seed)
        z = x @ wg.double().T
        ids, wts = _route64(torch.sqrt(torch.nn.functional.softplus(z)), bias.double())
    xq = _e4m3_rows(x) if fmt == "w4a8" else x
    out = torch.zeros((t, H), dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        row, col = (ids == e).nonzero(as_tuple=True)
        q13, s13, q2, s2 = _expert(fmt, e, seed)
        y = _ffn64(xq[row], _weight64(fmt, q13, s13), _weight64(fmt, q2, s2), fmt == "w4a8")
        out.index_add_(0, row, y * wts[row, col][:, None])
    if fmt == "ckpt":
        q1, s1, q3, s3, q2, s2 = _shared_fp8(seed)
        out += _ffn64(x, torch.cat([_fp8_64(q1, s1), _fp8_64(q3, s3)]), _fp8_64(q2, s2), False)
    else:
        q13, s13, q2, s2 = _expert(fmt, E, seed)
        out += _ffn64(xq, _weight64(fmt, q13, s13), _weight64(fmt, q2, s2), fmt == "w4a8")
    return out.view(1, t, H)
