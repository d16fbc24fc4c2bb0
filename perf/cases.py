"""The work this library is timed on: whole calls of its public entry points.

Four kinds of call, as the two programs that use the library make them:

  layer   RoutedMoE.forward (k3_moe_forward_bf16): a serving program with one
          K3 layer's experts resident in HBM, from one token to an 8K prefill
  native  NativeLayer.forward (k3_moe_native_forward_bf16): the K3 engine's
          whole MoE block (router, latent projections, experts, norm, shared
          expert, adds)
  expert  one routed expert's rows through the per-matrix entry points, as
          the engine's prefill loop issues them (gather, gate, up, SiTU, down,
          scatter)
  shared  the dense shared expert through the per-matrix Q8-128 entry points

Everything is seeded torch on the GPU. Expert bytes have the distribution of
the library's own synthetic store (uniform e2m1 codes, E8M0 exponents
121..125); router weights N(0, 0.02), token rows N(0, 1), as in its benchmark.
"""
import ctypes
import math
from types import SimpleNamespace

import numpy as np
import torch

from moonshine_amd import layer as L
from moonshine_amd import native as N
from moonshine_amd._lib import lib
from moonshine_amd.synth import ACT_SITU, ACT_SWIGLU, EXACT, MFMA, Config

ALIGN = 256

# (hidden, ffn, experts, top_k, activation, scale) of the routed layer
SHAPES = {
    "k3": (7168, 2048, 896, 16, ACT_SWIGLU, 2.5),        # the benchmark's K3 layer
    "reduced": (2048, 512, 64, 4, ACT_SWIGLU, 2.5),      # its reduced configuration
    "latent": (3584, 3072, 896, 16, ACT_SITU, 1.0),      # the K3 engine's expert stage
    "small": (1024, 1024, 40, 6, ACT_SITU, 1.5),          # a small generic layer
}
# the K3 block around the latent experts
NATIVE_HIDDEN, NATIVE_SHARED, EPS = 7168, 6144, 1e-5
BETA, LINEAR_BETA = 4.0, 25.0


def listed():
    return [
        # one token through the reduced layer: launches and latency only
        dict(name="decode-reduced", kind="layer", shape="reduced", tokens=1, precision=EXACT,
             zipf=False),
        # one token of K3 decode, the benchmark's headline call
        dict(name="decode-k3", kind="layer", shape="k3", tokens=1, precision=EXACT, zipf=False),
        # a handful of sequences decoded together, at the default precision
        dict(name="batch-5-exact", kind="layer", shape="k3", tokens=5, precision=EXACT,
             zipf=False),
        # batched decode of 64 sequences on the matrix path
        dict(name="batch-64", kind="layer", shape="k3", tokens=64, precision=MFMA, zipf=False),
        # a ragged prompt at the default (bit-exact) precision
        dict(name="prefill-333-exact", kind="layer", shape="k3", tokens=333, precision=EXACT,
             zipf=False),
        # a prefill chunk of 512 tokens
        dict(name="prefill-512", kind="layer", shape="k3", tokens=512, precision=MFMA, zipf=False),
        # an 8K prefill with skewed routing: a few heavy experts, many light ones
        dict(name="prefill-8192-zipf", kind="layer", shape="k3", tokens=8192, precision=MFMA,
             zipf=True),
        # one token through the engine's whole MoE block
        dict(name="native-decode", kind="native", tokens=1, precision=EXACT),
        # a small batch through the block at the default precision
        dict(name="native-batch-20-exact", kind="native", tokens=20, precision=EXACT),
        # a long prompt chunk through the block on the matrix path
        dict(name="native-prefill-2048", kind="native", tokens=2048, precision=MFMA),
        # the engine's own prefill loop: one expert's 77 rows, op by op
        dict(name="engine-expert-77", kind="expert", tokens=300, rows=77),
        # the engine's shared expert over a 300-token chunk, op by op
        dict(name="engine-shared-300", kind="shared", tokens=300),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer-decode", "layer-exact", "layer-exact", "layer-mfma", "layer-mfma",
                       "native-exact", "native-mfma", "expert", "shared"])
    if kind == "layer-decode":
        return dict(kind="layer", shape=rng.choice(sorted(SHAPES)), tokens=1,
                    precision=rng.choice([EXACT, MFMA]), zipf=rng.random() < 0.5)
    if kind == "layer-exact":
        return dict(kind="layer", shape=rng.choice(sorted(SHAPES)), tokens=_log_int(rng, 2, 333),
                    precision=EXACT, zipf=rng.random() < 0.5)
    if kind == "layer-mfma":
        return dict(kind="layer", shape=rng.choice(sorted(SHAPES)), tokens=_log_int(rng, 2, 8192),
                    precision=MFMA, zipf=rng.random() < 0.5)
    if kind == "native-exact":
        return dict(kind="native", tokens=_log_int(rng, 1, 96), precision=EXACT)
    if kind == "native-mfma":
        return dict(kind="native", tokens=_log_int(rng, 2, 2048), precision=MFMA)
    if kind == "expert":
        rows = _log_int(rng, 1, 300)
        return dict(kind="expert", tokens=max(300, rows), rows=rows)
    return dict(kind="shared", tokens=_log_int(rng, 1, 512))


# ---- inputs, made from the seed alone ---------------------------------------------------


def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 64 + part)
    return g


def _normal(shape, std, gen, mean=0.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std + mean).to(torch.bfloat16)


def _bias(experts, zipf, seed):
    g = _gen(seed, 1)
    if not zipf:
        return torch.randn(experts, generator=g, device="cuda") * 0.01
    rank = torch.randperm(experts, generator=g, device="cuda") + 1
    return (2.0 * rank.double() ** -1.1).float()


def _expert_spans(hidden, ffn):
    """(offset, bytes) of w1/w2/w3 packed and scale tensors, and one expert's span."""
    spans, off = [], 0
    for size in L.expert_tensor_sizes(hidden, ffn):
        spans.append((off, size))
        off += -(-size // ALIGN) * ALIGN
    return spans, off


def _expert_bytes(experts, hidden, ffn, seed):
    """[experts, span] bytes: uniform e2m1 codes, E8M0 exponents 121..125."""
    g = _gen(seed, 2)
    spans, span = _expert_spans(hidden, ffn)
    buf = torch.empty((experts, span), dtype=torch.uint8, device="cuda")
    buf.random_(0, 256, generator=g)
    for j, (off, size) in enumerate(spans):
        if j % 2 == 1:
            buf[:, off:off + size] = torch.randint(121, 126, (experts, size), dtype=torch.uint8,
                                                   device="cuda", generator=g)
    return buf


def _store(experts, hidden, ffn, seed):
    buf = _expert_bytes(experts, hidden, ffn, seed)
    spans, span = _expert_spans(hidden, ffn)
    base = np.arange(experts, dtype=np.uint64)[:, None] * np.uint64(span)
    table = base + np.array([o for o, _ in spans], dtype=np.uint64)[None, :]
    table += np.uint64(buf.data_ptr())
    return SimpleNamespace(buffer=buf, table=torch.from_numpy(table.view(np.int64)).cuda())


def _static(rows, cols, seed, part):
    """A Q8-128 static projection of N(0, 0.02): int8 codes and block scales."""
    w = torch.randn((rows, cols // 128, 128), generator=_gen(seed, part), device="cuda") * 0.02
    scales = w.abs().amax(dim=2) / 127.0
    codes = torch.clamp(torch.round(w / scales[:, :, None]), -127, 127).to(torch.int8)
    return codes.view(rows, cols).contiguous(), scales.contiguous()


def _native_statics(seed):
    D, H, S = SHAPES["latent"][0], NATIVE_HIDDEN, NATIVE_SHARED
    return dict(routed_down=_static(D, H, seed, 10), routed_up=_static(H, D, seed, 11),
                shared_gate=_static(S, H, seed, 12), shared_up=_static(S, H, seed, 13),
                shared_down=_static(H, S, seed, 14))


def _prepare_layer(case, seed):
    hidden, ffn, experts, top_k, act, scale = SHAPES[case["shape"]]
    T = case["tokens"]
    cfg = Config(case["shape"], T, hidden, experts, top_k, ffn, scale=scale, activation=act,
                 beta=BETA, linear_beta=LINEAR_BETA)
    moe = L.RoutedMoE(cfg, _normal((experts, hidden), 0.02, _gen(seed, 3)),
                      _bias(experts, case["zipf"], seed), _store(experts, hidden, ffn, seed))
    moe.workspace(T)
    x = _normal((T, hidden), 1.0, _gen(seed, 4))
    return dict(kind="layer", moe=moe, x=x, residual=_normal((T, hidden), 1.0, _gen(seed, 5)),
                out=torch.empty_like(x), precision=case["precision"],
                ids=torch.zeros((T, top_k), dtype=torch.int32, device="cuda"),
                weights=torch.zeros((T, top_k), dtype=torch.float32, device="cuda"))


def _prepare_native(case, seed):
    D, ffn, experts, top_k, act, scale = SHAPES["latent"]
    T, H = case["tokens"], NATIVE_HIDDEN
    cfg = N.NativeConfig("k3-native", T, H, D, experts, top_k, ffn, NATIVE_SHARED, scale=scale,
                         activation=act, beta=BETA, linear_beta=LINEAR_BETA, eps=EPS, seed=0)
    layer = N.NativeLayer(cfg, store=_store(experts, D, ffn, seed))
    # the checkpoint's tensors, copied into the layer's own
    layer.router_weight.copy_(_normal((experts, H), 0.02, _gen(seed, 3)).view(torch.int16))
    layer.router_bias_d.copy_(_bias(experts, False, seed))
    layer.norm.copy_(_normal((D,), 0.1, _gen(seed, 6), mean=1.0).view(torch.int16))
    statics = layer.statics()
    for name, (codes, scales) in _native_statics(seed).items():
        statics[name].data.copy_(codes)
        statics[name].scales.copy_(scales)
    layer.workspace(T)
    x = _normal((T, H), 1.0, _gen(seed, 4))
    return dict(kind="native", layer=layer, x=x,
                residual=_normal((T, H), 1.0, _gen(seed, 5)), out=torch.empty_like(x),
                precision=case["precision"],
                ids=torch.zeros((T, top_k), dtype=torch.int32, device="cuda"),
                weights=torch.zeros((T, top_k), dtype=torch.float32, device="cuda"))


def _expert_rows(case, seed):
    """Ascending token rows of the expert, a sample without repeats."""
    perm = torch.randperm(case["tokens"], generator=_gen(seed, 7), device="cuda")
    return perm[:case["rows"]].sort().values.to(torch.int32)


def _prepare_expert(case, seed):
    hidden, ffn = SHAPES["latent"][:2]
    n = case["rows"]
    bf = dict(dtype=torch.bfloat16, device="cuda")
    return dict(kind="expert", hidden=hidden, ffn=ffn, rows=n,
                x=_normal((case["tokens"], hidden), 1.0, _gen(seed, 4)),
                ids=_expert_rows(case, seed), weights=_expert_bytes(1, hidden, ffn, seed)[0],
                gathered=torch.empty((n, hidden), **bf), gate=torch.empty((n, ffn), **bf),
                up=torch.empty((n, ffn), **bf), act=torch.empty((n, ffn), **bf),
                y=torch.empty((n, hidden), **bf),
                out=torch.zeros((case["tokens"], hidden), **bf))


def _prepare_shared(case, seed):
    H, S, T = NATIVE_HIDDEN, NATIVE_SHARED, case["tokens"]
    bf = dict(dtype=torch.bfloat16, device="cuda")
    return dict(kind="shared", tokens=T, x=_normal((T, H), 1.0, _gen(seed, 4)),
                gate_w=_static(S, H, seed, 12), up_w=_static(S, H, seed, 13),
                down_w=_static(H, S, seed, 14), gate=torch.empty((T, S), **bf),
                up=torch.empty((T, S), **bf), act=torch.empty((T, S), **bf),
                out=torch.empty((T, H), **bf))


def prepare(case, seed):
    return {"layer": _prepare_layer, "native": _prepare_native, "expert": _prepare_expert,
            "shared": _prepare_shared}[case["kind"]](case, seed)


# ---- one pass ---------------------------------------------------------------------------


def _p(t, offset=0):
    return ctypes.c_void_p(t.data_ptr() + offset)


def _must(ok, what):
    if not ok:
        raise RuntimeError(f"{what} rejected its arguments or failed to launch")


def _run_expert(s):
    lb, st = lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    n, hidden, ffn, w = s["rows"], s["hidden"], s["ffn"], s["weights"]
    off = [o for o, _ in _expert_spans(hidden, ffn)[0]]
    gemm = lb.k3_rocm_mxfp4_gemm_bf16
    _must(lb.k3_rocm_gather_rows_bf16(_p(s["gathered"]), _p(s["x"]), _p(s["ids"]), n, hidden, st),
          "gather")
    _must(gemm(_p(s["gate"]), _p(w, off[0]), _p(w, off[1]), _p(s["gathered"]), n, ffn, hidden, st),
          "gate")
    _must(gemm(_p(s["up"]), _p(w, off[4]), _p(w, off[5]), _p(s["gathered"]), n, ffn, hidden, st),
          "up")
    _must(lb.k3_rocm_situ_bf16(_p(s["act"]), _p(s["gate"]), _p(s["up"]), n * ffn, BETA,
                               LINEAR_BETA, st), "situ")
    _must(gemm(_p(s["y"]), _p(w, off[2]), _p(w, off[3]), _p(s["act"]), n, hidden, ffn, st), "down")
    _must(lb.k3_rocm_scatter_rows_bf16(_p(s["out"]), _p(s["y"]), _p(s["ids"]), n, hidden, st),
          "scatter")
    return s["out"]


def _run_shared(s):
    lb, st = lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    H, S, T = NATIVE_HIDDEN, NATIVE_SHARED, s["tokens"]
    gemm = lb.k3_rocm_q8_128_gemm_bf16
    for name in ("gate", "up"):
        codes, scales = s[name + "_w"]
        _must(gemm(_p(s[name]), _p(codes), _p(scales), _p(s["x"]), T, S, H, st), name)
    _must(lb.k3_rocm_situ_bf16(_p(s["act"]), _p(s["gate"]), _p(s["up"]), T * S, BETA, LINEAR_BETA,
                               st), "situ")
    codes, scales = s["down_w"]
    _must(gemm(_p(s["out"]), _p(codes), _p(scales), _p(s["act"]), T, H, S, st), "down")
    return s["out"]


def run(state):
    if state["kind"] == "expert":
        return _run_expert(state)
    if state["kind"] == "shared":
        return _run_shared(state)
    layer = state["moe"] if state["kind"] == "layer" else state["layer"]
    out = layer.forward(state["x"], state["residual"], out=state["out"], ids=state["ids"],
                        weights=state["weights"], precision=state["precision"])
    return dict(out=out, ids=state["ids"], weights=state["weights"])


# ---- what a pass cannot do without --------------------------------------------------------


def _expert_weight_bytes(hidden, ffn):
    return 3 * (ffn * hidden // 2 + ffn * hidden // 32)


def _selected(experts, top_k, tokens):
    """Experts that `tokens` independent uniform choices of top_k touch, expected."""
    return experts * (1.0 - (1.0 - top_k / experts) ** tokens)


def work(case):
    T = case["tokens"]
    if case["kind"] == "expert":
        hidden, ffn = SHAPES["latent"][:2]
        n = case["rows"]
        return dict(bytes=_expert_weight_bytes(hidden, ffn) + n * (2 * hidden * 2 + 4),
                    flops=n * 6 * hidden * ffn)
    H, S = NATIVE_HIDDEN, NATIVE_SHARED
    q8 = 1 + 4 / 128
    if case["kind"] == "shared":
        return dict(bytes=int(3 * H * S * q8) + 2 * T * H * 2, flops=T * 6 * H * S)
    shape = case["shape"] if case["kind"] == "layer" else "latent"
    hidden, ffn, experts, top_k = SHAPES[shape][:4]
    nbytes = _selected(experts, top_k, T) * _expert_weight_bytes(hidden, ffn)
    flops = T * top_k * 6 * hidden * ffn
    width = hidden if case["kind"] == "layer" else H
    nbytes += experts * (2 * width + 4) + 3 * T * width * 2 + T * top_k * 8
    flops += 2 * T * experts * width
    if case["kind"] == "native":
        nbytes += (2 * hidden * H + 3 * S * H) * q8 + 2 * hidden
        flops += 2 * T * (2 * hidden * H + 3 * S * H)
    return dict(bytes=int(nbytes), flops=int(flops))


def tolerance(case):
    """EXACT precision and the per-matrix entry points have one stated summation order
    (include/k3_moe.h, include/k3_rocm_ops.h): the same bits from any implementation. One token
    runs it at every precision. The matrix precision states bf16 tolerance: against the exact
    order it measures rel 1.2e-3 (layer) and 1.6e-3 (whole block), worst element 1.8% of the
    larger of itself and the output's root mean square; ids and weights are the exact router's."""
    if case["kind"] in ("expert", "shared") or case["precision"] == EXACT or case["tokens"] == 1:
        return "exact"
    return {"rel": 6.4e-3 if case["kind"] == "native" else 4.8e-3, "max": 0.07}


# ---- the same results in 64 bits, in plain torch ------------------------------------------

E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _mxfp4(packed, scales, rows, cols):
    lut = torch.tensor(E2M1 + [-v for v in E2M1], dtype=torch.float64, device=packed.device)
    pairs = torch.stack((packed & 15, packed >> 4), dim=1).to(torch.int32)
    w = lut[pairs.view(rows, cols // 32, 32)]
    return (w * torch.exp2(scales.view(rows, cols // 32, 1).double() - 127.0)).view(rows, cols)


def _expert_f64(row, hidden, ffn):
    parts = [row[o:o + n] for o, n in _expert_spans(hidden, ffn)[0]]
    return (_mxfp4(parts[0], parts[1], ffn, hidden), _mxfp4(parts[4], parts[5], ffn, hidden),
            _mxfp4(parts[2], parts[3], hidden, ffn))


def _act_f64(g, u, kind):
    if kind == ACT_SWIGLU:
        return g * torch.sigmoid(g) * u
    return (BETA * torch.tanh(g / BETA) * torch.sigmoid(g) *
            (LINEAR_BETA * torch.tanh(u / LINEAR_BETA)))


def _route_f64(x, weight, bias, top_k, scale):
    score = torch.sigmoid(x @ weight.double().T)
    ids = torch.topk(score + bias.double(), top_k, dim=1).indices
    sel = score.gather(1, ids)
    return ids, sel / (1e-20 + sel.sum(dim=1, keepdim=True)) * scale


def _routed_f64(x, ids, weights, store, hidden, ffn, act):
    out = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        tok, rank = torch.nonzero(ids == e, as_tuple=True)
        gate, up, down = _expert_f64(store[e], hidden, ffn)
        rows = x[tok]
        y = _act_f64(rows @ gate.T, rows @ up.T, act) @ down.T
        out.index_add_(0, tok, y * weights[tok, rank, None])
    return out


def _q8_f64(w):
    codes, scales = w
    rows, cols = codes.shape
    return (codes.view(rows, cols // 128, 128).double() * scales[:, :, None].double()).view(rows,
                                                                                         cols)


def _shared_f64(x, gate, up, down):
    return _act_f64(x @ _q8_f64(gate).T, x @ _q8_f64(up).T, ACT_SITU) @ _q8_f64(down).T


def exact(case, seed):
    if case["kind"] == "expert":
        hidden, ffn = SHAPES["latent"][:2]
        x = _normal((case["tokens"], hidden), 1.0, _gen(seed, 4)).double()
        rows = _expert_rows(case, seed).long()
        gate, up, down = _expert_f64(_expert_bytes(1, hidden, ffn, seed)[0], hidden, ffn)
        out = torch.zeros_like(x)
        out[rows] = _act_f64(x[rows] @ gate.T, x[rows] @ up.T, ACT_SITU) @ down.T
        return out
    H, S, T = NATIVE_HIDDEN, NATIVE_SHARED, case["tokens"]
    if case["kind"] == "shared":
        return _shared_f64(_normal((T, H), 1.0, _gen(seed, 4)).double(), _static(S, H, seed, 12),
                           _static(S, H, seed, 13), _static(H, S, seed, 14))
    native = case["kind"] == "native"
    hidden, ffn, experts, top_k, act, scale = SHAPES["latent" if native else case["shape"]]
    width = H if native else hidden
    x = _normal((T, width), 1.0, _gen(seed, 4)).double()
    residual = _normal((T, width), 1.0, _gen(seed, 5)).double()
    ids, weights = _route_f64(x, _normal((experts, width), 0.02, _gen(seed, 3)),
                              _bias(experts, case.get("zipf", False), seed), top_k, scale)
    store = _expert_bytes(experts, hidden, ffn, seed)
    if not native:
        out = residual + _routed_f64(x, ids, weights, store, hidden, ffn, act)
    else:
        st = _native_statics(seed)
        routed = _routed_f64(x @ _q8_f64(st["routed_down"]).T, ids, weights, store, hidden, ffn,
                             act)
        norm = _normal((hidden,), 0.1, _gen(seed, 6), mean=1.0).double()
        normed = routed * torch.rsqrt(routed.square().mean(dim=1, keepdim=True) + EPS) * norm
        out = (residual + normed @ _q8_f64(st["routed_up"]).T +
               _shared_f64(x, st["shared_gate"], st["shared_up"], st["shared_down"]))
    # ids are whole numbers; a near-tie in 64 bits may order them otherwise
    return dict(out=out, ids=None, weights=weights)
