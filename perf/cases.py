"""Performance cases of the skinny decode GEMM library.

Every case is work that a decode engine has this library do, through its
public Python entry points, at sizes of the engine's own configurations: the
Qwen3-4B projections at decode batches and speculative-tree row counts of 1 to
128 rows (batch 32 with 4 tree rows each is the largest step the engine
builds), their tensor-parallel shards, and ragged shapes that fit no table.

Kinds:

* ``proj``   one projection of every layer, recorded in one graph over that
             many distinct weights and replayed, as a captured decode step
             runs it.  ``norm``: with the residual-add + RMSNorm prologue in
             front.  ``silu``: the fused gate/up + SiLU·mul projection.
             ``pad``: extra elements between the rows of x.
* ``call``   one eager call of a projection object.
* ``block``  the four projections of each layer (normed qkv, o, normed
             gate/up, down) in one graph, on the residual stream of the block.
* ``step``   the whole decode step (all layers and the normed lm_head) captured
             by ``GemmStep``; returns the logits.
* ``select`` the lm_head projection with per-row argmax / top-k selection.
* ``norm``   the stand-alone residual add + RMSNorm.
"""

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "kernel-rush-kawk_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from kernels import gemm as G  # noqa: E402
from kernels import step as S  # noqa: E402

DEV = "cuda:0"
BF16 = torch.bfloat16
EPS = 1e-6
HIDDEN, QKV, HEADS, INTER, VOCAB, LAYERS = 2560, 6144, 4096, 9728, 151936, 36
ROWS = 128  # most rows of a step


def _proj(name, M, N, K, norm=False, silu=False, layers=LAYERS, pad=0):
    return {"name": name, "kind": "proj", "M": M, "N": N, "K": K, "norm": norm, "silu": silu, "layers": layers,
            "pad": pad}


def listed():
    return [
        # An eager single-row call: what warm-up, self checks and uncaptured callers pay per projection.
        {"name": "call_o_m1", "kind": "call", "M": 1, "N": HIDDEN, "K": HEADS, "silu": False},
        # One sequence's decode step, attention input: all layers' normed qkv projections.
        _proj("qkv_normed_m1", 1, QKV, HIDDEN, norm=True),
        # Batch 4 decode, the long-K projection.
        _proj("down_m4", 4, HIDDEN, INTER),
        # Batch 16 decode, the smallest projection.
        _proj("o_m16", 16, HIDDEN, HEADS),
        # Batch 32 decode, the largest projection of a layer with its prologue and epilogue.
        _proj("gate_up_normed_m32", 32, 2 * INTER, HIDDEN, norm=True, silu=True),
        # Tree verification (64 rows), the long-K projection.
        _proj("down_m64", 64, HIDDEN, INTER),
        # A ragged shape outside every table: odd rows, channels and K stages, x rows with a stride.
        _proj("ragged_m13", 13, 3000, 1416, pad=24),
        # Token recycling after a verify step: the 8 best tokens of each of 64 rows.
        {"name": "select_m64_k8", "kind": "select", "M": 64, "N": VOCAB, "K": HIDDEN, "k": 8},
        # Tree verification of up to 16 sequences: the projections of some layers at 64 rows.
        {"name": "block_m64", "kind": "block", "M": 64, "layers": 8},
        # Tree verification of 32 sequences with 4 rows each.
        {"name": "block_m128", "kind": "block", "M": 128, "layers": 8},
        # One sequence's whole decode step, logits out.
        {"name": "step_m1", "kind": "step", "M": 1, "layers": LAYERS},
        # The whole decode step of a batch of 32.
        {"name": "step_m32", "kind": "step", "M": 32, "layers": LAYERS},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    M = _log_int(rng, 1, ROWS)
    kind = rng.choice(["proj"] * 6 + ["block", "block", "call", "select", "step", "norm"])
    if kind == "block":
        return {"kind": "block", "M": M, "layers": rng.randint(4, 12)}
    if kind == "step":
        return {"kind": "step", "M": M, "layers": rng.randint(8, LAYERS)}
    if kind == "select":
        tp = rng.choice([1, 1, 2, 4, 8])
        return {"kind": "select", "M": M, "N": VOCAB // tp, "K": HIDDEN, "k": rng.choice([1, 1, 4, 8])}
    if kind == "norm":
        return {"kind": "norm", "M": M, "K": 8 * _log_int(rng, 64, 1536)}
    tp = rng.choice([1, 1, 1, 2, 4, 8])  # tensor-parallel degree: N of qkv and gate_up, K of o and down
    which = rng.choice(["qkv", "o", "gate_up", "down", "ragged"])
    norm = silu = False
    pad = 0
    if which == "qkv":
        N, K, norm = QKV // tp, HIDDEN, rng.random() < 0.7
    elif which == "o":
        N, K = HIDDEN, HEADS // tp
    elif which == "gate_up":
        N, K, silu, norm = 2 * INTER // tp, HIDDEN, True, rng.random() < 0.7
    elif which == "down":
        N, K = HIDDEN, INTER // tp
    else:
        N, K = 2 * _log_int(rng, 128, 12288), 8 * _log_int(rng, 64, 1280)
        silu, norm, pad = rng.random() < 0.3, rng.random() < 0.2, rng.choice([0, 0, 8, 64])
    if kind == "call":
        return {"kind": "call", "M": M, "N": N, "K": K, "silu": silu}
    layers = max(4, min(LAYERS, int(1e9 / (2 * N * K))))
    return {"kind": "proj", "M": M, "N": N, "K": K, "norm": norm, "silu": silu, "layers": layers, "pad": pad}


# ----------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rnd(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device=DEV).mul_(scale).to(BF16)


def _gain(g, n):
    return torch.randn((n,), generator=g, device=DEV).mul_(0.1).add_(1.0).to(BF16)


def _weights(g, layers, N, K):
    return [_rnd(g, N, K, scale=0.02) for _ in range(layers)]


def _inputs(case, seed):
    """The operands of a case, from the seed alone (``step`` excepted: its
    model comes from ``synthetic_model``)."""
    g = _gen(seed)
    kind, M = case["kind"], case["M"]
    s = {}
    if kind in ("proj", "call"):
        N, K, pad = case["N"], case["K"], case.get("pad", 0)
        # A down projection reads post-SiLU·mul magnitudes, the others N(0, 1).
        s["x"] = _rnd(g, M, K + pad, scale=0.5 if K == INTER else 1.0)[:, :K]
        s["w"] = _weights(g, case.get("layers", 1), N, K)
        if case.get("norm"):
            s["d"], s["gain"] = _rnd(g, M, K), _gain(g, K)
    elif kind == "select":
        s["x"], s["w"] = _rnd(g, M, case["K"]), _rnd(g, case["N"], case["K"], scale=0.02)
    elif kind == "norm":
        K = case["K"]
        s["x"], s["d"], s["gain"] = _rnd(g, M, K), _rnd(g, M, K), _gain(g, K)
    elif kind == "block":
        s["x"], s["y"], s["attn"] = _rnd(g, M, HIDDEN), _rnd(g, M, HIDDEN), _rnd(g, M, HEADS)
        s["layers"] = [
            {"in": _gain(g, HIDDEN), "qkv": _rnd(g, QKV, HIDDEN, scale=0.02), "o": _rnd(g, HIDDEN, HEADS, scale=0.02),
             "post": _gain(g, HIDDEN), "gu": _rnd(g, 2 * INTER, HIDDEN, scale=0.02),
             "d": _rnd(g, HIDDEN, INTER, scale=0.02)}
            for _ in range(case["layers"])]
    elif kind == "step":
        s["model"] = S.synthetic_model(DEV, layers=case["layers"], seed=seed)
        s["x"], s["attn"] = _rnd(g, M, HIDDEN), _rnd(g, M, HEADS)
    else:
        raise ValueError(kind)
    return s


# ----------------------------------------------------------------- passes
def _capture(fn):
    """``fn`` recorded in one graph behind a warm-up call, and its outputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare(case, seed):
    s = _inputs(case, seed)
    kind, M = case["kind"], case["M"]
    s["kind"] = kind
    if kind in ("proj", "call"):
        N, K = case["N"], case["K"]
        op = G.SkinnyGateUp(M, N // 2, K, DEV) if case["silu"] else G.SkinnyMatmul(M, N, K, DEV)
        s["op"] = op
        if kind == "proj":
            if case["norm"]:
                xout = torch.empty((M, K), dtype=BF16, device=DEV)
                norm = (s["d"], s["gain"], xout, EPS)
                s["graph"], ys = _capture(lambda: [op(s["x"], w, norm=norm) for w in s["w"]])
                s["out"] = ys + [xout]
            else:
                s["graph"], s["out"] = _capture(lambda: [op(s["x"], w) for w in s["w"]])
    elif kind == "select":
        s["op"] = G.SkinnySelect(M, case["N"], case["K"], DEV, case["k"])
        s["idx"] = torch.empty((M, case["k"]), dtype=torch.int64, device=DEV)
        s["values"] = torch.empty((M, case["k"]), dtype=BF16, device=DEV)
    elif kind == "norm":
        s["xout"] = torch.empty_like(s["x"])
    elif kind == "block":
        qkv, o = G.SkinnyMatmul(M, QKV, HIDDEN, DEV), G.SkinnyMatmul(M, HIDDEN, HEADS, DEV)
        gu, d = G.SkinnyGateUp(M, INTER, HIDDEN, DEV), G.SkinnyMatmul(M, HIDDEN, INTER, DEV)
        s["ops"] = (qkv, o, gu, d)
        xa, xb = torch.empty_like(s["x"]), torch.empty_like(s["x"])

        def layers():
            cur, y, out = s["x"], s["y"], []
            for p in s["layers"]:
                out.append(qkv(cur, p["qkv"], norm=(y, p["in"], xa, EPS)))
                br = o(s["attn"], p["o"])
                act = gu(xa, p["gu"], norm=(br, p["post"], xb, EPS))
                y = d(act, p["d"])
                cur = xb
                out += [br, act, y]
            return out + [xa, xb]

        s["graph"], s["out"] = _capture(layers)
    elif kind == "step":
        step = S.GemmStep(s["model"], M)
        step.attn_out.copy_(s["attn"])
        step.capture(s["x"])
        s["step"] = step
    return s


def run(state):
    kind = state["kind"]
    if kind in ("proj", "block"):
        state["graph"].replay()
        return state["out"]
    if kind == "call":
        return state["op"](state["x"], state["w"][0])
    if kind == "select":
        state["op"].run(state["x"], state["w"], state["idx"], values=state["values"])
        return {"idx": state["idx"], "values": state["values"]}
    if kind == "norm":
        n = G.add_rms_norm(state["x"], state["d"], state["gain"], EPS, state["xout"])
        return {"n": n, "xout": state["xout"]}
    return state["step"].replay()


# ----------------------------------------------------------------- accounting
def _gemm_work(M, N, K, silu=False, norm=False, count=1):
    """Weights once per projection, its input and output, and for a normed
    one the residual, the branch, the gain and the residual written back."""
    nout = N // 2 if silu else N
    elems = N * K + M * K + M * nout + ((2 * M + 1) * K if norm else 0)
    return {"bytes": 2 * elems * count, "flops": 2 * M * N * K * count}


def _add(*parts):
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def work(case):
    kind, M = case["kind"], case["M"]
    if kind in ("proj", "call"):
        return _gemm_work(M, case["N"], case["K"], case["silu"], case.get("norm", False), case.get("layers", 1))
    if kind == "norm":
        return {"bytes": 2 * (4 * M + 1) * case["K"], "flops": 6 * M * case["K"]}
    if kind == "select":
        w = _gemm_work(M, case["N"], case["K"])
        # The logits stay inside; k indices and values come out.
        return {"bytes": w["bytes"] - 2 * M * case["N"] + 10 * M * case["k"], "flops": w["flops"]}
    L = case["layers"]
    layer = _add(_gemm_work(M, QKV, HIDDEN, norm=True, count=L), _gemm_work(M, HIDDEN, HEADS, count=L),
                 _gemm_work(M, 2 * INTER, HIDDEN, silu=True, norm=True, count=L), _gemm_work(M, HIDDEN, INTER, count=L))
    return layer if kind == "block" else _add(layer, _gemm_work(M, VOCAB, HIDDEN, norm=True))


def tolerance(case):
    """About four times the distance of a bf16 result from the 64-bit one
    (measured): one rounding for a plain projection, the prologue's and the
    epilogue's roundings on top where they run, and what travels through the
    layers of a block or step."""
    kind = case["kind"]
    if kind in ("proj", "call"):
        return {"rel": 7e-3 + (5e-3 if case["silu"] else 0.0) + (3e-3 if case.get("norm") else 0.0)}
    if kind == "select":
        # Near ties: sums in another order move a logit over a bf16 boundary now and then.
        return {"rel": 7e-3, "differ": 0.01}
    if kind == "norm":
        return {"rel": 1e-2}
    return {"rel": 2e-2 if kind == "block" else 3e-2}


# ----------------------------------------------------------------- 64 bits
def _mm64(x, w, rows=1 << 14):
    """x @ w.T in 64 bits, the weight converted ``rows`` rows at a time."""
    x = x.double()
    return torch.cat([x @ w[i:i + rows].double().t() for i in range(0, w.shape[0], rows)], dim=1)


def _silu_mul64(gu):
    n = gu.shape[1] // 2
    g = gu[:, :n]
    return g / (1.0 + torch.exp(-g)) * gu[:, n:]


def _norm64(x, d, gain):
    s = x.double() + d.double()
    return s, s * torch.rsqrt((s * s).mean(dim=-1, keepdim=True) + EPS) * gain.double()


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("proj", "call"):
        x, tail = s["x"], []
        if case.get("norm"):
            xout, x = _norm64(x, s["d"], s["gain"])
            tail = [xout]
        ys = [_silu_mul64(_mm64(x, w)) if case["silu"] else _mm64(x, w) for w in s["w"]]
        return ys[0] if kind == "call" else ys + tail
    if kind == "select":
        # The order of near-equal bf16 logits has no 64-bit counterpart.
        return {"idx": None, "values": torch.topk(_mm64(s["x"], s["w"]), case["k"], dim=-1).values}
    if kind == "norm":
        xout, n = _norm64(s["x"], s["d"], s["gain"])
        return {"n": n, "xout": xout}
    if kind == "block":
        cur, y, out = s["x"], s["y"], []
        for p in s["layers"]:
            xa, n = _norm64(cur, y, p["in"])
            out.append(_mm64(n, p["qkv"]))
            br = _mm64(s["attn"], p["o"])
            cur, n = _norm64(xa, br, p["post"])
            act = _silu_mul64(_mm64(n, p["gu"]))
            y = _mm64(act, p["d"])
            out += [br, act, y]
        return out + [xa, cur]
    m = s["model"]
    br = [_mm64(s["attn"], p.wo) for p in m.layers]
    cur, y = s["x"], torch.zeros_like(s["x"])
    for i, p in enumerate(m.layers):
        xa, n = _norm64(cur, y, p.in_norm)
        cur, n = _norm64(xa, br[i], p.post_norm)
        y = _mm64(_silu_mul64(_mm64(n, p.wgu)), p.wd)
    return _mm64(_norm64(cur, y, m.final_norm)[1], m.lm_head)
