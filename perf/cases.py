"""The workloads by which this library's speed is followed.

Each case is a piece of what an inference engine asks of the Q4 matmul path, called the way an engine calls it:
through ``HipQ4Backend``, launch by launch on the current stream, with the weights resident and the output buffers
in hand.  Seven kinds of work, told apart by ``"kind"``:

``gemv``     one activation row against one or several matrices (Q4, Q8_0 or Q3 blocks)
``token``    one token through the projections of several dense decoder layers, each as a dependent chain
``rows``     the decode step of several sequences at once (2..16 rows) through the same projections
``lm_head``  the vocabulary projection with the exact top-k behind it
``lora``     the q, k and v projections of several layers with a rank-r adapter on q and v, 1..128 rows
``gemm``     a prompt (17..2048 rows, f16 or f32 activations) against one matrix
``moe``      the mixture-of-experts FFN of one layer from the router logits on, 1..512 tokens, shared expert included
"""
import math

import torch

from lattice_amd import synth
from lattice_amd.backend import HipQ4Backend, LoraLayerData

BLOCK_BYTES = {"q4": 20, "q8": 34, "q3": 16}
EPS = 1e-6

_engine = None


def engine():
    """The process's backend: an engine opens one and keeps it."""
    global _engine
    if _engine is None:
        _engine = HipQ4Backend(0)
    return _engine


# ---- the cases -------------------------------------------------------------------------------------------------


def listed():
    return [
        # The smallest call there is: one row, one 2.6 MB matrix.  Stands for the many small projections of small
        # models, where the call itself is what is paid for.
        dict(name="gemv_q4_4096x1024", kind="gemv", fmt="q4", n=4096, k=1024, matrices=1),
        # One token through all 24 layers of the 2B-shaped model: decode of a single sequence, the reference's
        # headline use.
        dict(name="token_2b", kind="token", hidden=2048, kv=512, inter=6144, layers=24),
        # Eight sequences decoded together (continuous batching), six layers of the same model.
        dict(name="rows8_2b", kind="rows", rows=8, hidden=2048, kv=512, inter=6144, layers=6),
        # The largest single product of a token: 248 320 x 2048 with sampling's top-50 behind it.
        dict(name="lm_head_top50", kind="lm_head", vocab=248320, k=2048, top_k=50),
        # Decode over Q8_0 weights: the gate||up matrices of six layers.
        dict(name="gemv_q8_mlp", kind="gemv", fmt="q8", n=12288, k=2048, matrices=6),
        # Adapter serving: q, k and v of four layers for 64 rows, rank 16 on q and v.
        dict(name="lora_qkv_64", kind="lora", rows=64, hidden=2048, kv=512, rank=16, layers=4),
        # A long prompt through the up-projection of the 27B-shaped model: the largest case.
        dict(name="gemm_2048_up", kind="gemm", fmt="q4", dtype="f16", m=2048, n=17408, k=5120),
        # A short prompt through its down-projection (few, long rows).
        dict(name="gemm_512_down", kind="gemm", fmt="q4", dtype="f16", m=512, n=5120, k=17408),
        # A prompt of no round length with f32 activations, 2B-shaped gate||up.
        dict(name="gemm_333_f32", kind="gemm", fmt="q4", dtype="f32", m=333, n=12288, k=2048),
        # The same kind of prompt over Q8_0 weights.
        dict(name="gemm_q8_777", kind="gemm", fmt="q8", dtype="f16", m=777, n=5120, k=5120),
        # MoE decode of sixteen sequences: nearly every expert is read, each for two or three tokens.
        dict(name="moe_16", kind="moe", tokens=16, experts=64, top_k=8, hidden=2048, inter=512, shared=512),
        # MoE prompt at the most tokens one call takes: every expert serves dozens of tokens.
        dict(name="moe_512", kind="moe", tokens=512, experts=64, top_k=8, hidden=2048, inter=512, shared=512),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["gemv", "token", "rows", "lm_head", "lora", "gemm", "moe"], [3, 2, 2, 1, 2, 4, 3])[0]
    if kind == "gemv":
        # rows of any count, K any multiple of the block
        return dict(kind=kind, fmt=rng.choice(["q4", "q4", "q8", "q3"]), n=_log(rng, 64, 32768),
                    k=32 * _log(rng, 8, 544), matrices=rng.randint(1, 6))
    if kind in ("token", "rows"):
        hidden = 128 * _log(rng, 8, 40)
        case = dict(kind=kind, hidden=hidden, kv=128 * rng.randint(1, 8), inter=128 * rng.randint(hidden // 64, hidden // 32))
        if kind == "rows":
            return dict(case, rows=_log(rng, 2, 16), layers=rng.randint(1, 6))
        return dict(case, layers=rng.randint(2, max(2, min(24, 24 * 2048 * 6144 // (hidden * case["inter"])))))
    if kind == "lm_head":
        return dict(kind=kind, vocab=_log(rng, 32000, 248320), k=32 * _log(rng, 32, 160), top_k=_log(rng, 1, 256))
    if kind == "lora":
        return dict(kind=kind, rows=_log(rng, 1, 128), hidden=128 * _log(rng, 8, 32), kv=128 * rng.randint(1, 8),
                    rank=rng.choice([4, 8, 16, 16, 32, 64]), layers=rng.randint(1, 4))
    if kind == "gemm":
        k = 32 * _log(rng, 16, 544)
        return dict(kind=kind, fmt=rng.choice(["q4", "q4", "q4", "q8", "q3"]), dtype=rng.choice(["f16", "f16", "f32"]),
                    m=_log(rng, 17, 2048), n=_log(rng, 256, min(17408, 17408 * 5120 // k)), k=k)
    inter = 32 * _log(rng, 8, 32)
    top_k = rng.choice([2, 4, 8])
    return dict(kind=kind, tokens=_log(rng, 1, 512), experts=rng.choice([16, 32, 64, 128]), top_k=top_k,
                hidden=128 * _log(rng, 8, 24), inter=inter, shared=inter * rng.choice([1, 1, 2]))


# ---- inputs ----------------------------------------------------------------------------------------------------


def _blocks(fmt, n, k, gen):
    """Blocks of W[n, k] as the quantiser leaves them: the scale of a group of 32 normal weights, uniform codes."""
    nb = n * (k // 32)
    raw = torch.randint(0, 256, (nb, BLOCK_BYTES[fmt]), dtype=torch.uint8, device="cuda", generator=gen)
    levels = {"q4": 7.0, "q8": 127.0, "q3": 3.5}[fmt]
    scale = (torch.randn(nb, device="cuda", generator=gen).abs() * (0.02 / levels)).clamp_min(6.2e-5)
    raw[:, 0:2] = scale.to(torch.float16).view(torch.uint8).view(nb, 2)
    if fmt == "q8":
        raw[:, 2:].masked_fill_(raw[:, 2:] == 128, 129)  # the quantiser never emits -128
    else:
        zero = -8.0 if fmt == "q4" else -4.0
        raw[:, 2:4] = (zero * scale).to(torch.float16).view(torch.uint8).view(nb, 2)
    return raw.view(-1)


class State:
    """What a program holds between calls; ``go`` is one pass."""

    def __init__(self, be, own=False):
        self.be, self.own, self.go = be, own, None

    def __del__(self):
        if self.own:
            self.go = None
            self.be.close()


def _normal(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen)


def _empty(*shape):
    return torch.empty(shape, device="cuda")


def _prepare_gemv(case, gen):
    st = State(engine())
    be, n, k = st.be, case["n"], case["k"]
    call = {"q4": be.dispatch_matmul, "q8": be.dispatch_matmul_q8, "q3": be.dispatch_matmul_q3}[case["fmt"]]
    ws = [be.wrap_device_blocks(_blocks(case["fmt"], n, k, gen)) for _ in range(case["matrices"])]
    x, ys = _normal(gen, k), [_empty(n) for _ in ws]

    def go():
        for w, y in zip(ws, ys):
            call(x, w, y, 1, n, k)
        return ys
    st.go = go
    return st


def _layer_weights(be, case, gen):
    h, kv, inter = case["hidden"], case["kv"], case["inter"]
    w = lambda n, k: be.wrap_device_blocks(_blocks("q4", n, k, gen))  # noqa: E731
    return dict(qkv=w(h + 2 * kv, h), o=w(h, h), gate_up=w(2 * inter, h), down=w(h, inter),
                g1=0.1 * _normal(gen, h), g2=0.1 * _normal(gen, h))


def _prepare_token(case, gen):
    """Per layer one call: [o, gate||up, down, the next layer's qkv] with residual adds, norms and silu * up inside.
    Attention is not this library's work: o is fed with the q rows."""
    st = State(engine())
    be, h, inter, layers = st.be, case["hidden"], case["inter"], case["layers"]
    nqkv = h + 2 * case["kv"]
    lw = [_layer_weights(be, case, gen) for _ in range(layers)]
    embedding, residual, qkv = _normal(gen, h), _empty(h), _empty(layers, nqkv)
    chains = [[be.chain_step(lw[0]["qkv"], nqkv, h, norm=(embedding, None, lw[0]["g1"], EPS, residual), y=qkv[0])]]
    for i, w in enumerate(lw):
        steps = [be.chain_step(w["o"], h, h, x=qkv[i], add_residual=residual),
                 be.chain_step(w["gate_up"], 2 * inter, h, norm=(residual, None, w["g2"], EPS, None), silu_mul_pairs=True),
                 be.chain_step(w["down"], h, inter, from_previous=True, add_residual=residual)]
        if i + 1 < layers:
            nxt = lw[i + 1]
            steps.append(be.chain_step(nxt["qkv"], nqkv, h, norm=(residual, None, nxt["g1"], EPS, None), y=qkv[i + 1]))
        chains.append(steps)

    def go():
        for steps in chains:
            be.dispatch_chain(steps)
        return residual, qkv
    st.go = go
    return st


def _prepare_rows(case, gen):
    st = State(engine())
    be, h, kv, inter, rows = st.be, case["hidden"], case["kv"], case["inter"], case["rows"]
    lw = [_layer_weights(be, case, gen) for _ in range(case["layers"])]
    views = [[(w["qkv"], h, _empty(rows, h), None, 0), (w["qkv"], kv, _empty(rows, kv), None, h * (h // 32) * 20),
              (w["qkv"], kv, _empty(rows, kv), None, (h + kv) * (h // 32) * 20)] for w in lw]
    embedding = _normal(gen, rows, h)
    normed, att, res, out = (_empty(rows, h) for _ in range(4))
    gate_up = _empty(rows, 2 * inter)

    def go():
        x = embedding
        for w, v in zip(lw, views):
            be.dispatch_fused_residual_add_norm(x, None, None, normed, w["g1"], h, EPS, num_rows=rows)
            be.gemv_multi(normed, v, rows, h)
            be.gemv_batch(v[0][2], w["o"], att, rows, h, h)  # the q rows stand in for attention's result
            be.dispatch_matmul_fused(None, w["gate_up"], gate_up, 2 * inter, h, norm=(x, att, w["g2"], EPS, res), batch=rows)
            be.dispatch_matmul_fused(gate_up, w["down"], None, h, inter, silu_mul=True, add_residual=(res, out), batch=rows)
            x = out
        return out, [t for v in views for (_, _, t, _, _) in v]
    st.go = go
    return st


def _prepare_lm_head(case, gen):
    st = State(engine())
    be, vocab, k, top_k = st.be, case["vocab"], case["k"], case["top_k"]
    w, x = be.wrap_device_blocks(_blocks("q4", vocab, k, gen)), _normal(gen, k)
    st.go = lambda: be.lm_head_topk(x, w, vocab, k, top_k)
    return st


def _prepare_lora(case, gen, seed):
    be = HipQ4Backend(0)  # one adapter is loaded per backend
    st = State(be, own=True)
    h, kv, rows, rank = case["hidden"], case["kv"], case["rows"], case["rank"]
    be.load_lora_adapter([LoraLayerData(i, {name: synth.lora_pair(rank, h, n, seed=seed, tag="%s%d" % (name, i))
                                            for name, n in (("q_proj", h), ("v_proj", kv))})
                          for i in range(case["layers"])], scale=32.0 / rank)
    x = _normal(gen, rows, h)
    views = [[(be.wrap_device_blocks(_blocks("q4", n, h, gen)), n, _empty(rows, n), name)
              for name, n in (("q_proj", h), ("k_proj", kv), ("v_proj", kv))] for _ in range(case["layers"])]

    def go():
        for i, v in enumerate(views):
            be.gemv_multi(x, v, rows, h, layer_idx=i)
        return [t for v in views for (_, _, t, _) in v]
    st.go = go
    return st


def _prepare_gemm(case, gen):
    st = State(engine())
    be, m, n, k = st.be, case["m"], case["n"], case["k"]
    call = {"q4": be.dispatch_gemm, "q8": be.dispatch_gemm_q8, "q3": be.dispatch_gemm_q3}[case["fmt"]]
    w, x, y = be.wrap_device_blocks(_blocks(case["fmt"], n, k, gen)), _normal(gen, m, k), _empty(m, n)
    if case["dtype"] == "f16":
        x = x.to(torch.float16)

    def go():
        call(x, 0, w, y, 0, m, n, k)
        return y
    st.go = go
    return st


def _prepare_moe(case, gen):
    st = State(engine())
    be, t, e, h, inter, shared = (st.be, case["tokens"], case["experts"], case["hidden"], case["inter"], case["shared"])
    top_k = case["top_k"]
    w = lambda n, k: be.wrap_device_blocks(_blocks("q4", n, k, gen))  # noqa: E731
    gate_up, down = w(e * 2 * inter, h), w(e * h, inter)
    shared_gate_up, shared_down = w(2 * shared, h), w(h, shared)
    gate, logits, x, y = _normal(gen, h) / h ** 0.5, _normal(gen, t, e), _normal(gen, t, h), _empty(t, h)

    def go():
        be.moe_ffn(logits, gate_up, down, e, top_k, inter, shared_gate_up, shared_down, gate, shared, h, x, y)
        return y
    st.go = go
    return st


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind == "lora":
        return _prepare_lora(case, gen, seed)
    return {"gemv": _prepare_gemv, "token": _prepare_token, "rows": _prepare_rows, "lm_head": _prepare_lm_head,
            "gemm": _prepare_gemm, "moe": _prepare_moe}[kind](case, gen)


def run(state):
    return state.go()


# ---- what a pass cannot do without -----------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n, k, c = case["n"], case["k"], case["matrices"]
        return {"bytes": c * (n * (k // 32) * BLOCK_BYTES[case["fmt"]] + 4 * n) + 4 * k, "flops": 2 * c * n * k}
    if kind in ("token", "rows"):
        h, kv, inter, layers, rows = case["hidden"], case["kv"], case["inter"], case["layers"], case.get("rows", 1)
        weights = layers * (h * (h + 2 * kv) + h * h + 3 * h * inter)
        # weights and gammas, the embedding in, the residual and every layer's qkv out
        return {"bytes": weights // 32 * 20 + layers * 8 * h + 4 * rows * (2 * h + layers * (h + 2 * kv)),
                "flops": 2 * rows * weights}
    if kind == "lm_head":
        return {"bytes": case["vocab"] * (case["k"] // 32) * 20 + 4 * case["k"] + 8 * case["top_k"],
                "flops": 2 * case["vocab"] * case["k"]}
    if kind == "lora":
        h, kv, rows, rank, layers = case["hidden"], case["kv"], case["rows"], case["rank"], case["layers"]
        n, factors = h + 2 * kv, rank * (2 * h + h + kv)
        return {"bytes": layers * (n * (h // 32) * 20 + 2 * factors + 4 * rows * n) + 4 * rows * h,
                "flops": 2 * layers * rows * (n * h + factors)}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * (k // 32) * BLOCK_BYTES[case["fmt"]] + m * k * (2 if case["dtype"] == "f16" else 4) + 4 * m * n,
                "flops": 2 * m * n * k}
    t, e, top_k, h, inter, shared = (case[k] for k in ("tokens", "experts", "top_k", "hidden", "inter", "shared"))
    touched = e * (1 - (1 - top_k / e) ** t)  # experts that some token chose, on average
    return {"bytes": 3 * h * (touched * inter + shared) / 32 * 20 + 4 * t * e + 8 * t * h + 4 * h,
            "flops": 6 * t * h * (top_k * inter + shared)}


def tolerance(case):
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 1e-5}  # f32 activations and sums
    if kind == "token":
        return {"rel": 1e-4}  # the same through up to 24 dependent layers
    if kind == "lm_head":
        return {"rel": 1e-5, "differ": 0.01}
    if kind == "rows":
        return {"rel": 5e-3}  # activations rounded to f16 in up to 24 dependent products
    # f16 activations and dequantised weights, f32 sums
    return {"rel": 1e-3}
