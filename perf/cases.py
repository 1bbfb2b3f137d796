"""The work a serving engine has this library do, as cases that can be timed and compared.

Three kinds, each through the public Python entry points:

moe    MoeBlock.forward (or forward_seam) over a run of consecutive layers of the routed model the library is
       configured for (`MoeGeometry.qwen3_6`: 256 experts, top 8, hidden 2048, expert width 512, one gated shared
       expert): a layer's output is the next layer's residual.  1 to 63 tokens is decode (that many sequences, or a few
       with speculative tokens), 64 to 8192 a prefill chunk.
dense  DenseFfnBlock.forward, the feed-forward block of the dense sibling (hidden 5120, intermediate 17408, Q6_K).
head   LmHeadKernels.forward over the 248 320-token vocabulary and argmax per token: a greedy decode step's end.

`formats` of a MoE layer: "q6k" has Q6_K experts and a Q8_0 router, "shipped" is the layout of the model's published
file (gate/up Q6_K, down Q8_0, f32 router).  `routing` "zipf" adds the skewed per-expert bias of the benchmark
(`zipf_logit_bias`) to the router logits, "uniform" adds none.  `launch` "graph" replays one captured hipGraph, as a
decode engine does with a step of fixed shape; "eager" makes the calls from Python each time.
"""
import torch

import llmxabe_amd as X

EXPERTS, TOP_K, HIDDEN, WIDTH = 256, 8, 2048, 512
DENSE_HIDDEN, DENSE_WIDTH = 5120, 17408
VOCAB = 248320
Q6K_BYTES, Q8_BYTES = 210 / 256, 34 / 32   # per weight


def _moe(name, tokens, layers, formats="q6k", routing="uniform", launch="graph", seam=False):
    return {"name": name, "kind": "moe", "tokens": tokens, "layers": layers, "formats": formats, "routing": routing,
            "launch": launch, "seam": seam}


def listed():
    return [
        # one sequence, calls made one by one from the host: what an interactive user of the library waits for
        _moe("moe_decode_1_eager", 1, 8, launch="eager"),
        # three sequences, the benchmark's headline width, the step replayed as a graph
        _moe("moe_decode_3", 3, 8),
        # a handful of sequences at an odd count, on the layout the published file has
        _moe("moe_decode_13_shipped", 13, 6, formats="shipped"),
        # the widest decode batch of the configurations
        _moe("moe_decode_32", 32, 4),
        # a short prompt (or a wide verify step): below the matrix-core widths
        _moe("moe_prompt_45", 45, 4, launch="eager"),
        # a medium prompt with the skewed expert load real traffic shows
        _moe("moe_prefill_512_zipf", 512, 1, routing="zipf", launch="eager"),
        # a ragged last chunk of a prompt, published layout
        _moe("moe_prefill_1237_shipped", 1237, 1, formats="shipped", launch="eager"),
        # a full prefill chunk through consecutive layers, each layer's norm left by the layer before (forward_seam)
        _moe("moe_prefill_8192_seam", 8192, 2, launch="eager", seam=True),
        # the dense sibling: one sequence, a speculative verify step, a prefill chunk
        {"name": "dense_decode_1", "kind": "dense", "tokens": 1, "launch": "eager"},
        {"name": "dense_verify_7", "kind": "dense", "tokens": 7, "launch": "eager"},
        {"name": "dense_prefill_2048", "kind": "dense", "tokens": 2048, "launch": "eager"},
        # next-token logits and greedy choice for three sequences
        {"name": "head_3", "kind": "head", "tokens": 3, "format": "q8_0", "launch": "eager"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "dense", "head"))
    if kind == "decode":
        tokens = _log_int(rng, 1, 63)
        c = _moe("", tokens, 8 if tokens <= 4 else 6 if tokens <= 16 else 4, rng.choice(("q6k", "shipped")),
                 rng.choice(("uniform", "zipf")), rng.choice(("graph", "eager")))
    elif kind == "prefill":
        seam = rng.random() < 0.5
        c = _moe("", _log_int(rng, 64, 8191), 2 if seam else 1, rng.choice(("q6k", "shipped")),
                 rng.choice(("uniform", "zipf")), "eager", seam)
    elif kind == "dense":
        c = {"kind": "dense", "tokens": _log_int(rng, 1, 2047), "launch": "eager"}
    else:
        c = {"kind": "head", "tokens": rng.randint(1, 16), "format": rng.choice(("q8_0", "q6k", "bf16")),
             "launch": rng.choice(("graph", "eager"))}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- what a program holds before the call
def _quant(q, seed, elements):
    return X.QuantTensor(X.synth_quant(q, seed, elements, 0.02), q)


def _moe_layer(seed, formats):
    q6, q8 = X.ExpertQuant.Q6K, X.ExpertQuant.Q8_0
    shipped = formats == "shipped"
    stack, shared = EXPERTS * HIDDEN * WIDTH, HIDDEN * WIDTH
    router = (X.synth_normal_f32(seed + 1, EXPERTS * HIDDEN, 0.02) if shipped
              else X.synth_quant(q8, seed + 1, EXPERTS * HIDDEN, 0.02))
    return X.MoeLayerWeights(
        1.0 + X.synth_normal_f32(seed, HIDDEN, 0.1), router, None if shipped else q8,
        _quant(q6, seed + 2, stack), _quant(q6, seed + 3, stack), _quant(q8 if shipped else q6, seed + 4, stack),
        X.synth_normal_f32(seed + 5, HIDDEN, 0.02),
        _quant(q8, seed + 6, shared), _quant(q8, seed + 7, shared), _quant(q8, seed + 8, shared))


class _State:
    """Weights, inputs, buffers and handles of one case; `step` makes the calls, `out` holds what they write."""

    def __init__(self, case, seed):
        base = (int(seed) + 1) * 1_000_003
        getattr(self, "_" + case["kind"])(case, base)
        self.graph = None
        if case["launch"] == "graph":   # one eager step first, as a capture needs
            torch.cuda.synchronize()
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                self.step()
                stream.synchronize()
                self.graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(self.graph, stream=stream):
                    self.step()

    def _moe(self, case, base):
        tokens, layers = case["tokens"], case["layers"]
        weights = [_moe_layer(base + 100 * i, case["formats"]) for i in range(layers)]
        bias = torch.from_numpy(X.zipf_logit_bias(EXPERTS)).cuda() if case["routing"] == "zipf" else None
        block = X.MoeBlock(X.MoeGeometry.qwen3_6(X.moe_block_size(tokens), tokens))
        block.publish_tokens(tokens)
        x = X.synth_normal_f32(base + 99, tokens * HIDDEN, 1.0).view(tokens, HIDDEN)
        ffn_out, rows = torch.zeros_like(x), [torch.zeros_like(x), torch.zeros_like(x)]
        last = rows[(layers - 1) & 1]

        def step():
            cur = x
            for i, w in enumerate(weights):
                nxt = rows[i & 1]
                block.forward(w, cur, tokens, ffn_out, nxt, logit_bias=bias)
                cur = nxt

        def step_seam():
            cur = x
            for i, w in enumerate(weights):
                nxt = rows[i & 1]
                block.forward_seam(w, cur, tokens, None, nxt, logit_bias=bias, input_normed=i > 0, skip_readback=True,
                                   next_norm_weight=weights[i + 1].post_norm if i + 1 < layers else None)
                cur = nxt

        self.step = step_seam if case["seam"] else step
        self.out = {"l_out": last} if case["seam"] else {"l_out": last, "ffn_out": ffn_out}

    def _dense(self, case, base):
        tokens, count = case["tokens"], DENSE_HIDDEN * DENSE_WIDTH
        q = X.ExpertQuant.Q6K
        w = X.DenseFfnLayerWeights(1.0 + X.synth_normal_f32(base, DENSE_HIDDEN, 0.1),
                                   *(_quant(q, base + j, count) for j in (1, 2, 3)))
        block = X.DenseFfnBlock(DENSE_HIDDEN, DENSE_WIDTH, tokens)
        block.publish_tokens(tokens)
        x = X.synth_normal_f32(base + 99, tokens * DENSE_HIDDEN, 1.0).view(tokens, DENSE_HIDDEN)
        ffn_out, l_out = torch.zeros_like(x), torch.zeros_like(x)
        self.step = lambda: block.forward(w, x, tokens, ffn_out, l_out)
        self.out = {"l_out": l_out, "ffn_out": ffn_out}

    def _head(self, case, base):
        tokens, fmt = case["tokens"], case["format"]
        g = X.LmHeadGeometry.qwen3_6(tokens)
        if fmt == "bf16":
            head = X.HeadTensor.bf16(X.synth_normal_f32(base, g.elements(), 0.02).to(torch.bfloat16))
        elif fmt == "q6k":
            head = X.HeadTensor.q6_k(X.synth_quant(X.ExpertQuant.Q6K, base, g.elements(), 0.02))
        else:
            head = X.HeadTensor.q8_0(X.synth_quant(X.ExpertQuant.Q8_0, base, g.elements(), 0.02))
        kernels = X.LmHeadKernels(g)
        x = X.synth_normal_f32(base + 99, tokens * HIDDEN, 1.0).view(tokens, HIDDEN)
        logits = torch.zeros(tokens, VOCAB, device="cuda")
        rows = list(logits)
        values = torch.zeros(512, device="cuda")
        indices = torch.zeros(512, dtype=torch.int32, device="cuda")
        ids = torch.zeros(tokens, dtype=torch.int32, device="cuda")
        id_of = [ids[t:t + 1] for t in range(tokens)]

        def step():
            kernels.forward(head, x, tokens, logits)
            for t in range(tokens):
                kernels.argmax(rows[t], VOCAB, values, indices, id_of[t])

        self.step = step
        self.out = {"logits": logits, "ids": ids}


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    if state.graph is not None:
        state.graph.replay()
    else:
        state.step()
    return state.out


# ---------------------------------------------------------------- what a pass cannot do without
def _distinct_experts(tokens, routing):
    """Experts that `tokens` tokens select between them, for logits as these weights and inputs give them."""
    g = torch.Generator().manual_seed(1)
    logits = torch.randn(tokens, EXPERTS, generator=g) * (0.02 * HIDDEN ** 0.5)
    if routing == "zipf":
        logits += torch.from_numpy(X.zipf_logit_bias(EXPERTS))
    return len(torch.unique(torch.topk(logits, TOP_K, dim=1).indices))


def work(case):
    t = case["tokens"]
    if case["kind"] == "moe":
        shipped = case["formats"] == "shipped"
        matrix = HIDDEN * WIDTH
        expert = matrix * (2 * Q6K_BYTES + (Q8_BYTES if shipped else Q6K_BYTES))
        router = EXPERTS * HIDDEN * (4 if shipped else Q8_BYTES)
        layer = _distinct_experts(t, case["routing"]) * expert + 3 * matrix * Q8_BYTES + router + 2 * HIDDEN * 4
        rows = t * HIDDEN * 4   # residual in, l_out out, and ffn_out unless the seam leaves it away
        n = case["layers"]
        return {"bytes": n * (layer + rows * (2 if case["seam"] else 3)),
                "flops": n * t * 2 * (3 * (TOP_K + 1) * matrix + EXPERTS * HIDDEN)}
    if case["kind"] == "dense":
        weights = 3 * DENSE_HIDDEN * DENSE_WIDTH
        return {"bytes": weights * Q6K_BYTES + 3 * t * DENSE_HIDDEN * 4, "flops": 2 * t * weights}
    per = {"q8_0": Q8_BYTES, "q6k": Q6K_BYTES, "bf16": 2}[case["format"]]
    return {"bytes": VOCAB * HIDDEN * per + t * (HIDDEN + VOCAB) * 4, "flops": 2 * t * VOCAB * HIDDEN}


def tolerance(case):
    if case["kind"] == "head":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0}
    if case["tokens"] < 64:
        return {"rel": 1e-5, "max": 2e-4}   # fp32 sums throughout
    # fp16 operands: 2^-11 per rounded weight, activation and intermediate
    if case["kind"] == "moe" and case["seam"]:
        # The next layer routes on rows that carry that rounding: a token whose eighth and ninth expert are that close
        # may take the other one, which moves its row by a few per cent of the residual it is added to.
        return {"rel": 1e-3, "max": 0.5}
    return {"rel": 1e-3, "max": 1e-2}
