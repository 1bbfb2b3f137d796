"""The routed experts and the shared expert of one set of buffers on two streams at once, each with activation rows of
its own: the entry points share no scratch, so every pass equals the one made alone.  (hidden 4096: both sides go
through the digits of their activation rows; hidden 1024: only the routed experts do.)  And the MoE block's own second
stream, which reads weights that a copy on the caller's stream has just brought."""
import numpy as np
import pytest

from util import activations, make_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,tokens", [(4096, 512, 3), (4096, 512, 24), (1024, 512, 8)])
def test_routed_and_shared_expert_overlap(hidden, inter, tokens):
    import torch
    import llmxabe_amd as X

    q6, q8 = X.ExpertQuant.Q6K, X.ExpertQuant.Q8_0
    g = X.MoeGeometry(16, 4, hidden, inter, 32, tokens)
    n = 16 * hidden * inter
    stack = [X.QuantTensor(X.synth_quant(q6, 900 + i, n, 0.02), q6) for i in range(3)]
    shared = [X.QuantTensor(X.synth_quant(q8, 910 + i, hidden * inter, 0.02), q8) for i in range(3)]
    k = X.MoeKernels(g)
    b = k.buffers()
    k.set_valid_tokens(b, tokens)
    k.route_and_dispatch(b, X.synth_normal_f32(920, tokens * 16, 1.0))
    xr = [X.synth_normal_f32(930 + i, tokens * hidden, 1.0) for i in range(2)]
    xs = [X.synth_normal_f32(940 + i, tokens * hidden, 100.0) for i in range(2)]
    outs = [torch.zeros(tokens * hidden, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    want_r, want_s = [], []
    for i in range(2):
        k.grouped_forward_partial(b, *stack, xr[i])
        want_r.append(b.partial().cpu().numpy().copy())
        k.shared_expert(b, *shared, xs[i], outs[i])
        want_s.append(outs[i].cpu().numpy().copy())
        outs[i].zero_()
    torch.cuda.synchronize()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for i in range(2):
        for _ in range(20):
            with torch.cuda.stream(s1):
                k.grouped_forward_partial(b, *stack, xr[i])
            with torch.cuda.stream(s2):
                k.shared_expert(b, *shared, xs[i], outs[i])
        torch.cuda.synchronize()
        assert np.array_equal(b.partial().cpu().numpy().view(np.uint32), want_r[i].view(np.uint32)), i
        assert np.array_equal(outs[i].cpu().numpy().view(np.uint32), want_s[i].view(np.uint32)), i


@pytest.mark.parametrize("tokens", [320, 1100])
def test_weights_copied_on_the_callers_stream_right_before_a_forking_pass(oracle, tokens):
    import torch
    import llmxabe_amd as X

    g = X.MoeGeometry(8, 2, 512, 256, X.moe_block_size(tokens), tokens)   # (80 rows an expert and more: wide tiles, two streams)
    layers = [make_layer(oracle, g, seed=950 + 50 * i) for i in range(2)]
    of = lambda w: (w.shared_gate.bytes, w.shared_up.bytes, w.shared_down.bytes)
    hosts = [[t.cpu().pin_memory() for t in of(layer.dev)] for layer in layers]
    w = layers[0].dev
    x = activations(970, tokens, 512)
    blk = X.MoeBlock(g)
    want = []
    for i in range(2):
        for t, h in zip(of(w), hosts[i]):
            t.copy_(h)
        torch.cuda.synchronize()
        ffn = torch.zeros_like(x)
        blk.forward(w, x, tokens, ffn, torch.zeros_like(x))
        torch.cuda.synchronize()
        want.append((ffn, blk.shared_ungated().clone()))
    assert not torch.equal(want[0][0], want[1][0])
    outs, lout, stream = [torch.full_like(x, float("nan")) for _ in range(8)], torch.zeros_like(x), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for i, out in enumerate(outs):
            for t, h in zip(of(w), hosts[i % 2]):
                t.copy_(h, non_blocking=True)
            blk.forward(w, x, tokens, out, lout)
        stream.synchronize()
    for i, out in enumerate(outs):
        assert torch.equal(out.view(torch.int32), want[i % 2][0].view(torch.int32)), f"pass {i}"
    assert torch.equal(blk.shared_ungated().view(torch.int32), want[1][1].view(torch.int32))
