"""The routed experts and the shared expert of one set of buffers on two streams at once, each with activation rows of
its own: the entry points share no scratch, so every pass equals the one made alone.  (hidden 4096: both sides go
through the digits of their activation rows; hidden 1024: only the routed experts do.)"""
import numpy as np
import pytest

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
