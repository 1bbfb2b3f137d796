"""The combine at the widths of both its kernels (rows of at most 2048 elements, longer ones), with as many selections as the
short rows' kernel requests at once, fewer and more, against float64.

Tolerance.  The routed sum adds top_k values in order: at most top_k half ulps of the sum of magnitudes; the gate is a dot of
`hidden` terms (its error against sum |w x|, hidden half ulps at most, times the sigmoid's slope of 1/4) and the products and
sums behind it add two ulps of the terms."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def X():
    import llmxabe_amd as X
    return X


@pytest.mark.parametrize("hidden", [128, 1152, 2048, 2176])
@pytest.mark.parametrize("top_k,tokens", [(1, 5), (7, 3), (8, 70), (9, 4), (12, 65)])
def test_combine(X, hidden, top_k, tokens):
    import torch

    live = tokens - 1
    k = X.MoeKernels(X.MoeGeometry(16, top_k, hidden, 256, 32, tokens))
    b = k.buffers()
    k.set_valid_tokens(b, live)
    n, count = tokens * hidden, 16 * hidden * 256
    stacks = [X.QuantTensor(X.synth_quant(X.ExpertQuant.Q8_0, s, count, 0.05), X.ExpertQuant.Q8_0) for s in (6, 7, 8)]
    k.route_and_dispatch(b, X.synth_normal_f32(9, tokens * 16, 1.0))
    k.grouped_forward_partial(b, *stacks, X.synth_normal_f32(10, n, 1.0).view(tokens, hidden))
    part = b.partial()[:tokens * top_k * hidden]
    w = X.synth_normal_f32(2, hidden, 0.05)
    normed, shexp, residual = (X.synth_normal_f32(s, n, 1.0).view(tokens, hidden) for s in (3, 4, 5))
    gate = torch.zeros(tokens, device="cuda")
    routed, ffn, l_out = (torch.zeros(tokens, hidden, device="cuda") for _ in range(3))
    k.gate_and_combine(b, w, normed, shexp, residual, gate, routed, ffn, l_out)
    torch.cuda.synchronize()
    p = part.view(tokens, top_k, hidden).double()[:live]
    half = 2.0 ** -24
    assert bool(p.any())
    r, mag = p.sum(1), p.abs().sum(1)
    assert bool(((routed[:live].double() - r).abs() <= top_k * half * mag).all())
    z = normed[:live].double() @ w.double()
    g = torch.sigmoid(z)
    g_err = hidden * half * (normed[:live].double().abs() @ w.double().abs()) / 4 + 4 * half
    assert bool(((gate[:live].double() - g).abs() <= g_err).all())
    sh = shexp[:live].double()
    bound = top_k * half * mag + g_err[:, None] * sh.abs() + 4 * half * (mag + sh.abs() + residual[:live].double().abs())
    want = r + sh * g[:, None]
    assert bool(((ffn[:live].double() - want).abs() <= bound).all())
    assert bool(((l_out[:live].double() - want - residual[:live].double()).abs() <= bound).all())
    assert not routed[live:].any() and not ffn[live:].any() and not l_out[live:].any()


# (one 16-byte column per thread up to 1024 elements; k_gate_and_combine again for more than 2048 rows of at most 256)
@pytest.mark.parametrize("hidden,tokens", [(256, 2048), (256, 2049), (128, 2049), (384, 2049), (1024, 66), (1024, 2)])
def test_combine_on_both_sides_of_its_rules(X, hidden, tokens):
    test_combine(X, hidden, 8, tokens)
