"""Router logits at prefill widths: tiles of 64 and of 128 experts, chosen by how many workgroups there are, give a token's
logits the same bits."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", [None, "Q8_0"])
def test_a_tokens_logits_do_not_depend_on_the_tile(quant):
    import torch

    import llmxabe_amd as X

    hidden, experts, n = 2048, 256, 1700
    q = None if quant is None else X.ExpertQuant.Q8_0
    router = X.synth_normal_f32(1, experts * hidden, 0.02) if q is None else X.synth_quant(q, 1, experts * hidden, 0.02)
    x = X.synth_normal_f32(2, n * hidden, 1.0)
    rows = None
    for tokens in (300, 1024, 1088, 1535, 1536, n):   # around one and one and a half wide tiles per compute unit
        k = X.MoeKernels(X.MoeGeometry.qwen3_6(X.moe_block_size(tokens), tokens))
        b = k.buffers()
        k.set_valid_tokens(b, tokens)
        logits = torch.zeros(tokens * experts, device="cuda")
        k.router_logits(b, router, q, x[:tokens * hidden], logits)
        torch.cuda.synchronize()
        got = logits.view(tokens, experts)[:300].view(torch.int32)
        assert bool(got.any())
        assert rows is None or torch.equal(got, rows), tokens
        rows = got
