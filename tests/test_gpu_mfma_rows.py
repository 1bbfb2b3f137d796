"""The matrix-core grouped GEMM at the edges of its tiles: 32-row blocks, the narrow form's 64 rows, the wide form's 192, the
rule between the two, contractions of one superblock up, both formats, against the fp32 lanes of the same library.

Tolerance.  Weights are rounded to fp16 twice (scale, product) and activations once, each by a relative 2^-11 at most: over a
contraction of random signs a row's relative error in the 2-norm is about sqrt(3) 2^-11 / sqrt(3) = 4.9e-4 for gate and for up,
whose product carries sqrt(2) of that at SwiGLU's slope of about 1, one more rounding of the product, and the same again in
down: 1e-3 together.  Twice that is asked for; a row, block or step that is wrong is off by order 1."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROW_REL = 2e-3


@pytest.fixture(scope="module")
def X():
    import llmxabe_amd as X
    return X


def _weights(X, up, down, n):
    q = {"q6k": X.ExpertQuant.Q6K, "q8_0": X.ExpertQuant.Q8_0}
    return [X.QuantTensor(X.synth_quant(q[f], seed, n, 0.02), q[f]) for seed, f in ((1, up), (2, up), (3, down))]


def _close(got, want):
    got, want = got.double(), want.double()
    rel = (got - want).norm(dim=1) / want.norm(dim=1)
    assert float(want.norm(dim=1).min()) > 0
    assert float(rel.max()) <= ROW_REL, (int(rel.argmax()), float(rel.max()))


@pytest.mark.parametrize("up,down", [("q6k", "q6k"), ("q6k", "q8_0"), ("q8_0", "q6k")])
@pytest.mark.parametrize("hidden,inter", [(256, 256), (512, 256), (256, 768), (2048, 512), (1792, 1024), (256, 8192)])
@pytest.mark.parametrize("counts", [(1, 31, 32, 33), (63, 64, 65, 0), (191, 192, 193, 257), (385, 1, 0, 96), (160, 97, 224, 384)])
def test_experts_of_every_size(X, counts, hidden, inter, up, down):
    import torch

    experts, tokens = len(counts), sum(counts)
    g = X.MoeGeometry(experts, 1, hidden, inter, 32, tokens)
    weights = _weights(X, up, down, experts * hidden * inter)
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    pick = np.random.default_rng(tokens).permutation(np.repeat(np.arange(experts), counts))
    logits = torch.zeros(tokens, experts, device="cuda")
    logits[torch.arange(tokens), torch.from_numpy(pick)] = 5.0
    out = []
    for form in (1, 2, None):
        k = X.MoeKernels(g)
        if form is None:
            k.disable_tensor_cores()
        else:
            k.set_mfma_form(form)
        b = k.buffers()
        k.set_valid_tokens(b, tokens)
        k.route_and_dispatch(b, logits.view(-1))
        k.grouped_forward_partial(b, *weights, x)
        torch.cuda.synchronize()
        out.append(b.partial().clone()[:tokens * hidden].view(tokens, hidden))
    _close(out[0], out[2])
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32))


@pytest.mark.parametrize("experts", [191, 192, 193, 287, 288])
def test_gate_up_items_of_two_to_three_rounds(X, experts):
    # eight gate/up items per expert: 1528 to 2304, about two and three times the 768 workgroups that a chip of 256 CUs holds
    import torch

    hidden, inter, tokens = 512, 512, experts + 3
    g = X.MoeGeometry(experts, 1, hidden, inter, 32, tokens)
    weights = _weights(X, "q6k", "q8_0", experts * hidden * inter)
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    logits = torch.zeros(tokens, experts, device="cuda")
    logits[torch.arange(tokens), torch.arange(tokens) % experts] = 5.0
    out = []
    for form in (1, 2, None):
        k = X.MoeKernels(g)
        if form is None:
            k.disable_tensor_cores()
        else:
            k.set_mfma_form(form)
        b = k.buffers()
        k.set_valid_tokens(b, tokens)
        k.route_and_dispatch(b, logits.view(-1))
        k.grouped_forward_partial(b, *weights, x)
        torch.cuda.synchronize()
        out.append(b.partial().clone()[:tokens * hidden].view(tokens, hidden))
    _close(out[0], out[2])
    assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32))


@pytest.mark.parametrize("quant", ["q6k", "q8_0"])
@pytest.mark.parametrize("hidden,inter,widths", [(256, 16384, (383, 384, 385, 1000)), (512, 256, (64, 65, 97, 193)),
                                                 (1280, 11008, (576, 640, 769)),
                                                 # 128 tiles of gate/up in one row (wide from 97 tokens), 128 parts of down in two (from 193)
                                                 (256, 16384, (95, 96, 97, 192)), (4096, 12288, (192, 193, 384)),
                                                 (5120, 17408, (96, 97, 192, 193, 320))])
def test_unrouted_widths_across_the_rule(X, quant, hidden, inter, widths):
    import torch

    weights = _weights(X, quant, quant, hidden * inter)
    x = X.synth_normal_f32(9, max(widths) * hidden, 1.0).view(max(widths), hidden)
    rows = []
    for tokens in widths:
        g = X.MoeGeometry(1, 1, hidden, inter, 32, tokens)
        got = []
        for mma in (True, False):
            k = X.MoeKernels(g)
            if not mma:
                k.disable_tensor_cores()
            b = k.shared_only_buffers(True)
            k.set_valid_tokens(b, tokens)
            out = torch.zeros(tokens, hidden, device="cuda")
            (k.shared_expert_mma if mma else k.shared_expert)(b, *weights, x[:tokens], out)
            torch.cuda.synchronize()
            got.append(out)
        _close(*got)
        rows.append(got[0])
    for wider in rows[1:]:   # a token's row does not depend on the batch around it
        assert torch.equal(wider[:widths[0]].view(torch.int32), rows[0].view(torch.int32))


@pytest.mark.parametrize("quant", ["q6k", "q8_0"])
@pytest.mark.parametrize("hidden,inter", [(512, 6912), (768, 8704), (512, 11008), (1280, 4096)])
def test_long_down_contractions_in_parts(X, quant, hidden, inter):
    # three, two and one part (27, 34 and 43 superblocks), and none for want of a place for the planes; both tile forms; the block,
    # whose last launch adds the residual, against the separate calls
    import torch

    weights = _weights(X, quant, quant, hidden * inter)
    norm = 1.0 + X.synth_normal_f32(4, hidden, 0.1)
    rows = []
    for tokens, live in ((64, 64), (100, 97), (1024, 1000)):
        x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
        blk = X.DenseFfnBlock(hidden, inter, tokens)
        ffn, l_out = torch.full_like(x, -7.0), torch.full_like(x, -7.0)
        blk.publish_tokens(live)
        blk.forward(X.DenseFfnLayerWeights(norm, *weights), x, live, ffn, l_out)
        k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, tokens))
        got = []
        for mma in (True, False):
            if not mma:
                k.disable_tensor_cores()
            b = k.shared_only_buffers(True)
            k.set_valid_tokens(b, live)
            out = torch.full_like(x, -7.0)
            (k.shared_expert_mma if mma else k.shared_expert)(b, *weights, blk.normed().view(tokens, hidden), out)
            got.append(out)
        torch.cuda.synchronize()
        _close(got[0][:live], got[1][:live])
        assert torch.equal(ffn[:live].view(torch.int32), got[0][:live].view(torch.int32))
        assert torch.equal(l_out[:live], ffn[:live] + x[:live])
        for t in (ffn, l_out, got[0]):
            assert (t[live:] == -7.0).all()
        rows.append(ffn[:64])
    for wider in rows[1:]:   # a token's row does not depend on the batch around it
        assert torch.equal(wider.view(torch.int32), rows[0].view(torch.int32))


@pytest.mark.parametrize("quant", ["q6k", "q8_0"])
@pytest.mark.parametrize("hidden,inter", [(512, 6912), (4096, 12288)])
def test_few_live_tokens_in_buffers_of_more_than_1024(X, quant, hidden, inter):
    # there the down contraction is one chain at every width: float32 at the tolerance above, a row the same bits in every pass
    import torch

    weights, tokens = _weights(X, quant, quant, hidden * inter), 1025
    norm = 1.0 + X.synth_normal_f32(4, hidden, 0.1)
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, 257))
    k.disable_tensor_cores()
    b = k.shared_only_buffers(True)
    blk = X.DenseFfnBlock(hidden, inter, tokens)
    rows = []
    for live in (65, 257, 1025):
        ffn, l_out = torch.full_like(x, -7.0), torch.full_like(x, -7.0)
        blk.publish_tokens(live)
        blk.forward(X.DenseFfnLayerWeights(norm, *weights), x, live, ffn, l_out)
        n = min(live, 257)
        want = torch.zeros(257, hidden, device="cuda")
        k.set_valid_tokens(b, n)
        k.shared_expert(b, *weights, blk.normed().view(tokens, hidden)[:257].contiguous(), want)
        torch.cuda.synchronize()
        _close(ffn[:n], want[:n])
        assert torch.equal(l_out[:live], ffn[:live] + x[:live])
        assert (ffn[live:] == -7.0).all() and (l_out[live:] == -7.0).all()
        rows.append(ffn[:65].clone())
    for wider in rows[1:]:
        assert torch.equal(wider.view(torch.int32), rows[0].view(torch.int32))
