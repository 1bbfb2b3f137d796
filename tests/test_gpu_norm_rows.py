"""RMSNorm of many long rows: a row's bits do not depend on how many rows the launch has (few, many: other kernels), and the
dense block, whose norm launch writes the fp16 copy as well, gives the bits of its steps one by one."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def X():
    import llmxabe_amd as X
    return X


@pytest.mark.parametrize("width", [2052, 4096, 4100, 5120, 6140, 6144, 6148, 8196])
def test_a_row_is_the_same_bits_among_few_and_many(X, width):
    import torch

    rows = 1536
    x = X.synth_normal_f32(1, rows * width, 1.0).view(rows, width)
    w = 1.0 + X.synth_normal_f32(2, width, 0.1)
    many, few = torch.zeros_like(x), torch.zeros_like(x)
    X.LayerOpsKernels.rms_norm(x, w, many, rows, width, 1e-6)
    for r in (0, 1, 63, 700, rows - 1):
        X.LayerOpsKernels.rms_norm(x[r:r + 1], w, few[r:r + 1], 1, width, 1e-6)
        torch.cuda.synchronize()
        assert torch.equal(many[r].view(torch.int32), few[r].view(torch.int32)), r
    want = x.double() * torch.rsqrt((x.double() ** 2).mean(dim=1, keepdim=True) + 1e-6) * w.double()
    # (the fold of `width` squares, a quotient and a root, two products: a few hundred half ulps at most)
    assert float(((many.double() - want).abs() / want.abs().clamp_min(1e-30)).max()) < 3e-5


@pytest.mark.parametrize("hidden,tokens", [(512, 64), (2304, 64), (2304, 1535), (2304, 1536), (6144, 1600), (6400, 1540)])
def test_the_dense_block_is_its_steps(X, hidden, tokens):
    import torch

    inter, q = 256, X.ExpertQuant.Q6K
    w = [X.QuantTensor(X.synth_quant(q, s, hidden * inter, 0.02), q) for s in (1, 2, 3)]
    norm = 1.0 + X.synth_normal_f32(4, hidden, 0.1)
    x = X.synth_normal_f32(5, tokens * hidden, 1.0).view(tokens, hidden)
    block = X.DenseFfnBlock(hidden, inter, tokens)
    ffn, l_out = torch.zeros_like(x), torch.zeros_like(x)
    block.forward(X.DenseFfnLayerWeights(norm, *w), x, tokens, ffn, l_out)
    k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, tokens))
    b = k.shared_only_buffers(True)
    k.set_valid_tokens(b, tokens)
    normed, want = torch.zeros_like(x), torch.zeros_like(x)
    X.LayerOpsKernels.rms_norm(x, norm, normed, tokens, hidden, 1e-6)
    k.shared_expert_mma(b, *w, normed, want)
    torch.cuda.synchronize()
    assert torch.equal(ffn.view(torch.int32), want.view(torch.int32))
    assert torch.equal(l_out, want + x)


@pytest.mark.parametrize("hidden", [128, 1152, 5120])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_the_residual_is_added_wherever_rows_start(X, hidden, off):
    import torch

    tokens, live = 5, 4
    k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, 256, 32, tokens))
    b = k.shared_only_buffers(False)
    k.set_valid_tokens(b, live)
    n = tokens * hidden
    ffn, res, out = (X.synth_normal_f32(s, n + 4, 1.0)[off * (s == 2) + 2 * (s == 3) * (off > 0):][:n] for s in (1, 2, 3))
    before = out.clone()
    k.dense_ffn_add_residual(b, ffn, res, out)
    torch.cuda.synchronize()
    m = live * hidden
    assert torch.equal(out[:m], ffn[:m] + res[:m]) and torch.equal(out[m:], before[m:])
