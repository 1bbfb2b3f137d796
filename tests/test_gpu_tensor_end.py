"""A tensor's last row lies in windows whose last bytes no whole piece inside the tensor holds: the kernels that bring Q6_K
rows to LDS add those bytes by themselves.  The same bytes at the end of a tensor and further in give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def X():
    import llmxabe_amd as X
    return X


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("tokens", [1, 4, 13, 40, 70])
@pytest.mark.parametrize("hidden,inter", [(512, 256), (768, 512), (2048, 512)])
def test_an_expert_is_the_same_bits_first_and_last(X, hidden, inter, tokens):
    import torch

    experts = 8
    g = X.MoeGeometry(experts, 1, hidden, inter, 32, tokens)
    per = hidden * inter // 256 * 210
    stacks = []
    for seed in (1, 2, 3):
        b = X.synth_quant(X.ExpertQuant.Q6K, seed, experts * hidden * inter, 0.02)
        b[(experts - 1) * per:] = b[:per]
        stacks.append(X.QuantTensor(b, X.ExpertQuant.Q6K))
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    for forced in (False, True):
        out = []
        for expert in (0, experts - 1):
            k = X.MoeKernels(g)
            k.force_community(forced)
            b = k.buffers()
            k.set_valid_tokens(b, tokens)
            logits = torch.zeros(tokens, experts, device="cuda")
            logits[:, expert] = 5.0
            k.route_and_dispatch(b, logits.view(-1))
            k.grouped_forward_partial(b, *stacks, x)
            torch.cuda.synchronize()
            out.append(_bits(b.partial()).copy())
        assert np.array_equal(out[0], out[1]), (forced, hidden, inter, tokens)


@pytest.mark.parametrize("tokens", [1, 3, 13, 40])
@pytest.mark.parametrize("hidden,inter", [(512, 256), (2048, 512)])
def test_the_blocks_last_expert(X, hidden, inter, tokens):
    import torch

    q8 = X.ExpertQuant.Q8_0
    experts, n = 8, hidden * inter
    per = n // 256 * 210
    stacks = []
    for seed in (1, 2, 3):
        b = X.synth_quant(X.ExpertQuant.Q6K, seed, experts * n, 0.02)
        b[(experts - 1) * per:] = b[:per]
        stacks.append(X.QuantTensor(b, X.ExpertQuant.Q6K))
    quant = lambda seed: X.QuantTensor(X.synth_quant(q8, seed, n, 0.02), q8)
    w = X.MoeLayerWeights(1.0 + X.synth_normal_f32(4, hidden, 0.1), torch.zeros(experts * hidden, device="cuda"), None, *stacks,
                          X.synth_normal_f32(5, hidden, 0.02), quant(6), quant(7), quant(8))
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    out = []
    for expert in (0, experts - 1):
        blk = X.MoeBlock(X.MoeGeometry(experts, 1, hidden, inter, 32, tokens))
        bias = torch.zeros(experts, device="cuda")
        bias[expert] = 5.0
        ffn, lo = torch.zeros_like(x), torch.zeros_like(x)
        blk.forward(w, x, tokens, ffn, lo, logit_bias=bias)
        torch.cuda.synchronize()
        out.append(_bits(lo).copy())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("tokens", [1, 3, 8])
@pytest.mark.parametrize("vocab,hidden", [(777, 1024), (513, 1536), (800, 512)])
def test_a_heads_last_rows(X, vocab, hidden, tokens):
    import torch

    more = vocab + 64
    b = X.synth_quant(X.ExpertQuant.Q6K, 1, more * hidden, 0.02)
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    out = []
    for v in (vocab, more):
        k = X.LmHeadKernels(X.LmHeadGeometry(hidden, v, tokens))
        logits = torch.zeros(tokens, v, device="cuda")
        k.forward(X.HeadTensor.q6_k(b[: v * hidden // 256 * 210].clone()), x, tokens, logits)
        torch.cuda.synchronize()
        out.append(_bits(logits[:, :vocab].contiguous()).copy())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("tokens", [1, 4, 8, 70])
def test_a_dense_blocks_last_rows(X, tokens):
    """gate/up: the last of 4352 rows beside the same rows of a wider block (whose down rows are then longer: the
    intermediate rows are what is compared)."""
    import torch

    hidden, out = 2560, []
    rows = 4352
    more = rows + 256
    gate, up = (X.synth_quant(X.ExpertQuant.Q6K, s, more * hidden, 0.02) for s in (1, 2))
    x = X.synth_normal_f32(9, tokens * hidden, 1.0).view(tokens, hidden)
    for r in (rows, more):
        n = r * hidden // 256 * 210
        k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, r, 32, tokens))
        k.disable_tensor_cores()
        b = k.shared_only_buffers(False)
        k.set_valid_tokens(b, tokens)
        down = X.QuantTensor(X.synth_quant(X.ExpertQuant.Q6K, 3, r * hidden, 0.02), X.ExpertQuant.Q6K)
        o = torch.zeros(tokens, hidden, device="cuda")
        k.shared_expert(b, X.QuantTensor(gate[:n].clone(), X.ExpertQuant.Q6K), X.QuantTensor(up[:n].clone(), X.ExpertQuant.Q6K), down, x, o)
        torch.cuda.synchronize()
        out.append(_bits(b.shared_inter()).reshape(tokens, r)[:, :rows].copy())
    assert np.array_equal(out[0], out[1])
