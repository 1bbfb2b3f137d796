"""The fp32 regimes at matrix-core widths: their digits (csrc/digits.h) go through scratch of a bounded number of rows, part
by part, and every row is the one a narrow pass makes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


def test_wide_handles_carry_no_digits_of_every_row():
    # partial, the intermediate rows (fp32 and fp16), the fp16 activations, the router's planes, the shared expert's rows:
    # 880 MB for 8192 tokens of the model; the dense sibling's 2048 tokens: 234 MB
    import llmxabe_amd as X

    k = X.MoeKernels(X.MoeGeometry.qwen3_6(64, 8192))
    assert k.buffers().bytes() < 920e6
    k = X.MoeKernels(X.MoeGeometry(1, 1, 5120, 17408, 64, 2048))
    assert k.shared_only_buffers(True).bytes() < 260e6


@pytest.mark.parametrize("exact", [True, False])   # pairs; dispatch blocks (the matrix cores disabled)
@pytest.mark.parametrize("experts,top_k", [(16, 8), (256, 8), (8, 1)])   # (8, 1): `partial` has no room for the activations' digits
def test_routed_rows_of_a_wide_pass(exact, experts, top_k):
    import torch
    import llmxabe_amd as X

    H, I = 512, 256
    T, live = (1100, 1090) if top_k > 1 else (9000, 8990)
    q = X.ExpertQuant.Q6K
    st = [X.QuantTensor(X.synth_quant(q, 9200 + i, experts * H * I, 0.02), q) for i in range(3)]
    x = X.synth_normal_f32(9210, T * H, 1.0).view(T, H)
    logits = X.synth_normal_f32(9211, T * experts, 1.0).view(T, experts)

    def run(rows, tokens, lg, split=False):
        k = X.MoeKernels(X.MoeGeometry(experts, top_k, H, I, X.moe_block_size(rows.shape[0]), rows.shape[0]))
        k.set_exact_decode_regime(exact)
        k.disable_tensor_cores()
        b = k.buffers()
        k.set_valid_tokens(b, tokens)
        k.route_and_dispatch(b, lg.reshape(-1).contiguous())
        xr = rows.reshape(-1).contiguous()
        if split:
            for stage in (0, 1):
                k.grouped_forward_stage(b, *st, xr, stage)
        else:
            k.grouped_forward_partial(b, *st, xr)
        return _bits(b.partial()).reshape(-1, top_k, H)[:tokens].copy()

    wide = run(x, live, logits)
    assert np.array_equal(run(x, live, logits, split=True), wide)
    for at in (0, 300, live - 40):
        assert np.array_equal(run(x[at:at + 40], 40, logits[at:at + 40]), wide[at:at + 40]), at


@pytest.mark.parametrize("fused", [True, False])   # the dense block (norm and residual in the launches); the step by itself
def test_single_matrix_rows_of_a_wide_pass(fused):
    import torch
    import llmxabe_amd as X

    H, I, T, live = 2560, 512, 200, 131
    q = X.ExpertQuant.Q6K
    st = [X.QuantTensor(X.synth_quant(q, 9300 + i, H * I, 0.02), q) for i in range(3)]
    norm = 1.0 + X.synth_normal_f32(9305, H, 0.1)
    x = X.synth_normal_f32(9310, T * H, 1.0).view(T, H)

    def run(rows, tokens):
        rows, n = rows.contiguous(), rows.shape[0]
        out, lout = torch.full_like(rows, 7.0), torch.full_like(rows, 7.0)
        if fused:
            blk = X.DenseFfnBlock(H, I, n)
            blk.disable_tensor_cores()
            blk.forward(X.DenseFfnLayerWeights(norm, *st), rows, tokens, out, lout)
        else:
            k = X.MoeKernels(X.MoeGeometry(1, 1, H, I, 64, n))
            b = k.shared_only_buffers(False)
            k.set_valid_tokens(b, tokens)
            k.shared_expert(b, *st, rows.view(-1), out.view(-1))
        torch.cuda.synchronize()
        assert (out[tokens:] == 7.0).all() and (lout[tokens:] == 7.0).all()
        return np.stack([_bits(out)[:tokens], _bits(lout)[:tokens]])

    wide = run(x, live)
    for at, n in ((0, 7), (60, 9), (live - 5, 5)):
        assert np.array_equal(run(x[at:at + n], n), wide[:, at:at + n]), at
