"""The digit row contractions over the row lengths where their forms differ: rows that end in half a superblock (Q8_0 rows of
128 elements modulo 256: a wider window, a half that is not there), one to ten superblocks (the split between the
wavefronts changes at 3, 5 and 9), both formats, every pass width of a single matrix, pairs against dispatch blocks.

Tolerance: three contractions in a row, each held to 5e-7 of the peak (tests/test_gpu_digit_precision.py derives it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 3 * 5e-7


def _stacks(X, q, E, H, I, seed):
    import torch

    out = [X.QuantTensor(X.synth_quant(q, seed + i, E * H * I, 0.02), q) for i in range(3)]
    host = [X.dequantize(q, t.bytes).double().cpu().numpy() for t in out]
    torch.cuda.synchronize()
    return out, (host[0].reshape(E, I, H), host[1].reshape(E, I, H), host[2].reshape(E, H, I))


def _ffn64(host, e, x):
    g, u = host[0][e] @ x, host[1][e] @ x
    return host[2][e] @ (g / (1 + np.exp(-g)) * u)


ROUTED = [("q8", 128, 128), ("q8", 384, 128), ("q8", 640, 384), ("q8", 1152, 896), ("q8", 2176, 1280), ("q8", 512, 2176),
          ("q6", 256, 256), ("q6", 768, 1280), ("q6", 1792, 768), ("q6", 2304, 2560)]


@pytest.mark.parametrize("fmt,hidden,inter", ROUTED)
def test_routed_experts(fmt, hidden, inter):
    import torch
    import llmxabe_amd as X

    E, K = 5, 2
    q = X.ExpertQuant.Q8_0 if fmt == "q8" else X.ExpertQuant.Q6K
    st, host = _stacks(X, q, E, hidden, inter, 9000)
    for tokens, live in ((1, 1), (4, 3), (5, 5), (25, 23), (63, 63)):
        x = X.synth_normal_f32(9010 + tokens, tokens * hidden, 1.0)
        logits = X.synth_normal_f32(9011 + tokens, tokens * E, 1.0)
        got = []
        for blocks in (False, True) if tokens > 4 else (False,):
            k = X.MoeKernels(X.MoeGeometry(E, K, hidden, inter, 32, tokens))
            k.force_community(blocks)
            k.set_exact_decode_regime(not blocks)    # (pairs whatever the width)
            b = k.buffers()
            k.set_valid_tokens(b, live)
            k.route_and_dispatch(b, logits)
            k.grouped_forward_partial(b, *st, x)
            got.append(b.partial().cpu().numpy().reshape(tokens, K, hidden)[:live].copy())
        ids = b.topk_ids().cpu().numpy().reshape(tokens, K)
        wts = b.topk_weights().cpu().numpy().reshape(tokens, K)
        xs = x.double().cpu().numpy().reshape(tokens, hidden)
        ref = np.array([[wts[t, j] * _ffn64(host, ids[t, j], xs[t]) for j in range(K)] for t in range(live)])
        err = np.abs(got[0] - ref).max() / np.abs(ref).max()
        print(fmt, hidden, inter, tokens, f"{err:.2e}", flush=True)
        assert err <= TOL, (tokens, err)
        assert len(got) == 1 or np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), tokens


SHARED = [("q8", 2176, 128), ("q8", 2432, 384), ("q8", 2304, 1152), ("q8", 4096, 1664), ("q6", 2304, 768), ("q6", 2560, 1280),
          ("q6", 4096, 1792), ("q6", 5120, 2304), ("q8", 1152, 9472), ("q6", 2048, 5120)]


@pytest.mark.parametrize("fmt,hidden,inter", SHARED)
def test_single_matrix_rows(fmt, hidden, inter):
    # hidden above 2048, or a long intermediate row: the shared expert's (the dense block's) rows on the digits, one to
    # eight tokens per pass
    import torch
    import llmxabe_amd as X

    q = X.ExpertQuant.Q8_0 if fmt == "q8" else X.ExpertQuant.Q6K
    st, host = _stacks(X, q, 1, hidden, inter, 9100)
    x = X.synth_normal_f32(9110, 17 * hidden, 1.0).view(17, hidden)
    ref = np.array([_ffn64(host, 0, v) for v in x.double().cpu().numpy()])
    alone = None
    for tokens, live in ((1, 1), (2, 2), (3, 3), (4, 4), (7, 6), (8, 8), (17, 17)):
        k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, tokens))
        b = k.shared_only_buffers(False)
        k.set_valid_tokens(b, live)
        out = torch.full((tokens, hidden), 7.0, device="cuda")
        k.shared_expert(b, *st, x[:tokens].reshape(-1).contiguous(), out.view(-1))
        got = out.cpu().numpy()
        err = np.abs(got[:live] - ref[:live]).max() / np.abs(ref).max()
        print(fmt, hidden, inter, tokens, f"{err:.2e}", flush=True)
        assert err <= TOL, (tokens, err)
        assert (got[live:] == 7.0).all(), tokens     # rows past the live ones are not written
        one = torch.zeros_like(out)
        k.force_community(True)                      # a pass per token, in the kernel of a single matrix
        k.shared_expert(b, *st, x[:tokens].reshape(-1).contiguous(), one.view(-1))
        assert np.array_equal(got[:live].view(np.uint32), one.cpu().numpy()[:live].view(np.uint32)), tokens
        alone = got if tokens == 1 else alone
        assert np.array_equal(got[0].view(np.uint32), alone[0].view(np.uint32)), tokens


@pytest.mark.parametrize("hidden,inter", [(2048, 4352), (2304, 3840), (8448, 2048)])
def test_large_q6_k_matrices(hidden, inter):
    # gate, up and down too large for the caches: passes of one, two, up to four, eight and sixteen tokens, in kernels of their
    # own.  Odd numbers of superblocks and of sixteen-row sets, several row tiles per compute unit, shares of unequal size; rows
    # with marked superblocks (elements forty binary orders apart) and an infinity next to ordinary ones.
    import torch
    import llmxabe_amd as X

    q = X.ExpertQuant.Q6K
    st, host = _stacks(X, q, 1, hidden, inter, 9200)
    x = X.synth_normal_f32(9210, 36 * hidden, 1.0).view(36, hidden)
    x[1, 1::2] *= 2.0 ** -40
    x[6, 300] = 2.0 ** 30
    x[12, 5] = float("inf")
    x[17, 2::3] *= 2.0 ** -35
    finite = [t for t in range(36) if t not in (6, 12)]
    ref = np.array([_ffn64(host, 0, v) for v in x.double().cpu().numpy()[finite]])

    def run(rows, live):
        k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, len(rows)))
        b = k.shared_only_buffers(False)
        k.set_valid_tokens(b, live)
        out = torch.full(rows.shape, 7.0, device="cuda")
        k.shared_expert(b, *st, rows.reshape(-1).contiguous(), out.view(-1))
        return out.cpu().numpy()

    alone = np.concatenate([run(x[t:t + 1], 1) for t in range(36)])
    err = np.abs(alone[finite] - ref).max() / np.abs(ref).max()
    print(hidden, inter, f"{err:.2e}", flush=True)
    assert err <= TOL, err
    assert not np.isfinite(alone[12]).all()
    same = lambda a, b: np.array_equal(a, b, equal_nan=True)
    for tokens, live in ((2, 2), (3, 3), (4, 3), (5, 5), (8, 7), (9, 9), (16, 16), (17, 16), (19, 19), (24, 24), (33, 33), (36, 34)):
        got = run(x[:tokens], live)
        assert same(got[:live], alone[:live]), tokens
        assert (got[live:] == 7.0).all(), tokens
    # the dense block: one and two tokens are normalised inside gate/up
    norm = 1.0 + X.synth_normal_f32(9211, hidden, 0.1)
    x[12, 5], x[11, 7] = 2.0 ** 60, float("inf")
    for rows in (x[1:2], x[6:8], x[11:13], x[12:13], x[10:13]):
        rows = rows.contiguous()
        blk = X.DenseFfnBlock(hidden, inter, len(rows))
        ffn, l_out = torch.zeros_like(rows), torch.zeros_like(rows)
        blk.forward(X.DenseFfnLayerWeights(norm, *st), rows, len(rows), ffn, l_out)
        normed = torch.zeros_like(rows)
        X.LayerOpsKernels.rms_norm(rows, norm, normed, len(rows), hidden, 1e-6)
        got = blk.normed().view(len(rows), hidden)
        assert same(got.cpu().numpy(), normed.cpu().numpy())
        assert same(ffn.cpu().numpy(), run(normed, len(rows)))
        assert same(l_out.cpu().numpy(), (ffn + rows).cpu().numpy())


# (hidden, intermediate) of the kernels that scale the intermediate rows by superblocks: the smallest of both, odd numbers of
# superblocks (9 and 25, 9 and 33, 21 and 35: classes of down's without any, with one and two), more sets of sixteen gate/up rows than a wavefront holds sums of (73 superblocks), more
# shares of gate and up than compute units (81), down's widest tiles for sixteen wavefronts of four tokens (4096 on 256 compute units)
WHOLE = [(2048, 6144), (2048, 8192), (4096, 8192), (2304, 6400), (2304, 8448), (5376, 8960), (2048, 18688), (5376, 20736)]


def _ffn64_rows(X, st, x, hidden, inter):
    q = X.ExpertQuant.Q6K
    w = lambda i, rows, cols: X.dequantize(q, st[i].bytes).double().view(rows, cols)
    g, u = x @ w(0, inter, hidden).T, x @ w(1, inter, hidden).T
    return (g / (1 + (-g).exp()) * u) @ w(2, hidden, inter).T


@pytest.mark.parametrize("hidden,inter", WHOLE)
def test_intermediate_rows_scaled_by_superblocks(hidden, inter):
    # every pass width, one token's row being the same bits in all of them; rows with marked superblocks of the activations and
    # an infinity; the dense block, whose one and two tokens are normalised inside gate/up
    import torch
    import llmxabe_amd as X

    q = X.ExpertQuant.Q6K
    st = [X.QuantTensor(X.synth_quant(q, 9300 + i, hidden * inter, 0.02), q) for i in range(3)]
    x = X.synth_normal_f32(9310, 19 * hidden, 1.0).view(19, hidden)
    x[1, 1::2] *= 2.0 ** -40
    x[6, 300] = 2.0 ** 30
    x[12, 5] = float("inf")
    x[17, 2::3] *= 2.0 ** -35
    finite = [t for t in range(19) if t not in (6, 12)]
    ref = _ffn64_rows(X, st, x[finite].double(), hidden, inter)
    same = lambda a, b: np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)

    def run(rows, live):
        k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, len(rows)))
        b = k.shared_only_buffers(False)
        k.set_valid_tokens(b, live)
        out = torch.full(rows.shape, 7.0, device="cuda")
        k.shared_expert(b, *st, rows.reshape(-1).contiguous(), out.view(-1))
        return out

    alone = torch.cat([run(x[t:t + 1], 1) for t in range(19)])
    err = ((alone[finite] - ref).abs().max() / ref.abs().max()).item()
    print(hidden, inter, f"{err:.2e}", flush=True)
    assert err <= TOL, err
    assert not alone[12].isfinite().all()
    for tokens, live in ((2, 2), (3, 3), (4, 3), (5, 5), (8, 7), (16, 16), (17, 16), (19, 19)):
        got = run(x[:tokens], live)
        assert same(got[:live], alone[:live]), tokens
        assert (got[live:] == 7.0).all(), tokens
    norm = 1.0 + X.synth_normal_f32(9311, hidden, 0.1)
    x[12, 5], x[11, 7] = 2.0 ** 60, float("inf")
    for rows in (x[1:2], x[6:8], x[11:13], x[12:13], x[10:13]):
        rows = rows.contiguous()
        blk = X.DenseFfnBlock(hidden, inter, len(rows))
        ffn, l_out = torch.zeros_like(rows), torch.zeros_like(rows)
        blk.forward(X.DenseFfnLayerWeights(norm, *st), rows, len(rows), ffn, l_out)
        normed = torch.zeros_like(rows)
        X.LayerOpsKernels.rms_norm(rows, norm, normed, len(rows), hidden, 1e-6)
        assert same(blk.normed().view(len(rows), hidden), normed)
        assert same(ffn, run(normed, len(rows)))
        assert same(l_out, ffn + rows)


@pytest.mark.parametrize("hidden,inter", [(2048, 8192), (5376, 8960)])
@pytest.mark.parametrize("small", [1, 8, 9, 40])
def test_values_far_below_their_superblocks_largest(hidden, inter, small):
    # intermediate rows whose superblocks hold one large value, which down's weights ignore, and `small` ones 2^-32 of it, which
    # the 48-bit numbers hold to fourteen bits: up to eight are added by themselves, more take the whole superblock along.  float64
    # within TOL, and the same bits at every width
    import torch
    import llmxabe_amd as X

    q = X.ExpertQuant.Q6K
    st = [X.synth_quant(q, 9400 + i, hidden * inter, 0.02) for i in range(3)]
    factor = torch.zeros(inter, device="cuda")
    sbs = (0, 5, inter // 256 - 1)
    for sb in sbs:
        factor[256 * sb + 7] = 2.0 ** 16
        factor[256 * sb + 16 + 5 * torch.arange(small, device="cuda")] = 1.0
    for i in (0, 1):
        d = st[i].view(inter, hidden // 256, 210)[:, :, 208:]
        d.copy_((d.contiguous().view(torch.float16).float() * factor.view(-1, 1, 1)).half().view(torch.uint8))
    st[2].view(hidden, inter // 256, 210)[:, list(sbs), 192] = 0   # the scale of the large values' group
    st = [X.QuantTensor(t, q) for t in st]
    x = X.synth_normal_f32(9410, 19 * hidden, 1.0).view(19, hidden)
    ref = _ffn64_rows(X, st, x.double(), hidden, inter)

    def run(n):
        k = X.MoeKernels(X.MoeGeometry(1, 1, hidden, inter, 32, n))
        b = k.shared_only_buffers(False)
        k.set_valid_tokens(b, n)
        out = torch.full((n, hidden), 7.0, device="cuda")
        k.shared_expert(b, *st, x[:n].reshape(-1).contiguous(), out.view(-1))
        return out

    rows = run(19)
    err = ((rows - ref).abs().max(1).values / ref.abs().max(1).values).max().item()
    print(hidden, inter, small, f"{err:.2e}", flush=True)
    assert err <= TOL, err
    for n in (1, 2, 3, 4, 5, 8, 16):
        assert torch.equal(run(n).view(torch.int32), rows[:n].view(torch.int32)), n
