"""What the integer contraction of the fp32 regimes (csrc/digits.h) keeps of its fp32 operands.  An activation is a fixed-point
number relative to its group of sixteen, so the hard inputs are the ones an fp32 multiply-add never notices: an outlier
beside ordinary values where the weights' codes are zero (all that is left of the group is what lies far below its
largest), a group of which only the smallest value meets a weight, groups near the ends of the exponent range, and
infinities, which reach an output with their sign.  Every path that takes the contraction is held against float64: the LM
head, the step-by-step routed experts, the block's three launches, rows longer than 2048 elements.

Tolerance: a row of K elements is the fp32 sum of K / 16 exact group sums, each rounded a few times, so its error is a
random walk of at most about 2 K / 16 steps of 2^-25 of the partial sums, which the peak of the outputs bounds:
3 sqrt(2 * 2048 / 16) 2^-25 = 1.4e-6 of the peak at three sigma of the worst partial sum.  Measured 1.0e-7 to 2e-7; the
plain fp32 sums of the same rows 1.5e-7 to 3e-7.  5e-7 is asserted."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 5e-7


def _q8_0(codes, d):
    """codes int8 [rows][K], d float16 [rows]: block bytes and the values they encode."""
    rows, K = codes.shape
    b = np.zeros((rows, K // 32, 34), np.uint8)
    b[:, :, :2] = np.repeat(d.astype(np.float16).view(np.uint8).reshape(rows, 1, 2), K // 32, 1)
    b[:, :, 2:] = codes.reshape(rows, K // 32, 32).view(np.uint8)
    return b.reshape(-1), codes * d.astype(np.float16).astype(np.float64)[:, None]


def _q6_k(codes, d):
    """codes -32..31 [rows][K], every sub-block scale 16: ql[128] qh[64] scales[16] d."""
    rows, K = codes.shape
    c = (codes + 32).astype(np.uint8).reshape(rows, K // 256, 2, 4, 32)   # [half][quarter][32]
    b = np.zeros((rows, K // 256, 210), np.uint8)
    ql, qh = np.zeros((rows, K // 256, 2, 64), np.uint8), np.zeros((rows, K // 256, 2, 32), np.uint8)
    ql[..., :32] = (c[:, :, :, 0] & 15) | ((c[:, :, :, 2] & 15) << 4)
    ql[..., 32:] = (c[:, :, :, 1] & 15) | ((c[:, :, :, 3] & 15) << 4)
    for s in range(4):
        qh |= (c[:, :, :, s] >> 4) << (2 * s)
    b[:, :, :128], b[:, :, 128:192] = ql.reshape(rows, K // 256, 128), qh.reshape(rows, K // 256, 64)
    b[:, :, 192:208] = 16
    b[:, :, 208:] = d.astype(np.float16).view(np.uint8).reshape(rows, 1, 2)
    return b.reshape(-1), codes * 16.0 * d.astype(np.float16).astype(np.float64)[:, None]


def _matrix(rng, quant, rows, K, zero=None, d=None):
    hi = 127 if quant == "Q8_0" else 31
    codes = rng.integers(-hi, hi + 1, (rows, K)).astype(np.int8)
    if zero is not None:
        codes[:, zero] = 0
    d = np.full(rows, 2e-4 if quant == "Q8_0" else 6e-5) if d is None else d
    return (_q8_0 if quant == "Q8_0" else _q6_k)(codes, d)


def _rows(rng, kind, tokens, K):
    """activation rows of one kind, and the columns whose weights are zero"""
    x = rng.standard_normal((tokens, K)).astype(np.float32)
    zero = np.zeros(K, bool)
    if kind.startswith("outlier"):            # one outlier per group
        zero[3::16] = True
        x[:, zero] = float(kind.split("_")[1]) * np.where(rng.random(x[:, zero].shape) < 0.5, -1, 1)
    elif kind == "many_outliers":             # half of the group, at several magnitudes
        for i, m in ((0, 1e4), (2, 1e6), (5, 1e9), (6, 1e12), (9, 1e3), (11, 1e15), (13, 1e5), (15, 1e18)):
            zero[i::16] = True
            x[:, i::16] *= m
    elif kind == "smallest_only":             # weights only where the group's smallest value is
        zero[:] = True
        zero[7::16] = False
        x[:, 7::16] *= 2.0 ** -18
    elif kind == "tiny":
        x *= 2.0 ** -100
    elif kind == "huge":
        x *= 2.0 ** 100
    elif kind == "subnormal":
        x[:, ::2] *= np.float32(2.0 ** -140)  # (beside ordinary values)
    return x, zero


KINDS = ["plain", "outlier_1e3", "outlier_3e4", "outlier_1e8", "many_outliers", "smallest_only", "tiny", "huge", "subnormal"]


def _check(got, ref, label):
    assert np.all(np.isfinite(got)), label
    err = np.abs(got.astype(np.float64) - ref).max() / np.abs(ref).max()
    print(label, f"{err:.2e}")
    assert err <= TOL, (label, err)


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
@pytest.mark.parametrize("tokens", [1, 7])
def test_lm_head(quant, tokens):
    import torch
    import llmxabe_amd as X

    V, K = 300, 2048
    k = X.LmHeadKernels(X.LmHeadGeometry(K, V, tokens))
    for kind in KINDS:
        rng = np.random.default_rng(11)
        x, zero = _rows(rng, kind, tokens, K)
        raw, w = _matrix(rng, quant, V, K, zero)
        dev = torch.from_numpy(raw).cuda()
        head = X.HeadTensor.q8_0(dev) if quant == "Q8_0" else X.HeadTensor.q6_k(dev)
        out = torch.zeros(tokens, V, device="cuda")
        k.forward(head, torch.from_numpy(x).cuda(), tokens, out)
        _check(out.cpu().numpy(), x.astype(np.float64) @ w.T, ("head", quant, tokens, kind))


def _expert_stacks(X, rng, quant, E, H, I, zero_up, zero_down, d_rows=None):
    """gate, up and down stacks with the same zero columns in every expert, and their float64 values"""
    import torch

    q = X.ExpertQuant.Q8_0 if quant == "Q8_0" else X.ExpertQuant.Q6K
    out, host = [], []
    for rows, K, zero, d in ((I, H, zero_up, None), (I, H, zero_up, d_rows), (H, I, zero_down, None)):
        raw, val = zip(*(_matrix(rng, quant, rows, K, zero, d) for _ in range(E)))
        out.append(X.QuantTensor(torch.from_numpy(np.concatenate(raw)).cuda(), q))
        host.append(np.stack(val))
    return out, host


def _expert64(host, e, x):
    g, u = host[0][e] @ x, host[1][e] @ x
    return host[2][e] @ (g / (1 + np.exp(-g)) * u)


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
@pytest.mark.parametrize("tokens", [2, 9])
@pytest.mark.parametrize("hidden,inter", [(512, 256), (2048, 512), (2560, 512)])
def test_step_by_step_experts(quant, tokens, hidden, inter):
    # gate and up see the row kinds; a gate that saturates SwiGLU leaves silu(g) = g, so the row's error is the two products'
    import torch
    import llmxabe_amd as X

    E = 4
    g = X.MoeGeometry(E, 2, hidden, inter, 32, tokens)
    for kind in KINDS[:6]:
        rng = np.random.default_rng(12)
        x, zero = _rows(rng, kind, tokens, hidden)
        x /= np.abs(x[:, ~zero]).max()   # (the products stay in SwiGLU's range whatever the outliers are)
        st, host = _expert_stacks(X, rng, quant, E, hidden, inter, zero, None)
        k = X.MoeKernels(g)
        b = k.buffers()
        k.set_valid_tokens(b, tokens)
        logits = torch.from_numpy(rng.standard_normal((tokens, E)).astype(np.float32)).cuda()
        k.route_and_dispatch(b, logits)
        k.grouped_forward_partial(b, *st, torch.from_numpy(x).cuda())
        ids = b.topk_ids().cpu().numpy().reshape(tokens, 2)
        wts = b.topk_weights().cpu().numpy().reshape(tokens, 2)
        got = b.partial().cpu().numpy().reshape(tokens, 2, hidden)
        ref = np.array([[wts[t, j] * _expert64(host, ids[t, j], x[t].astype(np.float64)) for j in range(2)] for t in range(tokens)])
        # (three contractions in a row, the last one of 256 or 512 terms: their errors add)
        err = np.abs(got - ref).max() / np.abs(ref).max()
        print("steps", quant, tokens, hidden, kind, f"{err:.2e}")
        assert err <= 3 * TOL, (kind, err)


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
@pytest.mark.parametrize("tokens", [1, 9])
def test_intermediate_rows_with_outliers(quant, tokens):
    # one up row in sixteen is a thousand times larger, and the down matrix has zeros there: step by step and in the block
    import torch
    import llmxabe_amd as X

    E, H, I = 4, 512, 256
    rng = np.random.default_rng(13)
    g = X.MoeGeometry(E, 2, H, I, 32, tokens)
    d_rows = np.full(I, 2e-4 if quant == "Q8_0" else 6e-5)
    zero = np.zeros(I, bool)
    zero[5::16] = True
    d_rows[zero] *= 1000
    st, host = _expert_stacks(X, rng, quant, E, H, I, None, zero, d_rows)
    q8 = X.ExpertQuant.Q8_0
    sh = [X.QuantTensor(X.synth_quant(q8, 60 + i, H * I, 0.02), q8) for i in range(3)]
    x = torch.from_numpy(rng.standard_normal((tokens, H)).astype(np.float32)).cuda()
    w = X.MoeLayerWeights(torch.ones(H, device="cuda"), X.synth_normal_f32(61, E * H, 0.02), None, *st,
                          X.synth_normal_f32(62, H, 0.02), *sh)
    routed = []
    for fused in (True, False):
        blk = X.MoeBlock(g)
        blk.set_fused_decode(fused)
        blk.forward(w, x, tokens, torch.zeros_like(x), torch.zeros_like(x))
        b = blk.buffers()
        ids, wts = (t.cpu().numpy().reshape(tokens, 2) for t in (b.topk_ids(), b.topk_weights()))
        normed = blk.normed().cpu().numpy().reshape(tokens, H).astype(np.float64)
        routed.append(blk.routed().cpu().numpy().reshape(tokens, H))
        ref = np.array([sum(wts[t, j] * _expert64(host, ids[t, j], normed[t]) for j in range(2)) for t in range(tokens)])
        err = np.abs(routed[-1] - ref).max() / np.abs(ref).max()
        print("inter", quant, tokens, fused, f"{err:.2e}")
        assert err <= 3 * TOL, (fused, err)
    assert np.array_equal(routed[0].view(np.uint32), routed[1].view(np.uint32))


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
@pytest.mark.parametrize("tokens", [1, 9])
@pytest.mark.parametrize("hidden,inter", [(512, 256), (2048, 512)])
def test_normalised_rows_with_outliers(quant, tokens, hidden, inter):
    # norm weights of 2^24 on one channel in sixteen, where gate and up have zeros: the block's first launch writes the digits
    import torch
    import llmxabe_amd as X

    E = 4
    rng = np.random.default_rng(15)
    zero = np.zeros(hidden, bool)
    zero[9::16] = True
    st, host = _expert_stacks(X, rng, quant, E, hidden, inter, zero, None)
    q8 = X.ExpertQuant.Q8_0
    sh = [X.QuantTensor(X.synth_quant(q8, 70 + i, hidden * inter, 0.02), q8) for i in range(3)]
    norm = torch.where(torch.from_numpy(zero).cuda(), torch.tensor(2.0 ** 24, device="cuda"), torch.tensor(1.0, device="cuda"))
    x = torch.from_numpy(rng.standard_normal((tokens, hidden)).astype(np.float32)).cuda()
    router = X.synth_normal_f32(71, E * hidden, 0.02).view(E, hidden)
    router[:, torch.from_numpy(zero).cuda()] = 0.0
    w = X.MoeLayerWeights(norm, router.reshape(-1).contiguous(), None, *st, X.synth_normal_f32(72, hidden, 0.02), *sh)
    routed = []
    for fused in (True, False):
        blk = X.MoeBlock(X.MoeGeometry(E, 2, hidden, inter, 32, tokens))
        blk.set_fused_decode(fused)
        blk.forward(w, x, tokens, torch.zeros_like(x), torch.zeros_like(x))
        b = blk.buffers()
        ids, wts = (t.cpu().numpy().reshape(tokens, 2) for t in (b.topk_ids(), b.topk_weights()))
        normed = blk.normed().cpu().numpy().reshape(tokens, hidden).astype(np.float64)
        routed.append(blk.routed().cpu().numpy().reshape(tokens, hidden))
        ref = np.array([sum(wts[t, j] * _expert64(host, ids[t, j], normed[t]) for j in range(2)) for t in range(tokens)])
        err = np.abs(routed[-1] - ref).max() / np.abs(ref).max()
        print("norm", quant, tokens, hidden, fused, f"{err:.2e}")
        assert err <= 3 * TOL, (fused, err)
    assert np.array_equal(routed[0].view(np.uint32), routed[1].view(np.uint32))


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
@pytest.mark.parametrize("tokens", [1, 2, 4, 7])
def test_dense_rows_with_outliers(quant, tokens):
    # the norm launch of the dense block writes the digits; outliers in the normalised and in the intermediate rows
    import torch
    import llmxabe_amd as X

    H, I = 2560, 512
    rng = np.random.default_rng(16)
    zh, zi = np.zeros(H, bool), np.zeros(I, bool)
    zh[2::16], zi[11::16] = True, True
    d_rows = np.full(I, 2e-4 if quant == "Q8_0" else 6e-5)
    d_rows[zi] *= 1000
    st, host = _expert_stacks(X, rng, quant, 1, H, I, zh, zi, d_rows)
    norm = torch.where(torch.from_numpy(zh).cuda(), torch.tensor(2.0 ** 24, device="cuda"), torch.tensor(1.0, device="cuda"))
    x = torch.from_numpy(rng.standard_normal((tokens, H)).astype(np.float32)).cuda()
    blk = X.DenseFfnBlock(H, I, tokens)
    out, lout = torch.zeros_like(x), torch.zeros_like(x)
    blk.forward(X.DenseFfnLayerWeights(norm, *st), x, tokens, out, lout)
    normed = blk.normed().cpu().numpy().reshape(tokens, H).astype(np.float64)
    ref = np.array([_expert64(host, 0, normed[t]) for t in range(tokens)])
    err = np.abs(out.cpu().numpy() - ref).max() / np.abs(ref).max()
    print("dense", quant, tokens, f"{err:.2e}")
    assert err <= 3 * TOL, err


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
def test_infinities_and_nan_reach_the_outputs_as_in_plain_fp32(quant):
    # +-infinity by the sign of the product, NaN where it meets a zero code or another sign, everything else as it was
    import torch
    import llmxabe_amd as X

    V, K, tokens = 100, 2048, 3
    rng = np.random.default_rng(14)
    raw, w = _matrix(rng, quant, V, K)
    x = rng.standard_normal((tokens, K)).astype(np.float32)
    x[0, 100] = np.inf
    x[1, 700] = -np.inf
    x[1, 1900] = -np.inf
    x[2, 5] = np.nan
    dev = torch.from_numpy(raw).cuda()
    out = torch.zeros(tokens, V, device="cuda")
    X.LmHeadKernels(X.LmHeadGeometry(K, V, tokens)).forward(
        X.HeadTensor.q8_0(dev) if quant == "Q8_0" else X.HeadTensor.q6_k(dev), torch.from_numpy(x).cuda(), tokens, out)
    with np.errstate(invalid="ignore"):
        ref = np.stack([(w * x[t].astype(np.float64)).sum(1) for t in range(tokens)])
    got = out.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
    assert np.isinf(ref[0]).sum() > 50 and np.isinf(ref[1]).sum() > 20 and np.isnan(ref[2]).all()


@pytest.mark.parametrize("quant", ["Q8_0", "Q6_K"])
@pytest.mark.parametrize("tokens", [1, 3, 8])
def test_infinities_reach_the_gate_and_up_products(quant, tokens):
    # one activation of one token is infinite; gate's weight there is positive, so silu(g) is +infinity and the product has
    # the sign of up's weight (a NaN where that is zero); the other tokens' products are what they are without it
    import torch
    import llmxabe_amd as X

    H, I, col = 2560, 512, 1234
    rng = np.random.default_rng(17)
    make = _q8_0 if quant == "Q8_0" else _q6_k
    hi = 127 if quant == "Q8_0" else 31
    d = np.full(I, 2e-4 if quant == "Q8_0" else 6e-5)
    codes = [rng.integers(-hi, hi + 1, (I, H)).astype(np.int8) for _ in range(2)]
    codes[0][:, col] = 5
    codes[1][::7, col] = 0
    q = X.ExpertQuant.Q8_0 if quant == "Q8_0" else X.ExpertQuant.Q6K
    st = [X.QuantTensor(torch.from_numpy(make(c, d)[0]).cuda(), q) for c in codes]
    st.append(X.QuantTensor(torch.from_numpy(_matrix(rng, quant, H, I)[0]).cuda(), q))
    x = rng.standard_normal((tokens, H)).astype(np.float32)

    def products(rows, plain):
        k = X.MoeKernels(X.MoeGeometry(1, 1, H, I, 32, tokens))
        k.force_community(plain)
        b = k.shared_only_buffers(False)
        k.set_valid_tokens(b, tokens)
        out = torch.zeros(tokens * H, device="cuda")
        k.shared_expert(b, *st, torch.from_numpy(rows).cuda().view(-1), out)
        torch.cuda.synchronize()
        return b.shared_inter().cpu().numpy().reshape(tokens, I).copy()

    for plain in (False, True):
        finite = products(x, plain)
        y = x.copy()
        y[tokens - 1, col] = np.inf
        got, sign = products(y, plain), np.sign(codes[1][:, col].astype(int))
        assert np.array_equal(np.isposinf(got[-1]), sign > 0) and np.array_equal(np.isneginf(got[-1]), sign < 0)
        assert np.array_equal(np.isnan(got[-1]), sign == 0)
        assert np.array_equal(got[:-1].view(np.uint32), finite[:-1].view(np.uint32))
