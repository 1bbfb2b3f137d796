"""The shared expert's tiles in the launches of the routed ones (narrow tiles, an expert's share of at most 32 rows): the rows are those
of the separate calls, bit for bit."""
import pytest

from util import activations, make_layer

pytestmark = pytest.mark.gpu


# items of less than a round, of two to three (256 experts, 512 tokens) and of more (512 experts); a last tile of one and of 63
# rows; fewer live tokens than the buffers hold; the widest that goes along and, one token on, the narrowest that does not
@pytest.mark.parametrize("experts,top_k,hidden,inter,size,live", [
    (128, 2, 512, 256, 64, 64), (128, 2, 256, 512, 65, 65), (128, 2, 512, 256, 320, 1), (128, 8, 512, 512, 512, 127),
    (128, 8, 512, 256, 513, 512), (128, 8, 512, 256, 513, 513), (256, 8, 2048, 512, 512, 512), (512, 8, 512, 512, 1000, 1000)])
@pytest.mark.parametrize("routed_q,down_q,shared_q,shared_down_q", [
    ("Q6K", "Q6K", "Q8_0", "Q8_0"), ("Q6K", "Q8_0", "Q8_0", "Q6K"), ("Q8_0", "Q6K", "Q6K", "Q6K"), ("Q8_0", "Q8_0", "Q6K", "Q8_0")])
def test_rows_are_those_of_the_separate_calls(oracle, experts, top_k, hidden, inter, size, live, routed_q, down_q, shared_q, shared_down_q):
    import torch

    import llmxabe_amd as X

    q = lambda name: getattr(X.ExpertQuant, name)
    g = X.MoeGeometry(experts, top_k, hidden, inter, X.moe_block_size(size), size)
    w = make_layer(oracle, g, seed=60, expert_quant=q(routed_q), down_quant=q(down_q), shared_quant=q(shared_q),
                   shared_down_quant=q(shared_down_q)).dev
    x, other = activations(61, size, hidden), activations(62, size, hidden)
    blk = X.MoeBlock(g)
    ffn_out, l_out = torch.zeros_like(x), torch.zeros_like(x)
    for rows in (other, x):   # (the second pass finds another's rows in the buffers)
        blk.buffers().partial().fill_(float("nan"))
        blk.forward(w, rows, live, ffn_out, l_out)
    k = X.MoeKernels(g)
    b = k.buffers()
    k.set_valid_tokens(b, live)
    k.route_and_dispatch(b, blk.router_logits())
    k.grouped_forward_partial(b, w.gate_exps, w.up_exps, w.down_exps, blk.normed())
    shared = torch.zeros(size * hidden, device="cuda")
    k.shared_expert_mma(b, w.shared_gate, w.shared_up, w.shared_down, blk.normed(), shared)
    torch.cuda.synchronize()
    n = live * hidden
    assert torch.equal(blk.buffers().topk_ids()[:live * top_k], b.topk_ids()[:live * top_k])
    for got, want in ((blk.buffers().partial()[:n * top_k], b.partial()[:n * top_k]), (blk.shared_ungated()[:n], shared[:n])):
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)) and bool(want.isfinite().all())


def _small(X, oracle, buffers):
    g = X.MoeGeometry(128, 8, 512, 256, X.moe_block_size(buffers), buffers)
    return X.MoeBlock(g), make_layer(oracle, g, seed=70).dev, [activations(71 + i, buffers, 512) for i in range(2)]


def _bits(t):
    import torch

    return t.view(torch.int32)


# along with the routed tiles and, one token on, on a stream beside them: passes back to back on one block, alternating two inputs,
# eagerly and as a graph replayed with eager passes right before and behind it
@pytest.mark.parametrize("tokens", [512, 513])
def test_passes_back_to_back_on_either_side_of_the_rule(oracle, tokens):
    import torch

    import llmxabe_amd as X

    blk, w, xs = _small(X, oracle, tokens)
    blk.publish_tokens(tokens)
    out = lambda: [torch.full_like(xs[0], float("nan")) for _ in range(4)]
    want, got, before, behind = out(), out(), out(), out()

    def both(to):
        for i in range(2):
            blk.forward(w, xs[i], tokens, to[2 * i], to[2 * i + 1])

    shared = []
    for i in range(2):
        blk.forward(w, xs[i], tokens, want[2 * i], want[2 * i + 1])
        torch.cuda.synchronize()
        shared.append(blk.shared_ungated().clone())
    assert not torch.equal(want[0], want[2])
    same = lambda to: all(torch.equal(_bits(a), _bits(b)) for a, b in zip(to, want))
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        both(got)
        stream.synchronize()
        assert same(got)
        with torch.cuda.graph(graph, stream=stream):
            both(got)
        for _ in range(3):
            for t in got + before + behind:
                t.fill_(float("nan"))
            both(before)
            graph.replay()
            both(behind)
            stream.synchronize()
            assert same(before) and same(got) and same(behind)
            assert torch.equal(_bits(blk.shared_ungated()), _bits(shared[1]))


def test_live_counts_on_either_side_of_the_rule_in_turn(oracle):
    """One handle whose passes go along and fork in turn, without a drain between them: each gives the bits of the pass alone."""
    import torch

    import llmxabe_amd as X

    blk, w, xs = _small(X, oracle, 513)
    counts = (512, 513, 64, 513, 300, 513, 512)
    run = lambda x, n, to: blk.forward(w, x, n, to[0], to[1])
    out = lambda: [torch.full_like(xs[0], float("nan")) for _ in range(2)]
    want = []
    for i, n in enumerate(counts):
        want.append(out())
        run(xs[i % 2], n, want[-1])
        torch.cuda.synchronize()
    got = [out() for _ in counts]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for i, n in enumerate(counts):
            run(xs[i % 2], n, got[i])
        stream.synchronize()
    for n, a, b in zip(counts, got, want):
        for t, u in zip(a, b):
            assert torch.equal(_bits(t[:n]), _bits(u[:n])) and bool(t[:n].isfinite().all()) and bool(t[n:].isnan().all())


@pytest.mark.parametrize("captured,later", [(100, 513), (513, 100), (300, 512)])
def test_a_pass_captured_at_one_count_serves_another_published_later(oracle, captured, later):
    """The item counts come from the device: a graph of a pass that goes along (or forks) is replayed after a count on the rule's
    other side, or a larger one on the same, was published, and gives the bits of the eager pass of that count."""
    import torch

    import llmxabe_amd as X

    blk, w, xs = _small(X, oracle, 513)
    out = lambda: [torch.full_like(xs[0], float("nan")) for _ in range(2)]
    want = {}
    for n in (captured, later):
        want[n] = out()
        blk.forward(w, xs[0], n, want[n][0], want[n][1])
        torch.cuda.synchronize()
    got, eager = out(), out()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        blk.publish_tokens(captured)
        blk.forward(w, xs[0], captured, got[0], got[1])
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            blk.forward(w, xs[0], captured, got[0], got[1])
        for n in (captured, later, captured, later):
            for t in got + eager:
                t.fill_(float("nan"))
            blk.forward(w, xs[1], n, eager[0], eager[1])   # (publishes n)
            graph.replay()
            stream.synchronize()
            for t, u in zip(got, want[n]):
                assert torch.equal(_bits(t[:n]), _bits(u[:n])) and bool(t[:n].isfinite().all()) and bool(t[n:].isnan().all())
