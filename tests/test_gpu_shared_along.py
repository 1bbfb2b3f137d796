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
    x = activations(61, size, hidden)
    blk = X.MoeBlock(g)
    ffn_out, l_out = torch.zeros_like(x), torch.zeros_like(x)
    for _ in range(2):   # (the second pass finds the first's rows in the buffers)
        blk.buffers().partial().fill_(float("nan"))
        blk.forward(w, x, live, ffn_out, l_out)
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


# along with the routed tiles and, one token on, on a stream beside them: passes back to back on one block, alternating two inputs,
# eagerly and as a graph replayed with eager passes between the replays
@pytest.mark.parametrize("tokens", [512, 513])
def test_passes_back_to_back_on_either_side_of_the_rule(oracle, tokens):
    import torch

    import llmxabe_amd as X

    g = X.MoeGeometry(128, 8, 512, 256, X.moe_block_size(tokens), tokens)
    w = make_layer(oracle, g, seed=70).dev
    xs = [activations(71 + i, tokens, 512) for i in range(2)]
    blk = X.MoeBlock(g)
    blk.publish_tokens(tokens)
    out = lambda: [torch.zeros_like(xs[0]) for _ in range(4)]
    want, got = out(), out()

    def both(to):
        for i in range(2):
            blk.forward(w, xs[i], tokens, to[2 * i], to[2 * i + 1])

    for i in range(2):
        blk.forward(w, xs[i], tokens, want[2 * i], want[2 * i + 1])
        torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        both(got)
        stream.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        with torch.cuda.graph(graph, stream=stream):
            both(got)
        for _ in range(3):
            for t in got:
                t.zero_()
            graph.replay()
            blk.forward(w, xs[0], tokens, torch.zeros_like(xs[0]), torch.zeros_like(xs[0]))
            stream.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want))
