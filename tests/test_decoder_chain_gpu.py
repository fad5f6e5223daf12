"""A decoder layer's attention and feed-forward block as one launch each (ttmi_decoder_attention, ttmi_decoder_feed_forward), against 64 bits.

Tolerance: x is O(1), and values are rounded to 16 bits at up to six places (the normalised row, Q, K, V, probabilities, context; or the normalised
and the intermediate row), each by at most half of eps of an O(1) value and passed on by products whose rows have norm one; the result itself, up to 8, by
eps / 2 of it.  Six halves of eps and the result's own stay within 8 eps.
fp32: an element of a product is rounded at most 64 + 16 times (a wavefront's share of 4096 products by fours, then the wavefronts'), each time by 2^-24 of a
partial sum below 4 (rows of norm one against O(1) values): 2^-15.6 for signs that all agree, and three products follow one another: 2^-14.
"""
import ctypes

import pytest
import torch

from helpers import TORCH_DTYPES, TTMI_DTYPES, ok, ptr, stream

pytestmark = pytest.mark.gpu
TOLERANCE = {"f16": 8 * 2.0 ** -11, "bf16": 8 * 2.0 ** -8, "f32": 2.0 ** -14}


class Exchange:
    def __init__(self, ttmi, rows, heads, hidden, inner, keys, dt):
        size = ctypes.c_int64()
        ok(ttmi.ttmi_decoder_chain_workspace(rows, heads, hidden, inner, keys, TTMI_DTYPES[dt], ctypes.addressof(size)))
        assert size.value > 0
        self.memory = torch.zeros(size.value, dtype=torch.uint8, device="cuda")
        ok(ttmi.ttmi_chain_prepare(ptr(self.memory), size.value, stream()))
        self.turn = 0

    def next(self):
        self.turn = 1 - self.turn
        return 1 - self.turn


class Attention:
    def __init__(self, dt, rows, heads, past, grows, masked=True, seed=0):
        gen = torch.Generator().manual_seed(seed)
        h = heads * 64
        self.dt, self.rows, self.heads, self.hidden, self.past, self.grows = dt, rows, heads, h, past, grows
        self.keys = past + 1 if grows else past
        self.width = 3 * h if grows else h
        rnd = lambda *shape: torch.randn(shape, generator=gen)
        to = lambda t: t.to(TORCH_DTYPES[dt]).cuda()
        self.x, self.gamma, self.beta = to(rnd(rows, h)), to(1 + rnd(h) * 0.1), to(rnd(h) * 0.1)
        self.w_in, self.b_in, self.w_out, self.b_out = to(rnd(self.width, h) / h ** 0.5), to(rnd(self.width) * 0.1), to(rnd(h, h) / h ** 0.5), to(rnd(h) * 0.1)
        self.k_past, self.v_past = to(rnd(rows, heads, past, 64)), to(rnd(rows, heads, past, 64))
        self.mask = None
        if masked:
            self.mask = torch.zeros(rows, self.keys)
            self.mask[-1, :self.keys // 2] = -1e18
            self.mask = self.mask.cuda()

    def exchange(self, ttmi):
        return Exchange(ttmi, self.rows, self.heads, self.hidden, self.width, self.keys, self.dt)

    def outputs(self):
        made = lambda *shape: torch.full(shape, 7.0, dtype=TORCH_DTYPES[self.dt], device="cuda")
        grown = [made(self.rows, self.heads, self.keys, 64) for _ in range(2)] if self.grows else [None, None]
        return [made(self.rows, self.hidden), made(self.rows, self.heads, self.keys)] + grown

    def call(self, ttmi, outputs, exchange, turn, workgroups=0, patience=0, x=None):
        out, probs, k_out, v_out = outputs
        ok(ttmi.ttmi_decoder_attention(ptr(self.x if x is None else x), ptr(self.gamma), ptr(self.beta), 1e-6, ptr(self.w_in), ptr(self.b_in), ptr(self.w_out),
                                       ptr(self.b_out), ptr(self.k_past), ptr(self.v_past), ptr(k_out), ptr(v_out), ptr(self.mask), ptr(probs), ptr(out),
                                       ptr(exchange.memory), turn, self.rows, self.heads, self.hidden, self.keys, 0.125, TTMI_DTYPES[self.dt], workgroups,
                                       patience, stream()))

    def run(self, ttmi, exchange, workgroups=0, patience=0):
        outputs = self.outputs()
        self.call(ttmi, outputs, exchange, exchange.next(), workgroups, patience)
        torch.cuda.synchronize()
        return [o for o in outputs if o is not None]

    def exact(self):
        d = lambda t: t.double().cpu()
        h = self.hidden
        y = torch.nn.functional.layer_norm(d(self.x), (h,), d(self.gamma), d(self.beta), 1e-6) @ d(self.w_in).T + d(self.b_in)
        y = y.view(self.rows, -1, self.heads, 1, 64)
        k, v = d(self.k_past), d(self.v_past)
        if self.grows:
            k, v = torch.cat([k, y[:, 1]], 2), torch.cat([v, y[:, 2]], 2)
        scores = (y[:, 0] @ k.transpose(-1, -2))[:, :, 0] / 8
        if self.mask is not None:
            scores = scores + d(self.mask)[:, None]
        probs = scores.softmax(-1)
        out = d(self.x) + (probs[:, :, None] @ v).reshape(self.rows, h) @ d(self.w_out).T + d(self.b_out)
        return [out, probs] + ([k, v] if self.grows else [])


# one row, a full block; keys around the 64 of a wavefront, the fewest and the most; heads at both ends
@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("grows", [True, False])
@pytest.mark.parametrize("rows,heads,past", [(1, 12, 1), (8, 12, 40), (8, 12, 63), (16, 12, 64), (3, 16, 128), (5, 1, 200), (16, 16, 300), (2, 4, 511)])
def test_attention_as_one_launch(ttmi, dt, grows, rows, heads, past):
    case = Attention(dt, rows, heads, past, grows, masked=past > 1)
    exchange = case.exchange(ttmi)
    want = case.exact()
    first = case.run(ttmi, exchange)
    for got, exact in zip(first, want):
        assert (got.double().cpu() - exact).abs().max().item() <= TOLERANCE[dt]
    if grows:
        assert torch.equal(first[2][:, :, :past], case.k_past) and torch.equal(first[3][:, :, :past], case.v_past)
    for _ in range(3):  # the parts of the exchange memory take turns
        assert all(torch.equal(a, b) for a, b in zip(case.run(ttmi, exchange), first))


@pytest.mark.parametrize("grows", [True, False])
@pytest.mark.parametrize("dt,past", [("f16", 40), ("f16", 150), ("f32", 40), ("f32", 300)])
def test_any_number_of_workgroups_gives_the_same_bits(ttmi, grows, dt, past):
    """One workgroup does everything itself; few of them, with no patience, compute what they miss."""
    case = Attention(dt, 8, 12, past, grows)
    exchange = case.exchange(ttmi)
    want = case.run(ttmi, exchange)
    for workgroups, patience in [(1, 0), (7, 1), (100, 1), (0, 1)]:
        assert all(torch.equal(a, b) for a, b in zip(case.run(ttmi, exchange, workgroups, patience), want)), (workgroups, patience)


def _feed_forward(dt, rows, hidden, inner):
    gen = torch.Generator().manual_seed(rows)
    rnd = lambda *shape: torch.randn(shape, generator=gen)
    parts = [rnd(rows, hidden), 1 + rnd(hidden) * 0.1, rnd(hidden) * 0.1, rnd(inner, hidden) / hidden ** 0.5, rnd(inner) * 0.1, rnd(hidden, inner) / inner ** 0.5,
             rnd(hidden) * 0.1]
    return [t.to(TORCH_DTYPES[dt]).cuda() for t in parts]


def _run_feed_forward(ttmi, dt, parts, exchange, turn, workgroups=0, patience=0):
    x, gamma, beta, w1, b1, w2, b2 = parts
    out = torch.full_like(x, 7.0)
    ok(ttmi.ttmi_decoder_feed_forward(ptr(x), ptr(gamma), ptr(beta), 1e-12, ptr(w1), ptr(b1), ptr(w2), ptr(b2), ptr(out), ptr(exchange.memory), turn, x.shape[0],
                                      x.shape[1], w1.shape[0], TTMI_DTYPES[dt], workgroups, patience, stream()))
    return out


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("rows,hidden,inner", [(1, 768, 3072), (8, 768, 3072), (16, 1024, 4096), (16, 64, 64), (7, 320, 1088)])
def test_feed_forward_as_one_launch(ttmi, dt, rows, hidden, inner):
    inner = min(inner, 3072) if dt == "f32" else inner
    parts = _feed_forward(dt, rows, hidden, inner)
    exchange = Exchange(ttmi, rows, 0, hidden, inner, 0, dt)
    x, gamma, beta, w1, b1, w2, b2 = (t.double().cpu() for t in parts)
    want = x + (torch.nn.functional.layer_norm(x, (hidden,), gamma, beta, 1e-12) @ w1.T + b1).relu() @ w2.T + b2
    first = _run_feed_forward(ttmi, dt, parts, exchange, exchange.next())
    assert (first.double().cpu() - want).abs().max().item() <= TOLERANCE[dt]
    for workgroups, patience in [(0, 0), (1, 0), (5, 1), (0, 1)]:
        assert torch.equal(_run_feed_forward(ttmi, dt, parts, exchange, exchange.next(), workgroups, patience), first)


def test_replayed_from_a_graph(ttmi):
    """Three calls a graph, an odd number, and calls of its owner between the replays."""
    case = Attention("f16", 8, 12, 40, True)
    exchange = case.exchange(ttmi)
    other = Attention("f16", 8, 12, 40, True, seed=1).x
    want = case.run(ttmi, exchange)
    given, outputs = case.x.clone(), [case.outputs() for _ in range(3)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for o in outputs:
            case.call(ttmi, o, exchange, 2, x=given)
    for turn in range(5):
        given.copy_(case.x if turn % 2 == 0 else other)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for o in outputs for a, b in zip(o, outputs[0]))
        assert torch.equal(outputs[0][0], want[0]) == (turn % 2 == 0)
        assert all(torch.equal(a, b) for a, b in zip(case.run(ttmi, exchange), want))


def test_what_is_not_built_has_no_workspace(ttmi):
    size = ctypes.c_int64(7)
    for args in [(17, 12, 768, 768, 40, "f16"), (8, 12, 768, 768, 513, "f16"), (8, 17, 1088, 1088, 40, "f16"),
                 (8, 12, 768, 1536, 40, "f16"), (8, 0, 768, 4160, 0, "f16"), (8, 0, 800, 3072, 0, "f16"), (8, 0, 1088, 3072, 0, "f16"), (8, 0, 768, 3136, 0, "f32")]:
        ok(ttmi.ttmi_decoder_chain_workspace(*args[:5], TTMI_DTYPES[args[5]], ctypes.addressof(size)))
        assert size.value == 0, args


def _layer(seed=0, hidden=768, inner=3072):
    import turbo_transformers as tt
    from test_model_gpu import _OnmtLikeFfn

    torch.manual_seed(seed)
    return tt.PositionwiseFeedForward.from_onmt(_OnmtLikeFfn(hidden, inner).cuda().half())


def _recorded(side, call):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
    return graph, out


@pytest.mark.parametrize("rows", [1, 8, 16])
def test_recorded_calls_of_a_layer_are_replayed_in_any_order(rows):
    """Graphs of one and of two calls of one layer, between its own calls: each launch finds the part of the exchange memory whose turn it is."""
    layer = _layer()
    gen = torch.Generator().manual_seed(rows)
    xs = [torch.randn(rows, 1, 768, generator=gen).half().cuda() for _ in range(3)]
    want = [layer(x).clone() for x in xs]
    twice = layer(layer(xs[2])).clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        kept = [layer(xs[0]) for _ in range(8)]  # (results that the recorded calls find room in)
    side.synchronize()
    del kept
    one, out_one = _recorded(side, lambda: layer(xs[0]))
    other, out_other = _recorded(side, lambda: layer(xs[1]))
    two, out_two = _recorded(side, lambda: layer(layer(xs[2])))
    for order in ("1", "22", "121", "2", "3", "1331", "23", "3221", "111"):
        for o in (out_one, out_other, out_two):
            o.fill_(7.0)
        for kind in order:
            {"1": one, "2": other, "3": two}[kind].replay()
        torch.cuda.synchronize()
        for kind, out, exact in (("1", out_one, want[0]), ("2", out_other, want[1]), ("3", out_two, twice)):
            assert kind not in order or torch.equal(out, exact), order
        assert torch.equal(layer(xs[1]), want[1])


def test_a_call_that_is_recorded_before_any_is_made():
    """The exchange memory, where another layer's was before, is prepared by the graph itself."""
    given_back = _layer(1)
    x = torch.randn(8, 1, 768, generator=torch.Generator().manual_seed(5)).half().cuda()
    given_back(x)
    layer = _layer(2)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        layer(torch.randn(20, 1, 768, device="cuda").half())  # two launches: lays the weights out
        kept = [given_back(x) for _ in range(4)]
        side.synchronize()
    del given_back, kept
    graph, out = _recorded(side, lambda: layer(x))
    other, out_other = _recorded(side, lambda: layer(x))
    seen = []
    for g, o in ((graph, out), (graph, out), (other, out_other), (graph, out), (other, out_other)):
        o.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        seen.append(o.clone())
    want = layer(x)
    assert all(torch.equal(o, want) for o in seen)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(layer(x), want)
