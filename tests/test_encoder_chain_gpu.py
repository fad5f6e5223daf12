"""A stack of encoder layers over a few rows as one launch (ttmi_encoder_chain), against the same layers in 64 bits.

Tolerance: a layer rounds its values to 16 bits at eight places (the row, Q, K, V, probabilities, context, the second row, the intermediate
one), each by at most eps / 2 of an O(1) value, and every one reaches the output through a LayerNorm whose gain here is at most 2: sixteen halves of
eps per layer and O(1) value, of which the largest of some thousand is within 4.
"""
import ctypes

import pytest
import torch

from helpers import TORCH_DTYPES, TTMI_DTYPES, ok, ptr, stream

pytestmark = pytest.mark.gpu
EPS = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


class Stack:
    def __init__(self, dt, layers, heads, ffn, seed=0):
        gen = torch.Generator().manual_seed(seed)
        self.dt, self.layers, self.heads, self.hidden, self.ffn = dt, layers, heads, heads * 64, ffn
        h = self.hidden
        rnd = lambda *shape: torch.randn(shape, generator=gen)
        self.weights, self.space, self.turn = [], None, 1
        for _ in range(layers):
            w = [rnd(3 * h, h) / h ** 0.5, rnd(3 * h) * 0.1, rnd(h, h) / h ** 0.5, rnd(h) * 0.1, 1 + rnd(h) * 0.1, rnd(h) * 0.1,
                 rnd(ffn, h) / h ** 0.5, rnd(ffn) * 0.1, rnd(h, ffn) / ffn ** 0.5, rnd(h) * 0.1, 1 + rnd(h) * 0.1, rnd(h) * 0.1]
            self.weights.append([t.to(TORCH_DTYPES[dt]).cuda() for t in w])

    def input(self, batch, seq, seed):
        return torch.randn((batch, seq, self.hidden), generator=torch.Generator().manual_seed(seed)).to(TORCH_DTYPES[self.dt]).cuda()

    def exchange(self, ttmi):
        """The memory of calls of any number of rows, which take turns."""
        size = ctypes.c_int64()
        ok(ttmi.ttmi_encoder_chain_workspace(self.layers, 1, self.heads, self.hidden, self.ffn, TTMI_DTYPES[self.dt], ctypes.addressof(size)))
        assert size.value > 0
        if self.space is None:
            self.space = torch.zeros(size.value, dtype=torch.uint8, device="cuda")
            ok(ttmi.ttmi_chain_prepare(ptr(self.space), size.value, stream()))
        self.turn = 1 - self.turn
        return self.space

    def run(self, ttmi, x, mask=None, workgroups=0, patience=0):
        batch, seq, h = x.shape
        space, out = self.exchange(ttmi), torch.empty_like(x)
        out32 = torch.empty(x.shape, device="cuda") if self.dt == "bf16" else None
        pointers = (ctypes.c_void_p * (12 * self.layers))(*[w.data_ptr() for l in self.weights for w in l])
        ok(ttmi.ttmi_encoder_chain(ctypes.addressof(pointers), ptr(x), None, ptr(mask), ptr(out), ptr(out32), ptr(space), self.turn, self.layers, batch, seq,
                                   self.heads, h, self.ffn, 1e-12, TTMI_DTYPES[self.dt], workgroups, patience, stream()))
        torch.cuda.synchronize()
        if out32 is not None:
            assert torch.equal(out, out32.to(out.dtype)) or not torch.isfinite(out).all()
        return out

    def exact(self, x, mask=None):
        x = x.double().cpu()
        batch, seq, h = x.shape
        norm = lambda y, g, b: torch.nn.functional.layer_norm(y, (h,), g, b, 1e-12)
        for layer in self.weights:
            qkv_w, qkv_b, o_w, o_b, g1, b1, w1, c1, w2, c2, g2, b2 = (w.double().cpu() for w in layer)
            q, k, v = (x @ qkv_w.T + qkv_b).view(batch, seq, 3, self.heads, 64).permute(2, 0, 3, 1, 4)
            scores = q @ k.transpose(-1, -2) / 8
            if mask is not None:
                scores = scores + mask.double().cpu()[:, None, None, :]
            ctx = (scores.softmax(-1) @ v).permute(0, 2, 1, 3).reshape(batch, seq, h)
            x = norm(x + ctx @ o_w.T + o_b, g1, b1)
            y = torch.nn.functional.gelu(x @ w1.T + c1, approximate="tanh")
            x = norm(x + y @ w2.T + c2, g2, b2)
        return x


# one row, a row short of a block, full blocks, sequences that share it; heads and widths at both
# ends of the range, an intermediate row that the wavefronts share unevenly
SHAPES = [(1, 1), (1, 10), (1, 16), (4, 4), (16, 1), (3, 5), (1, 15)]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("layers,heads,ffn", [(2, 12, 3072), (2, 16, 4096), (1, 4, 256), (3, 5, 1088)])
def test_a_stack_as_one_launch(ttmi, dt, layers, heads, ffn):
    stack = Stack(dt, layers, heads, ffn)
    for batch, seq in SHAPES:
        x = stack.input(batch, seq, batch * 100 + seq)
        mask = None
        if seq > 2:
            mask = torch.zeros((batch, seq))
            mask[-1, seq // 2:] = -10000.0
            mask = mask.cuda()
        error = (stack.run(ttmi, x, mask).double().cpu() - stack.exact(x, mask)).abs().max().item()
        assert error <= 4 * 8 * EPS[dt] * layers, (batch, seq, error)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("batch,seq", [(1, 10), (2, 8)])
def test_any_number_of_workgroups_gives_the_same_bits(ttmi, dt, batch, seq):
    """One workgroup does everything itself; few of them, with no patience, compute what they miss."""
    stack = Stack(dt, 2, 12, 3072)
    x = stack.input(batch, seq, 5)
    want = stack.run(ttmi, x)
    for workgroups, patience in [(1, 0), (7, 1), (100, 1), (0, 1)]:
        assert torch.equal(stack.run(ttmi, x, None, workgroups, patience), want), (workgroups, patience)


@pytest.mark.parametrize("batch,seq", [(3, 5), (2, 8)])
def test_what_is_not_finite_stays_in_its_sequence(ttmi, batch, seq):
    """Among it the NaN that marks a word nobody has written."""
    stack = Stack("f16", 2, 12, 3072)
    x = stack.input(batch, seq, 9)
    want = stack.run(ttmi, x)
    bad = x.clone()
    bad[1].view(torch.int16)[:] = -1
    got = stack.run(ttmi, bad)
    assert torch.isnan(got[1]).all()
    bad[1] = float("inf")
    assert torch.isnan(stack.run(ttmi, bad)[1]).all()
    for b in (b for b in range(batch) if b != 1):
        assert torch.equal(got[b], want[b])
    masked = torch.zeros((batch, seq), device="cuda")
    masked[0] = torch.finfo(torch.float32).min  # a wholly masked sequence is the mean of its values, as a softmax has it
    assert torch.isfinite(stack.run(ttmi, x, masked)).all()


def test_replayed_from_a_graph(ttmi):
    """An odd number of calls, and calls of the owner of the exchange memory between the replays."""
    stack = Stack("f16", 2, 12, 3072)
    x, other = stack.input(1, 10, 3), stack.input(1, 10, 4)
    want = [stack.run(ttmi, x), stack.run(ttmi, other)]
    out, space, given = torch.empty_like(x), stack.space, x.clone()
    pointers = (ctypes.c_void_p * 24)(*[w.data_ptr() for l in stack.weights for w in l])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ok(ttmi.ttmi_encoder_chain(ctypes.addressof(pointers), ptr(given), None, None, ptr(out), None, ptr(space), 2, 2, 1, 10, 12, 768, 3072, 1e-12,
                                   TTMI_DTYPES["f16"], 0, 0, stream()))
    for turn in range(6):
        given.copy_([x, other][turn % 2])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[turn % 2]), turn
        assert torch.equal(stack.run(ttmi, other), want[1])


def test_what_is_not_built_has_no_workspace(ttmi):
    size = ctypes.c_int64(7)
    for args in [(2, 17, 12, 768, 3072, "f16"), (25, 8, 12, 768, 3072, "f16"), (2, 8, 12, 768, 3072, "f32"), (2, 8, 17, 1088, 3072, "f16"),
                 (2, 8, 3, 192, 768, "f16"), (2, 8, 12, 1536, 3072, "f16"), (2, 8, 12, 768, 3104, "f16"), (2, 8, 12, 768, 4160, "f16")]:
        ok(ttmi.ttmi_encoder_chain_workspace(*args[:5], TTMI_DTYPES[args[5]], ctypes.addressof(size)))
        assert size.value == 0, args


def test_a_recorded_stack_leaves_another_number_of_its_layers_alone():
    """Two stacks with the same first layer have exchange memory of two sizes: replays of the one between calls of the other."""
    import turbo_transformers as tt
    from test_model_gpu import _hf_bert

    model, cfg = _hf_bert(3, seed=11)
    encoder = tt.BertModel.from_torch(model.half(), torch.device("cuda:0"), "turbo").bertmodel_nopooler.encoder
    gen = torch.Generator().manual_seed(2)
    long, short = [torch.randn(1, 10, cfg.hidden_size, generator=gen).half().cuda() for _ in range(2)]
    layers = list(encoder.layer)

    def run(count, x):
        encoder.layer = layers[:count]
        return encoder(x)[0]

    want = [run(3, long).clone(), run(2, short).clone()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run(2, short)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        captured = run(2, short)
    for _ in range(4):
        assert torch.equal(run(3, long), want[0])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, want[1])


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("layers,heads,ffn", [(2, 12, 768), (1, 16, 1024)])
def test_a_stack_whose_inner_rows_are_as_wide_as_the_hidden_ones(ttmi, dt, layers, heads, ffn):
    """The narrowest that are run as one launch."""
    test_a_stack_as_one_launch(ttmi, dt, layers, heads, ffn)


class ResidualStack(Stack):
    """bf16, with the input before it was rounded, and the result before it is."""

    def __init__(self, layers, heads, ffn):
        super().__init__("bf16", layers, heads, ffn)

    def run(self, ttmi, x, x32):
        batch, seq, h = x.shape
        space, out, self.out32 = self.exchange(ttmi), torch.empty_like(x), torch.empty(x.shape, device="cuda")
        pointers = (ctypes.c_void_p * (12 * self.layers))(*[w.data_ptr() for l in self.weights for w in l])
        ok(ttmi.ttmi_encoder_chain(ctypes.addressof(pointers), ptr(x), ptr(x32), None, ptr(out), ptr(self.out32), ptr(space), self.turn, self.layers, batch, seq,
                                   self.heads, h, self.ffn, 1e-12, TTMI_DTYPES[self.dt], 0, 0, stream()))
        torch.cuda.synchronize()
        return out

    def exact(self, x, residual, stored=lambda r: r):
        """residual: what the first one is taken from; stored: what becomes of each of them before it is added."""
        x, residual = x.double().cpu(), residual.double().cpu()
        batch, seq, h = x.shape
        norm = lambda y, g, b: torch.nn.functional.layer_norm(y, (h,), g, b, 1e-12)
        for layer in self.weights:
            qkv_w, qkv_b, o_w, o_b, g1, b1, w1, c1, w2, c2, g2, b2 = [t.double().cpu() for t in layer]
            q, k, v = (t.reshape(batch, seq, self.heads, 64).permute(0, 2, 1, 3) for t in (x @ qkv_w.T + qkv_b).split(h, dim=-1))
            ctx = ((q @ k.transpose(-1, -2) / 8).softmax(-1) @ v).permute(0, 2, 1, 3).reshape(batch, seq, h)
            x = norm(stored(residual) + ctx @ o_w.T + o_b, g1, b1)
            y = torch.nn.functional.gelu(x @ w1.T + c1, approximate="tanh")
            residual = x = norm(stored(x) + y @ w2.T + c2, g2, b2)
        return x


@pytest.mark.parametrize("layers,heads,ffn", [(1, 12, 3072), (3, 12, 3072), (2, 16, 4096), (2, 5, 1088)])
@pytest.mark.parametrize("batch,seq", [(1, 1), (3, 5), (1, 16)])
@pytest.mark.parametrize("given", [True, False])
def test_the_residual_of_bf16_stays_in_fp32(ttmi, layers, heads, ffn, batch, seq, given):
    """From the input before it was rounded (where it is given) to the unrounded result.  What is added to a residual is small here, so that its eight
    roundings to 16 bits per layer, of at most 2^-8 / 2 of an O(1) value each and a 32nd of that behind the projection, stay below a quarter of one rounding of
    the residual itself: rms 2^-8 / 2 / sqrt(3) / 32 * sqrt(8) = 1.0e-4 per layer, and twice that is allowed.  The test shows that it would see a rounded one."""
    stack = ResidualStack(layers, heads, ffn)
    for layer in stack.weights:
        for w in (layer[2], layer[3], layer[8], layer[9]):
            w.mul_(1.0 / 32)  # (exact)
    x32 = torch.randn((batch, seq, stack.hidden), generator=torch.Generator().manual_seed(seq)).cuda()
    x = x32.bfloat16()
    out = stack.run(ttmi, x, x32=x32 if given else None)
    want = stack.exact(x, residual=x32 if given else x)
    rms = lambda t: t.double().cpu().pow(2).mean().sqrt().item()
    bound = 2 * layers * 2.0 ** -8 / 2 / 3 ** 0.5 / 32 * 8 ** 0.5
    rounded = stack.exact(x, residual=x32 if given else x, stored=lambda r: r.float().bfloat16().double())
    assert rms(rounded - want) > 1.5 * bound
    assert rms(stack.out32.double().cpu() - want) <= bound
    assert torch.equal(out, stack.out32.bfloat16())


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("inner", [256, 704])
def test_layers_with_inner_rows_narrower_than_the_hidden_ones(dt, inner):
    """Few rows through layers that are not run as one launch: the layers in fp32 on what is stored.  A layer rounds as in a stack as one launch, to two
    such tolerances (two layers)."""
    import turbo_transformers as tt
    from test_model_gpu import _hf_bert

    model, cfg = _hf_bert(2, seed=3, intermediate_size=inner)
    model = model.to(TORCH_DTYPES[dt])
    encoder = tt.BertEncoder.from_torch(model.encoder)
    x = torch.randn(2, 5, cfg.hidden_size, generator=torch.Generator().manual_seed(4)).to(TORCH_DTYPES[dt]).cuda()
    got = encoder(x)[0]
    with torch.no_grad():
        want = model.float().cpu().double().encoder(x.double().cpu(), attention_mask=None)[0]
    assert (got.double().cpu() - want).abs().max().item() <= 2 * 4 * 8 * EPS[dt]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
def test_recorded_stacks_are_replayed_in_any_order(dt):
    """One call of three layers and three of one layer each, recorded, between calls of their owner."""
    import turbo_transformers as tt
    from test_model_gpu import _hf_bert

    model, cfg = _hf_bert(3, seed=12)
    encoder = tt.BertEncoder.from_torch(model.to(TORCH_DTYPES[dt]).encoder)
    gen = torch.Generator().manual_seed(6)
    x, y = [torch.randn(1, 10, cfg.hidden_size, generator=gen).to(TORCH_DTYPES[dt]).cuda() for _ in range(2)]
    want = [encoder(x)[0].clone(), encoder(y)[0].clone()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        kept = [(encoder(x), encoder(x, output_hidden_states=True)) for _ in range(4)]  # (results that the recorded calls find room in)
    side.synchronize()
    del kept
    graphs = []
    for call in (lambda: encoder(x)[0], lambda: encoder(y, output_hidden_states=True)[0]):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = call()
        graphs.append((graph, out))
    for order in ((0, ), (1, ), (0, 1, 1), (1, 0), (0, 0, 0), (1, 1)):
        for k in order:
            graphs[k][1].fill_(7.0)
            graphs[k][0].replay()
        torch.cuda.synchronize()
        assert all(torch.equal(graphs[k][1], want[k]) for k in order), order
        assert torch.equal(encoder(y)[0], want[1]) and torch.equal(encoder(x, output_hidden_states=True)[0], want[0])


@pytest.mark.parametrize("dt,layers,heads,ffn", [("f16", 12, 12, 3072), ("bf16", 12, 12, 3072), ("bf16", 24, 16, 4096), ("f16", 24, 16, 4096)])
@pytest.mark.parametrize("batch,seq", [(1, 1), (1, 10), (3, 5), (2, 8)])
def test_whole_models_of_a_few_rows(dt, layers, heads, ffn, batch, seq):
    """BertModel with a padding mask, weights as the published models start from (N(0, 0.02)) with every bias and LayerNorm parameter perturbed, against the model in
    64 bits on what is stored.  Each layer rounds its values at eight places to half of eps at most, of O(1) values, independently, and the LayerNorms pass that on
    at a gain of about one: sqrt(8 * layers) eps / 2 / sqrt(3) rms."""
    import turbo_transformers as tt
    from test_model_gpu import _hf_bert

    model, cfg = _hf_bert(layers, seed=layers, hidden_size=heads * 64, num_attention_heads=heads, intermediate_size=ffn, vocab_size=500)
    model = model.to(TORCH_DTYPES[dt])
    ids = torch.randint(0, cfg.vocab_size, (batch, seq), generator=torch.Generator().manual_seed(seq)).cuda()
    keep = torch.ones(batch, seq, dtype=torch.int64)
    keep[-1, (seq + 1) // 2:] = 0
    hidden = tt.BertModel.from_torch(model, torch.device("cuda:0"), "turbo")(ids, attention_masks=keep.cuda())[0]
    with torch.no_grad():
        want = model.double()(input_ids=ids, attention_mask=keep.cuda()).last_hidden_state
    rows = keep.bool().cuda()
    error = (hidden.double() - want)[rows]
    assert bool(torch.isfinite(hidden.float()).all())
    assert error.pow(2).mean().sqrt().item() <= (8 * layers) ** 0.5 * EPS[dt] / 2 / 3 ** 0.5
