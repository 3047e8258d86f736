"""The decoder under the tools that trace it, which must take it whole: what it decides about the route of a layer in
Python may not break a graph, and a traced graph computes what the modules compute."""
import pytest
import torch
from torch._dynamo.source import ConstantSource
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.symbolic_shapes import DimDynamic, ShapeEnv

from macko_spmv_amd import llm


def _fake_model(mode, dim=256, hidden=704, heads=2):
    """Half-precision decoder with compressed projections on a GPU that need not exist."""
    with mode, torch.device("cuda"):
        default = torch.get_default_dtype()
        torch.set_default_dtype(torch.float16)
        try:
            model = llm.LlamaDecoder(100, dim, hidden, 2, heads, 48).requires_grad_(False)
        finally:
            torch.set_default_dtype(default)
        for layer in model.model.layers:
            for parent, name in llm.PROJECTIONS:
                module = getattr(layer, parent)
                rows, cols = getattr(module, name).weight.shape
                n = rows * cols // 2
                setattr(module, name, llm.MackoLinear(torch.empty(n, dtype=torch.float16), torch.empty(n // 2, dtype=torch.uint8),
                                                      torch.empty(rows + 1, dtype=torch.int32), rows, cols))
    return model


def _operators(function, *args):
    """Names of this package's operators in the one graph that Dynamo makes of a call."""
    graphs = []

    def backend(graph, example_inputs):
        graphs.append(graph)
        return graph.forward

    torch._dynamo.reset()
    torch.compile(function, fullgraph=True, backend=backend)(*args)
    assert len(graphs) == 1
    return [str(n.target).split(".")[1] for n in graphs[0].graph.nodes if str(n.target).startswith("macko_spmv.")]


def test_a_symbolic_number_of_tokens_stays_symbolic():
    # fake tensors alone, nothing compiled or recorded: the operators that an eager prompt goes through
    shapes = ShapeEnv()
    mode = FakeTensorMode(allow_non_fake_inputs=True, shape_env=shapes)
    layer = _fake_model(mode).model.layers[0]
    with mode, torch.no_grad(), torch.device("cuda"):
        # 19 is one number of tokens, which nothing may hold on to
        tokens = shapes.create_symintnode(shapes.create_symbol(19, source=ConstantSource("tokens"), dynamic_dim=DimDynamic.DYNAMIC), hint=19)
        x = torch.empty((1, tokens, 256), dtype=torch.float16)
        table, positions = torch.empty((1, 1, tokens, 128), dtype=torch.float16), torch.empty((tokens,), dtype=torch.long)
        assert layer.takes_fused(x)
        out = layer.forward_fused(x, table, table, positions)
    assert isinstance(out.shape[1], torch.SymInt) and not shapes.replacements


def test_decoder_compiles_as_one_graph():
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    model = _fake_model(mode)
    with mode, torch.no_grad(), torch.device("cuda"):
        for tokens in (1, 20):
            found = _operators(model, torch.empty((1, tokens), dtype=torch.long), torch.empty((tokens,), dtype=torch.long))
            per_layer = (["pack_rmsnorm"] + 3 * ["multiply_packed"] + ["prefill_rope_append", "prefill_attention", "multiply_packed",
                         "pack_rmsnorm", "multiply_packed", "multiply_packed", "pack_silu_mul", "multiply_packed"])
            if tokens == 1:
                per_layer = ["rmsnorm_rows"] + 4 * ["multiply"] + ["rmsnorm_rows"] + 3 * ["multiply"]
            assert found == 2 * per_layer + ["rmsnorm_rows"]
        norm, x = model.model.norm, torch.empty((3, 256), dtype=torch.float16)
        assert _operators(norm, x) == ["rmsnorm_rows"]
        # a batching rule, a tangent or a gradient goes through torch's own operators
        assert _operators(torch.func.vmap(norm), x) == []
        assert _operators(lambda a: torch.func.jvp(norm, (a,), (a,)), x) == []
    with mode, torch.enable_grad(), torch.device("cuda"):
        assert _operators(norm, torch.empty((3, 256), dtype=torch.float16, requires_grad=True)) == []


def test_one_graph_takes_prompts_of_any_length():
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    model, graphs = _fake_model(mode), []

    def backend(graph, example_inputs):
        graphs.append(graph)
        return graph.forward

    torch._dynamo.reset()
    with mode, torch.no_grad(), torch.device("cuda"):
        tokens, positions = torch.empty((1, 20), dtype=torch.long), torch.empty((20,), dtype=torch.long)
        torch._dynamo.mark_dynamic(tokens, 1)   # an error if the length becomes part of the graph
        torch._dynamo.mark_dynamic(positions, 0)
        compiled = torch.compile(model, fullgraph=True, backend=backend)
        compiled(tokens, positions)
        for length in (2, 16, 33):
            assert compiled(torch.empty((1, length), dtype=torch.long), torch.empty((length,), dtype=torch.long)).shape == (1, length, 100)
    assert len(graphs) == 1


@pytest.mark.parametrize("fuse", [True, False])
def test_decode_step_compiles_as_one_graph(fuse, monkeypatch):
    def stacked(parts):   # of tensors that hold nothing: the sizes
        return (torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts]),
                torch.empty(sum(p[3] for p in parts) + 1, dtype=torch.int32, device="cuda"), sum(p[3] for p in parts), parts[0][4])

    monkeypatch.setattr(llm, "concat_compressed", stacked)
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    model = _fake_model(mode)
    with mode, torch.no_grad(), torch.device("cuda"):
        engine = llm.DecodeEngine(model, fuse=fuse)
        found = _operators(engine.step, torch.empty((1,), dtype=torch.long), torch.empty((1,), dtype=torch.long))
    per_layer = ["multiply_rmsnorm", "decode_rope_attention_parts", "multiply_attention_axpby", "multiply_rmsnorm", "multiply_silu_mul_axpby"]
    if not fuse:
        per_layer = ["decode_rmsnorm", "multiply", "decode_rope_append", "decode_attention", "multiply_axpby",
                     "decode_rmsnorm", "multiply", "decode_silu_mul", "multiply_axpby"]
    assert found == 2 * per_layer + ["decode_norm_matvec"]


def _dense_model():
    torch.manual_seed(0)
    model = llm.LlamaDecoder(100, 64, 128, 2, 2, 32).requires_grad_(False)
    return model, torch.randint(0, 100, (1, 7)), torch.arange(7)


def test_symbolic_trace_of_norm_layer_and_decoder():
    model, tokens, positions = _dense_model()
    want = model(tokens, positions)
    assert torch.equal(torch.fx.symbolic_trace(model)(tokens, positions), want)
    x = torch.randn(1, 7, 64)
    assert torch.equal(torch.fx.symbolic_trace(model.model.norm)(x), model.model.norm(x))
    layer, cos = model.model.layers[0], torch.randn(1, 1, 7, 32)
    mask = torch.zeros(1, 1, 7, 32)
    assert torch.equal(torch.fx.symbolic_trace(layer)(x, cos, cos, positions, mask), layer(x, cos, cos, positions, mask))


def test_script_of_norm_layer_and_decoder():
    model, tokens, positions = _dense_model()
    want = model(tokens, positions)
    x, cos, mask = torch.randn(1, 7, 64), torch.randn(1, 1, 7, 32), torch.zeros(1, 1, 7, 32)
    normed, layered = model.model.norm(x), model.model.layers[0](x, cos, cos, positions, mask)
    assert torch.equal(torch.jit.script(model.model.norm)(x), normed)
    assert torch.equal(torch.jit.script(model.model.layers[0])(x, cos, cos, positions, mask), layered)
    scripted = torch.jit.script(model)
    for _ in range(3):   # the profiling executor specialises after the first calls
        assert torch.allclose(scripted(tokens, positions), want, rtol=1e-5, atol=1e-6)


def test_recorded_graphs_get_torchs_operators():
    """... which have a gradient and run on any device, whatever the call that was recorded ran on."""
    from torch.fx.experimental.proxy_tensor import make_fx

    mode = FakeTensorMode(allow_non_fake_inputs=True)
    model = _fake_model(mode)
    norm = model.model.norm
    with mode, torch.no_grad(), torch.device("cuda"):
        x = torch.empty((3, 256), dtype=torch.float16)
        exported = torch.export.export(norm, (x,), strict=True).graph
    with torch.no_grad():
        recorded = make_fx(norm)(x).graph
    for graph in (exported, recorded):
        assert not [n for n in graph.nodes if "macko_spmv" in str(n.target)]
    chosen = []
    with torch.no_grad():
        torch.jit.trace(lambda a: (chosen.append(llm._inference_half(x)), a + 1)[1], torch.zeros(1), check_trace=False)
        chosen.append(llm._inference_half(x))
    assert chosen == [False, True]


@pytest.mark.parametrize("tokens,positions", [((1, 20), (1, 20)), ((1, 20), (40,)), ((20,), (20,)), ((1, 20), (5, 4))])
def test_positions_that_do_not_fit_the_tokens_are_refused(tokens, positions):
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    model = _fake_model(mode)
    with mode, torch.no_grad(), torch.device("cuda"):
        with pytest.raises(RuntimeError):
            model(torch.empty(tokens, dtype=torch.long), torch.empty(positions, dtype=torch.long))


@pytest.mark.parametrize("shape", [(2, 2, 48, 128), (1, 2, 64, 128), (1, 4, 48, 64)])
def test_caches_that_do_not_fit_are_refused(shape):
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    model = _fake_model(mode)
    with mode, torch.no_grad(), torch.device("cuda"):
        attention = model.model.layers[1].self_attn
        attention.k_cache, attention.v_cache = torch.empty(shape, dtype=torch.float16), torch.empty(shape, dtype=torch.float16)
        with pytest.raises(RuntimeError):
            model(torch.empty((1, 20), dtype=torch.long), torch.empty((20,), dtype=torch.long))


class _Recorder(torch.Tensor):
    """A subclass with a meaning of its own for torch's operators, as a distributed or a quantised tensor has."""
    seen = []

    @staticmethod
    def __new__(cls):
        return torch.Tensor._make_wrapper_subclass(cls, (3, 256), dtype=torch.float16, device="cuda")

    @classmethod
    def __torch_dispatch__(cls, function, types, args, kwargs=None):
        cls.seen.append(str(function).split(".")[0])
        return cls()


def test_norm_of_a_tensor_subclass_goes_through_torchs_operators():
    norm = _fake_model(FakeTensorMode(allow_non_fake_inputs=True)).model.norm
    with torch.no_grad():
        norm(_Recorder())
    assert _Recorder.seen and set(_Recorder.seen) == {"aten"}


def test_operands_of_several_gpus_are_refused():
    """... by torch's operators; a kernel would read the other GPU's memory."""
    norm = _fake_model(FakeTensorMode(allow_non_fake_inputs=True)).model.norm
    with norm.weight.fake_mode, torch.no_grad():
        with pytest.raises(RuntimeError):
            norm(torch.empty((3, 256), dtype=torch.float16, device="cuda:1"))


def _takes_fused(change):
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    layer = _fake_model(mode).model.layers[0]
    with mode, torch.no_grad(), torch.device("cuda"):
        change(layer)
        return layer.takes_fused(torch.empty((1, 20, 256), dtype=torch.float16))


def test_layer_with_norm_weights_of_any_stride_goes_through_its_modules():
    def norm_weight(make):
        def change(layer):
            weight = make(torch.ones(512, dtype=torch.float16, device="cuda"))
            layer.post_attention_layernorm.weight = torch.nn.Parameter(weight, requires_grad=False)
        return change

    assert _takes_fused(lambda layer: None) and _takes_fused(norm_weight(lambda w: w[:256]))
    for make in (lambda w: w[:1].expand(256), lambda w: w[::2], lambda w: w[:1], lambda w: w[:256][None]):
        assert not _takes_fused(norm_weight(make))


@pytest.mark.parametrize("kind", [llm.Block, llm.Attention, llm.MLP, llm.RMSNorm, llm.MackoLinear])
def test_layer_calls_a_forward_that_was_replaced_in_its_class(kind, monkeypatch):
    kept = kind.forward
    monkeypatch.setattr(kind, "forward", lambda self, *args: kept(self, *args))
    assert not _takes_fused(lambda layer: None)
    monkeypatch.undo()
    assert _takes_fused(lambda layer: None)


@pytest.mark.parametrize("parent,name,rows,cols", [("self_attn", "q_proj", 256, 250), ("self_attn", "k_proj", 128, 256),
                                                   ("self_attn", "o_proj", 256, 251), ("mlp", "up_proj", 704, 255),
                                                   ("mlp", "up_proj", 696, 256), ("mlp", "down_proj", 256, 700)])
def test_layer_with_a_projection_that_does_not_fit_goes_through_its_modules(parent, name, rows, cols):
    """... which refuse it: a matrix of fewer columns must not be multiplied with the first of them."""
    def change(layer):
        n = rows * cols // 16 * 8
        setattr(getattr(layer, parent), name, llm.MackoLinear(
            torch.empty(n, dtype=torch.float16), torch.empty(n // 2, dtype=torch.uint8), torch.empty(rows + 1, dtype=torch.int32), rows, cols))

    assert not _takes_fused(change)
