"""Eager calls that go straight to the kernels' functions: they are left to the operators wherever something else than the
CUDA kernel would see the call, and give what the operators give."""
import numpy as np
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import macko_spmv_amd as mk


def test_calls_that_are_left_to_the_operators():
    cpu = (torch.zeros(8).half(), torch.zeros(4, dtype=torch.uint8), torch.zeros(3, dtype=torch.int32), 2, 8)
    x = torch.zeros(8).half()
    for args in ((cpu, x), (list(cpu), x), (cpu[:4], x), (None, x), (cpu, None), (cpu,), (cpu, x, x), (cpu[:3] + (2.0, 8), x)):
        assert mk._eager.multiply(*args) is NotImplemented
    for args in ((cpu, x, x, 1.0, 0.5), (cpu, x, x, 1, 0.5), (cpu, x, x)):
        assert mk._eager.multiply_axpby(*args) is NotImplemented
    assert mk._eager.multiply_packed_several([x], [x], [x], [2], 8, x, 1) is NotImplemented
    assert mk._eager.pack_rmsnorm(x, x, "1") is NotImplemented and mk._eager.multiply_batched(*cpu, x, x) is NotImplemented


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func.__name__)
        return func(*args, **(kwargs or {}))


class _Called(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(getattr(func, "__name__", str(func)))
        return func(*args, **(kwargs or {}))


@pytest.fixture
def case():
    g = torch.Generator(device="cuda").manual_seed(4)
    w = torch.randn(333, 200, device="cuda", generator=g) * (torch.rand(333, 200, device="cuda", generator=g) < 0.3)
    return mk.compress(w.half()), torch.randn(200, device="cuda", generator=g).half(), w.half()


@pytest.mark.gpu
def test_eager_calls_give_what_the_operators_give(case):
    c, x, w = case
    op = torch.ops.macko_spmv
    assert mk._plan_of(c) is not None
    bare = tuple(t.clone() if isinstance(t, torch.Tensor) else t for t in c)
    want = op.multiply(*c, x)
    for matrix in (c, bare, list(c)):
        assert torch.equal(mk.multiply(matrix, x), want)
    assert torch.equal(mk._eager.multiply(c, x), want) and mk._eager.multiply(list(c), x) is NotImplemented
    y = torch.ones(333, device="cuda").half()
    expect = y.clone()
    op.multiply_axpby(*c, x, expect, 2.0, 0.25)
    for matrix in (c, bare):
        into = y.clone()
        assert mk.multiply_axpby(matrix, x, into, 2.0, 0.25) is into and torch.equal(into, expect)
    X = torch.stack([x, -x, 2 * x])
    assert torch.equal(mk.multiply_batched(c, X), op.multiply_batched(*c, X))
    q = mk.compress_int8((w * 50).to(torch.int8))
    assert torch.equal(mk.multiply_int8(q, x), op.multiply_int8(*q, x))
    packed = mk.ops.pack_rmsnorm(X, torch.ones(200, device="cuda").half(), 1e-5)
    assert torch.equal(packed, op.pack_rmsnorm(X, torch.ones(200, device="cuda").half(), 1e-5))
    many = mk.ops.multiply_packed_several([c[0]] * 2, [c[1]] * 2, [c[2]] * 2, [332, 333], 200, packed, 3)
    assert all(torch.equal(a, b) for a, b in zip(many, op.multiply_packed_several([c[0]] * 2, [c[1]] * 2, [c[2]] * 2, [332, 333], 200, packed, 3)))
    # another stream, and a captured call
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert torch.equal(mk.multiply(c, x), want)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = mk.multiply(c, x)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.gpu
def test_what_looks_at_operators_still_sees_them(case):
    c, x, _ = case
    want = mk.multiply(c, x)
    with _Seen() as seen:
        assert torch.equal(mk.multiply(c, x), want)
        mk.multiply_batched(c, torch.stack([x, x]))
    assert any("multiply_planned" in n for n in seen.names) and any("multiply_batched" in n for n in seen.names)
    with _Called() as called:
        mk.multiply(c, x)
    assert any("multiply_planned" in n for n in called.names)
    assert torch.equal(torch.vmap(lambda v: mk.multiply(c, v))(torch.stack([x, -x])), mk.multiply_batched(c, torch.stack([x, -x])))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        mk.multiply(c, x)
    assert any("macko_spmv::multiply_planned" in e.key for e in profile.key_averages())
    leaf = x.clone().requires_grad_()
    with torch.enable_grad():   # whatever another test has left
        direct = torch.ops.macko_spmv.multiply_planned(*c, leaf, mk._plan_of(c))
        assert mk.multiply(c, leaf).requires_grad == direct.requires_grad
        assert mk._eager.multiply(c, leaf) is NotImplemented
    with torch.no_grad():
        assert mk._eager.multiply(c, leaf) is not NotImplemented
    with torch.inference_mode():
        assert torch.equal(mk.multiply(c, x), want)
    with torch.autocast("cuda"):
        assert mk._eager.multiply(c, x) is NotImplemented and torch.equal(mk.multiply(c, x), want)
    assert mk._eager.multiply(c, x) is not NotImplemented


@pytest.mark.gpu
def test_refused_calls_stay_refused(case):
    c, x, _ = case
    wide = torch.stack([x, x], 1)
    for call, error in ((lambda: mk.multiply(c, wide[:, 0]), AssertionError), (lambda: mk.multiply(c, x.cpu()), AssertionError),
                        (lambda: mk.multiply(c, x.float()), RuntimeError), (lambda: mk.multiply(c, x[:100]), RuntimeError),
                        (lambda: mk.multiply((c[0].float(),) + c[1:], x), RuntimeError),
                        (lambda: mk.multiply_axpby(c, x, torch.zeros(3, device="cuda").half(), 1.0, 1.0), RuntimeError),
                        (lambda: mk.multiply_axpby(c, x, torch.zeros(333, 2, device="cuda").half()[:, 0], 1.0, 1.0), AssertionError),
                        (lambda: mk.ops.multiply_packed_several([c[0]] * 4, [c[1]] * 4, [c[2]] * 4, [333] * 4, 200, x, 1), RuntimeError)):
        with pytest.raises(error):
            call()
    assert np.isfinite(mk.multiply(c, x).float().cpu().numpy()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,density", [(1, 8, 1.0), (3, 100, 0.0), (64, 130, 0.3), (4097, 64, 0.4), (5000, 700, 0.2), (20000, 50, 0.2),
                                               (12289, 257, 0.1), (300, 9000, 0.5), (9000, 9000, 0.02)])
def test_cuts_made_beside_the_rows_are_those_of_the_operator(rows, cols, density):
    g = torch.Generator(device="cuda").manual_seed(rows)
    keep = torch.rand(rows, cols, device="cuda", generator=g) < density * 2 * torch.rand(rows, 1, device="cuda", generator=g)
    m = (torch.randn(rows, cols, device="cuda", generator=g) * keep).half()
    c, general = mk.compress(m), torch.ops.macko_spmv.compress(m)
    assert type(c) is tuple and len(c) == 5 and all(torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b for a, b in zip(c, general))
    plan = torch.ops.macko_spmv.plan(c[2], rows, cols, c[0].numel())
    made = getattr(c[2], mk._PLAN_ATTRIBUTE)
    assert made is None if plan.numel() == 0 else torch.equal(made, plan)
    with pytest.raises(AssertionError):
        mk.compress(m.t()) if rows > 1 else mk.compress(m[:, ::2])
    with pytest.raises(RuntimeError):
        mk.compress(m.float())


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:.*overrid")
@pytest.mark.parametrize("key", ["Autograd", "AutogradCUDA", "ADInplaceOrView", "BackendSelect", "CUDA"])
def test_kernels_that_a_program_registers_see_the_calls(case, key):
    c, x, w = case
    X, y = torch.stack([x, -x]), torch.ones(333, device="cuda").half()
    seen = []

    def kernel(name, result):
        def f(*args):
            seen.append(name)
            return result
        return f

    made = torch.ops.macko_spmv.compress(w)
    cuts = torch.ops.macko_spmv.plan(made[2], 333, 200, made[0].numel())
    bare = tuple(t.clone() if isinstance(t, torch.Tensor) else t for t in c)
    calls = {"multiply_planned": (x, lambda: mk.multiply(c, x)), "multiply": (x, lambda: mk.multiply(bare, x)),
             "multiply_batched": (X, lambda: mk.multiply_batched(c, X)),
             "multiply_axpby_planned": (None, lambda: mk.multiply_axpby(c, x, y, 2.0, 0.25)), "multiply_axpby": (None, lambda: mk.multiply_axpby(bare, x, y, 2.0, 0.25)),
             "compress": (made, lambda: mk.compress(w)), "plan": (cuts, lambda: mk.compress(w))}
    before = y.clone()
    for name, (result, call) in calls.items():
        library = torch.library.Library("macko_spmv", "IMPL")
        seen.clear()
        try:
            library.impl(name, kernel(name, result), key, allow_override=True)
            got = call()
            assert seen == [name], key
            if name.startswith("multiply_axpby"):
                assert got is y and torch.equal(y, before)
            elif name.startswith("multiply"):
                assert got is result or torch.equal(got, result)
        finally:
            library._destroy()
        call()
        assert seen == [name]   # taken back
        y.copy_(before)
    assert torch.equal(mk.multiply(c, x), mk.multiply(bare, x)) and mk._eager.multiply(c, x) is not NotImplemented
