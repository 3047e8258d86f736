"""Forms of input that a layer of the decoder takes through its modules, and that it has to take as well where
hand-written kernels stand between the projections: memory that is not 16-byte aligned, norm weights of any stride,
projections that do not fit, infinite scores."""
import pytest
import torch

import macko_spmv_amd as mk
from macko_spmv_amd import llm

pytestmark = pytest.mark.gpu
ops = torch.ops.macko_spmv


def _elsewhere(t, by=1):
    """A copy of t whose memory starts `by` elements behind an aligned address, as storage of its own (offset 0)."""
    flat = torch.empty(t.numel() + by, device=t.device, dtype=t.dtype)
    moved = torch.from_dlpack(flat[by:].view(t.shape).copy_(t))
    assert moved.data_ptr() % 16 and moved.storage_offset() == 0
    return moved


def test_operators_between_the_projections_take_memory_of_any_alignment():
    g = torch.Generator(device="cuda").manual_seed(3)
    half = lambda *shape: torch.randn(shape, device="cuda", generator=g).half()
    x, up, w = half(19, 128), half(19, 128), half(128)
    assert torch.equal(ops.rmsnorm_rows(_elsewhere(x), _elsewhere(w), 1e-5), ops.rmsnorm_rows(x, w, 1e-5))
    assert torch.equal(ops.pack_rmsnorm(_elsewhere(x), _elsewhere(w), 1e-5), ops.pack_rmsnorm(x, w, 1e-5))
    assert torch.equal(ops.pack_silu_mul(_elsewhere(x), _elsewhere(up)), ops.pack_silu_mul(x, up))
    k, v, cos, sin, kc, vc = half(19, 128), half(19, 128), half(19, 64), half(19, 64), half(2, 30, 64), half(2, 30, 64)
    pos = torch.arange(19, device="cuda")
    q1, k1, v1 = x.clone(), kc.clone(), vc.clone()
    ops.prefill_rope_append(q1, k, v, cos, sin, pos, k1, v1)
    q2, k2, v2 = _elsewhere(x), _elsewhere(kc), _elsewhere(vc)
    ops.prefill_rope_append(q2, _elsewhere(k), _elsewhere(v), _elsewhere(cos), _elsewhere(sin), pos, k2, v2)
    assert torch.equal(q1, q2) and torch.equal(k1, k2) and torch.equal(v1, v2)
    assert torch.equal(ops.prefill_attention(q2, k2, v2, pos, 0.125), ops.prefill_attention(q1, k1, v1, pos, 0.125))


def test_norm_takes_memory_of_any_alignment():
    norm = llm.RMSNorm(64).cuda().half().requires_grad_(False)
    x = torch.randn(5, 64, device="cuda").half()
    want = norm(x.float()).double()   # fp32: through torch
    # one rounding to fp16 of a value with a few fp32 roundings in it
    assert torch.allclose(norm(_elsewhere(x)).double(), want, rtol=2.0 ** -10, atol=2.0 ** -24)


@pytest.mark.parametrize("tokens", [1, 19])
def test_compiled_decoder_gives_what_the_eager_one_gives(tokens):
    with torch.no_grad():
        model, _ = llm.build_model(0.4, sparse=True, n_layers=2, dim=256, hidden=704, n_heads=2, vocab=1000, max_len=48)
        prompt, pos = torch.randint(0, 1000, (1, tokens), device="cuda"), torch.arange(tokens, device="cuda")
        want = model(prompt, pos)
        caches = [layer.self_attn.k_cache.clone() for layer in model.model.layers]
        for layer in model.model.layers:
            layer.self_attn.k_cache.zero_()
        torch._dynamo.reset()
        got = torch.compile(model, fullgraph=True, backend="aot_eager")(prompt, pos)
        assert torch.equal(got, want)
        assert all(torch.equal(layer.self_attn.k_cache, kept) for layer, kept in zip(model.model.layers, caches))


def _small_model(**change):
    return llm.build_model(0.4, sparse=True, **{**dict(n_layers=1, dim=256, hidden=704, n_heads=2, vocab=1000, max_len=48), **change})[0]


@pytest.mark.parametrize("make", [lambda w: w[:1].expand(256), lambda w: w[::2]])
def test_layer_takes_norm_weights_of_any_stride(make):
    with torch.no_grad():
        model = _small_model()
        prompt, pos = torch.randint(0, 1000, (1, 19), device="cuda"), torch.arange(19, device="cuda")
        norm = model.model.layers[0].post_attention_layernorm
        weight = make(1 + 0.1 * torch.randn(512, device="cuda").half())
        norm.weight = torch.nn.Parameter(weight.contiguous(), requires_grad=False)
        want = model(prompt, pos).float()
        norm.weight = torch.nn.Parameter(weight, requires_grad=False)
        # the same weights, through the modules: fp16 activations rounded in other places
        assert torch.allclose(model(prompt, pos).float(), want, rtol=2e-2, atol=2e-2)


def test_layer_refuses_a_projection_of_fewer_columns():
    with torch.no_grad():
        model = _small_model()
        weight = torch.randn(256, 250, device="cuda").half()
        model.model.layers[0].self_attn.q_proj = llm.MackoLinear(*mk.compress(weight))
        prompt, pos = torch.randint(0, 1000, (1, 19), device="cuda"), torch.arange(19, device="cuda")
        with pytest.raises(RuntimeError):
            model(prompt, pos)


@pytest.mark.parametrize("head_dim", [64, 128])
def test_attention_of_infinite_and_nan_operands(head_dim):
    """As a softmax in torch has it: scores of -inf weigh nothing, and everything where nothing else is left; +inf, NaN
    and what a weight of zero meets in the values become NaN."""
    heads, tokens, max_len = 5, 40, 64
    g = torch.Generator(device="cuda").manual_seed(head_dim)
    q, kc, vc = (torch.randn(shape, device="cuda", generator=g).half().abs_() for shape in
                 ((tokens, heads * head_dim), (heads, max_len, head_dim), (heads, max_len, head_dim)))
    inf = float("inf")
    kc[0, 0], kc[1, :3], kc[2, 5, 7], kc[3, 33, 0] = -inf, -inf, inf, float("nan")
    vc[4, 20, 3], vc[0, 0, 1], vc[0, tokens:], kc[0, tokens:] = inf, inf, float("nan"), float("nan")
    pos = torch.arange(tokens, device="cuda")
    scale = head_dim ** -0.5

    def reference(q, last, h):
        scores = (q.double()[None] @ kc[h, :last + 1].double().t().contiguous())[0] * scale
        weights = torch.softmax(scores, -1)
        return (weights[:, None] * vc[h, :last + 1].double()).sum(0)

    packed = ops.prefill_attention(q, kc, vc, pos, scale)
    steps, tiles = heads * head_dim // 64, (tokens + 15) // 16
    rows = packed.view(steps, tiles, 2, 4, 16, 8).permute(1, 4, 0, 3, 2, 5).reshape(tiles * 16, -1)
    assert not rows[tokens:].any()
    seen = 0
    for h in range(heads):
        for t in range(tokens):
            want, got = reference(q[t, h * head_dim:(h + 1) * head_dim], t, h), rows[t, h * head_dim:(h + 1) * head_dim].double()
            # a value of a later token of the same 16 may be met by a weight of zero; torch's masked softmax meets all of them
            if h == 4 and t < 20:
                want = torch.where(torch.isinf(vc[4, 20].double()) & torch.isnan(got), got, want)
            assert torch.equal(want.isnan(), got.isnan()) and torch.equal(want.isinf(), got.isinf()), (h, t)
            seen += int(want.isnan().any())
            ok = want.isfinite()
            # weights and result rounded to fp16
            assert torch.allclose(got[ok], want[ok], rtol=2.0 ** -9, atol=2.0 ** -20), (h, t)
    assert seen > 50
    # one token, in pieces
    cos, sin = torch.ones(max_len, head_dim // 2, device="cuda"), torch.zeros(max_len, head_dim // 2, device="cuda")
    for last in (0, 2, 6, 39):
        k, v = kc[:, last].reshape(-1).contiguous(), vc[:, last].reshape(-1).contiguous()
        parts = ops.decode_rope_attention_parts(q[last].contiguous(), k, v, cos, sin, pos[last:last + 1], kc.clone(), vc.clone(), scale)
        whole = ops.decode_rope_attention(q[last].contiguous(), k, v, cos, sin, pos[last:last + 1], kc.clone(), vc.clone(), scale)
        sums = parts[:heads * 4 * head_dim].view(heads, 4, head_dim)
        pairs = parts[heads * 4 * head_dim:].view(heads, 4, 2)
        weight = torch.exp(pairs[..., 0] - pairs[..., 0].max(1, keepdim=True).values)
        merged = (weight[..., None] * sums).sum(1) / (weight * pairs[..., 1]).sum(1)[:, None]
        got, want = merged.double(), whole.view(heads, head_dim).double()
        assert torch.equal(want.isnan(), got.isnan()) and torch.equal(want.isinf(), got.isinf()), last
        ok = want.isfinite()
        assert torch.allclose(got[ok], want[ok], rtol=2.0 ** -9, atol=2.0 ** -20), last
