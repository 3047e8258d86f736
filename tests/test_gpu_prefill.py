"""The kernels that work all tokens of a prompt between the projections, against plain torch in float64 at the
edges of their tiles (16 tokens, 32 cache positions, 64 columns), and the layer built from them against the
module path."""
import ctypes

import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import macko_spmv_amd as mk
from macko_spmv_amd import llm
from tests import helpers

pytestmark = pytest.mark.gpu
ops = torch.ops.macko_spmv


def _unpack(packed, cols, batch):
    """Operand order back to [batch, cols], and what lies beyond them."""
    steps, tiles = (cols + 63) // 64, (batch + 15) // 16
    # [step, tile, s, q, n, 8] -> [tile, n, step, q, s, 8]
    full = packed.view(steps, tiles, 2, 4, 16, 8).permute(1, 4, 0, 3, 2, 5).reshape(tiles * 16, steps * 64)
    rest = full.clone()
    rest[:batch, :cols] = 0
    return full[:batch, :cols], rest


@pytest.mark.parametrize("batch,cols", [(1, 64), (2, 72), (15, 4096), (16, 512), (17, 1376), (33, 16392), (128, 4096)])
def test_norm_and_gate_in_operand_order(batch, cols):
    g = torch.Generator(device="cuda").manual_seed(cols + batch)
    x, up = (torch.randn(batch, cols, device="cuda", generator=g).half() for _ in range(2))
    w = (1 + 0.1 * torch.randn(cols, device="cuda", generator=g)).half()
    xd = x.double()
    want = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    got, rest = _unpack(ops.pack_rmsnorm(x, w, 1e-5), cols, batch)
    # one rounding to fp16 of a value with a few fp32 roundings in it
    assert torch.allclose(got.double(), want, rtol=2.0 ** -10, atol=2.0 ** -24) and not rest.any()
    assert torch.equal(ops.rmsnorm_rows(x, w, 1e-5), got)
    want = xd / (1 + torch.exp(-xd)) * up.double()
    got, rest = _unpack(ops.pack_silu_mul(x, up), cols, batch)
    assert torch.allclose(got.double(), want, rtol=2.0 ** -10, atol=2.0 ** -24) and not rest.any()


@pytest.mark.parametrize("batch,n_heads,head_dim,max_len,start", [(1, 1, 64, 1, 0), (2, 3, 128, 40, 0), (16, 2, 64, 16, 0), (17, 4, 128, 33, 0),
                                                                  (31, 2, 64, 200, 7), (128, 32, 128, 512, 0), (100, 2, 128, 900, 640)])
def test_rope_append_and_attention(batch, n_heads, head_dim, max_len, start):
    g = torch.Generator(device="cuda").manual_seed(batch + max_len)
    width = n_heads * head_dim
    q, k, v = (torch.randn(batch, width, device="cuda", generator=g).half() for _ in range(3))
    inv = 1.0 / (10000.0 ** (torch.arange(0, head_dim, 2, device="cuda").float() / head_dim))
    ang = torch.outer(torch.arange(max_len, device="cuda").float(), inv)
    ang = torch.cat((ang, ang), dim=-1)
    positions = start + torch.arange(batch, device="cuda")
    if batch == 31:
        positions = positions.flip(0).contiguous()   # any order
    cos, sin = ang.cos().half()[positions], ang.sin().half()[positions]
    kc, vc = (torch.randn(n_heads, max_len, head_dim, device="cuda", generator=g).half() for _ in range(2))
    top = int(positions.max())
    kc[:, top + 1:] = float("nan")   # what lies behind the context is not used
    vc[:, top + 1:] = float("nan")
    kc0, vc0 = kc.clone(), vc.clone()

    def rope(t):
        t = t.double().view(batch, n_heads, head_dim)
        rot = torch.cat((-t[..., head_dim // 2:], t[..., :head_dim // 2]), dim=-1)
        return t * cos.double()[:, None] + rot * sin.double()[:, None]

    q_in = q.clone()
    ops.prefill_rope_append(q, k, v, cos, sin, positions, kc, vc)
    assert torch.allclose(q.double().view(batch, n_heads, head_dim), rope(q_in), rtol=2.0 ** -10, atol=2.0 ** -20)
    assert torch.allclose(kc[:, positions].double().transpose(0, 1), rope(k), rtol=2.0 ** -10, atol=2.0 ** -20)
    assert torch.equal(vc[:, positions].transpose(0, 1).reshape(batch, width), v)
    keep = torch.ones(max_len, dtype=torch.bool, device="cuda")
    keep[positions] = False
    assert torch.equal(kc[:, keep].view(torch.int16), kc0[:, keep].view(torch.int16))
    assert torch.equal(vc[:, keep].view(torch.int16), vc0[:, keep].view(torch.int16))

    scale = head_dim ** -0.5
    got, rest = _unpack(ops.prefill_attention(q, kc, vc, positions, scale), width, batch)
    assert not rest.any()
    qd, kd, vd = q.float().view(batch, n_heads, head_dim), kc.float()[:, :top + 1], vc.float()[:, :top + 1]
    for h in range(n_heads):
        s = (qd[:, h] @ kd[h].t()) * scale
        s = s.masked_fill(torch.arange(top + 1, device="cuda")[None, :] > positions[:, None], float("-inf"))
        p = torch.softmax(s, dim=-1)
        want = p @ vd[h]
        # weights rounded to fp16 (2^-11 each) and one rounding of the result
        bound = 2.0 ** -10 * want.abs() + 2.0 ** -10 * (p @ vd[h].abs()) + 2.0 ** -20
        assert ((got[:, h * head_dim:(h + 1) * head_dim].float() - want).abs() <= bound).all(), h


@pytest.mark.parametrize("batch,rows,cols", [(1, 7, 64), (5, 100, 200), (40, 333, 1000), (130, 4100, 512)])
def test_product_of_packed_vectors_with_residual(batch, rows, cols):
    rng = np.random.default_rng(rows)
    dense = helpers.random_sparse(rng, rows, cols, 0.4)
    c = mk.compress(torch.from_numpy(dense).cuda())
    x = rng.standard_normal((batch, cols)).astype(np.float16)
    up = np.full((batch, cols), 30.0, dtype=np.float16)
    gate = torch.from_numpy(x).cuda()
    packed = ops.pack_silu_mul(gate, torch.from_numpy(up).cuda())
    staged = _unpack(packed, cols, batch)[0].cpu().numpy().astype(np.float64)
    r = rng.standard_normal((batch, rows)).astype(np.float16)
    d64 = dense.astype(np.float64)
    for residual in (None, torch.from_numpy(r).cuda()):
        y = ops.multiply_packed(*c, packed, batch, residual).cpu().double().numpy()
        want = staged @ d64.T + (r.astype(np.float64) if residual is not None else 0.0)
        bound = 2.0 ** -11 * np.abs(want) + 2.0 ** -25 + (cols + 3) * 2.0 ** -24 * (np.abs(staged) @ np.abs(d64).T + np.abs(want))
        assert (np.abs(y - want) <= bound).all()


@pytest.mark.parametrize("batch,rows,cols,density", [(2, (4, 0, 7), 64, 0.5), (17, (100, 52, 333), 200, 0.4), (128, (512, 512, 512), 1000, 0.1),
                                                     (100, (1376, 1377), 512, 0.5), (33, (4096, 8, 4100), 640, 0.05), (130, (48, 4), 4104, 0.9),
                                                     (64, (12400, 12400), 128, 0.3), (5, (21,), 72, 0.4)])
def test_product_of_packed_vectors_with_several_matrices(batch, rows, cols, density):
    rng = np.random.default_rng(sum(rows))
    dense = [helpers.random_sparse(rng, r, cols, density) for r in rows]
    c = [mk.compress(torch.from_numpy(d).cuda()) for d in dense]
    x = rng.standard_normal((batch, cols)).astype(np.float16)
    x[batch - 1, 3] = np.inf     # sums that are not finite are computed again, from their own matrix
    up = torch.full((batch, cols), 30.0, device="cuda", dtype=torch.float16)
    packed = ops.pack_silu_mul(torch.from_numpy(x).cuda(), up)
    staged = _unpack(packed, cols, batch)[0].cpu().numpy().astype(np.float64)
    got = ops.multiply_packed_several([m[0] for m in c], [m[1] for m in c], [m[2] for m in c], list(rows), cols, packed, batch)
    assert [tuple(y.shape) for y in got] == [(batch, r) for r in rows]
    for y, d in zip(got, dense):
        y, d64 = y.cpu().double().numpy(), d.astype(np.float64)
        used = d64[:, 3] != 0                    # rows that multiply the infinite element
        finite = np.ones_like(y, dtype=bool)
        finite[batch - 1, used] = False
        assert not np.isfinite(y[~finite]).any() and np.isfinite(y[finite]).all()
        x64 = np.where(np.isfinite(staged), staged, 0.0)
        want = x64 @ d64.T
        bound = 2.0 ** -11 * np.abs(want) + 2.0 ** -25 + (cols + 3) * 2.0 ** -24 * (np.abs(x64) @ np.abs(d64).T)
        assert (np.abs(y - want) <= bound)[finite].all()


@pytest.mark.parametrize("batch,rows,cols,offset,ldx", [(1, 40, 64, 0, 64), (17, 333, 200, 3, 211), (40, 100, 71, 1, 72)])
def test_packing_and_residual_in_place_through_the_c_abi(batch, rows, cols, offset, ldx):
    vp, i32, i64 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64
    lib = ctypes.CDLL(mk.HIP_LIBRARY_PATH)
    lib.macko_packed_bytes.argtypes = [i32, i32, ctypes.POINTER(i64)]
    lib.macko_pack_f16.argtypes = [vp, i32, i32, i64, vp, vp]
    lib.macko_spmv_f16_packed.argtypes = [vp, vp, vp, vp, vp, vp, i32, i32, i64, i32, i64, vp]
    rng = np.random.default_rng(rows)
    dense = helpers.random_sparse(rng, rows, cols, 0.4)
    c = mk.compress(torch.from_numpy(dense).cuda())
    flat = torch.from_numpy(rng.standard_normal(offset + batch * ldx).astype(np.float16)).cuda()
    x = flat[offset:].view(batch, ldx)[:, :cols]
    size = i64(-1)
    assert lib.macko_packed_bytes(cols, batch, ctypes.byref(size)) == 0
    packed = torch.full((size.value // 2,), 7.0, dtype=torch.float16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.macko_pack_f16(x.data_ptr(), cols, batch, ldx, packed.data_ptr(), stream) == 0
    got, rest = _unpack(packed, cols, batch)
    assert torch.equal(got, x) and not rest.any()
    r = rng.standard_normal((batch, rows)).astype(np.float16)
    y = torch.from_numpy(r).cuda()   # the residual is where the result goes
    assert lib.macko_spmv_f16_packed(c[0].data_ptr(), c[1].data_ptr(), c[2].data_ptr(), packed.data_ptr(), y.data_ptr(), y.data_ptr(),
                                     rows, cols, c[0].numel(), batch, rows, stream) == 0
    x64, d64 = x.cpu().double().numpy(), dense.astype(np.float64)
    want = x64 @ d64.T + r.astype(np.float64)
    bound = 2.0 ** -11 * np.abs(want) + 2.0 ** -25 + (cols + 3) * 2.0 ** -24 * (np.abs(x64) @ np.abs(d64).T + np.abs(want))
    assert (np.abs(y.cpu().double().numpy() - want) <= bound).all()
    # refused before any launch
    assert lib.macko_pack_f16(x.data_ptr(), 63, batch, ldx, packed.data_ptr(), stream) == -1
    assert lib.macko_pack_f16(x.data_ptr(), cols, batch, cols - 1, packed.data_ptr(), stream) == -1


def test_operators_have_fake_implementations():
    M = torch.randn((128, 128), dtype=torch.float16, device="cuda")
    c = mk.compress(M)
    x, w = torch.randn(5, 128, device="cuda").half(), torch.ones(128, device="cuda").half()
    packed = ops.pack_rmsnorm(x, w, 1e-5)
    torch.library.opcheck(ops.pack_rmsnorm, (x, w, 1e-5))
    torch.library.opcheck(ops.rmsnorm_rows, (x, w, 1e-5))
    torch.library.opcheck(ops.pack_silu_mul, (x, x.clone()))
    torch.library.opcheck(ops.multiply_packed, (*c, packed, 5, x))
    kc, vc = torch.zeros(2, 30, 64, device="cuda").half(), torch.zeros(2, 30, 64, device="cuda").half()
    pos, cs = torch.arange(5, device="cuda"), torch.ones(5, 64, device="cuda").half()
    torch.library.opcheck(ops.prefill_rope_append, (x.clone(), x.clone(), x.clone(), cs, cs, pos, kc, vc))
    torch.library.opcheck(ops.prefill_attention, (x, kc, vc, pos, 0.125))


@pytest.mark.parametrize("dim,hidden,heads,t", [(256, 688, 4, 2), (256, 704, 2, 19), (512, 1376, 8, 64)])
@torch.no_grad()
def test_fused_layers_against_the_module_path(dim, hidden, heads, t):
    cfg = dict(n_layers=2, dim=dim, hidden=hidden, n_heads=heads, vocab=1000, max_len=80)
    model, _ = llm.build_model(0.4, sparse=True, **cfg)
    prompt, pos = torch.randint(0, 1000, (1, t), device="cuda"), torch.arange(t, device="cuda")
    x = model.model.embed_tokens(prompt)
    assert all(layer.takes_fused(x) for layer in model.model.layers)
    fused = model(prompt, pos).float()
    caches = [layer.self_attn.k_cache.clone() for layer in model.model.layers]
    # a hook on one projection sends its layer (only) through the modules
    calls = []
    handle = model.model.layers[1].mlp.up_proj.register_forward_hook(lambda *a: calls.append(1))
    mixed = model(prompt, pos).float()
    assert calls and not model.model.layers[1].takes_fused(x) and model.model.layers[0].takes_fused(x)
    handle.remove()
    for layer in model.model.layers:
        layer.mlp.register_forward_pre_hook(lambda *a: None)
    plain = model(prompt, pos).float()
    assert not any(layer.takes_fused(x) for layer in model.model.layers)
    # fp16 activations between the parts, rounded in other places
    assert torch.allclose(fused, plain, rtol=2e-2, atol=2e-2) and torch.allclose(mixed, plain, rtol=2e-2, atol=2e-2)
    for kept, layer in zip(caches, model.model.layers):
        assert torch.allclose(kept.float(), layer.self_attn.k_cache.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("part", ["attention", "mlp", "both"])
@pytest.mark.parametrize("dim,hidden,heads,t", [(256, 688, 4, 2), (256, 704, 2, 19), (512, 1376, 8, 64)])
@torch.no_grad()
def test_what_a_fused_layer_adds(dim, hidden, heads, t, part):
    """The increment of the layer's two halves, each alone (the other's last projection is zero) and together, against
    float64; weights large enough for the scores to matter."""
    g = torch.Generator(device="cuda").manual_seed(dim + t)
    layer, max_len, hd = llm.Block(dim, hidden, heads, 80).half().cuda(), 80, dim // heads
    dense = {}
    for parent, name in llm.PROJECTIONS:
        rows, cols = getattr(getattr(layer, parent), name).weight.shape
        w = torch.randn(rows, cols, device="cuda", generator=g).mul_(0.1).half()
        llm.prune_rows_(w, 0.4)
        if (part, name) in (("attention", "down_proj"), ("mlp", "o_proj")):
            w.zero_()
        dense[name] = w.double()
        setattr(getattr(layer, parent), name, llm.MackoLinear(*mk.compress(w)))
    for norm in (layer.input_layernorm, layer.post_attention_layernorm):
        norm.weight.copy_(1 + 0.3 * torch.randn(dim, device="cuda", generator=g))
    x = torch.randn(1, t, dim, device="cuda", generator=g).half()
    pos = torch.arange(t, device="cuda")
    ang = torch.outer(pos.float(), 1.0 / (10000.0 ** (torch.arange(0, hd, 2, device="cuda").float() / hd)))
    ang = torch.cat((ang, ang), -1)
    cos, sin = ang.cos().half(), ang.sin().half()
    assert layer.takes_fused(x)
    got = layer(x, cos[None, None], sin[None, None], pos, llm._FUSED_CAUSAL)

    def normed(v, norm):
        return v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + norm.eps) * norm.weight.double()

    def rope(v):
        return v * cos.double() + torch.cat((-v[..., hd // 2:], v[..., :hd // 2]), -1) * sin.double()

    x64 = x[0].double()
    n = normed(x64, layer.input_layernorm)
    q, k, v = ((n @ dense[name].t().contiguous()).view(t, heads, hd).transpose(0, 1) for name in ("q_proj", "k_proj", "v_proj"))
    q, k = rope(q), rope(k)
    out = torch.empty(t, heads, hd, device="cuda", dtype=torch.float64)
    for h in range(heads):
        scores = (q[h] @ k[h].t().contiguous()) * hd ** -0.5
        out[:, h] = scores.masked_fill(pos[None] > pos[:, None], float("-inf")).softmax(-1) @ v[h]
    after = x64 + out.reshape(t, -1) @ dense["o_proj"].t().contiguous()
    n = normed(after, layer.post_attention_layernorm)
    gate, up = n @ dense["gate_proj"].t().contiguous(), n @ dense["up_proj"].t().contiguous()
    after = after + (gate * torch.sigmoid(gate) * up) @ dense["down_proj"].t().contiguous()
    # about ten roundings to fp16 on the way (2^-11 at most, 2^-12.8 in the mean, each), those of q and k times
    # scores of a few units: 2^-8
    off = lambda a, b: float((a.double() - b).norm() / b.norm())
    assert off(got[0].double() - x64, after - x64) < 2.0 ** -8
    assert off(layer.self_attn.k_cache[0, :, :t], k) < 2.0 ** -9 and off(layer.self_attn.v_cache[0, :, :t], v) < 2.0 ** -9
    assert not layer.self_attn.k_cache[:, :, t:].any() and not layer.self_attn.v_cache[:, :, t:].any()


def test_gradients_take_the_modules():
    layer = llm.Block(256, 704, 2, 48).half().cuda().requires_grad_(False)
    for parent, name in llm.PROJECTIONS:
        module = getattr(layer, parent)
        setattr(module, name, llm.MackoLinear(*mk.compress(getattr(module, name).weight.detach())))
    x = torch.randn(1, 19, 256, device="cuda").half()
    norm = layer.input_layernorm
    with torch.enable_grad():
        assert layer.takes_fused(x)
        assert not layer.takes_fused(x.clone().requires_grad_())
        norm.weight.requires_grad_()
        assert not layer.takes_fused(x)
        leaf = x.clone().requires_grad_()
        norm(leaf).float().pow(2).sum().backward()
        want = x.double().requires_grad_()
        (want * torch.rsqrt(want.pow(2).mean(-1, keepdim=True) + norm.eps)).pow(2).sum().backward()
        assert norm.weight.grad is not None and leaf.grad.shape == x.shape
        # the squared norm does not depend on x but for eps: what is left is rounding
        assert leaf.grad.abs().max() < 0.05 and want.grad.abs().max() < 1e-3
    with torch.no_grad():
        assert layer.takes_fused(x)


@torch.no_grad()
def test_layer_keeps_a_given_mask_and_strided_positions():
    model, _ = llm.build_model(0.4, sparse=True, n_layers=1, dim=256, hidden=704, n_heads=2, vocab=1000, max_len=48)
    layer, t = model.model.layers[0], 20
    pos = torch.arange(t, device="cuda")
    x = model.model.embed_tokens(torch.randint(0, 1000, (1, t), device="cuda"))
    cos, sin = (table[pos].half()[None, None] for table in (model.cos, model.sin))
    assert layer.takes_fused(x)
    causal = layer(x, cos, sin, pos, llm._FUSED_CAUSAL)
    spread = torch.stack((pos, pos), 1)[:, 0]
    assert not spread.is_contiguous() and torch.equal(layer(x, cos, sin, spread, llm._FUSED_CAUSAL), causal)
    with pytest.raises(TypeError):   # no mask is no call of the layer
        layer(x, cos, sin, pos, None)
    # a mask that lets a token see only itself is not the causal one
    own = torch.full((1, 1, t, 48), float("-inf"), device="cuda", dtype=torch.float16)
    own[0, 0, pos, pos] = 0
    masked = layer(x, cos, sin, pos, own)
    handle = layer.mlp.register_forward_pre_hook(lambda *a: None)   # through the modules
    want = layer(x, cos, sin, pos, own)
    handle.remove()
    assert torch.equal(masked, want) and not torch.allclose(masked, causal, rtol=2e-2, atol=2e-2)


def test_norm_goes_the_general_way_where_the_kernel_cannot():
    """Unaligned tokens, forward-mode derivatives, vmap: as torch's own operators take them."""
    norm = llm.RMSNorm(64).cuda().half().requires_grad_(False)
    flat = torch.randn(5 * 64 + 8, device="cuda").half()
    x = flat[:320].view(5, 64)
    want = norm(x.float()).double()   # fp32: through torch
    unaligned = flat[1:321].view(5, 64)
    unaligned.copy_(x.clone())
    got = norm(unaligned)
    assert torch.allclose(got.double(), want, rtol=2.0 ** -10, atol=2.0 ** -24)
    x = unaligned.clone()
    assert torch.equal(torch.func.vmap(norm)(x), norm(unaligned))
    y, tangent = torch.func.jvp(norm, (x,), (x,))
    # the norm does not change with its input's length, up to eps and the rounding of x times the weight
    assert torch.equal(y, norm(unaligned)) and tangent.abs().max() < 1e-2


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func.__name__)
        return func(*args, **(kwargs or {}))


@pytest.mark.filterwarnings("ignore:.*overrid")
@pytest.mark.parametrize("t,max_len,start", [(2, 80, 0), (19, 80, 40), (64, 80, 16)])
@torch.no_grad()
def test_layer_in_one_call(monkeypatch, t, max_len, start):
    # the same operators one by one and in one call; what looks at operators, and a kernel that a program registers, sees them
    model, _ = llm.build_model(0.4, sparse=True, n_layers=2, dim=256, hidden=712, n_heads=4, vocab=1000, max_len=max_len)
    layers = model.model.layers
    prompt = torch.randint(0, 1000, (1, t), device="cuda")
    pos = torch.arange(start, start + t, device="cuda").repeat_interleave(2)[::2]   # not contiguous

    def outputs():
        for layer in layers:
            layer.self_attn.k_cache.fill_(0.25)
            layer.self_attn.v_cache.fill_(0.5)
        logits = model(prompt, pos)
        return [logits] + [c.clone() for layer in layers for c in (layer.self_attn.k_cache, layer.self_attn.v_cache)]

    taken = []
    one_call = mk.eager_prefill_layer

    def watched(*args):
        out = one_call(*args)
        taken.append(out is not NotImplemented)
        return out

    monkeypatch.setattr(mk, "eager_prefill_layer", watched)
    got = outputs()
    assert taken == [True, True]
    with _Seen() as seen:
        observed = outputs()
    assert taken == [True, True, False, False]
    monkeypatch.setattr(mk, "eager_prefill_layer", lambda *args: NotImplemented)
    want = outputs()
    for a, b, c in zip(got, want, observed):
        assert torch.equal(a, b) and torch.equal(a, c)
    assert sum(name.startswith("multiply_packed_silu") for name in seen.names) == 2
    monkeypatch.setattr(mk, "eager_prefill_layer", watched)
    for key in ("Autograd", "CUDA"):
        library, calls = torch.library.Library("macko_spmv", "IMPL"), []
        try:
            library.impl("prefill_attention", lambda q, *rest: (calls.append(1), mk._packed_like(q, q.shape[1], q.shape[0]).zero_())[1], key,
                         allow_override=True)
            model(prompt, pos)
        finally:
            library._destroy()
        assert len(calls) == 2, key


def test_layer_in_one_call_refuses_what_the_operators_refuse():
    model, _ = llm.build_model(0.4, sparse=True, n_layers=1, dim=256, hidden=704, n_heads=2, vocab=1000, max_len=48)
    layer = model.model.layers[0]
    x, pos = torch.zeros(1, 5, 256, device="cuda").half(), torch.arange(5, device="cuda")
    table = torch.ones(1, 1, 5, 128, device="cuda").half()
    with torch.no_grad():
        assert torch.isfinite(layer.forward_fused(x, table, table, pos)).all()
        for args in ((x, table, table, pos[:4]), (x, table[..., :64], table, pos), (x.float(), table, table, pos), (x, table, table, pos.int())):
            with pytest.raises(RuntimeError):
                layer.forward_fused(*args)
    assert mk.eager_prefill_layer(x.cpu(), table, table, pos) is NotImplemented


class _Subclass(torch.Tensor):
    pass


def test_layer_in_one_call_looks_at_every_argument():
    model, _ = llm.build_model(0.4, sparse=True, n_layers=1, dim=256, hidden=704, n_heads=2, vocab=1000, max_len=48)
    layer = model.model.layers[0]
    att, mlp = layer.self_attn, layer.mlp
    first, second = layer.input_layernorm, layer.post_attention_layernorm
    x, pos = torch.randn(1, 5, 256, device="cuda").half(), torch.arange(5, device="cuda")
    table = torch.ones(1, 1, 5, 128, device="cuda").half()
    args = [x, table, table.clone(), pos, att.k_cache, att.v_cache, att.head_dim ** -0.5, first.weight, first.eps, second.weight, second.eps]
    for linear in (att.q_proj, att.k_proj, att.v_proj, att.o_proj, mlp.gate_proj, mlp.up_proj, mlp.down_proj):
        args += [linear.c_0, linear.c_1, linear.c_2, linear.c_3, linear.c_4]
    # what the layer hands over with gradients off, and on where none of them asks for one
    for enabled in (False, True):
        with torch.set_grad_enabled(enabled):
            taken = mk.eager_prefill_layer(*[a.detach() if isinstance(a, torch.Tensor) else a for a in args])
            assert torch.equal(taken.detach(), layer.forward_fused(x, table, table, pos))
    refused = lambda place, value: mk.eager_prefill_layer(*args[:place], value, *args[place + 1:]) is NotImplemented  # noqa: E731
    with torch.no_grad():
        assert mk.eager_prefill_layer(*args) is not NotImplemented
        for place, value in enumerate(args):
            if isinstance(value, torch.Tensor):
                assert refused(place, value.cpu()) and refused(place, value.detach().as_subclass(_Subclass)) and refused(place, None), place
            elif isinstance(value, float):
                assert refused(place, 1) and refused(place, torch.tensor(value)), place
            else:
                assert refused(place, float(value)) and refused(place, True), place
        assert refused(0, x[0]) and refused(0, x.expand(2, 5, 256)) and refused(4, att.k_cache[0])
        assert mk.eager_prefill_layer(*args[:-1]) is NotImplemented and mk.eager_prefill_layer(*args, 1) is NotImplemented
    with torch.enable_grad():
        assert refused(0, x.clone().requires_grad_())
    with torch.autograd.forward_ad.dual_level(), torch.no_grad():
        assert refused(0, torch.autograd.forward_ad.make_dual(x, x))


def test_product_of_gate_and_up_is_an_operator():
    w = torch.randn(72, 64, device="cuda").half()
    c, x = mk.compress(w), torch.randn(5, 64, device="cuda").half()
    ops = torch.ops.macko_spmv
    packed = ops.pack_rmsnorm(x, torch.ones(64, device="cuda").half(), 1e-5)
    torch.library.opcheck(ops.multiply_packed_silu, ([c[0]] * 2, [c[1]] * 2, [c[2]] * 2, 72, 64, packed, 5))
    for rows, batch, n in ((72, 17, 2), (56, 5, 2), (72, 5, 1), (76, 5, 2)):
        with pytest.raises(RuntimeError):
            ops.multiply_packed_silu([c[0]] * n, [c[1]] * n, [c[2]] * n, rows, 64, packed, batch)
