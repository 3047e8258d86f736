"""Decode attention left in pieces and merged by the product that consumes it, against the one-workgroup-per-head
kernel and a float64 merge of the pieces; and the products that build their input while staging it, at the edges of
what travels in registers (two 16-byte pieces, or four columns, per thread)."""
import numpy as np
import pytest
import torch

import macko_spmv_amd as mk
from tests import helpers

pytestmark = pytest.mark.gpu
PARTS = 4


def _tables(max_len, head_dim):
    inv = 1.0 / (10000.0 ** (torch.arange(0, head_dim, 2, device="cuda").float() / head_dim))
    ang = torch.outer(torch.arange(max_len, device="cuda").float(), inv)
    return ang.cos().contiguous(), ang.sin().contiguous()


def _merged(parts, n_heads, head_dim):
    p = parts.double().cpu()
    o = p[:n_heads * PARTS * head_dim].view(n_heads, PARTS, head_dim)
    ml = p[n_heads * PARTS * head_dim:].view(n_heads, PARTS, 2)
    w = torch.exp(ml[:, :, 0] - ml[:, :, 0].max(dim=1, keepdim=True).values)
    return ((w[:, :, None] * o).sum(1) / (w * ml[:, :, 1]).sum(1)[:, None]).reshape(-1)


@pytest.mark.parametrize("n_heads,head_dim,max_len", [(1, 64, 1), (4, 64, 40), (32, 128, 300), (3, 128, 17), (5, 64, 1300), (2, 128, 4096)])
def test_pieces_against_the_whole(n_heads, head_dim, max_len):
    ops = torch.ops.macko_spmv
    torch.manual_seed(max_len)
    cos, sin = _tables(max_len, head_dim)
    kc = torch.randn(n_heads, max_len, head_dim, device="cuda").half()
    vc = torch.randn(n_heads, max_len, head_dim, device="cuda").half()
    # positions around the piece and load boundaries (32 or 64 rows per load, 4 loads, 4 pieces)
    wanted = (0, 1, 2, 3, 4, 31, 32, 63, 64, 127, 128, 129, 255, 256, 511, 512, 513, 1025, 2049, max_len - 1)
    for pos in sorted({p for p in wanted if p < max_len}):
        q, k, v = (torch.randn(n_heads * head_dim, device="cuda").half() for _ in range(3))
        position = torch.tensor([pos], device="cuda")
        kc1, vc1, kc2, vc2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
        kc2[:, pos + 1:] = float("nan")  # what lies behind the context is not read
        vc2[:, pos + 1:] = float("nan")
        want = ops.decode_rope_attention(q, k, v, cos, sin, position, kc1, vc1, head_dim ** -0.5).double().cpu()
        parts = ops.decode_rope_attention_parts(q, k, v, cos, sin, position, kc2, vc2, head_dim ** -0.5)
        assert torch.equal(kc1[:, :pos + 1], kc2[:, :pos + 1]) and torch.equal(vc1[:, :pos + 1], vc2[:, :pos + 1])
        got = _merged(parts, n_heads, head_dim)
        # one rounding to fp16, and fp32 sums of up to 4096 weights from a 2^-20 exponential
        assert torch.allclose(got, want, rtol=2.0 ** -10, atol=1e-4), pos


@pytest.mark.parametrize("n_heads,head_dim,rows,density", [(1, 64, 100, 0.5), (4, 64, 700, 0.3), (32, 128, 4096, 0.5), (40, 128, 333, 0.9),
                                                           (128, 64, 64, 1.0), (72, 128, 200, 0.2)])
def test_product_of_merged_pieces(n_heads, head_dim, rows, density):
    rng = np.random.default_rng(rows)
    cols = n_heads * head_dim
    dense = helpers.random_sparse(rng, rows, cols, density)
    c = mk.compress(torch.from_numpy(dense).cuda())
    g = torch.Generator(device="cuda").manual_seed(rows)
    o = torch.randn(n_heads, PARTS, head_dim, device="cuda", generator=g)
    ml = torch.stack((torch.randn(n_heads, PARTS, device="cuda", generator=g) * 3,
                      1.0 + torch.rand(n_heads, PARTS, device="cuda", generator=g) * 40), dim=-1)
    ml[:, 2, 0], ml[:, 2, 1], o[:, 2] = -3.0e38, 0.0, 0.0   # a piece without positions
    parts = torch.cat((o.reshape(-1), ml.reshape(-1))).contiguous()
    y0 = torch.randn(rows, device="cuda", generator=g).half()
    y = y0.clone()
    mk.multiply_attention_axpby(c, parts, head_dim, y, 0.5, -2.0)
    a = _merged(parts, n_heads, head_dim).numpy().astype(np.float16).astype(np.float64)
    d64 = dense.astype(np.float64)
    want = 0.5 * (d64 @ a) - 2.0 * y0.cpu().double().numpy()
    # every staged element may round one unit away from the float64 merge; then the product's own bound
    bound = 2.0 ** -10 * np.abs(want) + (2.0 ** -10 + (cols + 4) * 2.0 ** -24) * (np.abs(d64) @ np.abs(a)) + 2.0 ** -24
    assert (np.abs(y.cpu().double().numpy() - want) <= bound).all()


@pytest.mark.parametrize("rows,cols,density", [(64, 8, 1.0), (300, 1000, 0.3), (4096, 8184, 0.1), (4200, 8192, 0.3), (500, 8200, 0.5),
                                               (600, 16384, 0.2), (5000, 16392, 0.05), (40, 40000, 0.3)])
def test_staged_functions_at_the_edges_of_the_registers(rows, cols, density):
    rng = np.random.default_rng(cols)
    dense = helpers.random_sparse(rng, rows, cols, density)
    d64 = dense.astype(np.float64)
    c = mk.compress(torch.from_numpy(dense).cuda())
    x, w, up = (rng.standard_normal(cols).astype(np.float16) for _ in range(3))
    xf = x.astype(np.float64)

    def check(got, staged, extra):
        n = staged.astype(np.float16).astype(np.float64)
        want = d64 @ n + extra
        bound = 2.0 ** -10 * np.abs(want) + (2.0 ** -10 + (cols + 4) * 2.0 ** -24) * (np.abs(d64) @ np.abs(n)) + 2.0 ** -24
        assert (np.abs(got.cpu().double().numpy() - want) <= bound).all()

    check(mk.multiply_rmsnorm(c, torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), 1e-5),
          xf / np.sqrt((xf ** 2).mean() + 1e-5) * w.astype(np.float64), 0.0)
    y0 = rng.standard_normal(rows).astype(np.float16)
    y = torch.from_numpy(y0.copy()).cuda()
    mk.multiply_silu_mul_axpby(c, torch.from_numpy(x).cuda(), torch.from_numpy(up).cuda(), y, 1.0, 1.0)
    check(y, xf / (1 + np.exp(-xf)) * up.astype(np.float64), y0.astype(np.float64))


def test_operators_have_fake_implementations():
    ops = torch.ops.macko_spmv
    torch.manual_seed(4)
    cos, sin = _tables(48, 64)
    q, k, v = (torch.randn(256, device="cuda").half() for _ in range(3))
    kc, vc = torch.randn(4, 48, 64, device="cuda").half(), torch.randn(4, 48, 64, device="cuda").half()
    position = torch.tensor([5], device="cuda")
    torch.library.opcheck(ops.decode_rope_attention_parts, (q, k, v, cos, sin, position, kc, vc, 0.125))
    parts = ops.decode_rope_attention_parts(q, k, v, cos, sin, position, kc, vc, 0.125)
    M = torch.randn((300, 256), dtype=torch.float16, device="cuda")
    torch.library.opcheck(ops.multiply_attention_axpby, (*mk.compress(M), parts, 64, torch.zeros(300, device="cuda").half(), 1.0, 1.0))
