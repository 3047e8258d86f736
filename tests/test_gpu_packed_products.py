"""Products of vectors in operand order, of one and of several matrices, by every kernel that takes them, against float64.

Bound: the sum in fp32 of n terms in any order (n * 2^-24 of the sum of the terms' magnitudes) and one rounding to fp16 (2^-11
of the value, 2^-25 where it is subnormal)."""
import ctypes

import numpy as np
import pytest
import torch

import macko_spmv_amd as mk
from tests import helpers, packed_products

pytestmark = pytest.mark.gpu
ops = torch.ops.macko_spmv
vp, i32, i64 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64


def _pack(lib, x):
    batch, cols = x.shape
    size = i64(-1)
    assert lib.macko_packed_bytes(cols, batch, ctypes.byref(size)) == 0
    packed = torch.empty(size.value // 2, dtype=torch.float16, device="cuda")
    lib.macko_pack_f16.argtypes = [vp, i32, i32, i64, vp, vp]
    assert lib.macko_pack_f16(x.data_ptr(), cols, batch, cols, packed.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    return packed


def _check(y, x, dense, residual=None):
    """x: finite but for column 1 of one vector, which a padding entry never stands for."""
    y = y.cpu().double().numpy()
    x64, d64 = np.where(np.isfinite(x), x, 0).astype(np.float64), dense.astype(np.float64)
    spoiled = (~np.isfinite(x)).any(axis=1)[:, None] & (dense[:, 1] != 0)[None, :]
    assert not np.isfinite(y[spoiled]).any() and np.isfinite(y[~spoiled]).all()
    want = x64 @ d64.T
    size = np.abs(x64) @ np.abs(d64).T
    if residual is not None:
        want, size = want + residual.astype(np.float64), size + np.abs(residual).astype(np.float64)
    bound = 2.0 ** -11 * np.abs(want) + 2.0 ** -25 + (dense.shape[1] + 3) * 2.0 ** -24 * size
    assert (np.abs(y - want) <= bound)[~spoiled].all()


@pytest.mark.parametrize("product", packed_products.PRODUCTS, ids=str)
def test_products_of_packed_vectors(product):
    dense = packed_products.matrices(product)
    c = [mk.compress(torch.from_numpy(m).cuda()) for m in dense]
    rng = np.random.default_rng(product.cols)
    x = rng.standard_normal((product.batch, product.cols)).astype(np.float16)
    x[product.batch // 2, 1] = np.inf
    lib = ctypes.CDLL(mk.HIP_LIBRARY_PATH)
    packed = _pack(lib, torch.from_numpy(x).cuda())
    if len(c) > 1:
        args = ([m[0] for m in c], [m[1] for m in c], [m[2] for m in c], list(product.rows), product.cols, packed, product.batch)
        got = ops.multiply_packed_several(*args)
        for y, m in zip(got, dense):
            _check(y, x, m)
        for y, again in zip(got, ops.multiply_packed_several(*args)):
            assert torch.equal(y.view(torch.int16), again.view(torch.int16))
        return
    (rows,), one = product.rows, c[0]
    y = ops.multiply_packed(*one, packed, product.batch, None)
    _check(y, x, dense[0])
    assert torch.equal(y.view(torch.int16), ops.multiply_packed(*one, packed, product.batch, None).view(torch.int16))
    # a residual; results of an odd row length that start at an odd element
    r = rng.standard_normal((product.batch, rows)).astype(np.float16)
    _check(ops.multiply_packed(*one, packed, product.batch, torch.from_numpy(r).cuda()), x, dense[0], r)
    lib.macko_spmv_f16_packed.argtypes = [vp, vp, vp, vp, vp, vp, i32, i32, i64, i32, i64, vp]
    ldy = rows + 2 + (rows + 1) % 2
    flat = torch.full((product.batch * ldy + 1,), 7.0, dtype=torch.float16, device="cuda")
    into = flat[1:].view(product.batch, ldy)
    into[:, :rows] = torch.from_numpy(r).cuda()
    assert lib.macko_spmv_f16_packed(one[0].data_ptr(), one[1].data_ptr(), one[2].data_ptr(), packed.data_ptr(), into.data_ptr(), into.data_ptr(),
                                     rows, product.cols, one[0].numel(), product.batch, ldy, torch.cuda.current_stream().cuda_stream) == 0
    _check(into[:, :rows], x, dense[0], r)
    assert (into[:, rows:] == 7.0).all() and flat[0] == 7.0


def test_matrices_of_unequal_densities():
    batch, rows, cols, densities = (packed_products.UNEQUAL[k] for k in ("batch", "rows", "cols", "densities"))
    rng = np.random.default_rng(cols)
    dense = [helpers.random_sparse(rng, r, cols, d, scale=0.05) for r, d in zip(rows, densities)]
    c = [mk.compress(torch.from_numpy(m).cuda()) for m in dense]
    x = rng.standard_normal((batch, cols)).astype(np.float16)
    packed = _pack(ctypes.CDLL(mk.HIP_LIBRARY_PATH), torch.from_numpy(x).cuda())
    got = ops.multiply_packed_several([m[0] for m in c], [m[1] for m in c], [m[2] for m in c], list(rows), cols, packed, batch)
    for y, m, one in zip(got, dense, c):
        _check(y, x, m)
        assert torch.equal(y, ops.multiply_packed(*one, packed, batch, None))


def test_rows_at_the_end_of_the_longest_array():
    # 32 entries, in the first columns, for each of the last two rows; what the array holds elsewhere is no row's
    entries, rows, cols, batch = (packed_products.LONG_ARRAY[k] for k in ("entries", "rows", "cols", "batch"))
    values = torch.zeros(entries, dtype=torch.float16, device="cuda")
    values[:1 << 20] = 100.0
    values[-64:] = 1.0
    deltas = torch.zeros(entries // 2, dtype=torch.uint8, device="cuda")
    row_ptr = torch.full((rows + 1,), entries - 64, dtype=torch.int32, device="cuda")
    row_ptr[-2:] = torch.tensor([entries - 32, entries], dtype=torch.int32)
    x = np.random.default_rng(1).standard_normal((batch, cols)).astype(np.float16)
    packed = _pack(ctypes.CDLL(mk.HIP_LIBRARY_PATH), torch.from_numpy(x).cuda())
    y = ops.multiply_packed(values, deltas, row_ptr, rows, cols, packed, batch, None)
    assert not y[:, :-2].any()
    want = x[:, :32].astype(np.float64).sum(axis=1)
    bound = 2.0 ** -11 * np.abs(want) + 33 * 2.0 ** -24 * np.abs(x[:, :32].astype(np.float64)).sum(axis=1)
    for row in (-2, -1):
        assert (np.abs(y[:, row].cpu().double().numpy() - want) <= bound).all()


@pytest.mark.parametrize("batch,rows,cols,density", packed_products.SUMS)
def test_long_sums_are_as_exact_as_the_other_kernel_s(batch, rows, cols, density):
    # How many results are not the exact one rounded to fp16: the error of the sum in fp32, in units of what a rounding hides.  Of
    # 400000 results and more at least 300 are; counts of so many differ by chance by 6 % (one standard deviation) and by 25 % hardly
    # ever; with half of the parts of a sum it is 1.5 times as many.
    generator = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.randn((batch, cols), device="cuda", generator=generator, dtype=torch.float16)
    packed = _pack(ctypes.CDLL(mk.HIP_LIBRARY_PATH), x)
    dense = []
    for r in rows:
        w = torch.randn((r, cols), device="cuda", generator=generator, dtype=torch.float16).mul_(0.02)
        dense.append(w.mul_(torch.rand((r, cols), device="cuda", generator=generator) < density))
    c = [mk.compress(w) for w in dense]
    together = ops.multiply_packed_several([m[0] for m in c], [m[1] for m in c], [m[2] for m in c], list(rows), cols, packed, batch)
    wrong = [0, 0]
    for y, w, one in zip(together, dense, c):
        exact = (x.double() @ w.double().T).half()
        wrong[0] += int((y != exact).sum())
        wrong[1] += int((ops.multiply_packed(*one, packed, batch, None) != exact).sum())
    print("not the rounded result:", wrong, "of", batch * sum(rows), flush=True)
    assert wrong[1] > 100 and wrong[0] <= 1.25 * wrong[1]


def _check_gated(c, rows, cols, batch, x):
    """Twice the same bits, and those of the products in one launch and the gate behind them."""
    packed = _pack(ctypes.CDLL(mk.HIP_LIBRARY_PATH), x)
    args = ([m[0] for m in c], [m[1] for m in c], [m[2] for m in c])
    got = ops.multiply_packed_silu(*args, rows, cols, packed, batch)
    for again in (ops.multiply_packed_silu(*args, rows, cols, packed, batch), mk.ops.multiply_packed_silu(*args, rows, cols, packed, batch)):
        assert torch.equal(again.view(torch.int16), got.view(torch.int16))
    want = ops.pack_silu_mul(*ops.multiply_packed_several(*args, [rows, rows], cols, packed, batch))
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(), want.nan_to_num())


# the gate's product: pairs of units of four rows over row blocks, columns that fill up no block of 64, vectors that
# fill up no block of 16, one chunk and several, matrices of one density and of two that are launched one by one
@pytest.mark.parametrize("rows,cols,batch,densities", [
    (64, 64, 2, (0.5, 0.5)), (72, 100, 16, (0.3, 0.3)), (1376, 512, 17, (0.5, 0.5)), (1376, 512, 128, (0.1, 0.1)),
    (2752, 1024, 33, (0.9, 0.85)), (5504, 2048, 100, (0.5, 0.5)), (11008, 4096, 128, (0.5, 0.5)), (11000, 1000, 130, (0.2, 0.2)),
    (11016, 640, 250, (0.4, 0.4)), (11008, 1024, 128, (0.9, 0.05)), (4096, 4096, 5, (0.05, 0.05)), (28672, 512, 64, (0.1, 0.12)),
    (1376, 512, 40, (0.0, 0.0))])
@pytest.mark.parametrize("special", (False, True))
def test_product_of_gate_and_up(rows, cols, batch, densities, special):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(rows + cols + batch)
    c = []
    for density in densities:
        w = torch.randn((rows, cols), device="cuda", generator=generator, dtype=torch.float16).mul_(0.1)
        w.mul_(torch.rand((rows, cols), device="cuda", generator=generator) < density)
        w[rows // 2] = 0
        c.append(mk.compress(w))
    x = torch.randn((batch, cols), device="cuda", generator=generator, dtype=torch.float16)
    if special:
        x[batch // 2, cols // 3] = float("inf")
        x[0, cols - 1] = float("nan")
    _check_gated(c, rows, cols, batch, x)


# ... by every kernel that takes two matrices (test_packed_routes_host.py)
@pytest.mark.parametrize("rows,cols,batch,density,kernel", packed_products.GATED)
def test_product_of_gate_and_up_by_every_kernel(rows, cols, batch, density, kernel):
    c = [mk.compress(torch.from_numpy(m).cuda()) for m in packed_products.gate_and_up(rows, cols, density)]
    x = torch.from_numpy(np.random.default_rng(batch).standard_normal((batch, cols)).astype(np.float16)).cuda()
    _check_gated(c, rows, cols, batch, x)
