"""The product with several vectors on the matrix cores, at the sizes where it can go wrong: edges of the
16-row and 16-vector tiles and of the 64-column steps, chunks that end inside a row's entries, the smallest
and largest shapes of a launch, unaligned vectors, Inf / NaN / subnormal operands.

Bound: the exact product of the fp16 data, rounded once to fp16 (half a unit in the last place: 2^-11 of the
value, 2^-25 where it is subnormal), after a sum in fp32 of n terms in any order (n * 2^-24 of the sum of the
terms' magnitudes).
"""
import ctypes

import numpy as np
import pytest
import torch

import macko_spmv
import macko_spmv_amd
from oracle import macko_oracle as mo
from tests import helpers

pytestmark = pytest.mark.gpu


def _check(Y, dense, X, label):
    d64, x64 = dense.astype(np.float64), X.astype(np.float64)
    want = x64 @ d64.T
    size = np.abs(x64) @ np.abs(d64).T
    bound = 2.0 ** -11 * np.abs(want) + 2.0 ** -25 + (dense.shape[1] + 2) * 2.0 ** -24 * size
    err = np.abs(Y.astype(np.float64) - want)
    assert Y.shape == want.shape and not (err > bound).any(), f"{label}: {(err > bound).sum()} out of bound, worst {err.max()}"


def _case(rng, rows, cols, density, batch, scale=0.05):
    dense = helpers.random_sparse(rng, rows, cols, density, scale=scale)
    if rows > 6:
        dense[rng.integers(0, rows, size=max(1, rows // 9))] = 0
    return dense, rng.standard_normal((batch, cols)).astype(np.float16)


@pytest.mark.parametrize("rows,cols,density,batch", [
    (1, 64, 1.0, 4), (3, 65, 0.5, 5), (15, 71, 0.9, 15), (16, 72, 0.3, 16), (17, 127, 0.3, 17), (33, 128, 1.0, 31),
    (47, 129, 0.2, 33), (48, 1000, 0.5, 63), (49, 1023, 0.05, 64), (777, 3333, 0.25, 65), (1030, 515, 0.4, 127),
    (4096, 1024, 0.1, 128), (4100, 777, 0.5, 129), (1025, 4096, 0.5, 200), (11008, 512, 0.3, 40), (12289, 320, 0.7, 80),
    (12288, 200, 0.6, 128), (50000, 96, 0.5, 24), (64, 28000, 0.4, 20), (5, 90000, 0.02, 6), (700, 6000, 0.003, 48)])
def test_edges_of_tiles_and_chunks(rows, cols, density, batch):
    rng = np.random.default_rng(rows * 7 + cols + batch)
    dense, X = _case(rng, rows, cols, density, batch)
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    Y = macko_spmv.multiply_batched(c, torch.from_numpy(X).cuda())
    _check(Y.cpu().numpy(), dense, X, f"{rows}x{cols} d={density} b={batch}")
    # the same again, bit for bit: no sum depends on the order in which waves run
    assert torch.equal(Y, macko_spmv.multiply_batched(c, torch.from_numpy(X).cuda()))


# many rows and more than 16 vectors through the entry point, which packs X from 100000 elements on (12000 where a row is not
# 16-byte aligned) and has the kernel whose waves scatter or multiply for 65 and more of them here; every shape of that
# kernel: test_gpu_packed_products.py
@pytest.mark.parametrize("rows,cols,density,batch", [
    (12288, 300, 0.05, 17), (12285, 512, 0.1, 32), (12289, 513, 0.3, 33), (24575, 128, 0.5, 64), (12001, 1281, 0.2, 65), (11009, 767, 0.45, 128),
    (11500, 1025, 0.08, 128), (24001, 250, 0.3, 129), (49000, 70, 0.4, 40), (12288, 2000, 0.03, 100)])
def test_many_rows(rows, cols, density, batch):
    rng = np.random.default_rng(rows + cols + batch)
    dense, X = _case(rng, rows, cols, density, batch)
    dense[5::97] = 0                                                      # rows without entries
    full = np.arange(3, rows, 211)
    dense[full] = rng.standard_normal((full.size, cols)).astype(np.float16)   # more entries in a chunk than a pass holds
    dense[-1] = 0
    dense[-1, -1] = 1.0                                                   # one entry behind padding entries
    dense[::13, cols // 5:cols // 5 * 4] = 0                              # gaps wider than a lane's columns
    X[batch // 2, 1] = np.inf
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    Y = macko_spmv.multiply_batched(c, torch.from_numpy(X).cuda())
    got, finite = Y.cpu().numpy(), dense[:, 1] == 0   # a padding entry stands on column 15 at the first, never on column 1
    exact = np.where(np.isfinite(X), X, 0).astype(np.float16)
    spoiled = got[batch // 2]
    assert np.isfinite(spoiled[finite]).all() and not np.isfinite(spoiled[~finite]).any()
    spoiled[~finite] = (exact[batch // 2].astype(np.float64) @ dense.astype(np.float64).T).astype(np.float16)[~finite]
    _check(got, dense, exact, f"{rows}x{cols} d={density} b={batch}")
    assert torch.equal(Y.view(torch.int16), macko_spmv.multiply_batched(c, torch.from_numpy(X).cuda()).view(torch.int16))


@pytest.mark.parametrize("batch", [5, 16, 17, 100])
@pytest.mark.parametrize("offset,ldx,ldy", [(0, 1008, 304), (0, 1001, 301), (1, 1003, 300), (3, 1016, 303), (8, 1024, 302)])
def test_strided_and_unaligned_with_and_without_workspace(batch, offset, ldx, ldy):
    rng = np.random.default_rng(batch + ldx + offset)
    rows, cols = 300, 1001
    dense, _ = _case(rng, rows, cols, 0.3, 1)
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    flat = rng.standard_normal(offset + batch * ldx).astype(np.float16)
    flat_gpu = torch.from_numpy(flat).cuda()
    X = np.lib.stride_tricks.as_strided(flat[offset:], (batch, cols), (2 * ldx, 2))
    lib = ctypes.CDLL(macko_spmv_amd.HIP_LIBRARY_PATH)
    vp, i32, i64 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64
    lib.macko_spmv_f16_batched_ws.argtypes = [vp, vp, vp, vp, vp, i32, i32, i64, i32, i64, i64, vp, i64, vp]
    lib.macko_spmv_f16_batched_workspace.argtypes = [vp, i32, i32, i64, i32, i64, ctypes.POINTER(i64)]
    wanted = i64(-1)
    assert lib.macko_spmv_f16_batched_workspace(flat_gpu.data_ptr() + 2 * offset, rows, cols, c[0].numel(), batch, ldx,
                                                ctypes.byref(wanted)) == 0
    assert wanted.value >= 0
    scratch = torch.full((max(1, wanted.value),), 0xff, dtype=torch.uint8, device="cuda")
    for given in (0, wanted.value):
        Y = torch.full((batch, ldy), 7.0, dtype=torch.float16, device="cuda")
        rc = lib.macko_spmv_f16_batched_ws(c[0].data_ptr(), c[1].data_ptr(), c[2].data_ptr(), flat_gpu.data_ptr() + 2 * offset,
                                           Y.data_ptr(), rows, cols, c[0].numel(), batch, ldx, ldy,
                                           scratch.data_ptr() if given else None, given,
                                           torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        Y = Y.cpu().numpy()
        _check(Y[:, :rows], dense, X, f"offset {offset} ldx {ldx} workspace {given}")
        assert (Y[:, rows:] == 7.0).all()


@pytest.mark.parametrize("batch", [5, 40])
def test_inf_nan_and_subnormal_operands(batch):
    rng = np.random.default_rng(batch)
    rows, cols = 150, 900
    dense, X = _case(rng, rows, cols, 0.2, batch)
    dense[:, 300:312] = 0                      # columns no row stores ...
    dense[:, 299] = dense[:, 312] = 0.5        # (and no padding entry stands on)
    X[1, 300:312] = np.inf                     # ... and what no row may read
    X[2, 305] = np.nan
    X[3, :] = np.where(rng.random(cols) < 0.5, np.float16(3e-7), np.float16(-5e-8))   # subnormal halves
    dense[7, ::3] = np.float16(6e-8)
    X[0, 10] = -np.inf                         # read by the rows that store column 10
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    Y = macko_spmv.multiply_batched(c, torch.from_numpy(X).cuda()).cpu().numpy()
    values = c[0].cpu().numpy().view(np.uint16)
    for b in range(batch):
        want = mo.spmv(values, c[1].cpu().numpy(), c[2].cpu().numpy(), rows, cols, X[b]).view(np.float16)
        assert np.array_equal(np.isnan(Y[b]), np.isnan(want)) and np.array_equal(np.isinf(Y[b]), np.isinf(want)), b
        ok = np.isfinite(want)
        assert np.array_equal(Y[b][~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)])
        assert np.allclose(Y[b][ok].astype(np.float64), want[ok].astype(np.float64), rtol=2.0 ** -10, atol=1e-4 if b != 3 else 2.0 ** -23)


def test_malformed_matrices_end_and_stay_inside():
    # entries that decode to columns beyond cols, and row pointers that point anywhere: the call returns and the
    # rows that are well-formed are right
    rng = np.random.default_rng(9)
    rows, wide, cols, batch = 300, 900, 600, 20
    dense = helpers.random_sparse(rng, rows, wide, 0.2)
    dense[::3, cols:] = 0
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    X = rng.standard_normal((batch, cols)).astype(np.float16)
    Y = macko_spmv.multiply_batched((c[0], c[1], c[2], rows, cols), torch.from_numpy(X).cuda()).cpu().numpy()
    _check(Y[:, ::3], dense[::3, :cols], X, "columns beyond cols")
    for broken in (lambda p: p.flip(0), lambda p: p * 0 - 5, lambda p: p + 2 ** 30, lambda p: p * 0 + int(p[-1])):
        wrong = broken(c[2]).contiguous()
        out = macko_spmv.multiply_batched((c[0], c[1], wrong, rows, cols), torch.from_numpy(X).cuda())
        torch.cuda.synchronize()
        assert out.shape == (batch, rows)
    good = macko_spmv.compress(torch.from_numpy(np.ascontiguousarray(dense[:, :cols])).cuda())
    _check(macko_spmv.multiply_batched(good, torch.from_numpy(X).cuda()).cpu().numpy(), dense[:, :cols], X, "next call")


def test_captured_and_replayed():
    rng = np.random.default_rng(4)
    dense, X = _case(rng, 500, 1111, 0.3, 50)
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    Xg = torch.from_numpy(X).cuda()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        want = macko_spmv.multiply_batched(c, Xg)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = macko_spmv.multiply_batched(c, Xg)
        for k in range(4):
            got.zero_()
            Xg.mul_(-1.0)
            graph.replay()
            stream.synchronize()
            assert torch.equal(got, macko_spmv.multiply_batched(c, Xg))
            assert torch.equal(got, want if k % 2 else -want)
    torch.cuda.current_stream().wait_stream(stream)
