"""Which products of several vectors go through the gather kernels and which to the matrix cores, and the gather
kernels' launches of eight, four, two and one vectors on the matrices that stay with them.  Bounds as in
test_gpu_batched_tile."""
import ctypes

import numpy as np
import pytest
import torch

import macko_spmv
import macko_spmv_amd
from oracle import macko_oracle as mo
from tests import helpers
from tests.test_gpu_batched_tile import _check

pytestmark = pytest.mark.gpu

vp, i32, i64 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64


def _library():
    lib = ctypes.CDLL(macko_spmv_amd.HIP_LIBRARY_PATH)
    lib.macko_spmv_f16_batched.argtypes = [vp, vp, vp, vp, vp, i32, i32, i64, i32, i64, i64, vp]
    lib.macko_spmv_f16_batched_workspace.argtypes = [vp, i32, i32, i64, i32, i64, ctypes.POINTER(i64)]
    return lib


def _on_matrix_cores(rows, cols, density, batch):
    # vectors that are not 16-byte aligned want scratch memory from 12000 elements on, and only on the matrix cores
    assert batch >= 4 and batch * cols >= 12000
    entries = int(rows * cols * density / (1 - (1 - density) ** 16)) // 8 * 8   # with padding entries, independent zeros
    wanted = i64(-1)
    assert _library().macko_spmv_f16_batched_workspace(2, rows, cols, entries, batch, cols | 1, ctypes.byref(wanted)) == 0
    return wanted.value > 0


def test_route_follows_rows_entries_and_vectors():
    # (measured where the two are clearly apart)
    for rows, cols, density, batch in [(28672, 4096, 0.05, 5), (28672, 4096, 0.05, 8), (28672, 4096, 0.1, 8), (28672, 8192, 0.05, 8),
                                       (28672, 8192, 0.1, 6), (28672, 8192, 0.2, 8), (8192, 28672, 0.05, 4)]:
        assert not _on_matrix_cores(rows, cols, density, batch), (rows, cols, density, batch)
    for rows, cols, density, batch in [(4096, 4096, 0.05, 8), (4096, 4096, 0.5, 5), (11008, 4096, 0.5, 8), (11008, 4096, 0.05, 16),
                                       (28672, 4096, 0.05, 16), (28672, 8192, 0.5, 12), (20000, 300, 0.1, 64)]:
        assert _on_matrix_cores(rows, cols, density, batch), (rows, cols, density, batch)


# 28672 x 1200 at 0.09 stays with the gather kernels for 8 vectors, 28672 x 2048 at 0.05 for 3, 5 and 8; fewer than 64
# columns always do; 9, 15: next to them
@pytest.mark.parametrize("rows,cols,density", [(28672, 1200, 0.09), (28672, 2048, 0.05), (300, 63, 0.5), (5000, 17, 0.3), (1, 1, 1.0)])
def test_products_around_the_gather_kernels_launches(rows, cols, density):
    rng = np.random.default_rng(rows + cols)
    dense = helpers.random_sparse(rng, rows, cols, density, scale=0.05)
    dense[rows // 2] = 0
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    X = rng.standard_normal((15, cols)).astype(np.float16)
    for batch in (2, 3, 4, 5, 8, 9, 15):
        Y = macko_spmv.multiply_batched(c, torch.from_numpy(X[:batch]).cuda())
        _check(Y.cpu().numpy(), dense, X[:batch], f"{rows}x{cols} d={density} b={batch}")


@pytest.mark.parametrize("rows,density", [(384, 0.6), (9000, 0.3)])   # rows split between waves, rows of one wave
def test_vectors_too_far_apart_for_the_matrix_cores(rows, density):
    # their offsets do not fit 32 bits: launches of eight, four, two and one
    rng = np.random.default_rng(rows)
    cols, batch, ldx = 4096, 15, 1 << 28
    dense = helpers.random_sparse(rng, rows, cols, density, scale=0.05)
    X = rng.standard_normal((batch, cols)).astype(np.float16)
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    wide = torch.empty((batch, ldx), dtype=torch.float16, device="cuda")
    wide[:, :cols] = torch.from_numpy(X).cuda()
    Y = torch.empty((batch, rows), dtype=torch.float16, device="cuda")
    assert _library().macko_spmv_f16_batched(c[0].data_ptr(), c[1].data_ptr(), c[2].data_ptr(), wide.data_ptr(), Y.data_ptr(), rows, cols,
                                             c[0].numel(), batch, ldx, rows, torch.cuda.current_stream().cuda_stream) == 0
    _check(Y.cpu().numpy(), dense, X, f"{rows} rows")


@pytest.mark.parametrize("batch", [2, 4, 8])
@pytest.mark.parametrize("rows,cols", [(28672, 1200), (400, 63)])
def test_inf_and_nan_where_no_row_has_an_entry(rows, cols, batch):
    rng = np.random.default_rng(cols + batch)
    dense = helpers.random_sparse(rng, rows, cols, 0.09 if cols > 63 else 0.5, scale=0.05)
    dense[:, 30:42] = 0
    dense[:, 29] = dense[:, 42] = 0.5          # no padding entry in between
    X = rng.standard_normal((batch, cols)).astype(np.float16)
    X[0, 30:42] = np.inf
    X[1, 35] = np.nan
    X[batch - 1, 10] = -np.inf                 # read by the rows that store column 10
    c = macko_spmv.compress(torch.from_numpy(dense).cuda())
    Y = macko_spmv.multiply_batched(c, torch.from_numpy(X).cuda()).cpu().numpy()
    for b in range(batch):
        want = mo.spmv(c[0].cpu().numpy().view(np.uint16), c[1].cpu().numpy(), c[2].cpu().numpy(), rows, cols, X[b]).view(np.float16)
        assert np.array_equal(np.isnan(Y[b]), np.isnan(want)) and np.array_equal(np.isinf(Y[b]), np.isinf(want)), b
        ok = np.isfinite(want)
        assert ok.any() and np.array_equal(Y[b][np.isinf(want)], want[np.isinf(want)])
        # each within 2^-11 of the exact sum, plus a few fp32 roundings of terms below 16 in all
        assert np.allclose(Y[b][ok].astype(np.float64), want[ok].astype(np.float64), rtol=2.0 ** -10, atol=1e-4)
