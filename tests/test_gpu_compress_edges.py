"""The compressor at the edges of its lanes (8 columns), tiles (512) and rounds (2048), on rows that start at
any element: bit for bit what the checker gives."""
import ctypes
import time

import numpy as np
import pytest
import torch

import macko_spmv_amd as mk
from oracle import macko_oracle as mo

pytestmark = pytest.mark.gpu
COLS = (1, 3, 7, 8, 9, 15, 17, 63, 505, 511, 512, 513, 1000, 2041, 2048, 2055, 4096, 4099)


@pytest.mark.parametrize("int8", (False, True))
@pytest.mark.parametrize("density", (0.0, 0.02, 0.3, 0.97, 1.0))
@pytest.mark.parametrize("offset", (0, 1))
def test_compress_at_edges(int8, density, offset):
    rng = np.random.default_rng(int(density * 100) + offset)
    for cols in COLS:
        rows = int(rng.integers(1, 12))
        flat = rng.standard_normal(rows * cols + offset)
        flat = np.clip(np.rint(flat * 60), -128, 127).astype(np.int8) if int8 else flat.astype(np.float16)
        flat[rng.random(flat.size) >= density] = 0
        dense = flat[offset:].reshape(rows, cols)
        if rows > 3:
            dense[2] = 0
        if not int8 and density == 0.3:
            dense[0, cols // 2:] = -0.0
            dense[rows - 1, cols // 2] = np.nan
        M = torch.from_numpy(flat).cuda()[offset:].view(rows, cols)
        got = (mk.compress_int8 if int8 else mk.compress)(M)
        values, deltas, row_ptr, n = (mo.compress_int8 if int8 else mo.compress)(dense)
        v = got[0].cpu().numpy()
        assert np.array_equal(v if int8 else v.view(np.uint16), values), (cols, rows)
        assert np.array_equal(got[1].cpu().numpy(), deltas), (cols, rows)
        assert np.array_equal(got[2].cpu().numpy(), row_ptr), (cols, rows)


@pytest.mark.parametrize("int8", (False, True))
@pytest.mark.parametrize("density", (0.0, 0.0004, 0.05, 0.97))
def test_rows_of_several_waves(int8, density):
    # few long rows: pieces that end with the row, before it or after it, pieces without entries, rows without
    rng = np.random.default_rng(int(density * 10000))
    for rows, cols, offset in ((1, 8192, 0), (3, 8193, 1), (2, 9215, 0), (5, 12288, 0), (64, 16385, 1), (7, 49152, 0)):
        flat = rng.standard_normal(rows * cols + offset)
        flat = np.clip(np.rint(flat * 60), -128, 127).astype(np.int8) if int8 else flat.astype(np.float16)
        flat[rng.random(flat.size) >= density] = 0
        dense = flat[offset:].reshape(rows, cols)
        if rows > 2:
            dense[1] = 0
            dense[2, 1024:cols - 1024] = 0
            dense[0, cols // 2:] = 0
        if not int8:
            dense[rows - 1, cols // 2] = np.nan
        M = torch.from_numpy(flat).cuda()[offset:].view(rows, cols)
        got = (mk.compress_int8 if int8 else mk.compress)(M)
        values, deltas, row_ptr, n = (mo.compress_int8 if int8 else mo.compress)(dense)
        v = got[0].cpu().numpy()
        assert np.array_equal(v if int8 else v.view(np.uint16), values), (cols, rows)
        assert np.array_equal(got[1].cpu().numpy(), deltas), (cols, rows)
        assert np.array_equal(got[2].cpu().numpy(), row_ptr), (cols, rows)


# the last shapes whose rows are shared and the first whose are not; matrices of more than 128 MB, which are read past the cache
@pytest.mark.parametrize("rows,cols,int8", [
    (512, 2048, False), (512, 2047, False), (513, 2048, False), (1280, 8192, False), (1280, 8191, False), (1281, 8192, False),
    (512, 2048, True), (1280, 8192, True), (1280, 53001, False), (40, 1700001, False), (1280, 104999, True)])
def test_which_rows_several_waves_share(rows, cols, int8):
    rng = np.random.default_rng(rows + cols)
    dense = np.zeros((rows, cols), dtype=np.int8 if int8 else np.float16)
    for r in range(rows):
        at = np.flatnonzero(rng.random(cols, dtype=np.float32) < (0.0, 0.001, 0.05, 0.5)[r % 4])
        dense[r, at] = rng.integers(1, 100, size=at.size)
    dense[3::8, cols // 3:] = 0
    got = (mk.compress_int8 if int8 else mk.compress)(torch.from_numpy(dense).cuda())
    values, deltas, row_ptr, n = (mo.compress_int8 if int8 else mo.compress)(dense)
    v = got[0].cpu().numpy()
    assert np.array_equal(got[2].cpu().numpy(), row_ptr)
    assert np.array_equal(v if int8 else v.view(np.uint16), values)
    assert np.array_equal(got[1].cpu().numpy(), deltas)


@pytest.mark.parametrize("int8", (False, True))
def test_the_longest_row(int8):
    # 2^31 - 1 columns; non-zeros in the first, a middle and the last piece, one of them the last column
    cols = 2 ** 31 - 1
    at = torch.tensor([5, 4096, 2 ** 30 + 3, 2 ** 31 - 4099, 2 ** 31 - 520, 2 ** 31 - 2], device="cuda")
    M = torch.zeros(1, cols, dtype=torch.int8 if int8 else torch.float16, device="cuda")
    M[0, at] = torch.arange(1, 7, device="cuda", dtype=M.dtype)
    values, deltas, row_ptr = (mk.compress_int8 if int8 else mk.compress)(M)[:3]
    gap = torch.diff(at, prepend=torch.tensor([-1], device="cuda")) - 1
    place = torch.cumsum((gap >> 4) + 1, 0) - 1   # an entry for every 16 columns of a gap, and the non-zero's
    entries = int(place[-1]) + 1
    assert row_ptr.tolist() == [0, entries] and values.numel() == (entries + 7) // 8 * 8
    assert torch.equal(values.nonzero()[:, 0], place) and values[place].tolist() == [1, 2, 3, 4, 5, 6]
    nibbles = torch.stack((deltas & 15, deltas >> 4), 1).view(-1)
    assert torch.equal(nibbles[place], (gap & 15).to(torch.uint8)) and not nibbles[entries:].any()
    others = nibbles[:entries] != 15
    others[place] = False
    assert not others.any()


# the scan over the rows: 8 rows a thread, 8192 a slice, 24576 a round of the total, each one short of it, whole and one over
@pytest.mark.parametrize("rows", (1, 7, 8, 9, 8191, 8192, 8193, 16383, 16385, 24575, 24576, 24577, 49161))
def test_scan_of_the_rows(rows):
    rng = np.random.default_rng(rows)
    dense = rng.standard_normal((rows, 5)).astype(np.float16)
    dense[rng.random((rows, 5)) >= 0.4] = 0
    got = mk.compress(torch.from_numpy(dense).cuda())
    values, deltas, row_ptr, n = mo.compress(dense)
    assert np.array_equal(got[2].cpu().numpy(), row_ptr)
    assert np.array_equal(got[0].cpu().numpy().view(np.uint16), values)
    assert np.array_equal(got[1].cpu().numpy(), deltas)


# ... as the C interface has it: without a total, with one when row_ptr is complete, with one before it is
@pytest.mark.parametrize("rows", (1, 8, 8191, 8193, 16385, 24576, 24577, 49161))
@pytest.mark.parametrize("int8", (False, True))
def test_scan_of_the_rows_by_every_entry_point(rows, int8):
    rng = np.random.default_rng(rows)
    dense = rng.integers(-3, 4, (rows, 5)).astype(np.int8 if int8 else np.float16)
    row_ptr = (mo.compress_int8 if int8 else mo.compress)(dense)[2]
    M = torch.from_numpy(dense).cuda()
    lib, kind = ctypes.CDLL(mk.HIP_LIBRARY_PATH), "i8" if int8 else "f16"
    stream, other = torch.cuda.current_stream(), torch.cuda.Stream()
    pointer, i32 = ctypes.c_void_p, ctypes.c_int32
    for ending in ("count", "count_total", "count_early"):
        entry = getattr(lib, f"macko_compress_{kind}_{ending}")
        entry.argtypes = [pointer, i32, i32, pointer] + ([pointer] if ending != "count" else []) + [pointer]
        for with_total in (False, True) if ending != "count" else (False,):
            got = torch.full((rows + 1,), -1, dtype=torch.int32, device="cuda")
            total = torch.full((1,), -1, dtype=torch.int32).pin_memory()
            at = total.data_ptr() if with_total else None
            torch.cuda.synchronize()
            assert entry(M.data_ptr(), rows, 5, got.data_ptr(), *(() if ending == "count" else (at,)), stream.cuda_stream) == 0
            if ending == "count_total" and with_total:   # who sees the word finds row_ptr complete: read by a stream that waits for nothing
                until = time.monotonic() + 5.0
                while int(total) == -1 and time.monotonic() < until:
                    pass
                with torch.cuda.stream(other):
                    seen = got.to("cpu", non_blocking=False)
                assert np.array_equal(seen.numpy(), row_ptr)
            torch.cuda.synchronize()
            assert np.array_equal(got.cpu().numpy(), row_ptr)
            assert int(total) == (row_ptr[-1] if with_total else -1)
