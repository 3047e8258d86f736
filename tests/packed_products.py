"""Products of vectors in operand order that test_gpu_packed_products.py runs, and the kernel each of them takes
(test_packed_routes_host.py)."""
import dataclasses

import numpy as np

from tests import helpers


@dataclasses.dataclass(frozen=True)
class Product:
    batch: int
    rows: tuple        # of each matrix
    cols: int
    density: float
    kernel: str        # with 256 compute units
    empty: int = -1    # the matrix without entries

    def __str__(self):
        return f"{self.kernel[5:9]}{self.kernel[16:]}-{self.batch}x{self.cols}"


PRODUCTS = [
    # lanes of 16 entries: a matrix without entries among others, in front of and behind them
    Product(17, (12288, 512, 4096), 257, 0.4, "spmv_pipe_kernel<1,16,true>", empty=1),
    Product(129, (2048, 2048, 2049), 300, 0.4, "spmv_pipe_kernel<4,16,true>", empty=0),
    # ... and arrays that end in the middle of a lane's entries
    Product(17, (9001,), 257, 0.3, "spmv_pipe_kernel<1,16,false>"),
    Product(129, (6143,), 257, 0.45, "spmv_pipe_kernel<4,16,false>"),
    # columns in several chunks: every width of vectors and of lanes, one and several matrices, the last one of any rows
    Product(17, (9003,), 1300, 0.1, "spmv_pipe_kernel<1,8,false>"),
    Product(32, (6140, 512, 2049), 1411, 0.12, "spmv_pipe_kernel<1,8,true>"),
    Product(31, (4096, 4096, 4093), 1300, 0.3, "spmv_pipe_kernel<1,16,true>"),
    Product(33, (12285,), 1281, 0.08, "spmv_pipe_kernel<2,8,false>"),
    Product(64, (8000, 2048, 2050), 1300, 0.1, "spmv_pipe_kernel<2,8,true>"),
    Product(63, (12285,), 1301, 0.4, "spmv_pipe_kernel<2,16,false>"),
    Product(40, (4096, 4096, 4095), 1300, 0.35, "spmv_pipe_kernel<2,16,true>"),
    Product(65, (12289,), 1281, 0.1, "spmv_pipe_kernel<4,8,false>"),
    Product(127, (4096, 4100, 4099), 1300, 0.08, "spmv_pipe_kernel<4,8,true>"),
    Product(128, (12287,), 1337, 0.5, "spmv_pipe_kernel<4,16,false>"),
    Product(128, (4096, 4096, 4094), 1300, 0.45, "spmv_pipe_kernel<4,16,true>"),
]

# an array that ends as near to 2^31 entries as is taken, and a row there that leaves more columns than that free
LONG_ARRAY = dict(entries=2 ** 31 - 8200, rows=524288, cols=16384, batch=17, kernel="spmv_pipe_kernel<1,16,false>")

# matrices of so unequal densities that each has a launch of its own: batch, rows of each, cols, their densities
UNEQUAL = dict(batch=16, rows=(11008, 11006), cols=1300, densities=(0.95, 0.03))


# sums that are long enough to show in the rounded results: batch, rows of each of several matrices (the kernel of two roles), cols,
# density; the matrices one by one go through the other kernel
SUMS = [(128, (4096, 4096, 4096), 4096, 0.5), (40, (4096, 4096, 4096), 4096, 0.3), (20, (4096, 4096, 4096), 4096, 0.4),
        (100, (4096, 4096, 4096), 2048, 0.1)]



# silu(gate) * up in one launch: rows of each of the two matrices, cols, vectors, density, and the kernel that is meant; every variant that
# takes several matrices
GATED = [
    (11256, 137, 20, 0.25, "spmv_pipe_kernel<1,8,true>"), (7912, 435, 31, 0.35, "spmv_pipe_kernel<1,16,true>"),
    (9016, 213, 53, 0.15, "spmv_pipe_kernel<2,8,true>"), (8952, 279, 37, 0.4, "spmv_pipe_kernel<2,16,true>"),
    (11192, 119, 110, 0.3, "spmv_pipe_kernel<4,8,true>"), (7800, 339, 119, 0.35, "spmv_pipe_kernel<4,16,true>"),
    (712, 619, 14, 0.4, "spmv_tile_kernel<1,1,1,true,true>"), (1576, 651, 23, 0.2, "spmv_tile_kernel<1,1,2,true,true>"),
    (488, 463, 60, 0.4, "spmv_tile_kernel<1,2,1,true,true>"), (736, 1027, 76, 0.2, "spmv_tile_kernel<1,2,2,true,true>"),
    (2728, 775, 12, 0.15, "spmv_tile_kernel<2,1,1,true,true>"), (2120, 1497, 22, 0.25, "spmv_tile_kernel<2,1,2,true,true>"),
    (1064, 971, 109, 0.7, "spmv_tile_kernel<2,2,1,true,true>"), (1192, 1677, 98, 0.07, "spmv_tile_kernel<2,2,2,true,true>"),
    (5736, 419, 11, 0.7, "spmv_tile_kernel<3,1,1,true,true>"), (4360, 1147, 28, 0.7, "spmv_tile_kernel<3,1,2,true,true>"),
    (5136, 487, 45, 0.9, "spmv_tile_kernel<3,2,1,true,true>"), (2504, 1249, 107, 0.3, "spmv_tile_kernel<3,2,2,true,true>"),
]


def gate_and_up(rows, cols, density):
    rng = np.random.default_rng(rows + cols)
    both = [helpers.random_sparse(rng, rows, cols, density, scale=0.1) for _ in range(2)]
    for m in both:
        m[rows // 2] = 0
    return both

def matrices(product):
    """The product's matrices: rows without entries, full rows, rows of one entry behind padding entries and gaps wider than
    a lane's columns; the stored arrays end 8 entries behind a multiple of 16."""
    rng = np.random.default_rng(sum(product.rows) + product.cols + product.batch)
    out = []
    for k, rows in enumerate(product.rows):
        if k == product.empty:
            out.append(np.zeros((rows, product.cols), dtype=np.float16))
            continue
        m = helpers.random_sparse(rng, rows, product.cols, product.density, scale=0.05)
        m[::13, product.cols // 5:product.cols // 5 * 4] = 0
        m[5::97] = 0
        full = np.arange(3, rows, 211)
        m[full] = rng.standard_normal((full.size, product.cols)).astype(np.float16)   # more entries in a chunk than a pass holds
        m[7] = 0
        m[7, -1] = 1.0
        m[0] = 0
        m[0, :(8 - stored_entries(m)) % 16] = 0.5
        out.append(m)
    return out


def stored_entries(m):
    """Entries of a compressed fp16 matrix: its non-zeros, and one for every 16 columns of the distance to the non-zero before."""
    padded = np.zeros((m.shape[0], m.shape[1] + 1), dtype=bool)
    padded[:, 0] = True   # a non-zero in front of the row
    padded[:, 1:] = m != 0
    at = np.flatnonzero(padded)
    gap = np.diff(at)
    first = at[1:] % (m.shape[1] + 1) == 0
    return int((((gap - 1) >> 4) + 1)[~first].sum())
