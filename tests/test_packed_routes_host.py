"""Which kernel products of packed vectors launch, asked of the host code itself without a GPU (tile_routes.cpp)."""
import os
import subprocess

import pytest

from macko_spmv_amd import _build
from oracle import macko_oracle as mo
from tests import packed_products

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    directory = tmp_path_factory.mktemp("routes")
    obj, program = str(directory / "routes.o"), str(directory / "routes")
    include = os.path.join(os.path.dirname(HERE), "include")
    csrc = os.path.join(os.path.dirname(_build.__file__), "csrc")
    subprocess.run([_build._hipcc(), "-x", "hip", "--cuda-host-only", "-fuse-cuid=none", "-std=c++17", "-O1", "-fPIE", "-I" + include, "-I" + csrc,
                    "-c", os.path.join(HERE, "tile_routes.cpp"), "-o", obj], check=True)
    subprocess.run(["g++", "-pie", "-Wl,--defsym=__hip_fatbin=0", obj, "-o", program], check=True)

    def ask(cols, batch, matrices, residual=False, gated=False):
        line = " ".join(str(v) for v in (cols, batch, 2 if gated else int(residual), len(matrices), *(v for m in matrices for v in m)))
        return subprocess.run([program], input=line + "\n", stdout=subprocess.PIPE, text=True, check=True).stdout.split()  # an answer for each launch

    return ask


@pytest.mark.parametrize("product", packed_products.PRODUCTS, ids=str)
def test_the_products_take_the_kernels_they_are_meant_for(routes, product):
    sizes = []
    for k, m in enumerate(packed_products.matrices(product)):
        values, _, _, n = mo.compress(m)
        assert n == packed_products.stored_entries(m)
        assert k == product.empty or values.size % 16 == 8
        sizes.append((m.shape[0], values.size))
    launches = routes(product.cols, product.batch, sizes)
    assert [name.split(":")[0] for name in launches] == [product.kernel]
    if len(sizes) == 1:
        assert routes(product.cols, product.batch, sizes, residual=True) == launches


def test_the_longest_array_takes_the_kernel_it_is_meant_for(routes):
    long = packed_products.LONG_ARRAY
    assert routes(long["cols"], long["batch"], [(long["rows"], long["entries"])])[0].split(":")[0] == long["kernel"]
    assert routes(long["cols"], long["batch"], [(long["rows"], long["entries"] + 8)])[0] == "refused"


@pytest.mark.parametrize("rows,densities,batch,launches", [
    (11008, (0.5, 0.5), 16, 1), (11008, (0.9, 0.1), 16, 2), (11008, (0.1, 0.9), 128, 2), (11008, (0.7, 0.2), 2, 2), (11008, (0.5, 0.48), 128, 1),
    (4096, (0.5, 0.5, 0.5), 128, 1), (4096, (0.9, 0.1, 0.1), 16, 3), (4096, (0.9, 0.1, 0.1), 128, 1), (4096, (0.1, 0.9, 0.9), 2, 3),
    (512, (0.9, 0.1, 0.1), 16, 1), (4096, (0.3, 0.0, 0.3), 64, 1), (4096, (0.0, 0.0, 0.0), 64, 1)])
def test_matrices_of_unequal_densities_share_a_launch_where_it_takes_less_time(routes, rows, densities, batch, launches):
    sizes = [(rows, int(rows * 4096 * d) // 8 * 8) for d in densities]
    got = routes(4096, batch, sizes)
    assert len(got) == launches and got[0] != "refused"
    if launches > 1:   # each as it is launched on its own
        assert got == [routes(4096, batch, [size])[0] for size in sizes]


def test_the_unequal_matrices_are_launched_apart(routes):
    unequal = packed_products.UNEQUAL
    sizes = [(rows, int(rows * unequal["cols"] * max(d, 1 / 16)) // 8 * 8) for rows, d in zip(unequal["rows"], unequal["densities"])]
    assert len(routes(unequal["cols"], unequal["batch"], sizes)) == 2


@pytest.mark.parametrize("batch,rows,cols,density", packed_products.SUMS)
def test_long_sums_of_both_kernels(routes, batch, rows, cols, density):
    sizes = [(r, int(r * cols * density) // 8 * 8) for r in rows]
    together = routes(cols, batch, sizes)
    assert len(together) == 1 and together[0].startswith("spmv_pipe_kernel")
    assert all(routes(cols, batch, [size])[0].startswith("spmv_tile_kernel") for size in sizes)


@pytest.mark.parametrize("rows,cols,batch,density,kernel,chunk", [
    (26268, 576, 41, 0.128, "spmv_pipe_kernel<2,8,false>", 640), (16546, 640, 39, 0.085, "spmv_pipe_kernel<2,8,false>", 640),
    (28369, 110, 64, 0.2, "spmv_pipe_kernel<2,8,false>", 128), (28379, 244, 21, 0.17, "spmv_pipe_kernel<1,8,false>", 256),
    # rows that fill a pass, whose last round of units they do not
    (9831, 242, 64, 0.61, "spmv_pipe_kernel<2,16,false>", 384), (25680, 242, 138, 0.758, "spmv_pipe_kernel<4,16,false>", 384)])
def test_columns_that_fit_into_one_chunk(routes, rows, cols, batch, density, kernel, chunk):
    name, _, lds = routes(cols, batch, [(rows, int(rows * cols * density) // 8 * 8)])[0].split(":")
    pad = 2 * (16 * int(kernel.split(",")[1]) + 8)   # bytes behind a row; 48 rows, twice, and one pad in front
    assert name == kernel and int(lds) == pad + 96 * (2 * chunk + pad)


# Products between the two kernels: few rows in each workgroup, few columns, far more columns than rows; sums that would have fewer parts
# by the kernel of two roles.  us, by it and by the other one: 652 x 79, 215 vectors 4.89 and 4.04, 2164 x 221, 125 5.30 and 4.17, 4962 x 20544, 38
# 53.9 and 39.7, 5466 x 16693, 38 44.4 and 33.9; 4963 x 570, 82 vectors 5.9 and 7.2, but with half of the parts.
@pytest.mark.parametrize("rows,cols,batch,density,kernel", [
    (652, 79, 215, 0.914, "spmv_tile_kernel"), (1071, 191, 37, 0.3, "spmv_tile_kernel"), (2164, 221, 125, 0.389, "spmv_tile_kernel"),
    (2904, 293, 86, 0.448, "spmv_tile_kernel"), (4962, 20544, 38, 0.104, "spmv_tile_kernel"), (5466, 16693, 38, 0.113, "spmv_tile_kernel"),
    (8061, 13857, 23, 0.216, "spmv_tile_kernel"), (4963, 570, 82, 0.178, "spmv_tile_kernel"), (4421, 626, 79, 0.082, "spmv_tile_kernel"),
    (11008, 4096, 128, 0.5, "spmv_pipe_kernel"), (28672, 1024, 64, 0.1, "spmv_pipe_kernel"), (6149, 1024, 205, 0.507, "spmv_pipe_kernel"),
    (11514, 64, 172, 0.082, "spmv_pipe_kernel"), (26429, 225, 36, 0.695, "spmv_pipe_kernel")])
def test_the_choice_holds_for_products_of_any_size(routes, rows, cols, batch, density, kernel):
    assert routes(cols, batch, [(rows, int(rows * cols * density) // 8 * 8)])[0].startswith(kernel)


@pytest.mark.parametrize("rows,cols,batch,density", [(11008, 576, 128, 0.3), (12000, 513, 64, 0.35)])
def test_rows_of_more_than_512_columns_are_several_parts(routes, rows, cols, batch, density):
    # one chunk of 576 columns would hold them, as one block
    name, _, lds = routes(cols, batch, [(rows, int(rows * cols * density) // 8 * 8)])[0].split(":")
    assert name.startswith("spmv_pipe_kernel<") and ",16," in name and int(lds) == 528 + 96 * (2 * 384 + 528)


def test_several_matrices_leave_the_kernel_that_looks_them_up_row_by_row_sooner(routes):
    # gate and up of dim 1024, 17 vectors at 0.1: 5.26 us by the kernel of two roles, 5.61
    sizes = [(2752, 2752 * 1024 // 10 // 8 * 8)] * 2
    assert routes(1024, 17, sizes)[0].startswith("spmv_pipe_kernel")


@pytest.mark.parametrize("rows,cols,batch,density,kernel", packed_products.GATED)
def test_gate_and_up_take_the_kernel_they_are_meant_for(routes, rows, cols, batch, density, kernel):
    sizes = [(rows, -(-packed_products.stored_entries(m) // 8) * 8) for m in packed_products.gate_and_up(rows, cols, density)]
    launches = routes(cols, batch, sizes, gated=True)
    assert [name.split(":")[0] for name in launches] == [kernel]
    assert launches == routes(cols, batch, sizes)   # row blocks are whole units of eight rows where they are gated, of four otherwise


def test_several_matrices_of_few_columns_are_launched_as_each_of_them(routes):
    # a compiled graph, which launches gate and up one by one, gives the bits of the eager layer (dim 256, hidden 704)
    sizes = [(704, int(704 * 256 * 0.4) // 8 * 8)] * 2
    for gated in (False, True):
        assert routes(256, 19, sizes, gated=gated)[0].startswith("spmv_tile_kernel")
    assert routes(256, 19, sizes[:1])[0].startswith("spmv_tile_kernel")
