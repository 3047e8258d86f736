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

    def ask(cols, batch, matrices, residual=False):
        line = " ".join(str(v) for v in (cols, batch, int(residual), len(matrices), *(v for m in matrices for v in m)))
        return subprocess.run([program], input=line + "\n", stdout=subprocess.PIPE, text=True, check=True).stdout.split()

    return ask


@pytest.mark.parametrize("product", packed_products.PRODUCTS, ids=str)
def test_the_products_take_the_kernels_they_are_meant_for(routes, product):
    sizes = []
    for k, m in enumerate(packed_products.matrices(product)):
        values, _, _, n = mo.compress(m)
        assert n == packed_products.stored_entries(m)
        assert k == product.empty or values.size % 16 == 8
        sizes.append((m.shape[0], values.size))
    assert routes(product.cols, product.batch, sizes)[0] == product.kernel
    if len(sizes) == 1:
        assert routes(product.cols, product.batch, sizes, residual=True)[0] == product.kernel


def test_the_longest_array_takes_the_kernel_it_is_meant_for(routes):
    long = packed_products.LONG_ARRAY
    assert routes(long["cols"], long["batch"], [(long["rows"], long["entries"])])[0] == long["kernel"]
    assert routes(long["cols"], long["batch"], [(long["rows"], long["entries"] + 8)])[0] == "refused"
