"""The grid-stride walks of the kernels (acme-ecp_amd/csrc/crm_index.hpp), built for the host: every
tile is taken once and no index wraps, up to the largest batch an int counts."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INT_MAX = 2**31 - 1


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    exe = tmp_path_factory.mktemp("index") / "index_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "acme-ecp_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "native", "index_check.cpp")], check=True)
    return lambda *a: [int(x) for x in subprocess.run([str(exe)] + [str(v) for v in a], check=True,
                                                       capture_output=True, text=True).stdout.split()]


# the last rows below 2^31, where tile 64 x 256 workgroups ahead passes it
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 16384, INT_MAX - 64 * 256, INT_MAX - 1, INT_MAX])
@pytest.mark.parametrize("blocks", [1, 7, 256])
def test_training_tiles(walk, rows, blocks):
    taken, last, wrapped = walk(rows, 64, blocks)
    assert (taken, last, wrapped) == (-(-rows // 64), (rows - 1) // 64 * 64, 0)


# rows on both sides of 2^31 and 2^32, with the levels of 28-level columns of that many
@pytest.mark.parametrize("row", [0, 1, 2**31 - 1, 2**31, 2**32 - 1, 2**32, 28 * (2**31 - 1) - 1])
@pytest.mark.parametrize("nrad", [1, 16, 76695845, 2**31 - 1])
def test_level_of_a_row(walk, row, nrad):
    if row // nrad <= INT_MAX:
        assert walk(row, nrad, 0, 0) == [row // nrad]


def test_gcm_kernels_count_rows_with_it():
    src = open(os.path.join(ROOT, "acme-ecp_amd", "csrc", "crm_glue.hip")).read()
    assert src.count("(long)nrad * crm_nz") + src.count("(long)nrad * pver") >= 6
    for product in ("nrad * crm_nz", "nrad * pver"):
        assert src.count(product) == src.count("(long)" + product)


def test_training_kernel_walks_its_tiles_with_it():
    src = open(os.path.join(ROOT, "acme-ecp_amd", "csrc", "crm_mlp.hip")).read()
    body = src[src.index("k_train("):src.index("k_reduce(")]
    assert "tiles_of(n, TROWS, blockIdx.x, gridDim.x)" in body and "int tile" not in body
