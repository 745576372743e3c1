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


def test_training_kernel_walks_its_tiles_with_it():
    src = open(os.path.join(ROOT, "acme-ecp_amd", "csrc", "crm_mlp.hip")).read()
    body = src[src.index("k_train("):src.index("k_reduce(")]
    assert "tiles_of(n, TROWS, blockIdx.x, gridDim.x)" in body and "int tile" not in body
