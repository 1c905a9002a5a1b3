"""Host-side checks of the products' plan and placement (weed_amd/csrc/matmul_plan.h), which need no GPU: every tile goes to one
workgroup, and the shapes of the GPU tests are planned as those tests say."""
import os
import subprocess

import pytest

from test_gpu_dense_ops import LARGE_TILES, PLACED, SHORT_SUMS
from test_zz_no_alloc import LARGE_IN_A_GRAPH, SCRATCH_BEFORE

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "plan_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", os.path.join(HERE, "plan_check.cpp"), "-o", exe], check=True)

    def run(*args):
        out = subprocess.run([exe] + [str(int(a)) for a in args], capture_output=True, text=True)
        assert out.returncode == 0, out.stdout + out.stderr
        return out.stdout.strip()

    return run


def _plan(check, M, N, K, batch=1, most=64, b_along_k=True, a_along_k=False):
    """Dense operands: off the 16-byte grid where what one of them is contiguous along is no multiple of four."""
    off_grid = (K if a_along_k else M) % 4 != 0 or (K if b_along_k else N) % 4 != 0
    words = check(M, N, K, batch, most, off_grid, b_along_k).split()
    return {k: int(v) for k, v in zip(words[::2], words[1::2])}


def test_every_tile_goes_to_one_workgroup(check):
    assert check() == "OK"


def test_large_tiles_of_the_gpu_tests(check):
    plans = [_plan(check, *shape, b_along_k=b, a_along_k=a) for a in (True, False) for b in (True, False) for shape in LARGE_TILES]
    assert all(p["tile"] == 256 and not p["strips"] for p in plans)
    assert [p["splits"] for p in plans] == 4 * [1, 1, 1, 3, 3]
    infinite = _plan(check, 2709, 921, 1501)
    assert (infinite["tile"], infinite["splits"], infinite["strips"]) == (256, 5, 0)


def test_placed_workgroups_of_the_gpu_tests(check):
    plans = [_plan(check, M, N, K, batch, 64 if batch == 1 else 1, a_along_k=True) for batch, M, N, K in PLACED]
    assert all(p["placed"] and not p["strips"] for p in plans)
    assert sum(p["wgs"] % 8 != 0 for p in plans) >= 5
    assert [p["tile"] for p in plans] == 6 * [128] + 2 * [256]
    assert [p["splits"] for p in plans] == [1, 1, 1, 1, 1, 5, 1, 5]
    assert [p["three"] for p in plans] == [1, 1, 0, 1, 0, 0, 0, 0]


def test_short_sums_of_the_gpu_tests(check):
    assert all(_plan(check, *shape)["three"] for shape in SHORT_SUMS)
    assert not _plan(check, 3331, 2309, 129)["three"] and not _plan(check, 2048, 4096, 128)["three"]


def test_captured_products_of_the_gpu_tests(check):
    plans = [_plan(check, *shape) for shape in LARGE_IN_A_GRAPH]
    assert [(p["tile"], p["splits"], p["strips"]) for p in plans] == [(128, 4, 0), (256, 5, 0), (256, 4, 0), (256, 3, 1), (256, 1, 0)]
    M, N, K = SCRATCH_BEFORE
    scratch = _plan(check, M, N, K)["splits"] * M * N
    rooms = [scratch // (m * n) for m, n, _ in LARGE_IN_A_GRAPH[:3]]
    assert rooms == [3, 3, 1]
    assert [_plan(check, *shape, most=room)["splits"] for shape, room in zip(LARGE_IN_A_GRAPH, rooms)] == [3, 2, 1]


@pytest.mark.parametrize("M,N,K,strips", [(1030, 4096, 4096, 1), (1100, 8192, 4096, 1), (2052, 4100, 1024, 1), (4100, 4100, 1024, 1),
                                          (4099, 4099, 1024, 1), (1000, 4100, 4096, 0), (1001, 4096, 4096, 0), (129, 16400, 4096, 0)])
def test_strips_are_taken_where_they_are_planned_to_be_faster(check, M, N, K, strips):
    """A few rows or columns more than whole rounds of tiles, and where the last round has room for them."""
    assert _plan(check, M, N, K)["strips"] == strips
