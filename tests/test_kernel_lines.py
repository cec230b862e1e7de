"""Where one kernel hands over to another, as the library's own rules say it (host code of the built library, no GPU).  Each case lies in
a range that was measured slower on the other side of its line."""
import pytest

from wllm_amd.kernels import library


@pytest.fixture(scope="module")
def lib():
    return library.load()


@pytest.mark.parametrize("m,n,k,out", [
    (333, 2048, 2048, 0), (333, 2560, 2048, 0), (192, 8192, 2048, 0), (260, 2048, 768, 0), (200, 2560, 2048, 0),    # one or two workgroups a unit
    (400, 2048, 4096, 0), (288, 2560, 4096, 0), (400, 4096, 2048, 0),                                               # four
    (80, 8192, 768, 0),                                                 # one tile of rows, one workgroup a unit
    (140, 32768, 2048, 1), (129, 32768, 768, 1),                        # two a unit, one with all rows and one without
    (65, 32768, 2048, 1), (96, 32768, 2048, 1),                         # one tile of rows, two and more a unit
    (333, 32768, 2048, 1), (260, 32768, 2048, 1), (333, 2048, 16384, 1), (600, 2048, 4096, 1),                      # five and more
    (128, 32768, 2048, 0), (256, 2048, 16384, 0), (64, 32768, 2048, 0)])                                            # full tiles, few rows
def test_float32_tiles_leave_out_rows_where_the_launch_gets_shorter(lib, m, n, k, out):
    assert lib.wllm_gemm_f32_leaves_out(m, n, k) == out
