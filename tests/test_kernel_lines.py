"""Where one kernel hands over to another, as the library's own rules say it (host code of the built library, no GPU).  Each case lies in
a range that was measured slower on the other side of its line."""
import numpy as np
import pytest

from wllm_amd.kernels import attention_plan, hip_backend, library


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


@pytest.mark.parametrize("m,k,norm,takes", [
    (1, 256, 0, 1), (8, 256, 0, 1), (9, 256, 0, 0), (16, 512, 0, 0), (16, 960, 0, 0), (16, 1024, 0, 1), (17, 1024, 0, 0), (32, 512, 0, 0), (25, 768, 0, 0),
    (13, 2048, 0, 1), (14, 2048, 0, 0), (8, 3072, 0, 1), (9, 3072, 0, 0),
    (8, 512, 1, 1), (9, 512, 1, 0), (16, 1024, 1, 0), (9, 1536, 1, 0), (13, 2048, 1, 1), (14, 2048, 1, 0)])
def test_gated_products_keep_x_whole_where_that_pays(lib, m, k, norm, takes):
    assert lib.wllm_gated_rows_take(m, k, norm) == takes


@pytest.mark.parametrize("n,nh,nkv,d,rot,by_heads", [
    (1, 1, 1, 32, 32, 0), (64, 14, 2, 64, 64, 0), (1, 14, 2, 64, 64, 0),                              # at most one round of pairs
    (1, 8, 1, 256, 256, 1), (64, 8, 1, 256, 256, 1), (65, 8, 1, 256, 256, 0), (42, 16, 4, 128, 128, 1), (43, 16, 4, 128, 128, 0),
    (64, 32, 8, 128, 128, 1), (64, 16, 16, 256, 256, 1), (64, 40, 40, 64, 64, 1), (65, 40, 40, 64, 64, 0), (128, 64, 64, 64, 64, 0),
    (16, 16, 16, 256, 36, 0), (16, 2100, 1000, 4, 8, 0), (16, 16, 16, 260, 256, 0)])                  # sizes that the other kernel does not take
def test_the_rotation_goes_by_heads_where_that_pays(lib, n, nh, nkv, d, rot, by_heads):
    assert lib.wllm_rope_by_heads(n, nh, nkv, d, rot, 16) == by_heads


@pytest.mark.parametrize("nh,nkv,portion,decoded,pays", [
    (8, 1, (448, 896), (60, 1500), True), (16, 16, (448, 896), (32, 1500), True), (64, 8, (448, 3000), (8, 2048), True),
    (16, 16, (448, 896), (256, 300), False), (32, 8, (64, 64), (128, 4000), False), (40, 40, (448, 896), (60, 4000), False),
    (64, 8, (448, 3000), (128, 1500), True), (64, 8, (448, 3000), (256, 1500), True), (40, 40, (448, 3000), (40, 1500), True)])
def test_portions_run_beside_decoded_tokens_where_that_pays(nh, nkv, portion, decoded, pays):
    count, keys = decoded
    q_len, ctx_len = np.array([portion[0]] + [1] * count), np.array([portion[1]] + [keys] * count)
    items, _, _, prefill, rows = attention_plan.build_work_items(q_len, ctx_len, nh // nkv, nkv, 0)
    assert hip_backend.HipBackend.portions_pay_beside(prefill, rows, items.shape[0]) is pays


@pytest.mark.parametrize("rows,columns,k,tile", [
    (300, 250, 3072, None), (2048, 64, 3072, None), (1024, 128, 3072, None), (2049, 64, 3072, (64, 64)), (300, 512, 3072, (64, 64)),
    (512, 512, 4096, None), (1024, 250, 4096, None), (2048, 128, 4096, None), (640, 512, 4096, (64, 64)),
    (256, 64, 4096, (64, 64)), (257, 64, 2048, (64, 64))])
def test_gated_products_of_few_tiles_and_many_keys_are_the_librarys(rows, columns, k, tile):
    """Beyond 256 rows; up to there the tiles of 128 take twice as long."""
    assert hip_backend.HipBackend.block_gated_tile(rows, columns, k) == tile


def test_products_of_one_round_refuse_more(lib):
    """257 tiles of 64 by 64; 256 pieces times two tiles."""
    fn = lib.wllm_gemm_block
    fn.argtypes = hip_backend._SIGNATURES["wllm_gemm_block"]
    sizes = [(64 * 257, 64, 64, 64, 1), (64, 64 * 256 + 1, 64, 64 * 257, 1), (65, 64, 64 * 256, 64, 256)]
    for m, n, k, stride, splits in sizes:
        out, partial = (None, 4096) if splits > 1 else (4096, None)
        assert fn(4096, 4096, out, partial, m, n, k, stride, splits, 0, 0.0, 0.0, 0.0, 64, 64, None) == -1
