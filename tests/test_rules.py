"""Which kernel takes a call: the rules of the kernel library that need no GPU to be asked."""
import pytest

from yalis_amd.ops.build import load_kernels
from yalis_amd.ops.hip import HipOps


@pytest.fixture(scope="module")
def lib():
    return load_kernels()


# tokens, heads, kv heads, requests, tokens of the longest span, keys, window
@pytest.mark.parametrize("step,form", [
    ((128, 32, 32, 128, 1, 20, 0), 0), ((128, 32, 32, 128, 1, 256, 0), 0), ((128, 32, 8, 128, 1, 2000, 64), 0),  # few keys: a wave a token
    ((200, 32, 8, 100, 2, 2, 0), 1),  # (two tokens of four heads fill half a tile)
    ((128, 32, 32, 128, 1, 300, 0), 2), ((128, 32, 8, 128, 1, 2000, 0), 2), ((231, 32, 32, 32, 200, 301, 0), 2), ((180, 32, 16, 60, 3, 203, 0), 2),
    ((352, 32, 32, 352, 1, 300, 0), 1), ((128, 32, 4, 128, 1, 2000, 0), 1), ((500, 32, 32, 100, 5, 5, 0), 1),
    ((2000, 32, 32, 1, 2000, 2000, 0), 1), ((8320, 32, 8, 64, 130, 130, 0), 1), ((1, 4096, 4096, 1, 1, 300, 0), 1),
])
def test_float32_attention_of_several_requests(lib, step, form):
    assert lib.yk_attn_f32_form(*step) == form


def test_what_is_taken_whole_is_not_refused_where_slices_would_do(lib):
    for n in (512, 1360, 2048, 3072, 4096, 5120, 6144, 8192, 28672):
        for k in (1024, 2048, 4096, 8192, 14336):
            for m in range(65, 2101, 13):
                whole, either = lib.yk_gemm_block_plan(m, n, k, 0, 0), lib.yk_gemm_block_plan(m, n, k, 1, 0)
                assert either >= 0 or whole < 0, (m, n, k)
                assert whole < 0 or whole % 256 == 1
                assert either < 0 or either % 256 > 1 or either == whole


@pytest.mark.parametrize("m", [129, 160, 192, 224, 256])
@pytest.mark.parametrize("n,k", [(8192, 28672), (8192, 22016), (7168, 20480), (6144, 16384), (5120, 13824), (4096, 14336), (3072, 8192)])
def test_long_matrices_are_cut_along_k(lib, m, n, k):
    plan = lib.yk_gemm_block_plan(m, n, k, 1, 0)
    assert plan >= 0 and plan % 256 > 1
    assert HipOps.long_matrix_tiles(m, n, k) and not HipOps.long_matrix_tiles(m, n, k, True)
    assert lib.yk_gemm_block_plan(m, n, k - 32, 1, 0) < 0  # then they are gemm_tile's
    assert HipOps.long_matrix_tiles(128, n, k, True) and not HipOps.long_matrix_tiles(257, n, k)


# rows, columns, K of a product with pairs (1) or an activation (2): faster without its pass in the product, and sizes beside them that are not
@pytest.mark.parametrize("m,n,k,kind", [(107, 2048, 8192, 1), (105, 2048, 4096, 1), (98, 3584, 28672, 1), (128, 4096, 2048, 1), (106, 14336, 8192, 1), (2366, 8192, 4096, 1),
                                        (2962, 4096, 5120, 1), (207, 8192, 5120, 2), (251, 7168, 5120, 2), (1300, 8192, 4096, 2)])
def test_long_products_that_leave_units_idle_keep_their_pass(lib, m, n, k, kind):
    assert lib.yk_gemm_block_plan(m, n, k, 0, kind) < 0


@pytest.mark.parametrize("m,n,k,kind", [(107, 2048, 768, 1), (103, 16384, 2048, 1), (999, 16384, 2048, 1), (1005, 8192, 4096, 1), (3985, 16384, 3072, 1), (512, 16384, 3072, 1),
                                        (8192, 28672, 4096, 1), (129, 2048, 1024, 2), (512, 8192, 2048, 2), (4096, 16384, 4096, 2)])
def test_products_that_gain_by_their_pass_have_it(lib, m, n, k, kind):
    assert lib.yk_gemm_block_plan(m, n, k, 0, kind) >= 0


# rows, columns, K of products that were slower in large tiles, whole or in slices, than by the kernels and the library beside them
@pytest.mark.parametrize("m,n,k", [(103, 1024, 3072), (110, 512, 3072), (103, 2560, 1024), (122, 3072, 1024), (536, 3584, 5120), (660, 1536, 3072),
                                   (3195, 1360, 8192), (893, 8192, 28672), (1844, 4096, 28672), (373, 8192, 6144), (364, 8192, 5120)])
def test_products_that_are_not_for_large_tiles(lib, m, n, k):
    assert lib.yk_gemm_block_plan(m, n, k, 1, 0) < 0 and lib.yk_gemm_block_plan(m, n, k, 0, 0) < 0


# rows beyond those that are taken apart at a time walk along K again, which pays where columns are many
@pytest.mark.parametrize("m,n,k,taken", [(1681, 916, 7264, False), (5677, 632, 6592, False), (2247, 848, 15788, False), (1472, 916, 7264, True), (2009, 7724, 5428, True),
                                         (2000, 6144, 4096, True), (8192, 2048, 8192, True)])
def test_float32_products_of_several_passes(lib, m, n, k, taken):
    assert (lib.yk_gemm_split_plan(m, n, k) > 0) == taken
