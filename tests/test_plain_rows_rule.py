"""Which products of few rows in the plain kernels leave their segments' sums in a workspace: a rule of the native library (the host
alone answers)."""
import pytest

from denno_beta_amd.build import load_library
from denno_beta_amd.kernels import ops


@pytest.fixture(scope="module")
def lib():
    """(The library as such: a question that launches nothing needs no GPU.)"""
    lib = load_library("gemm")
    ops._declare("gemm", lib)
    return lib


# (columns of a K in one kernel for 1 to 5, 6 to 8 and 9 to 16 rows; 0: none of those asked)
@pytest.mark.parametrize("N,longest", [(8, (3072, 2048, 3072)), (511, (3072, 2048, 3072)), (512, (4096, 3072, 4096)), (768, (7680, 6400, 6400)),
                                       (1024, (12288, 7680, 7680)), (1536, (16384, 16384, 4096)), (2048, (16384, 16384, 4096)), (2049, (16384, 7680, 4096)), (4095, (16384, 7680, 7680)), (4096, (16384, 16384, 7680)),
                                       (16384, (16384, 16384, 7680))])
def test_longest_inner_size_of_the_one_kernel(lib, N, longest):
    for rows, K in zip(((1, 5), (6, 8), (9, 16)), longest):
        for M in rows:
            assert lib.dn_gemm_work_floats(M, N, K, 0) == 0
            assert lib.dn_gemm_work_floats(M, N, K + 4, 0) == (K // 128 + 1) * M * N
    assert lib.dn_gemm_work_floats(17, N, 1024, 0) == 8 * 17 * N


@pytest.mark.parametrize("M,N,K,one", [(8, 8192, 252, True), (8, 16384, 252, False), (8, 16384, 256, True), (1, 16384, 252, False), (16, 16384, 132, True)])
def test_a_short_inner_size_beside_many_columns(lib, M, N, K, one):
    assert lib.dn_gemm_work_floats(M, N, K, 0) == (0 if one else 2 * M * N)
    # (either kernel writes a fused projection's cache; one of a single segment does not)
    assert lib.dn_gemm_plain_qkv_takes(0, K, 0, M, N, K, ops.F32) == 1
    assert lib.dn_gemm_plain_qkv_takes(0, 128, 0, M, N, 128, ops.F32) == 0
