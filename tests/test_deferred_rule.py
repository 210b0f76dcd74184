"""What `linear_deferred_shares` says is what the product behind it takes: one rule, the native one (the host alone answers)."""
import pytest
import torch

from denno_beta_amd.build import load_library
from denno_beta_amd.kernels import ops


@pytest.fixture(scope="module", autouse=True)
def gemm():
    """(The library as such: a question that launches nothing needs no GPU.)"""
    with pytest.MonkeyPatch.context() as m:
        lib = load_library("gemm")
        ops._declare("gemm", lib)
        m.setitem(ops._libs, "gemm", lib)
        yield


@pytest.mark.parametrize("M,N,K,shares", [
    (64, 1600, 6400, 0), (65, 1600, 6400, 4), (128, 1600, 6400, 4), (129, 1600, 6400, 2), (256, 1600, 6400, 2), (256, 1600, 1600, 2), (256, 1600, 448, 0),
    (257, 1280, 5120, 2), (300, 1280, 5120, 2), (512, 1280, 5120, 3), (257, 64, 4096, 4), (512, 1600, 6400, 0), (300, 1280, 1280, 2), (512, 1024, 1024, 2),
    (512, 1280, 1280, 0), (300, 1280, 960, 0), (513, 1280, 5120, 0), (513, 64, 4096, 0), (300, 2048, 4096, 0), (300, 1280, 5152, 0)])
def test_shares_of_a_deferred_product(M, N, K, shares):
    w = ops.PackedMatrix(torch.empty(0, dtype=torch.bfloat16), (N, K))
    assert ops.linear_deferred_shares(M, w) == shares
    assert ops.linear_deferred_shares(M, torch.empty(0)) == 0


@pytest.mark.parametrize("M", [65, 72, 128, 129, 136, 192, 203, 256])
@pytest.mark.parametrize("N", [64, 768, 1024, 1280, 1600, 2032])
def test_a_long_k_is_cut_alike_deferred_and_not(M, N):
    """From K = 4,096 on the product that adds into the stream itself cuts K too: into the same shares, so that a row is the same bits with its
    sum deferred and without."""
    for K in (4096, 5120, 6400, 8192):
        w = ops.PackedMatrix(torch.empty(0, dtype=torch.bfloat16), (N, K))
        floats = ops._libs["gemm"].dn_gemm_work_floats(M, N, K, ops.PACKED_W)
        assert floats == ops.linear_deferred_shares(M, w) * M * N, (M, N, K)
    for K in (1280, 1600, 3072):      # (cut only where the sum is deferred)
        assert ops.linear_deferred_shares(M, ops.PackedMatrix(torch.empty(0, dtype=torch.bfloat16), (N, K))) == 2
