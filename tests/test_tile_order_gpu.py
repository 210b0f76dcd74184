"""The many-rows product where the order of its tiles, or the waves' taking turns, can go wrong: numbers of tiles that the eight
XCDs do not share evenly, bands of rows that end early, fewer stages along K than are in flight."""
import pytest
import torch

from test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K", [(257, 160, 64), (1025, 1600, 128), (2300, 1284, 192), (4097, 960, 320), (8192, 168, 256), (513, 8000, 64),
                                   (1500, 3840, 1280), (5000, 1280, 640)])
def test_every_tile_is_made_once(M, N, K):
    a, w, bias = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(N, K, seed=N, dtype=torch.bfloat16, scale=K ** -0.5), rnd(N, seed=3)
    wp, out, stream = ops().pack_matrix(w), torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV), rnd(M, N, seed=4)
    want = a.float() @ w.float().t() + bias
    ops().linear(a, wp, bias, out=out)
    # (32-bit sums of K products of numbers about 1 x K^-1/2, rounded to bfloat16: half a place of 2^-8 of the largest, about 6)
    assert (out.float() - want).abs().max().item() < 2e-2
    x = stream.clone()
    ops().linear(a, wp, bias, residual=x)
    assert (x - (stream + want)).abs().max().item() < 1e-3
