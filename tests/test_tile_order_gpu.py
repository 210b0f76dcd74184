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


@pytest.mark.parametrize("M,N,K", [(257, 1280, 5120), (320, 1280, 1280), (384, 1024, 4096), (512, 1280, 5120), (511, 96, 4096)])
def test_sums_left_for_the_norm_beyond_256_rows(M, N, K):
    o = ops()
    a, w, bias = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(N, K, seed=N, dtype=torch.bfloat16, scale=0.05), rnd(N, seed=3)
    wp, x0, gamma, beta = o.pack_matrix(w), rnd(M, N, seed=4), rnd(N, seed=5), rnd(N, seed=6)
    shares = o.linear_deferred_shares(M, wp)
    assert shares >= 2
    part = o.linear_deferred(a, wp)
    assert part.shape == (shares, M, N)
    x, out = x0.clone(), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    o.layernorm_join(x, part, bias, gamma, beta, 1e-5, out)
    want = (x0.double() + a.double() @ w.double().t() + bias.double()).float()
    assert torch.allclose(x, want, atol=2e-3, rtol=1e-4)
    assert torch.equal(out, o.layernorm(x, gamma, beta, 1e-5, torch.empty_like(out)))
