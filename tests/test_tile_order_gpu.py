"""The many-rows product where the order of its tiles, or the waves' taking turns, can go wrong: numbers of tiles that the eight
XCDs do not share evenly, bands of rows that end early, fewer stages along K than are in flight."""
import math

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


@pytest.mark.parametrize("M,N,K", [(1028, 7200, 64), (1028, 7200, 128), (2300, 4000, 192), (2300, 4000, 1536), (1028, 7200, 1600), (2300, 4000, 2496),
                                   (2300, 4000, 2560), (1028, 7200, 2624), (2300, 7204, 4160)])
def test_waves_in_step_and_in_turns(M, N, K):
    """Tiles of 256 x 160, the ones whose waves may take turns: on both sides of the K from which they do (1,600 for 32-bit results, 2,560 for
    bfloat16), fewer stages of 64 along K than are asked for ahead, numbers of stages that leave every place of the three last; one band of rows
    and several, the last one short; columns beyond the last whole tile."""
    o = ops()
    assert o._lib_quiet("gemm").dn_gemm_tile(M, N, K) == 256160
    a, w, bias = rnd(M, K, seed=M, dtype=torch.bfloat16), rnd(N, K, seed=N, dtype=torch.bfloat16, scale=0.7 * K ** -0.5), rnd(N, seed=3)
    wp, out, stream = o.pack_matrix(w), torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV), rnd(M, N, seed=4)
    want = a.double() @ w.double().t() + bias.double()
    o.linear(a, wp, bias, out=out)
    # (bfloat16 rounds a number below 8 by at most 2^-6)
    assert want.abs().max().item() < 8 and (out.double() - want).abs().max().item() <= 2.0 ** -6 + 1e-4
    x = stream.clone()
    o.linear(a, wp, bias, residual=x)
    # (partial sums below 8 are off by at most 2^-22 a step, K steps)
    assert (x.double() - (stream.double() + want)).abs().max().item() <= (K + 2) * 2.0 ** -22


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
    # (a share's sum stays below 32, where a step rounds by at most 2^-20; the steps' errors go both ways: six times their root mean square)
    assert part.abs().max().item() < 32 and (x - want).abs().max().item() < 6 * math.sqrt(K / 3) * 2.0 ** -20
    assert torch.equal(out, o.layernorm(x, gamma, beta, 1e-5, torch.empty_like(out)))
