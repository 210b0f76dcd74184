"""Products of very many columns (a vocabulary): 32-bit rows of any length and place, on both sides of every border between the kernels and tiles."""
import pytest
import torch

from test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def within(got, a, w, epilogue=None):
    want = a.double() @ w.double().t()
    want = epilogue(want) if epilogue else want
    # (partial sums of K products about K^-1/2 stay below 8, where a step rounds by at most 2^-22)
    assert want.abs().max().item() < 8 and (got.double() - want).abs().max().item() <= (a.shape[1] + 2) * 2.0 ** -22


@pytest.mark.parametrize("M", [16, 17, 33, 64, 65, 128, 129, 203, 256, 257, 600])
@pytest.mark.parametrize("N,K", [(257, 128), (2049, 1024), (12287, 512), (12289, 576), (16385, 512), (16449, 512), (50257, 128), (50257, 512)])
@pytest.mark.parametrize("beyond", [0, 1, 3])
def test_rows_of_any_length_and_place(M, N, K, beyond):
    a, w = rnd(M, K, seed=M, dtype=BF), rnd(N, K, seed=N + 1000, dtype=BF, scale=K ** -0.5)
    held = torch.full((1 + (M + 1) * (N + beyond),), 7.0, device=DEV)
    rows = held[1:].view(M + 1, N + beyond)      # (a first element 4 bytes behind a multiple of 16)
    ops().linear(a, ops().pack_matrix(w), None, out=rows[:M, :N])
    within(rows[:M, :N], a, w)
    assert held[0].item() == 7.0 and bool((rows[M] == 7.0).all()) and bool((rows[:M, N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(17, 12288, 1024), (33, 12288, 512), (64, 16384, 1024), (64, 16448, 1024), (40, 20480, 1600), (65, 16384, 512), (65, 16448, 512), (128, 20480, 512),
                                   (203, 8192, 512), (203, 8256, 512), (256, 16384, 1600)])
def test_tiles_of_wide_products(M, N, K):
    """Few to some hundreds of rows, tiles of 64 and of more columns: rows of A in rows and packed, bias and activation, both types of result."""
    a, w, bias = rnd(M, K, seed=M, dtype=BF), rnd(N, K, seed=N + 1000, dtype=BF, scale=K ** -0.5), rnd(N, seed=3)
    wp, exact = ops().pack_matrix(w), torch.empty(M, N, device=DEV)
    tile = ops()._lib_quiet("gemm").dn_gemm_tile(M, N, K)
    if M <= 64:
        assert tile == (64064 if N <= 16384 else 64128)
    else:
        assert (tile in (64064, 128064)) == (((M + 127) // 128) * ((N + 63) // 64) <= 256)
    ops().linear(a, wp, None, out=exact)
    within(exact, a, w)
    packed = torch.empty_like(exact)
    ops().linear(ops().pack_matrix(a), wp, None, out=packed)
    assert torch.equal(packed, exact)
    ended, rounded = torch.empty_like(exact), torch.empty(M, N, dtype=BF, device=DEV)
    ops().linear(a, wp, bias, out=ended, epilogue="relu2")
    ops().linear(a, wp, bias, out=rounded, epilogue="relu2")
    assert torch.equal(ended, torch.relu(exact + bias) ** 2)
    assert torch.equal(rounded, ended.to(BF))


@pytest.mark.parametrize("M", [17, 64])
def test_activations_with_numbers_stay_where_they_were(M):
    """Products of 17 to 64 wide rows with an activation that only the few-rows kernel ends are one kernel still."""
    N, K = 12288, 512
    a, w = rnd(M, K, seed=M, dtype=BF), rnd(N, K, seed=N + 1000, dtype=BF, scale=K ** -0.5)
    out = torch.empty(M, N, device=DEV)
    assert ops().linear_act(a, ops().pack_matrix(w), "silu", out, cols=N)
    want = a.double() @ w.double().t()
    assert (out.double() - want * torch.sigmoid(want)).abs().max().item() < 1e-5
