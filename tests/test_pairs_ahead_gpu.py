"""Products of up to 16 rows: the pairs of steps a wave asks for at once follow from K (one to four), with remainders of a pair, of a step, of a
wave's share, and K below one pair; with and without the second half of the rows."""
import pytest
import torch

from denno_beta_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [32, 64, 520, 1024, 1288, 1600, 2080, 5000])
@pytest.mark.parametrize("M", [1, 2, 8, 9, 16])
@pytest.mark.parametrize("N", [2064, 4100])
def test_pairs_ahead(M, N, K):
    torch.manual_seed(M * 7 + K)
    a = torch.randn(M, K, device="cuda").bfloat16()
    w = torch.randn(N, K, device="cuda").bfloat16()
    bias = torch.randn(N, device="cuda")
    stream = torch.randn(M, N, device="cuda")
    got = torch.empty(M, N, device="cuda")
    ops.linear(a, ops.pack_matrix(w), bias=bias, out=got)
    into = stream.clone()
    ops.linear(a, ops.pack_matrix(w), bias=bias, residual=into)
    exact = a.double() @ w.double().t() + bias.double()
    # (sums of K products in 32 bits: every partial sum lies within the sum of the magnitudes, and K + 2 of them are rounded)
    bound = (K + 2) * 2.0 ** -23 * (a.double().abs() @ w.double().abs().t() + bias.double().abs())
    assert ((got.double() - exact).abs() <= bound).all()
    assert ((into.double() - stream.double() - exact).abs() <= bound + 2.0 ** -23 * (stream.double().abs() + exact.abs())).all()
