"""How products of many rows leave: through LDS in whole pieces of 16 bytes where rows and columns allow it, four columns at a time elsewhere: the same bits."""
import pytest
import torch

from test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def operands(M, N, K):
    w = ops().pack_matrix((rnd(N, K, seed=2) * K ** -0.5).to(BF))
    return rnd(M, K, seed=1).to(BF), w, rnd(N, seed=3)


@pytest.mark.parametrize("M", [257, 600, 1025, 2049])
@pytest.mark.parametrize("N,K", [(128, 64), (1600, 128), (5120, 192), (6400, 64), (4800, 1280), (2056, 96)])
@pytest.mark.parametrize("epilogue", ["none", "gelu_tanh"])
def test_rows_of_any_stride_have_the_same_bits(M, N, K, epilogue):
    """Rows at multiples of 16 bytes, and rows 8 bytes longer (four columns at a time); both against 32-bit results of the same product."""
    a, w, bias = operands(M, N, K)
    whole, wider = torch.full((M + 1, N), 7.0, dtype=BF, device=DEV), torch.full((M + 1, N + 4), 7.0, dtype=BF, device=DEV)
    ops().linear(a, w, bias, out=whole[:M], epilogue=epilogue)
    ops().linear(a, w, bias, out=wider[:M, :N], epilogue=epilogue)
    assert torch.equal(whole[:M], wider[:M, :N])
    assert bool((whole[M] == 7.0).all()) and bool((wider[M] == 7.0).all()) and bool((wider[:M, N:] == 7.0).all())
    exact = torch.empty(M, N, device=DEV)
    ops().linear(a, w, bias, out=exact, epilogue=epilogue)
    # (the same sums, rounded once more: half a unit of 8 bits)
    assert bool(((whole[:M].float() - exact).abs() <= 2.0 ** -8 * exact.abs() + 1e-30).all())


@pytest.mark.parametrize("M", [257, 601, 1100, 2049])
@pytest.mark.parametrize("heads,kv_heads,dh,ps", [(25, 25, 64, 16), (16, 4, 64, 16), (8, 2, 48, 32), (5, 5, 80, 24), (20, 20, 64, 64), (3, 3, 16, 16), (12, 3, 128, 16)])
def test_queries_and_keys_of_many_rows_go_to_their_places(M, heads, kv_heads, dh, ps):
    """Against the product alone and the cache write alone, bit for bit: runs of slots that begin anywhere, rows without a slot, pages in any order."""
    K, qw, kvw = 128, heads * dh, kv_heads * dh
    N, pages = qw + 2 * kvw, M // ps + 3
    a, w, bias = operands(M, N, K)
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(4))
    slot = torch.arange(M) + 3
    slots = (order[slot // ps] * ps + slot % ps).to(torch.int32)
    slots[5::97] = -1
    slots = slots.to(DEV)
    new = lambda: (torch.full((pages, kv_heads, ps, dh), 7.0, dtype=BF, device=DEV), torch.full((pages, kv_heads, dh, ps), 7.0, dtype=BF, device=DEV))      # noqa: E731
    k0, v0 = new()
    plain = torch.empty(M, N, dtype=BF, device=DEV)
    ops().linear(a, w, bias, out=plain)
    ops().kv_write(plain, qw, qw + kvw, slots, k0, v0)
    for wide in (qw, N):
        k1, v1 = new()
        out = torch.full((M, wide), 7.0, dtype=BF, device=DEV)
        q = ops().linear_qkv(a, w, bias, out, slots, k1, v1, qw)
        assert torch.equal(q, plain[:, :qw]) and torch.equal(k1, k0) and torch.equal(v1, v0)
        assert wide == qw or torch.equal(out, plain)
