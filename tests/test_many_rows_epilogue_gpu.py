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


def into_cache(M, heads, kv_heads, dh, ps, beyond, q_more=0, K=128, packed=False):
    """The fused projection's queries and pages against the product alone with its keys and values put into the pages by torch, bit for bit."""
    qw, kvw = heads * dh + q_more, kv_heads * dh
    N, pages = qw + 2 * kvw, M // ps + 4
    a, w, bias = operands(M, N, K)
    a = ops().pack_matrix(a) if packed else a
    slot = torch.arange(M) + 3
    order = torch.cat([torch.randperm(pages - 1, generator=torch.Generator().manual_seed(4)), torch.tensor([pages - 1])])      # (the last page is nobody's)
    slots = (order[slot // ps] * ps + slot % ps).to(torch.int32)
    slots[5::97] = -1
    plain = torch.empty(M, N, dtype=BF, device=DEV)
    ops().linear(a, w, bias, out=plain)
    new = lambda: (torch.full((pages, kv_heads, ps, dh), 7.0, dtype=BF, device=DEV), torch.full((pages, kv_heads, dh, ps), 7.0, dtype=BF, device=DEV))      # noqa: E731
    k0, v0 = new()
    has = (slots >= 0).nonzero()[:, 0].to(DEV)
    page, off = slots.to(DEV).long()[has] // ps, slots.to(DEV).long()[has] % ps
    k0[page, :, off] = plain[has, qw:qw + kvw].view(-1, kv_heads, dh)
    v0[page, :, :, off] = plain[has, qw + kvw:].view(-1, kv_heads, dh)
    for wide in (qw, N):
        k1, v1 = new()
        rows = torch.full((M + 1, wide + beyond), 7.0, dtype=BF, device=DEV)
        q = ops().linear_qkv(a, w, bias, rows[:M, :wide], slots.to(DEV), k1, v1, qw)
        assert torch.equal(q, plain[:, :qw]) and torch.equal(k1, k0) and torch.equal(v1, v0)
        assert bool((rows[M] == 7.0).all()) and bool((rows[:M, wide:] == 7.0).all())
        assert wide == qw or torch.equal(rows[:M, :wide], plain)


# (dims that are multiples of 4 alone, of 8, of 16; widths of queries, and of keys, that end inside a block of 16 columns)
HEADS = [(8, 8, 40, 16), (16, 16, 24, 16), (16, 16, 20, 24), (5, 3, 20, 16), (6, 2, 20, 32), (8, 8, 72, 64), (8, 2, 104, 16), (3, 1, 100, 16), (9, 9, 4, 16),
         (7, 3, 12, 48), (4, 4, 64, 16), (4, 2, 48, 24)]


@pytest.mark.parametrize("M", [16, 64, 257, 513, 2049])
@pytest.mark.parametrize("heads,kv_heads,dh,ps", HEADS)
@pytest.mark.parametrize("beyond", [0, 4])
def test_heads_of_any_multiple_of_four(M, heads, kv_heads, dh, ps, beyond):
    """A block of 16 columns may hold the end of one head and the beginning of the next, or queries and keys, or keys and values."""
    into_cache(M, heads, kv_heads, dh, ps, beyond)


@pytest.mark.parametrize("M", [65, 203, 257, 300])
@pytest.mark.parametrize("heads,kv_heads,dh,ps", [(40, 40, 20, 16), (30, 30, 24, 24), (24, 24, 40, 16), (12, 12, 100, 16), (29, 3, 72, 32), (60, 20, 36, 16), (25, 25, 64, 16)])
@pytest.mark.parametrize("beyond", [0, 4])
def test_wide_heads_of_any_multiple_of_four(M, heads, kv_heads, dh, ps, beyond):
    """2,048 columns and more: the tiles of 65 to 512 rows."""
    into_cache(M, heads, kv_heads, dh, ps, beyond)


@pytest.mark.parametrize("M", [64, 300, 2049])
@pytest.mark.parametrize("q_more", [4, 8, 12])
@pytest.mark.parametrize("dh", [40, 64])
def test_queries_that_end_inside_a_block(M, q_more, dh):
    """Whole heads of 16 dims behind queries that are no whole blocks."""
    into_cache(M, 10, 10, dh, 16, 0, q_more)


@pytest.mark.parametrize("M", [1100, 2049])
@pytest.mark.parametrize("heads,kv_heads,dh,K", [(40, 40, 40, 1280), (16, 16, 100, 96), (64, 64, 20, 64), (25, 25, 64, 1280)])
def test_large_tiles_with_heads_of_any_multiple_of_four(M, heads, kv_heads, dh, K):
    """Thousands of columns: the tiles of 128 and 256 rows, in both widths of a stage."""
    into_cache(M, heads, kv_heads, dh, 16, 0, K=K)


@pytest.mark.parametrize("M,K", [(17, 1024), (32, 1088), (33, 512), (64, 576)])
@pytest.mark.parametrize("heads,kv_heads,dh", [(64, 64, 64), (65, 64, 64), (128, 128, 64), (103, 103, 40), (200, 4, 64), (131, 129, 64)])
@pytest.mark.parametrize("packed", [False, True])
def test_few_rows_of_very_many_columns_write_the_cache(M, K, heads, kv_heads, dh, packed):
    """Few rows and 12,288 columns or more: tiles of 64 x 64, and of 64 x 128 where those are more than the CUs."""
    assert ops()._lib_quiet("gemm").dn_gemm_tile(M, (heads + 2 * kv_heads) * dh, K) == (64064 if (heads + 2 * kv_heads) * dh <= 16384 else 64128)
    into_cache(M, heads, kv_heads, dh, 16, 0, K=K, packed=packed)


@pytest.mark.parametrize("K", [1216, 1280, 2240, 2304])
@pytest.mark.parametrize("epilogue", ["gelu_tanh", "gelu_erf"])
def test_tiles_of_256_by_160_in_step_and_in_turns(K, epilogue):
    """On both sides of the borders from which their waves take turns: the results in 32-bit, rounded."""
    M, N = 1500, 6400
    assert ops()._lib("gemm").dn_gemm_tile(M, N, K) == 256160
    a, w, bias = operands(M, N, K)
    got, exact = torch.full((M + 1, N), 7.0, dtype=BF, device=DEV), torch.empty(M, N, device=DEV)
    ops().linear(a, w, bias, out=got[:M], epilogue=epilogue)
    ops().linear(a, w, bias, out=exact, epilogue=epilogue)
    assert bool(((got[:M].float() - exact).abs() <= 2.0 ** -8 * exact.abs() + 1e-30).all()) and bool((got[M] == 7.0).all())
