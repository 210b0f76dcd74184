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
        assert (tile in (64064, 64096, 128064)) == (((M + 127) // 128) * ((N + 63) // 64) <= 256)
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


# the first product beyond a round of 64 x 64, the last round of 64 x 96, the first beyond it, the last round of 128 x 64, the first beyond that
WIDE = [(203, 4160, 64096), (203, 6144, 64096), (203, 6208, 128064), (256, 8192, 128064), (256, 8256, 0), (65, 8256, 64096), (128, 12288, 64096), (320, 3264, 64064),
        (320, 3328, 64096), (320, 4896, 64096), (320, 4904, 128064), (384, 5440, 128064), (385, 4096, 128064), (512, 2304, 64096), (512, 4104, 0), (511, 3072, 64096)]


@pytest.mark.parametrize("M,N,tile", WIDE)
@pytest.mark.parametrize("K", [64, 192, 448, 1280])
def test_one_round_of_wide_products(M, N, tile, K):
    """65 to 512 rows of a wide product: every tile on both sides of the border to the next, fewer stages than are in flight and more."""
    assert ops()._lib_quiet("gemm").dn_gemm_wide_tile(M, N, K) == tile and ops()._lib_quiet("gemm").dn_gemm_wide_tile(M, N, K + 32) == 0
    a, w, bias = rnd(M, K, seed=M, dtype=BF), rnd(N, K, seed=N + 1000, dtype=BF, scale=K ** -0.5), rnd(N, seed=3)
    wp, exact, rounded, x0 = ops().pack_matrix(w), torch.empty(M, N, device=DEV), torch.full((M + 1, N), 7.0, dtype=BF, device=DEV), rnd(M, N, seed=4)
    ops().linear(a, wp, None, out=exact)
    within(exact, a, w)
    ops().linear(a, wp, bias, out=rounded[:M])
    assert torch.equal(rounded[:M], (exact + bias).to(BF)) and bool((rounded[M] == 7.0).all())
    ops().linear(a, wp, bias, out=rounded[:M], epilogue="gelu_tanh")
    # (half a unit of 8 bits, and what the kernel's tanh is off by)
    assert torch.allclose(rounded[:M].float(), torch.nn.functional.gelu(exact + bias, approximate="tanh"), rtol=2.0 ** -8, atol=2e-6)
    x = x0.clone()
    ops().linear(a, wp, bias, residual=x)
    assert (x - (x0 + (exact + bias))).abs().max().item() <= 2.0 ** -20      # (one more rounding of sums below 16)
    if M <= 256:
        ops().linear(ops().pack_matrix(a), wp, bias, out=rounded[:M])
        assert torch.equal(rounded[:M], (exact + bias).to(BF))


@pytest.mark.parametrize("M", [136, 203, 300, 320])
@pytest.mark.parametrize("heads,kv_heads,dh,ps", [(25, 25, 64, 16), (24, 24, 64, 16), (24, 4, 128, 16), (25, 25, 48, 32), (20, 20, 80, 24)])
def test_wide_fused_projections_write_the_cache(M, heads, kv_heads, dh, ps):
    """Against the product alone and the cache write alone, bit for bit: runs of slots that begin anywhere, rows without a slot."""
    K, qw, kvw = 128, heads * dh, kv_heads * dh
    N, pages = qw + 2 * kvw, M // ps + 3
    a, w, bias = rnd(M, K, seed=1).to(BF), ops().pack_matrix((rnd(N, K, seed=2) * K ** -0.5).to(BF)), rnd(N, seed=3)
    slots = torch.arange(M, dtype=torch.int32) + 3
    slots[5::97] = -1
    slots = slots.to(DEV)
    new = lambda: (torch.full((pages, kv_heads, ps, dh), 7.0, dtype=BF, device=DEV), torch.full((pages, kv_heads, dh, ps), 7.0, dtype=BF, device=DEV))      # noqa: E731
    (k0, v0), (k1, v1) = new(), new()
    plain, out = torch.empty(M, N, dtype=BF, device=DEV), torch.empty(M, qw, dtype=BF, device=DEV)
    ops().linear(a, w, bias, out=plain)
    ops().kv_write(plain, qw, qw + kvw, slots, k0, v0)
    q = ops().linear_qkv(a, w, bias, out, slots, k1, v1, qw)
    assert torch.equal(q, plain[:, :qw]) and torch.equal(k1, k0) and torch.equal(v1, v0)


@pytest.mark.parametrize("K", [64, 448, 4160])
def test_tiles_of_64_by_128_beyond_512_rows(K):
    """The list's tile that wide products of up to 512 rows have no use for."""
    o = ops()
    tile, wide = o._lib_quiet("gemm").dn_gemm_tile, o._lib_quiet("gemm").dn_gemm_wide_tile
    M, N = next((M, N) for M in range(300, 4200, 60) for N in range(2056, 9000, 104) if tile(M, N, K) == 64128 and wide(M, N, K) == 0)
    a, w = rnd(M, K, seed=M, dtype=BF), rnd(N, K, seed=N + 1000, dtype=BF, scale=K ** -0.5)
    out = torch.empty(M, N, device=DEV)
    o.linear(a, o.pack_matrix(w), None, out=out)
    within(out, a, w)


@pytest.mark.parametrize("M", [64, 65, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("N,K", [(3001, 1024), (4095, 512), (4097, 512), (1001, 4096), (1023, 4160), (1025, 4096), (2050, 1056)])
def test_some_rows_of_any_length(M, N, K):
    """Up to 128 rows of fewer than 4,096 columns, no multiple of 4, up to 192 of up to 1,024, and those on the other side of each border, from packed rows and from rows."""
    a, w = rnd(M, K, seed=M, dtype=BF), rnd(N, K, seed=N + 1000, dtype=BF, scale=K ** -0.5)
    wp = ops().pack_matrix(w)
    got = [torch.full((M + 1, N), 7.0, device=DEV) for _ in range(2)]
    ops().linear(a, wp, None, out=got[0][:M]), ops().linear(ops().pack_matrix(a), wp, None, out=got[1][:M])
    within(got[0][:M], a, w)
    assert torch.equal(got[0], got[1]) and bool((got[0][M] == 7.0).all())
