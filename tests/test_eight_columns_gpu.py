"""Products of up to 8 rows with 8 columns a workgroup, against the same rows among 16, which the kernel with 16 columns takes: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(16, 8), (24, 40), (8, 64), (320, 320), (1000, 200), (768, 768), (1024, 1000), (1024, 1024), (1600, 1600), (1024, 4096), (1280, 5120), (1600, 6400), (2048, 8192),
         (64, 16392), (2048, 136), (2056, 1024)]


def _case(N, K):
    from denno_beta_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(N + K)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    return make(16, K).bfloat16(), ops.pack_matrix((make(N, K) * K ** -0.5).bfloat16()), make(N), make


@pytest.mark.parametrize("N,K", SIZES)
def test_the_bits_of_sixteen_columns(N, K):
    from denno_beta_amd.kernels import ops
    a, w, bias, make = _case(N, K)
    x0 = make(16, N)
    for dtype, epilogue in ((torch.float32, "none"), (torch.bfloat16, "gelu_tanh")):
        want = ops.linear(a, w, bias, out=torch.empty(16, N, dtype=dtype, device="cuda"), epilogue=epilogue)
        for M in (1, 2, 7, 8):
            wide = torch.full((M, N + 8), 7.0, dtype=dtype, device="cuda")
            ops.linear(a[:M], w, bias, out=wide[:, :N], epilogue=epilogue)
            assert torch.equal(wide[:, :N], want[:M]) and bool((wide[:, N:] == 7.0).all()), M
    want = ops.linear(a, w, bias, residual=x0.clone())
    for M in (1, 3, 8):
        assert torch.equal(ops.linear(a[:M], w, bias, residual=x0[:M].clone()), want[:M]), M


@pytest.mark.parametrize("N,K", SIZES)
def test_against_64_bits(N, K):
    from denno_beta_amd.kernels import ops
    a, w, bias, make = _case(N, K)
    a, x0, rows = a[:8], make(8, N), w.rows().double()
    exact, size = a.double() @ rows.t() + bias.double(), a.double().abs() @ rows.abs().t() + bias.double().abs()
    # (sums of K products in 32 bits: every partial sum lies within the sum of the magnitudes, and K + 2 of them are rounded)
    bound = (K + 2) * 2.0 ** -23 * size
    for M in (1, 5, 8):
        got = ops.linear(a[:M], w, bias, out=torch.empty(M, N, device="cuda"))
        assert bool(((got.double() - exact[:M]).abs() <= bound[:M]).all())
        into = ops.linear(a[:M], w, bias, residual=x0[:M].clone())
        total = x0[:M].double() + exact[:M]
        assert bool(((into.double() - total).abs() <= bound[:M] + 2.0 ** -23 * total.abs()).all())
