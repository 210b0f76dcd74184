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


@pytest.mark.parametrize("N,K", [s for s in SIZES if s[0] % 16 == 0])
def test_the_next_norms_statistics_by_eights(N, K):
    from denno_beta_amd.kernels import ops
    a, w, bias, make = _case(N, K)
    gamma, beta, next_w = 1 + 0.1 * make(N), make(N), ops.pack_matrix((make(96, N) * N ** -0.5).bfloat16())
    for M in (1, 5, 8):
        assert ops.norm_stream_block(M, w) == 8 and ops.norm_stream_block(9, w) == 16
        x, y = make(M, N), None
        copies = []
        for block in (16, 8):
            y = x.clone()
            copy, stats = ops.norm_stream_buffers(M, N, "cuda", block)
            ops.linear_norm_out(a[:M], w, bias, y, gamma, copy, stats)
            rows = y.double().view(M, N // block, block)
            assert torch.allclose(stats[:, :, 0].double(), rows.mean(-1), rtol=1e-5, atol=1e-6)
            assert torch.allclose(stats[:, :, 1].double(), ((rows - rows.mean(-1, keepdim=True)) ** 2).sum(-1), rtol=1e-5, atol=1e-5)
            c1, c2 = ops.norm_folded(next_w.rows(), None, gamma, beta)
            copies.append((y, copy, ops.linear_norm_in(copy, stats, c1, c2, 1e-5, next_w, torch.empty(M, 96, dtype=torch.bfloat16, device="cuda"))))
        (y16, c16, o16), (y8, c8, o8) = copies
        assert torch.equal(y16, y8) and torch.equal(c16, c8)
        assert torch.equal(o16, o8)


def test_rows_beyond_eight_take_no_statistics_by_eights():
    from denno_beta_amd.kernels import ops
    a, w, bias, make = _case(64, 64)
    copy, stats = ops.norm_stream_buffers(9, 64, "cuda", 8)
    with pytest.raises(Exception):
        ops.linear_norm_out(a[:9], w, bias, make(9, 64), make(64), copy, stats)
