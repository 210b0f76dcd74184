"""The norm inside a product of 17 to 64 rows: its statistics go straight into LDS beside the operands, and the sums of K's last rounds."""
import pytest
import torch

from denno_beta_amd.kernels import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("M", [17, 31, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("K,N", [(1024, 2560), (1024, 96), (1056, 3072), (1280, 5120), (1600, 4800), (2016, 2592), (2048, 1600)])
@pytest.mark.parametrize("no_mean", [False, True])
def test_rows_are_the_bits_of_sixteen_rows(M, K, N, no_mean):
    """Against the kernel of up to 16 rows, whose sums stand in the same order, bit for bit, and against 64 bits; with statistics at multiples
    of 16 bytes and 8 bytes behind one."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    x0, a, gamma, beta = make(64, K) + 0.3, make(64, 1024).to(BF), 1 + 0.1 * make(K), 0.1 * make(K)
    before, w, bias = ops.pack_matrix((make(K, 1024) * 0.03).to(BF)), ops.pack_matrix((make(N, K) * K ** -0.5).to(BF)), make(N)
    c1, c2 = ops.norm_folded(w.rows(), bias, gamma, None if no_mean else beta, no_mean)

    def product(rows, apart=0):
        x, (copy, stats) = x0[rows].clone(), ops.norm_stream_buffers(len(x0[rows]), K, "cuda")
        ops.linear_norm_out(a[rows], before, None, x, gamma, copy, stats)
        if apart:
            held = torch.empty(stats.numel() + 2, device="cuda")
            held[2:] = stats.view(-1)
            stats = held[2:].view(stats.shape)
        out = torch.empty(len(x), N, dtype=BF, device="cuda")
        return x, ops.linear_norm_in(copy, stats, c1, c2, 1e-5, w, out, no_mean=no_mean)
    x, out = product(slice(0, M))
    for at in range(0, M, 16):
        xs, few = product(slice(at, min(at + 16, M)))
        assert torch.equal(x[at:at + 16], xs) and torch.equal(out[at:at + 16], few)
    assert torch.equal(product(slice(0, M), apart=1)[1], out)
    y = x.double()
    d = y if no_mean else y - y.mean(-1, keepdim=True)
    y = d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * gamma.double() + (0 if no_mean else beta.double())
    exact = y @ w.rows().double().T + bias.double()
    # (rows and results are rounded to 8 bits: 2^-9 of each operand's size, and of the result's)
    assert float((out.double() - exact).norm() / exact.norm()) < 2.0 ** -8


@pytest.mark.parametrize("M", [17, 40, 64])
@pytest.mark.parametrize("K", [1024, 1088, 2048, 2304, 2560, 2592, 4096, 4864, 5120, 6400, 7680])
def test_every_round_of_k_is_in_the_sums(M, K):
    """Into the stream, K in rounds of four and of five pairs a wave, whole and not: the bits of 16 rows."""
    N = 1280
    g = torch.Generator(device="cuda").manual_seed(M + K)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    a, w, bias, gamma, x0 = make(64, K).to(BF), ops.pack_matrix((make(N, K) * K ** -0.5).to(BF)), make(N), make(N), make(64, N)

    def product(rows):
        x, (copy, stats) = x0[rows].clone(), ops.norm_stream_buffers(len(x0[rows]), N, "cuda")
        ops.linear_norm_out(a[rows], w, bias, x, gamma, copy, stats)
        return x, stats
    x, stats = product(slice(0, M))
    for at in range(0, M, 16):
        xs, few = product(slice(at, min(at + 16, M)))
        assert torch.equal(x[at:at + 16], xs) and torch.equal(stats[at:at + 16], few)
    exact = x0[:M].double() + a[:M].double() @ w.rows().double().T + bias.double()
    # (32-bit sums: K terms of size 1 / sqrt(K), 2^-24 of the partial sums each)
    assert float((x.double() - exact).norm() / exact.norm()) < 1e-6
