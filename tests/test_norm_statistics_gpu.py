"""The statistics that a product of up to 64 rows leaves for the norm behind it: one order of sums, whichever kernel has the rows."""
import numpy as np
import pytest
import torch

from denno_beta_amd.kernels import ops

pytestmark = pytest.mark.gpu


def sums_of_sixteen(first, others):
    """Lane 0's sum of 16 lanes: neighbours (`first` does the first step), pairs, halves of 8 mirrored, 16 mirrored."""
    lanes, v = np.arange(16), first
    for partner in others:
        v = (v + v[..., partner(lanes)]).astype(np.float32)
    return v[..., 0]


STEPS = [lambda i: i ^ 2, lambda i: i // 8 * 8 + 7 - i % 8, lambda i: 15 - i]


def statistics(rows):
    """[M, N] 32-bit -> [M, N / 16, 2]: mean and sum of squared distances of each 16 columns, every step rounded to 32 bits; the first step
    of the squares' sum is one multiply-add (in 64 bits its sum is off by 2^-53, which the rounding to 24 bits behind it does not see)."""
    x = rows.cpu().numpy().reshape(rows.shape[0], -1, 16)
    other = x[..., np.arange(16) ^ 1]
    mean = sums_of_sixteen((x + other).astype(np.float32), STEPS) * np.float32(1 / 16)
    d = (x - mean[..., None]).astype(np.float32)
    squares = (d * d).astype(np.float32)
    first = (d.astype(np.float64) ** 2 + squares[..., np.arange(16) ^ 1].astype(np.float64)).astype(np.float32)
    return torch.from_numpy(np.stack([mean, sums_of_sixteen(first, STEPS)], axis=-1))


@pytest.mark.parametrize("M", [1, 5, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(1024, 1024), (1600, 1600), (1280, 5120), (2048, 1032)])
def test_statistics_are_of_sixteen_columns_in_one_order(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    a, w = make(64, K).bfloat16(), ops.pack_matrix((make(N, K) * K ** -0.5).bfloat16())
    bias, gamma, x0 = make(N), 1 + 0.1 * make(N), make(64, N)
    x = x0[:M].clone()
    copy, stats = ops.norm_stream_buffers(M, N, "cuda")
    ops.linear_norm_out(a[:M], w, bias, x, gamma, copy, stats)
    assert tuple(stats.shape) == (M, N // 16, 2) and torch.equal(stats.cpu(), statistics(x))
    # and the norm in the product behind it: a row's bits are those that it has among 16 rows
    if M > 16:
        return
    x16, (copy16, stats16) = x0[:16].clone(), ops.norm_stream_buffers(16, N, "cuda")
    ops.linear_norm_out(a[:16], w, bias, x16, gamma, copy16, stats16)
    assert torch.equal(x16[:M], x) and torch.equal(copy16[:M], copy) and torch.equal(stats16[:M], stats)
    nxt = ops.pack_matrix((make(96, N) * N ** -0.5).bfloat16())
    c1, c2 = ops.norm_folded(nxt.rows(), None, gamma, make(N))
    out = ops.linear_norm_in(copy, stats, c1, c2, 1e-5, nxt, torch.empty(M, 96, dtype=torch.bfloat16, device="cuda"))
    out16 = ops.linear_norm_in(copy16, stats16, c1, c2, 1e-5, nxt, torch.empty(16, 96, dtype=torch.bfloat16, device="cuda"))
    assert torch.equal(out, out16[:M])
