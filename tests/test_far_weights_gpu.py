"""Products of few rows whose weights are not all finite: a column has what its own weights make of it, whatever the others are."""
import pytest
import torch

from denno_beta_amd.kernels import ops

pytestmark = pytest.mark.gpu

INF = float("inf")


def _far(N, K):
    """(weights, the same with some that are not finite, the columns that have them): the first steps of K in the first columns, and others."""
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    far = w.clone()
    places = [(0, 0, INF), (3, 5, -INF), (7, 31, float("nan")), (9, 16, INF), (N - 1, K - 1, INF), (N // 2, K // 2, -INF)]
    for n, k, v in places:
        far[n, k] = v
    return w, far, sorted({n for n, _, _ in places})


def _columns_of_their_own(far, near, a, far_w, cols):
    others = [n for n in range(far.shape[1]) if n not in cols]
    assert torch.equal(far[:, others], near[:, others])
    want = a.double().cpu() @ far_w.double().cpu()[cols].t()
    got = far[:, cols].double().cpu()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[~want.isnan()], want[~want.isnan()])      # (infinities, each with its sign)


# (numbers of steps of 32 that no wave shares evenly: the last step alone, waves with a step less than others, and with none)
@pytest.mark.parametrize("K", [32, 40, 96, 200, 736, 1024, 1056, 1600, 2048, 5120])
def test_a_column_keeps_its_infinities_to_itself(K):
    for N in (48, 1024, 2064, 2576):
        w, far_w, cols = _far(N, K)
        packed = ops.pack_matrix(w), ops.pack_matrix(far_w)
        for M in (1, 8, 9, 16, 17, 40, 64):
            a = (1.0 + torch.rand(M, K, device="cuda")).bfloat16() * torch.where(torch.rand(M, 1, device="cuda") < 0.5, -1.0, 1.0).bfloat16()
            near, far = (ops.linear(a, x, out=torch.empty(M, N, device="cuda")) for x in packed)
            _columns_of_their_own(far, near, a, far_w, cols)


@pytest.mark.parametrize("M", [1, 8, 16, 64])
@pytest.mark.parametrize("K", [1024, 1600])
def test_behind_a_norm_in_the_product(M, K):
    N = 1600
    w, far_w, cols = _far(N, K)
    copy, stats = ops.norm_stream_buffers(M, K, "cuda")
    x, gamma = torch.zeros(M, K, device="cuda"), torch.ones(K, device="cuda")
    rows = torch.randn(M, K, device="cuda").bfloat16()
    ops.linear_norm_out(rows if M <= 16 else ops.pack_matrix(rows), ops.pack_matrix(torch.eye(K, device="cuda").bfloat16()), None, x, gamma, copy, stats)
    c1, c2 = ops.norm_folded(w, None, gamma, None)
    near, far = (ops.linear_norm_in(copy, stats, c1, c2, 1e-5, ops.pack_matrix(m), torch.empty(M, N, dtype=torch.bfloat16, device="cuda")) for m in (w, far_w))
    others = [n for n in range(N) if n not in cols]
    assert torch.equal(far[:, others], near[:, others]) and bool(near.isfinite().all()) and not bool(far[:, cols].isfinite().any())
