"""Products whose epilogue is an activation with numbers of its own, against the product and the activation one after the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 8, 9, 16, 17, 40, 64, 65, 100, 200, 257, 500, 1100, 2100]


def _operands(M, N, K):
    from denno_beta_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    return make(M, K).bfloat16(), ops.pack_matrix((make(N, K) * K ** -0.5).bfloat16()), make(N), make


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", [(2048, 512), (4096, 1024), (100, 72), (8192, 2048)])
def test_xielu(M, N, K):
    from denno_beta_amd.kernels import ops
    a, w, bias, _ = _operands(M, N, K)
    numbers = torch.tensor([0.9, 1.3], device="cuda")
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    z = ops.linear(a, w, bias, out=torch.empty(M, N, device="cuda"))
    did = ops.linear_act(a, w, "xielu", out, bias=bias, numbers=numbers)
    assert did or (M > 64 and (M <= 256 or K % 32 != 0))      # (beyond 64 rows: only where the many-rows kernel takes the product)
    if did:
        zd = z.double()
        low = zd.clamp(max=0)
        want = torch.where(zd > 0, 0.9 * zd * zd + 0.5 * zd, 1.3 * (torch.expm1(low) - low) + 0.5 * zd)
        # one rounding to bfloat16 (half of a last place: up to 2^-8 of the value), and where the function's terms cancel their own rounding in 32-bit
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-6 * (1 + zd.abs())).all())


def test_xielu_of_large_infinite_and_missing_values():
    from denno_beta_amd.kernels import ops
    for M in (3, 40, 300):
        K = N = 64
        w = ops.pack_matrix(torch.eye(64, device="cuda").bfloat16())
        a = torch.zeros(M, K, dtype=torch.bfloat16, device="cuda")
        a[0, :7] = torch.tensor([float("inf"), -1e30, -100.0, -0.5, -1e-20, 1e20, -3e38])
        z = ops.linear(a, w, out=torch.empty(M, N, device="cuda"))
        if not torch.equal(z[0, 1:7], a[0, 1:7].float()):      # (0 times infinity: the row's other columns are not numbers)
            a[0, 0] = 0.0
            z = ops.linear(a, w, out=torch.empty(M, N, device="cuda"))
        numbers = torch.tensor([0.9, 1.3], device="cuda")
        out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        assert ops.linear_act(a, w, "xielu", out, numbers=numbers)
        ref = ops.activate(z, "xielu", torch.empty_like(out), lower=numbers)
        assert torch.equal(out.isnan(), ref.isnan())
        both = ~ref.isnan()
        assert torch.allclose(out[both].float(), ref[both].float(), rtol=2.0 ** -7, atol=1e-30)


@pytest.mark.parametrize("M", [1, 2, 8, 9, 16, 17, 33, 64, 65, 300])
@pytest.mark.parametrize("N,K", [(1024, 64), (3072, 1024), (56, 40)])
def test_silu_and_decays_have_the_bits_of_two_kernels(M, N, K):
    from denno_beta_amd.kernels import ops
    a, w, bias, make = _operands(M, N, K)
    rates, cols = make(N).exp(), N - 8
    z = ops.linear(a, w, out=torch.empty(M, N, device="cuda"))
    out = torch.empty(M, N, device="cuda")
    did = ops.linear_act(a, w, "silu", out, cols=cols)
    assert did == (M <= 64)
    want = z.clone()
    ops.activate(want[:, :cols], "silu", want[:, :cols])
    if did:
        assert torch.equal(out, want)
    did = ops.linear_act(a, w, "exp_neg_softplus", out, bias=bias, numbers=rates)
    assert did == (M <= 64)
    if did:
        assert torch.equal(out, ops.activate(z, "exp_neg_softplus", torch.empty_like(z), bias=bias, lower=rates))
