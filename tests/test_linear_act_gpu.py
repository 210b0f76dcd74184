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


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", [(2048, 512), (4096, 1024), (100, 72), (8192, 2048)])
def test_xielu_has_the_bits_of_two_kernels(M, N, K):
    from denno_beta_amd.kernels import ops
    a, w, bias, _ = _operands(M, N, K)
    numbers = torch.tensor([0.9, 1.3], device="cuda")
    for b in (None, bias):
        out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        z = ops.linear(a, w, b, out=torch.empty(M, N, device="cuda"))
        if ops.linear_act(a, w, "xielu", out, bias=b, numbers=numbers):
            assert torch.equal(out, ops.activate(z, "xielu", torch.empty_like(out), lower=numbers))
        else:
            assert M > 64 and (M <= 256 or K % 32 != 0)


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


@pytest.mark.parametrize("M", [1, 2, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("first,rest,K", [(128, 1544, 1024), (16, 3, 8), (64, 3000, 512), (80, 40000, 40)])
def test_two_products_of_the_same_rows(M, first, rest, K):
    from denno_beta_amd.kernels import ops
    a, w1, _, make = _operands(M, first, K)
    w2 = ops.pack_matrix((make(rest, K) * K ** -0.5).bfloat16())
    both, v1, v2 = ops.stacked(w1, w2)
    assert torch.equal(v1.rows(), w1.rows()) and torch.equal(v2.rows(), w2.rows()) and both.shape == (first + rest, K)
    low, z = ops.linear_two(a, both, first)
    one = ops.linear(a, both, out=torch.empty(M, first + rest, device="cuda"))
    assert torch.equal(z, one[:, first:]) and torch.equal(low, one[:, :first].bfloat16())
    # (up to 64 rows the order of a sum follows from K alone: the products one after the other have the same bits)
    assert torch.equal(z, ops.linear(a, w2, out=torch.empty(M, rest, device="cuda")))
    assert torch.equal(low, ops.linear(a, w1, out=torch.empty(M, first, dtype=torch.bfloat16, device="cuda")))


@pytest.mark.parametrize("M", [1, 2, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("n1,n2,K", [(512, 1024, 64), (64, 8, 8), (256, 2560, 72), (2560, 5120, 16)])
def test_two_products_of_neighbouring_columns(M, n1, n2, K):
    from denno_beta_amd.kernels import ops
    _, w1, _, make = _operands(M, n1, K)
    w2, low, rate, bias = ops.pack_matrix((make(n2, K) * K ** -0.5).bfloat16()), make(M, 2 * K).bfloat16(), make(n1).exp(), make(n1 + n2)
    both = ops.stacked(w1, w2)[0]
    g, gate = ops.linear_pair(low, both, n1, bias, rate)
    z = ops.linear(low[:, :K], w1, out=torch.empty(M, n1, device="cuda"))
    assert torch.equal(g, ops.activate(z, "exp_neg_softplus", torch.empty_like(z), bias=bias[:n1].contiguous(), lower=rate))
    assert torch.equal(gate, ops.linear(low[:, K:], w2, bias[n1:].contiguous(), out=torch.empty(M, n2, device="cuda")))
    with pytest.raises(Exception):      # (a bias for the first columns only: the kernel would read beyond it)
        ops.linear_pair(low, both, n1, bias[:n1], rate)


def test_matrices_that_do_not_stack():
    from denno_beta_amd.kernels import ops
    _, w1, _, make = _operands(1, 24, 64)      # (24 rows are one and a half blocks)
    _, w2, _, _ = _operands(1, 16, 72)
    assert ops.stacked(w1, w1) is None and ops.stacked(w2, w1) is None and ops.stacked(make(16, 64).bfloat16(), w1) is None


@pytest.mark.parametrize("M", [1, 8, 16, 17, 64])
def test_xielu_behind_a_norm_that_is_left_to_the_product(M):
    """A feed-forward with xielu is handed a norm of the stream that nobody has run yet (steps of few rows): the same bits as with its rows."""
    from denno_beta_amd.kernels import ops
    from denno_beta_amd.parts import FEED_FORWARDS, NORMS
    from denno_beta_amd.parts.base import LazyNorm, Runtime, StreamStats
    W, inner = 1024, 2048
    g = torch.Generator(device="cuda").manual_seed(M)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    tensors = dict(up=(make(inner, W) * W ** -0.5).bfloat16(), down=(make(W, inner) * inner ** -0.5).bfloat16(), numbers=make(2), gamma=1 + 0.1 * make(W))
    runtime = Runtime(torch.bfloat16, torch.device("cuda"))
    ffn = FEED_FORWARDS.make(("dense_mlp", dict(width=W, inner=inner, activation="xielu", up_weight="up", up_bias=None, down_weight="down", down_bias=None,
                                                activation_params="numbers")))
    norm = NORMS.make(("layernorm", dict(width=W, eps=1e-5, weight_name="gamma")))
    ffn.bind(tensors, runtime), norm.bind(tensors, runtime)
    ffn.prepare_lazy_norm(norm)
    x, stream = make(M, W), StreamStats(*ops.norm_stream_buffers(M, W, "cuda"), norm)
    stream.written = True
    assert ffn.takes_lazy_norm(M, norm)
    mine, want = x.clone(), x.clone()
    ffn.forward(LazyNorm(norm, x, torch.bfloat16, stream), None, mine)
    ffn.forward(norm.forward(x, torch.bfloat16), None, want)
    assert torch.equal(mine, want) and not torch.equal(mine, x)
