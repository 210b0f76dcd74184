"""The 32-bit kernels on the matrix cores against the kernels that run the same sums as chains of fused multiply-adds:
the same bits, whichever of them a step takes."""
import math

import pytest
import torch

from test_kernels_gpu import i32, ops, paged_case, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(65, 64, 128), (65, 1, 4), (129, 63, 1), (200, 65, 127), (64 * 9, 257, 129), (130, 200, 1600),
                                   (67, 130, 250), (300, 96, 34), (70, 66, 16), (131, 300, 32), (65, 200, 33), (194, 70, 36), (66, 129, 63), (257, 65, 64),
                                   (66, 70, 65), (130, 64, 68),
                                   (65, 16449, 33), (1030, 2001, 64), (1030, 2001, 20), (129, 16384, 1)])
def test_a_product_of_many_rows_has_the_few_rows_bits(dtype, M, N, K):
    """Numbers of very different sizes, so that another order or another rounding shows; ends of tiles, of slabs, of segments."""
    g = torch.Generator().manual_seed(M + N + K)
    a = (torch.randn(M, K, generator=g) * torch.exp2(torch.randint(-12, 13, (M, K), generator=g).float())).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=g) * torch.exp2(torch.randint(-12, 13, (N, K), generator=g).float())).to(dtype).to(DEV)
    bias = rnd(N, seed=1)
    many = torch.zeros(M, N, device=DEV)
    ops().linear(a, w, bias, out=many)
    stream, few_stream = rnd(M, N, seed=2), rnd(M, N, seed=2)
    ops().linear(a, w, bias, residual=stream)
    # one order of summation, spelled out: segments of 128 with one rounding a step (64-bit products are exact)
    rows = torch.tensor(sorted({0, 1, 31, 32, 63, 64, M - 1}))
    a64, w64 = a[rows].double().cpu(), w.double().cpu()
    total = torch.zeros(len(rows), N)
    for seg in range(0, K, 128):
        acc = torch.zeros(len(rows), N)
        for k in range(seg, min(K, seg + 128)):
            acc = (a64[:, k:k + 1] * w64[None, :, k] + acc.double()).float()
        total = total + acc
    want = total + bias.cpu()
    # (64 bits round the sum once before 32 bits do: two roundings differ from one in a few of a thousand million cases)
    assert (many[rows].cpu() != want).float().mean() < 1e-4, (M, N, K)
    if K % 4 == 0:      # the kernel for few rows takes these
        few = torch.zeros(M, N, device=DEV)
        for m in range(0, M, 64):
            ops().linear(a[m:m + 64], w, bias, out=few[m:m + 64])
            ops().linear(a[m:m + 64], w, bias, residual=few_stream[m:m + 64])
        assert torch.equal(many, few) and torch.equal(stream, few_stream), (M, N, K)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("a_exp,w_exp", [(-70, -70), (-64, -66), (-63, -63), (-127, 0), (0, -127), (-40, -100)])
def test_products_below_the_smallest_normal_number(dtype, a_exp, w_exp):
    """Operands, products or partial sums (or all) are subnormal: kept by the matrix instruction as by the multiply-adds."""
    M, N, K = 130, 70, 260
    g = torch.Generator().manual_seed(K)
    a, w = ((torch.randn(n, K, generator=g).double() * 2.0 ** e).to(dtype).to(DEV) for n, e in ((M, a_exp), (N, w_exp)))
    many, few = torch.zeros(M, N, device=DEV), torch.zeros(M, N, device=DEV)
    ops().linear(a, w, None, out=many)
    for m in range(0, M, 64):
        ops().linear(a[m:m + 64], w, None, out=few[m:m + 64])
    assert torch.equal(many, few)
    assert ((many != 0) & (many.abs() < 2.0 ** -126)).float().mean() > 0.02
    # (a step rounds by at most half of the smallest subnormal number, or by 2^-24 of a sum that is itself below 64 times the operands' sizes)
    exact = a.double() @ w.double().t()
    assert (many.double() - exact).abs().max() <= K * max(2.0 ** -150, 2.0 ** (a_exp + w_exp + 6 - 24))


@pytest.mark.parametrize("dh,q_exp,v_exp", [(64, -130, 0), (64, 0, -130), (128, -127, -127), (48, -140, -128)])
def test_portions_of_subnormal_queries_and_values(dh, q_exp, v_exp):
    """Scores and weighted values below the smallest normal number: the portions' kernel and the narrow one give the same bits."""
    q, k, v, bt, tiles, T = paged_case([300, 64, 133], [100, 64, 1], 2, 2, dh, 16, torch.float32, seed=dh)
    q, v = (q.double() * 2.0 ** q_exp).float(), (v.double() * 2.0 ** v_exp).float()
    narrow, wide = torch.zeros(T, 2 * dh, device=DEV), torch.zeros(T, 2 * dh, device=DEV)
    # (a scale that brings the scores back to about 1: a dot product rounded among subnormal numbers then shows)
    args = (q[:, 2 * dh:4 * dh], k, v, bt, tiles, 2, 2.0 ** min(-q_exp, 126) / math.sqrt(dh), 0)
    ops().attention(args[0], narrow, *args[1:])
    ops().attention(args[0], wide, *args[1:], tiles_wide=paged_case.wide)
    assert torch.equal(narrow, wide) and bool(torch.isfinite(wide).all()) and (wide != 0).float().mean() > 0.9
    if v_exp < -120:
        assert (wide.abs() < 2.0 ** -126).float().mean() > 0.9


@pytest.mark.parametrize("H,Hkv,dh,ps,kw", [
    (2, 2, 16, 16, {}), (3, 1, 32, 16, {}), (2, 2, 48, 48, {}), (4, 2, 64, 16, {}), (2, 2, 64, 64, dict(window=70)), (2, 1, 80, 32, {}),
    (2, 2, 96, 16, dict(window=33)), (1, 1, 112, 16, {}), (2, 1, 128, 32, {}), (2, 2, 64, 16, dict(chunk=50, sink=True)),
    (2, 2, 64, 32, dict(window=40, keep_first=5, softcap=20.0)), (2, 2, 32, 16, dict(bias=True))])
def test_portions_have_the_narrow_kernels_bits(H, Hkv, dh, ps, kw):
    """Portions that end at every place in a tile of rows and start at every place in a tile of keys; the cache holds NaN
    beyond a request's tokens and in pages that no request has, and infinities in tokens that come later."""
    seq_lens, new_rows = [300, 64, 133, 1, 430, 129, 65], [1, 64, 21, 1, 300, 129, 16]
    q, k, v, bt, tiles, T = paged_case(seq_lens, new_rows, H, Hkv, dh, ps, torch.float32, seed=H + dh)
    used = torch.zeros(k.shape[0], ps, dtype=torch.bool)
    for s, n in enumerate(seq_lens):
        for p in range(n):
            used[int(bt[s, p // ps]), p % ps] = True
    spare = ~used.to(DEV)
    k.masked_fill_(spare[:, None, :, None], math.nan), v.masked_fill_(spare[:, None, None, :], math.nan)
    last = int(bt[4, 429 // ps])
    v[last, :, :, 429 % ps] = math.inf
    kw = dict(kw)
    window = kw.pop("window", 0)
    if kw.get("bias"):
        kw["bias"] = rnd(H, 100, seed=3)
    args = (k, v, bt, tiles, H, 1 / math.sqrt(dh), window)
    narrow, wide = torch.zeros(T, H * dh, device=DEV), torch.zeros(T, H * dh, device=DEV)
    ops().attention(q[:, H * dh:2 * H * dh], narrow, *args, **kw)
    ops().attention(q[:, H * dh:2 * H * dh], wide, *args, tiles_wide=paged_case.wide, **kw)
    assert torch.equal(narrow.nan_to_num(nan=7e30), wide.nan_to_num(nan=7e30)), (narrow - wide).abs().nan_to_num().max()
    assert torch.isfinite(wide[:-17]).float().mean() > 0.9
