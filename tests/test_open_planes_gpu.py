"""An average over depth whose last plane has still to take a sublayer's result, in one kernel, against the kernels it stands for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [1, 63, 256, 257, 512, 1000, 1024, 1025, 2048, 4095, 4096, 4097])
@pytest.mark.parametrize("n", [1, 2, 4, 5, 9])
def test_one_kernel_gives_the_bits_of_three(width, n):
    from denno_beta_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(width * 16 + n)
    T = 3
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    for dtype, has_scale, then_dtype in ((torch.float32, True, torch.bfloat16), (torch.bfloat16, False, torch.float32), (torch.float32, True, None)):
        hist, y = make(n + 1, T, width), make(T, width + 4).to(dtype)[:, :width]
        weight, scale, w, next_w = make(width), make(width) if has_scale else None, make(n), make(width)
        mine, theirs = hist.clone(), hist.clone()
        then = None if then_dtype is None else (next_w, 1e-6, torch.empty(T, width, dtype=then_dtype, device="cuda"))
        planes = ops.OpenPlanes(mine, n - 1, y, weight, scale, 0.37, 1e-5, then=then)
        ops.depth_mix(planes, n, w, mine[n])
        ops.rmsnorm_add(y, weight, scale, 0.37, 1e-5, theirs[n - 1])
        ops.depth_mix(theirs, n, w, theirs[n])
        assert torch.equal(mine, theirs)
        if then is not None and width <= 4096:
            assert planes.normed is then[2]
            assert torch.equal(then[2], ops.rmsnorm(theirs[n], next_w, 1e-6, torch.empty_like(then[2])))
        else:
            assert planes.normed is None


def test_a_plane_that_is_read_has_taken_the_result():
    from denno_beta_amd.kernels import ops
    hist, y, w = torch.randn(3, 2, 64, device="cuda"), torch.randn(2, 64, device="cuda"), torch.ones(64, device="cuda")
    want = ops.rmsnorm_add(y, w, None, 1.0, 1e-5, hist[1].clone())
    planes = ops.OpenPlanes(hist, 1, y, w, None, 1.0, 1e-5)
    assert torch.equal(planes[1], want) and torch.equal(planes[1], want)      # (once)
