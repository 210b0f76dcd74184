"""Queries, keys and values of the 32-bit turn, turned and taken to the cache in one launch, against the turn and the cache write one after the other."""
import pytest
import torch

from denno_beta_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,dk,dv,kept,dims,page", [(16, 8, 64, 64, 64, 64, 16), (4, 4, 48, 32, 48, 16, 32), (25, 5, 80, 80, 80, 80, 16), (3, 1, 33, 47, 48, 32, 16),
                                                      (2, 2, 128, 128, 128, 0, 16), (2, 1, 256, 200, 256, 256, 48), (8, 2, 96, 16, 96, 94, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 8, 257, 1023, 1025])      # (all a row's vectors at once, four workgroups a row, two, one)
def test_one_launch_has_the_bits_of_two(H, G, dk, dv, kept, dims, page, dtype, T):
    g = torch.Generator(device="cuda").manual_seed(H * 1000 + dk + T)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    width = (H + G) * dk + G * dv
    z = make(T, width + 12)[:, :width + 4]      # (a gate's columns behind them, rows further apart than that)
    positions = torch.randint(0, 5000, (T,), generator=g, device="cuda", dtype=torch.int32)
    freq = (10000.0 ** (-torch.arange(dims // 2, device="cuda", dtype=torch.float64) * 2 / max(dims, 1))).float()
    pages = T // page + 2
    slots = torch.randperm(pages * page, generator=g, device="cuda")[:T].to(torch.int32)
    if T > 4:
        slots[3] = -1
    pool = lambda *s: torch.full(s, 9.0, dtype=dtype, device="cuda")   # noqa: E731
    mine, theirs = [(pool(pages, G, page, kept), pool(pages, G, kept, page)) for _ in range(2)]
    q = ops.norm_turn_write(z, H, G, dk, dv, positions, pool(T, H * kept), slots, *mine, freq=freq if dims else None, as_runs=True)
    want, kv = torch.zeros(T, H * kept, dtype=dtype, device="cuda"), torch.zeros(T, 2 * G * kept, dtype=dtype, device="cuda")
    ops.rotary_runs(z, positions, freq, [(want, 0, H, dk, dims, 0, kept), (kv, H * dk, G, dk, dims, 0, kept), (kv, (H + G) * dk, G, dv, 0, G * kept, kept)])
    ops.kv_write(kv, 0, G * kept, slots, *theirs)
    assert torch.equal(q, want)
    assert torch.equal(mine[0], theirs[0]) and torch.equal(mine[1], theirs[1])
    # (not written: the pools stay as they are)
    kept_pools = [t.clone() for t in mine]
    ops.norm_turn_write(z, H, G, dk, dv, positions, q, slots, *mine, freq=freq if dims else None, write=False, as_runs=True)
    assert torch.equal(q, want) and all(torch.equal(a, b) for a, b in zip(mine, kept_pools))
