"""The 32-bit attention of portions goes through its tiles in an order that depends on how many there are: every row is there whatever it is."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("requests,H", [(1, 1), (4, 32), (8, 16), (43, 3), (5, 51), (8, 32), (27, 19), (16, 33)])
@pytest.mark.parametrize("extras", [{}, dict(softcap=3.0)])
def test_all_rows_around_one_and_two_workgroups_a_cu(requests, H, extras):
    # (a request of up to 128 rows is one tile, two workgroups a head: 2, 256, 256, 258, 510, 512, 1,026 and 1,056 of them)
    from denno_beta_amd.kernels import ops
    g = torch.Generator().manual_seed(requests + H)
    dh, ps = 16, 16
    counts = [int(x) for x in torch.randint(1, 129, (requests,), generator=g)]
    counts[0] = 128
    longest = -(-max(counts) // ps)
    tables = torch.arange(requests * longest, dtype=torch.int32).view(requests, longest).cuda()
    k, v = (torch.randn(shape, generator=g).cuda() for shape in ((requests * longest, H, ps, dh), (requests * longest, H, dh, ps)))
    T = sum(counts)
    q = torch.randn(T, H * dh, generator=g).cuda()
    wide, narrow, first = [], [], 0
    for s, n in enumerate(counts):
        wide.append((s, first, n, 0))
        narrow += [(s, first + i, min(16, n - i), i) for i in range(0, n, 16)]
        first += n
    wide.sort(key=lambda t: -(t[2] + t[3]))
    wide, narrow = (torch.tensor(t, dtype=torch.int32).t().contiguous().cuda() for t in (wide, narrow))
    mine, theirs = torch.full((T, H * dh), 7.0, device="cuda"), torch.empty(T, H * dh, device="cuda")
    ops.attention(q, mine, k, v, tables, narrow, H, dh ** -0.5, tiles_wide=wide, **extras)
    ops.attention(q, theirs, k, v, tables, narrow, H, dh ** -0.5, **extras)      # (the kernel for tiles of 16 rows: the same bits)
    assert torch.equal(mine, theirs)


@pytest.mark.parametrize("counts,start", [([1], 0), ([16], 0), ([17], 0), ([1, 2, 3], 0), ([8, 8, 8], 20), ([33, 64, 5], 15), ([100], 63), ([128, 130], 64)])
@pytest.mark.parametrize("dh", [16, 48, 64, 96, 128])
@pytest.mark.parametrize("extras", [dict(softcap=3.0), dict(window=24, softcap=3.0, keep_first=5), dict(bias=70), dict(softcap=3.0, bias=7, chunk=32)])
def test_keys_that_no_row_of_a_wave_reads(counts, start, dh, extras):
    """A soft cap or a bias is worked out for runs of 16 keys that a wave's rows read: the bits of the kernel for tiles of 16 rows, at every edge of a run."""
    from denno_beta_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(sum(counts) + start + dh)
    make = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    H, G, ps = 4, 2, 16
    if "bias" in extras:
        extras = dict(extras, bias=make(H, extras["bias"]))
    longest = -(-(max(counts) + start) // ps)
    tables = torch.arange(len(counts) * longest, dtype=torch.int32).view(len(counts), longest).cuda()
    k, v, T = make(len(counts) * longest, G, ps, dh), make(len(counts) * longest, G, dh, ps), sum(counts)
    q = 2 * make(T, H * dh)
    wide, narrow, first = [], [], 0
    for s, n in enumerate(counts):
        wide += [(s, first + i, min(128, n - i), start + i) for i in range(0, n, 128)]
        narrow += [(s, first + i, min(16, n - i), start + i) for i in range(0, n, 16)]
        first += n
    wide, narrow = (torch.tensor(t, dtype=torch.int32).t().contiguous().cuda() for t in (wide, narrow))
    mine, theirs = torch.full((T, H * dh), 7.0, device="cuda"), torch.empty(T, H * dh, device="cuda")
    ops.attention(q, mine, k, v, tables, narrow, H, dh ** -0.5, tiles_wide=wide, **extras)
    ops.attention(q, theirs, k, v, tables, narrow, H, dh ** -0.5, **extras)
    assert torch.equal(mine, theirs)
