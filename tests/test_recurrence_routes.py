"""Which of a step's requests go through their recurrences in chunks: by each request's own rows, whatever else is in the step and whether it is captured."""
import random
from types import SimpleNamespace

import pytest

from denno_beta_amd.parts.recurrent import walk


def routes(lengths, padding=None, rows_min=96, dk=64):
    """-> the kernel of each request (and that no request has two), the launches; padding (T, S): the tables of a captured step."""
    starts = [0]
    for n in lengths:
        starts.append(starts[-1] + n)
    T, S = padding or (starts[-1], len(lengths))
    ctx = SimpleNamespace(T=T, S=S, rows_of_requests=None if padding else (min(lengths), max(lengths)))
    got, launches = [""] * len(lengths), []

    def in_chunks(least):
        launches.extend(["chunks", "rows"] if least else ["chunks"])
        for i, n in enumerate(lengths):
            got[i] += "chunks" if n >= least else "rows"

    def by_rows():
        launches.append("rows")
        for i in range(len(lengths)):
            got[i] += "rows"
    walk(ctx, dk, rows_min, in_chunks, by_rows)
    return got, launches


def test_by_the_requests_own_rows():
    rng = random.Random(1)
    for _ in range(300):
        rows_min = rng.choice([32, 96])
        lengths = [rng.choice([1, 5, 31, 32, 95, 96, 97, 350, 1024]) for _ in range(rng.randint(1, 12))]
        got, launches = routes(lengths, rows_min=rows_min)
        assert got == ["chunks" if n >= rows_min else "rows" for n in lengths]
        assert len(launches) == len(set(got))      # (none for nobody)
        T, S = sum(lengths) + rng.randint(0, 300), len(lengths) + rng.randint(0, 4)
        assert routes(lengths, (T, S), rows_min)[0] == got
    assert routes([40] * 4, (192, 4))[1] == ["chunks", "rows"] and routes([20] * 4, (95, 4))[1] == ["rows"]      # (no room for a request of 96 rows)
    assert routes([200, 200], dk=40) == (["rows", "rows"], ["rows"])


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["wide", "rows", "head"])
@pytest.mark.parametrize("lengths", [[200, 1, 96, 40, 95, 1], [3, 350, 97], [17, 1]])
@pytest.mark.parametrize("padding", [0, 34])
def test_each_request_has_the_bits_it_has_alone(mode, lengths, padding):
    import torch

    from test_kernels_gpu import ops
    from test_scan_chunks_gpu import DEV, chunks, operands, per_row
    from test_sequence_kernels_gpu import tables
    heads, dk, dv, least = 2, 64, 40, 96
    row_start, slots, T = tables(lengths + [0] * (padding > 0), [i if i != 1 else 7 for i in range(len(lengths))] + [-1] * (padding > 0))
    if mode == "rows":
        r, k, v, kw, rate, bias = per_row(heads, heads, dk, dv, T + padding, 0.5)
        numbers = dict(kw, rate=rate, bias=bias)
    else:
        r, k, v, kw = operands(mode, heads, heads, dk, dv, T + padding, 0.5)
        numbers = dict(kw)

    def step(rows, state, row_start, slots, how, least=0):
        out = torch.full((rows.stop - rows.start, heads * dv), 7.0, device=DEV)
        n = {a: t[rows] if t is not None and t.dim() == 2 else t for a, t in numbers.items()}
        a = (state, row_start, slots, heads, dk, dv, out)
        if how == "chunks" and mode == "rows":
            ops().delta_chunks(r[rows], k[rows], v[rows], n["beta"], n["w"], n["rate"], n["bias"], *a, rows_min=least)
        elif how == "chunks":
            ops().scan_chunks(r[rows], k[rows], v[rows], n["w"], *a, **{x: t for x, t in n.items() if x != "w"}, rows_min=least)
        elif mode == "head":
            ops().state_scan(r[rows], k[rows], v[rows], None, None, *a, read_after=True, w_head=n["w_head"])
        elif mode == "wide":
            ops().state_scan(r[rows], k[rows], v[rows], n["w"], None, *a, beta=n["beta"], beta_logits=True)
        else:
            ops().state_scan(r[rows], k[rows], v[rows], n["w"], None, *a, beta=n["beta"], beta_logits=True, w_rows=True, w_rate=n["rate"], w_bias=n["bias"])
        return out
    first = torch.randn(9, heads * dk * dv, device=DEV)
    together = first.clone()
    got = step(slice(0, T + padding), together, row_start, slots, "chunks", least)
    alone = first.clone()
    for s, n in enumerate(lengths):
        rows = slice(int(row_start[s]), int(row_start[s + 1]))
        table, slot = torch.tensor([0, n], dtype=torch.int32, device=DEV), slots[s:s + 1].contiguous()
        want = step(rows, alone, table, slot, "chunks" if n >= least else "rows")
        assert torch.equal(got[rows], want)
    assert torch.equal(together, alone)
    assert bool((got[T:] == 7.0).all())
