"""The scan against the recurrence in 64 bits.  The scan's two ways of reading its rows (16 bytes a lane, or number by number where an operand's rows do not begin at 16 bytes) and its
places for rows beyond a request's last: the same bits."""
import pytest
import torch

import kernel_refs as R
from test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MODES = ["before", "bonus", "after", "head", "rows", "from_decay", "delta", "delta_rows"]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("heads,dk,dv", [(2, 4, 4), (3, 16, 20), (2, 28, 16), (2, 64, 12), (1, 100, 8), (2, 128, 32), (1, 256, 4)])
@pytest.mark.parametrize("lengths", [[1, 1, 1], [15, 16, 17], [33, 1, 64], [5]])
def test_the_scan_reads_its_rows_either_way(mode, heads, dk, dv, lengths):
    o, T, n = ops(), sum(lengths), heads * dk
    starts = torch.tensor([0] + [sum(lengths[:i + 1]) for i in range(len(lengths))], dtype=torch.int32, device=DEV)
    slots = torch.tensor([3, 0, 2][:len(lengths)], dtype=torch.int32, device=DEV)
    wide = [rnd(T, n, seed=1) * dk ** -0.5, rnd(T, n, seed=2) * dk ** -0.5, rnd(T, heads * dv, seed=3), torch.sigmoid(rnd(T, n, seed=4))]
    per_row, beta, u, state = torch.sigmoid(rnd(T, heads, seed=5)), rnd(T, heads, seed=6), rnd(n, seed=7), rnd(4, heads * dk * dv, seed=8)

    def run(moved):
        # (rows one number longer, from the second number on: none of them begins at 16 bytes for long)
        r, k, v, w = (torch.nn.functional.pad(x, (1, 0))[:, 1:] if moved else x for x in wide)
        st, out = state.clone(), torch.full((T, heads * dv), 7.0, device=DEV)
        kw = dict(bonus=dict(u=u), after=dict(read_after=True), head=dict(w=None, w_head=per_row[0].contiguous(), read_after=True),
                  rows=dict(w=per_row, w_rows=True, read_after=True), from_decay=dict(k=None, key_from_decay=True),
                  delta=dict(beta=beta, beta_logits=True), delta_rows=dict(beta=beta, beta_logits=True, w=per_row, w_rows=True),
                  before={})[mode]
        a = dict(dict(r=r, k=k, v=v, w=w, u=None), **kw)
        o.state_scan(a.pop("r"), a.pop("k"), a.pop("v"), a.pop("w"), a.pop("u"), st, starts, slots, heads, dk, dv, out, **a)
        return st, out

    (s0, o0), (s1, o1) = run(False), run(True)
    assert torch.equal(s0, s1) and torch.equal(o0, o1)
    assert torch.equal(s0[1], state[1]) and bool(torch.isfinite(o0).all()) and not bool((o0 == 7.0).any())


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("heads,dk,dv,lengths", [(2, 4, 4, [1, 1, 1]), (3, 16, 20, [15, 16, 17]), (2, 28, 16, [3, 2, 40]), (2, 64, 12, [33, 1, 64]),
                                                 (1, 100, 8, [5]), (2, 128, 32, [17, 31, 2]), (1, 256, 4, [18, 1, 16]), (2, 256, 8, [1, 1])])
def test_the_scan_in_64_bits(mode, heads, dk, dv, lengths):
    """Every row and every state against the plain recurrence in 64 bits: the sizes of heads, fetches that end early, single rows."""
    o, T, n = ops(), sum(lengths), heads * dk
    starts = torch.tensor([0] + [sum(lengths[:i + 1]) for i in range(len(lengths))], dtype=torch.int32, device=DEV)
    slots = torch.tensor([3, 0, 2][:len(lengths)], dtype=torch.int32, device=DEV)
    x = dict(r=rnd(T, n, seed=1) * dk ** -0.5, k=rnd(T, n, seed=2) * dk ** -0.5, v=rnd(T, heads * dv, seed=3), w=torch.sigmoid(rnd(T, n, seed=4)), u=None)
    per_row, beta, state = torch.sigmoid(rnd(T, heads, seed=5)), rnd(T, heads, seed=6), rnd(4, heads * dk * dv, seed=8)
    x.update(dict(bonus=dict(u=rnd(n, seed=7)), after=dict(read_after=True), head=dict(w=None, w_head=per_row[0].contiguous(), read_after=True),
                  rows=dict(w=per_row, w_rows=True, read_after=True), from_decay=dict(k=None, key_from_decay=True),
                  delta=dict(beta=beta, beta_logits=True), delta_rows=dict(beta=beta, beta_logits=True, w=per_row, w_rows=True), before={})[mode])

    def run(fn, as_):
        a = {name: as_(t) if torch.is_tensor(t) else t for name, t in x.items()}
        st, out = as_(state.clone()), as_(torch.zeros(T, heads * dv, device=DEV))
        fn(a.pop("r"), a.pop("k"), a.pop("v"), a.pop("w"), a.pop("u"), st, starts, slots, heads, dk, dv, out, **a)
        return st, out
    got, want = run(o.state_scan, lambda t: t), run(R.state_scan, lambda t: t.double())
    # (sums of dk products of numbers about dk^-1/2 and 1, carried over up to 64 rows by factors below 1: some hundreds of roundings of
    # numbers below 16, by at most 2^-21 each, in both directions)
    for a, b in zip(got, want):
        assert b.abs().max() < 64 and (a.double() - b).abs().max() <= 40 * 2.0 ** -21


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("heads,dk,dv,n,rows,moved", [(64, 16, 20, 17, 3, False), (64, 64, 8, 17, 18, False), (64, 64, 8, 17, 18, True), (64, 64, 8, 16, 18, False),
                                                      (9, 64, 8, 116, 130, False), (32, 128, 4, 33, 17, False), (32, 128, 4, 33, 17, True), (3, 256, 4, 342, 3, False),
                                                      (2, 256, 4, 3, 18, False)])
def test_many_waves_and_few_have_the_same_bits(mode, heads, dk, dv, n, rows, moved):
    """A step of many requests may read its operands as it goes where few requests have them read ahead: on both sides of the numbers of
    waves at which that changes, every request is what it is in a step of its own."""
    o, T = ops(), n * rows
    pad = lambda x: torch.nn.functional.pad(x, (1, 0))[:, 1:] if moved else x      # noqa: E731
    g = heads if mode == "from_decay" else 1      # (one head of queries and keys for all, and little to hold)
    x = dict(r=pad(rnd(T, g * dk, seed=1) * dk ** -0.5), k=pad(rnd(T, g * dk, seed=2) * dk ** -0.5), v=pad(rnd(T, heads * dv, seed=3)),
             w=pad(torch.sigmoid(rnd(T, heads * dk, seed=4))), u=None)
    per_row, beta = torch.sigmoid(rnd(T, heads, seed=5)), rnd(T, heads, seed=6)
    x.update(dict(bonus=dict(u=rnd(heads * dk, seed=7)), after=dict(read_after=True), head=dict(w=None, w_head=per_row[0].contiguous(), read_after=True),
                  rows=dict(w=per_row, w_rows=True, read_after=True), from_decay=dict(k=None, key_from_decay=True),
                  delta=dict(beta=beta, beta_logits=True), delta_rows=dict(beta=beta, beta_logits=True, w=per_row, w_rows=True), before={})[mode])
    state = rnd(n, heads * dk * dv, seed=8)

    def run(a, b):
        y = {name: t[a * rows:b * rows] if torch.is_tensor(t) and t.dim() == 2 else t for name, t in x.items()}
        if moved is False:
            y = {name: t.contiguous() if torch.is_tensor(t) else t for name, t in y.items()}
        st, out = state[a:b].clone(), torch.full(((b - a) * rows, heads * dv), 7.0, device=DEV)
        starts = torch.arange(b - a + 1, dtype=torch.int32, device=DEV) * rows
        o.state_scan(y.pop("r"), y.pop("k"), y.pop("v"), y.pop("w"), y.pop("u"), st, starts, torch.arange(b - a, dtype=torch.int32, device=DEV), heads, dk,
                     dv, out, qk_heads=g, **y)
        return st, out
    st, out = run(0, n)
    for a in (0, n // 2, n - 1):
        s1, o1 = run(a, a + 1)
        assert torch.equal(s1, st[a:a + 1]) and torch.equal(o1, out[a * rows:(a + 1) * rows])
    assert bool(torch.isfinite(out).all()) and not bool((out == 7.0).any())
