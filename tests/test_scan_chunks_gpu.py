"""The recurrences in chunks of 16 rows against the recurrence in 64 bits: sizes of heads, requests that end inside a chunk, and what is no number."""
import pytest
import torch

import kernel_refs as R
from test_kernels_gpu import ops, rnd
from test_sequence_kernels_gpu import close, tables

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(mode, heads, qk_heads, dk, dv, T, fade):
    """r, k (unit vectors that point almost the same way), v, then decays and beta's arguments, as views of wider rows."""
    C = 2 * qk_heads * dk + heads * dv
    x = rnd(T, C + 3, seed=1)[:, 1:1 + C]      # (rows that begin at any number)
    r, k, v = x[:, :qk_heads * dk], x[:, qk_heads * dk:2 * qk_heads * dk], x[:, 2 * qk_heads * dk:]
    unit = lambda t: torch.nn.functional.normalize(t.reshape(T, qk_heads, dk), dim=-1).reshape(T, -1)      # noqa: E731
    k.copy_(unit(k + 2.0 * rnd(1, qk_heads * dk, seed=2)))
    r.copy_(unit(r) * dk ** -0.5)
    if mode == "head":
        return r, k, v, dict(w=None, w_head=torch.exp(-fade * torch.rand(heads, device=DEV)))
    return r, k, v, dict(w=torch.exp(-fade * torch.rand(T, heads * dk, device=DEV)), beta=rnd(T, heads + 2, seed=4)[:, 1:1 + heads] * 2)


@pytest.mark.parametrize("mode", ["wide", "head"])
@pytest.mark.parametrize("dk,dv,heads,qk_heads", [(16, 16, 2, 2), (64, 128, 4, 2), (48, 33, 3, 1), (128, 40, 2, 2), (80, 7, 2, 1), (32, 64, 6, 3), (96, 16, 1, 1),
                                                  (112, 50, 2, 2), (64, 300, 1, 1), (16, 1, 1, 1)])
@pytest.mark.parametrize("lengths", [[40], [16, 1, 33], [1, 15, 17, 200, 3], [64, 63, 65], [2, 2, 5]])
@pytest.mark.parametrize("fade", [0.02, 1.0, 200.0])
def test_chunks_in_64_bits(mode, dk, dv, heads, qk_heads, lengths, fade):
    slot_of = [4, 0, -1, 2, 1][:len(lengths)]
    row_start, slots, T = tables(lengths, slot_of)
    r, k, v, kw = operands(mode, heads, qk_heads, dk, dv, T, fade)
    state = torch.randn(5, heads * dk * dv + 11, device=DEV)
    n = heads * dk * dv
    d = lambda t: t.cpu().double() if torch.is_tensor(t) else t      # noqa: E731
    want_state, want = d(state), torch.zeros(T, heads * dv, dtype=torch.float64)
    R.scan_chunks(d(r), d(k), d(v), d(kw["w"]), want_state[:, :n], row_start.cpu(), slots.cpu(), heads, dk, dv, want, qk_heads=qk_heads,
                  **{a: d(t) for a, t in kw.items() if a != "w"})
    got_state, got = state.clone(), torch.full((T + 1, heads * dv), 7.0, device=DEV)
    ops().scan_chunks(r, k, v, kw["w"], got_state[:, :n], row_start, slots, heads, dk, dv, got[:T], qk_heads=qk_heads,
                      **{a: t for a, t in kw.items() if a != "w"})
    real = [t for s, m in enumerate(lengths) for t in range(int(row_start[s]), int(row_start[s]) + m) if slot_of[s] >= 0]
    close(got[real], want[real]), close(got_state, want_state)
    rest = [t for t in range(T + 1) if t not in real]
    assert bool((got[rest] == 7.0).all()) and torch.equal(got_state[3], state[3])      # (rows and slots of no request)


@pytest.mark.parametrize("mode", ["wide", "head"])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("which", ["v", "k", "r"])
def test_what_is_no_number_does_not_reach_rows_before_it(mode, bad, which):
    heads, dk, dv, T, at = 2, 64, 40, 50, 21
    row_start, slots, _ = tables([T], [0])
    r, k, v, kw = operands(mode, heads, heads, dk, dv, T, 0.5)
    got = []
    for spoilt in (False, True):
        x = dict(r=r.clone(), k=k.clone(), v=v.clone())
        if spoilt:
            x[which][at, 5] = bad
        out = torch.zeros(T, heads * dv, device=DEV)
        ops().scan_chunks(x["r"], x["k"], x["v"], kw["w"], torch.zeros(1, heads * dk * dv, device=DEV), row_start, slots, heads, dk, dv, out,
                          **{a: t for a, t in kw.items() if a != "w"})
        got.append(out)
    close(got[1][:at], got[0][:at]), close(got[1][:, dv:], got[0][:, dv:])      # (rows before it, and the other head)
    assert not bool(torch.isfinite(got[1][at]).all())
    if which == "v":      # (a value's column alone)
        keep = [j for j in range(heads * dv) if j != 5]
        close(got[1][:, keep], got[0][:, keep])
    if which == "r":
        close(got[1][at + 1:], got[0][at + 1:])


def per_row(heads, qk_heads, dk, dv, T, fade):
    """The operands of the delta rule with one decay a row: beta's and the decay's arguments, rate and bias."""
    r, k, v, kw = operands("wide", heads, qk_heads, dk, dv, T, fade)
    return r, k, v, dict(beta=kw["beta"], w=rnd(T, heads, seed=6)), rnd(heads, seed=7).abs() * fade, rnd(heads, seed=8)


def chunks(mode, r, k, v, kw, state, row_start, slots, heads, dk, dv, qk_heads=None):
    out = torch.zeros(len(r), heads * dv, device=DEV)
    if mode == "rows":
        kw, rate, bias = kw
        ops().delta_chunks(r, k, v, kw["beta"], kw["w"], rate, bias, state, row_start, slots, heads, dk, dv, out, qk_heads)
    else:
        ops().scan_chunks(r, k, v, kw["w"], state, row_start, slots, heads, dk, dv, out, qk_heads=qk_heads, **{a: t for a, t in kw.items() if a != "w"})
    return out


@pytest.mark.parametrize("mode,which", [("wide", "beta"), ("wide", "w"), ("rows", "beta"), ("rows", "w"), ("rows", "v"), ("rows", "k"), ("rows", "r")])
@pytest.mark.parametrize("at", [0, 15, 16, 21, 49])
def test_no_number_among_the_numbers_of_a_row(mode, which, at):
    """Beta's argument, decays and the operands of the rule with one decay a row: rows before it and other heads have none of it."""
    heads, dk, dv, T = 2, 64, 40, 50
    row_start, slots, _ = tables([T], [0])
    r, k, v, kw = operands("wide", heads, heads, dk, dv, T, 0.5)
    if mode == "rows":
        r, k, v, kw, rate, bias = per_row(heads, heads, dk, dv, T, 0.5)
    got = []
    for spoilt in (False, True):
        x = dict(r=r.clone(), k=k.clone(), v=v.clone(), **{a: t.clone() for a, t in kw.items()})
        if spoilt:
            x[which][at, 0] = float("nan")      # (of head 0)
        numbers = {a: x[a] for a in kw}
        got.append(chunks(mode, x["r"], x["k"], x["v"], (numbers, rate, bias) if mode == "rows" else numbers, torch.zeros(1, heads * dk * dv, device=DEV),
                          row_start, slots, heads, dk, dv))
    close(got[1][:at], got[0][:at]), close(got[1][:, dv:], got[0][:, dv:])
    assert not bool(torch.isfinite(got[1][at, :dv]).all())


@pytest.mark.parametrize("T", [1, 16, 40, 200])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf")])
def test_an_infinite_state_stays_infinite(T, bad):
    """Constant decays: as row after row, an entry that has overflowed stays what it is, and so do its column's results."""
    heads, dk, dv = 2, 64, 40
    row_start, slots, _ = tables([T], [0])
    r, k, v, kw = operands("head", heads, heads, dk, dv, T, 0.1)
    state = torch.randn(1, heads * dv * dk, device=DEV)
    state.view(heads, dv, dk)[1, 7, 3] = bad
    one, many = state.clone(), state.clone()
    want = torch.zeros(T, heads * dv, device=DEV)
    ops().state_scan(r, k, v, None, None, one, row_start, slots, heads, dk, dv, want, read_after=True, w_head=kw["w_head"])
    got = chunks("head", r, k, v, kw, many, row_start, slots, heads, dk, dv)
    for a, b in ((got, want), (many, one)):
        fine = torch.isfinite(b)
        assert torch.equal(a[~fine], b[~fine])
        close(a[fine], b[fine])
    assert int((~torch.isfinite(many)).sum()) == 1 and bool(torch.isinf(want[:, dv + 7]).all())


@pytest.mark.parametrize("mode", ["wide", "rows", "head"])
@pytest.mark.parametrize("S", [63, 64, 65, 128, 130, 200])
def test_many_requests(mode, S):
    """A chunk finds its request among 64 at a time: empty requests, ones that end inside a chunk, and ones without a slot among them."""
    heads, dk, dv = 2, 16, 20
    lengths = [[17, 0, 5, 40, 16, 1, 33, 0, 3][i % 9] for i in range(S)]
    row_start, slots, T = tables(lengths, [-1 if i % 7 == 3 else S - 1 - i for i in range(S)])
    r, k, v, kw = operands("wide" if mode == "rows" else mode, heads, heads, dk, dv, T, 0.5)
    if mode == "rows":
        r, k, v, kw, rate, bias = per_row(heads, heads, dk, dv, T, 0.5)
    state = torch.randn(S, heads * dk * dv, device=DEV)
    one, many, want = state.clone(), state.clone(), torch.zeros(T, heads * dv, device=DEV)
    how = dict(head=dict(read_after=True, w_head=kw.get("w_head")), wide=dict(beta=kw.get("beta"), beta_logits=True),
               rows=dict(beta=kw.get("beta"), beta_logits=True, w_rows=True))[mode]
    if mode == "rows":
        how.update(w_rate=rate, w_bias=bias)
    ops().state_scan(r, k, v, kw["w"], None, one, row_start, slots, heads, dk, dv, want, **how)
    got = chunks(mode, r, k, v, (kw, rate, bias) if mode == "rows" else kw, many, row_start, slots, heads, dk, dv)
    close(got, want), close(many, one)


@pytest.mark.parametrize("dk,heads,qk_heads", [(64, 4, 2), (48, 3, 1), (16, 2, 2)])
@pytest.mark.parametrize("lengths", [[1, 15, 40], [200]])
def test_one_decay_a_row_from_rows_that_begin_anywhere(dk, heads, qk_heads, lengths):
    """Rows of r and k that begin at no multiple of 16 bytes: the bits of rows that do."""
    dv = 24
    row_start, slots, T = tables(lengths, [2, 0, 1][:len(lengths)])
    r, k, v, kw, rate, bias = per_row(heads, qk_heads, dk, dv, T, 0.5)
    assert r.data_ptr() % 16 != 0 and r.stride(0) % 4 != 0
    state = torch.randn(3, heads * dk * dv, device=DEV)
    one, many = state.clone(), state.clone()
    want = chunks("rows", r.contiguous(), k.contiguous(), v.contiguous(), (kw, rate, bias), one, row_start, slots, heads, dk, dv, qk_heads)
    got = chunks("rows", r, k, v, (kw, rate, bias), many, row_start, slots, heads, dk, dv, qk_heads)
    assert torch.equal(got, want) and torch.equal(many, one)


@pytest.mark.parametrize("mode", ["wide", "rows", "head"])
@pytest.mark.parametrize("T", [1, 20])
def test_results_whose_rows_lie_far_apart(mode, T):
    """Rows 2^24 numbers apart and more; with 20 rows the other request's one is walked row by row."""
    heads, dk, dv, far = 2, 16, 20, (1 << 24) + 4
    row_start, slots, rows = tables([T, 1], [0, 1])
    r, k, v, kw = operands("wide" if mode == "rows" else mode, heads, heads, dk, dv, rows, 0.5)
    if mode == "rows":
        r, k, v, kw, rate, bias = per_row(heads, heads, dk, dv, rows, 0.5)
    held = torch.full((rows * far,), 7.0, device=DEV)
    out, near = held.as_strided((rows, heads * dv), (far, 1)), torch.full((rows, heads * dv), 7.0, device=DEV)
    state = torch.zeros(2, heads * dk * dv, device=DEV)
    for to in (out, near):
        if mode == "rows":
            ops().delta_chunks(r, k, v, kw["beta"], kw["w"], rate, bias, state.clone(), row_start, slots, heads, dk, dv, to, rows_min=T if T > 1 else 0)
        else:
            ops().scan_chunks(r, k, v, kw["w"], state.clone(), row_start, slots, heads, dk, dv, to, **{a: t for a, t in kw.items() if a != "w"},
                              rows_min=T if T > 1 else 0)
    assert torch.equal(out, near) and bool((held.view(rows, far)[:, heads * dv:] == 7.0).all())
