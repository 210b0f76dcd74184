"""The scan's two ways of reading its rows (16 bytes a lane, or number by number where an operand's rows do not begin at 16 bytes) and its
places for rows beyond a request's last: the same bits."""
import pytest
import torch

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
