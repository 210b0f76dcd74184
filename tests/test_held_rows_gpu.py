"""The norms that hold a row in registers and the kernels whose rows are cut among workgroups, at the widths where their cases meet: a last
column alone in its place, a row that is a multiple of 256, the widest row held and the first that is not."""
import pytest
import torch

from test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# a sum of squares over n columns in 32 bits, then a handful of roundings: far under 1e-5 of a number of about 1 to 6; bfloat16: half a place
# of 2^-8 beside it
TOL = {torch.float32: dict(atol=2e-5, rtol=1e-5), torch.bfloat16: dict(atol=2e-5, rtol=2 ** -8)}


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [1, 64, 65, 255, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097])
def test_rmsnorm_and_the_sum_behind_it(width, dtype):
    o, R = ops(), 3
    wide = rnd(R + 2, width + 5, seed=width).to(dtype)
    x, w, scale, nw = wide[:, :width], rnd(width, seed=1), rnd(width, seed=2), rnd(width, seed=3)
    rows = torch.tensor([4, 0, 2], dtype=torch.int32, device=DEV)
    for weight in (w, None):
        out = torch.full((R, width + 3), 7.0, dtype=dtype, device=DEV)
        o.rmsnorm(x, weight, 1e-5, out[:, :width], rows=rows)
        want = rms(x[rows.long()].double(), 1e-5) * (1.0 if weight is None else w.double())
        assert torch.allclose(out[:, :width].double(), want, **TOL[dtype]) and (out[:, width:] == 7).all()
    for weight, sc, gate, norm in ((w, scale, None, nw), (None, None, rnd(R, width, seed=5), None), (w, None, rnd(R, width, seed=6), nw)):
        y, stream = x[:R], rnd(R, width + 4, seed=7)
        mine, then = stream.clone()[:, :width], torch.empty(R, width, dtype=dtype, device=DEV)
        o.rmsnorm_add(y, weight, sc, 0.37, 1e-5, mine, gate=gate, then=(norm, 1e-6, then))
        v = y.double() * (1.0 if gate is None else torch.sigmoid(gate.double()))
        v = rms(v, 1e-5) * (1.0 if weight is None else w.double()) * (1.0 if sc is None else sc.double())
        want = stream[:, :width].double() + 0.37 * v
        assert torch.allclose(mine.double(), want, **TOL[torch.float32])
        # (the norm of the row as it was stored: a row of one column may be near zero, where its norm is steep)
        assert torch.allclose(then.double(), rms(mine.double(), 1e-6) * (1.0 if norm is None else nw.double()), **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [1, 63, 64, 65, 256, 4097])
def test_a_sum_with_nothing_beside_it(width, dtype):
    o, R = ops(), 5
    y, w, stream = rnd(R, width + 3, seed=1, dtype=dtype)[:, :width], rnd(width, seed=2), rnd(R, width + 2, seed=3)
    mine = stream.clone()
    o.rmsnorm_add(y, w, None, 0.37, 1e-5, mine[:, :width])
    want = stream[:, :width].double() + 0.37 * rms(y.double(), 1e-5) * w.double()
    assert torch.allclose(mine[:, :width].double(), want, **TOL[torch.float32]) and torch.equal(mine[:, width:], stream[:, width:])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 256, 257, 512, 513, 769, 1023, 1024, 1025, 1280, 1281, 2560, 2561, 4097])
def test_activations_over_cut_rows(n, dtype):
    o, T = ops(), 3
    z, bias, two = rnd(T, n + 3, seed=n)[:, :n], rnd(n, seed=1), torch.tensor([0.7, 0.4], device=DEV)
    low = rnd(n, seed=2).abs()
    x = z.double() + bias.double()
    for kind, lower, want in (("silu", None, torch.nn.functional.silu(x)), ("exp_neg_softplus", low, torch.exp(-low.double() * torch.nn.functional.softplus(x))),
                              ("xielu", two, torch.where(x > 0, two[0].double() * x * x + x / 2, two[1].double() * (torch.expm1(x) - x) + x / 2))):
        out = torch.full((T, n + 2), 7.0, dtype=dtype, device=DEV)
        o.activate(z, kind, out[:, :n], bias=bias, lower=lower)
        assert torch.allclose(out[:, :n].double(), want, **TOL[dtype]) and (out[:, n:] == 7).all()
    mine = z.clone()
    o.activate(mine, "silu", mine, bias=bias)
    assert torch.allclose(mine.double(), torch.nn.functional.silu(x), **TOL[torch.float32])


@pytest.mark.parametrize("heads,dv", [(1, 1), (5, 16), (3, 63), (3, 64), (3, 65), (2, 128), (2, 129), (2, 256), (2, 257), (2, 512), (2, 513), (1, 1024),
                                      (2, 1025), (1, 2048), (1, 2049), (1, 3072), (2, 3073), (1, 4096), (1, 4097)])
@pytest.mark.parametrize("gate_first", [False, True])
def test_head_norms_hold_their_heads(heads, dv, gate_first):
    o, T = ops(), 3
    x, g, w = rnd(T, heads * dv + 4, seed=dv)[:, :heads * dv], rnd(T, heads * dv + 1, seed=2)[:, :heads * dv], rnd(heads, dv, seed=3)
    out = torch.empty(T, heads * dv, device=DEV)
    o.head_norm(x, w.flatten(), 1e-5, out, heads, gate=g, gate_kind="silu", gate_first=gate_first)
    act, v = torch.nn.functional.silu(g.double()), x.double()
    v = v * act if gate_first else v
    v = rms(v.view(T, heads, dv), 1e-5) * w.double()
    v = v.reshape(T, -1) * (1.0 if gate_first else act)
    assert torch.allclose(out.double(), v, **TOL[torch.float32])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dim", [(1, 2), (3, 64), (25, 80)])
def test_turned_runs_of_many_rows_and_few(heads, dim, dtype):
    """Up to 1,024 rows a row's pairs are cut among workgroups, beyond them not: the same numbers, places beside them untouched."""
    o, T = ops(), 1025
    src, pos = rnd(T, 2 * heads * dim, seed=dim), torch.arange(T, device=DEV, dtype=torch.int32)
    freq = 100.0 ** (-torch.arange(0, dim, 2, device=DEV).float() / dim)

    def turned(a, b):
        q, v = (torch.full((b - a, heads * dim + 1), 7.0, dtype=dtype, device=DEV) for _ in range(2))
        o.rotary_runs(src[a:b], pos[a:b], freq, [(q, 0, heads, dim, dim, 0, dim), (v, heads * dim, heads, dim, 0, 0, dim)])
        return q, v
    many, few = turned(0, T), [torch.cat(x) for x in zip(turned(0, 1), turned(1, T))]
    angle = (pos.double()[:, None] * freq.double()).repeat(1, heads)
    x = src[:, :heads * dim].double()
    even = x[:, 0::2] * torch.cos(angle) - x[:, 1::2] * torch.sin(angle)
    # (an angle of up to 1,024 is off by up to 2^-14 in 32 bits; bfloat16 rounds numbers of up to 8 by up to 2^-6)
    assert (many[0][:, 0:-1:2].double() - even).abs().max() < 4e-2 and bool((many[0][:, -1] == 7).all())
    assert torch.equal(many[1][:, :-1], src[:, heads * dim:].to(dtype))
    assert all(torch.equal(m, f) for m, f in zip(many, few))
