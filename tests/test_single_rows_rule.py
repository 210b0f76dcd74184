"""Which steps of single rows in the plain kernels are one kernel: a rule of the native library (the host alone answers)."""
import pytest

from denno_beta_amd.build import load_library
from denno_beta_amd.kernels import ops


@pytest.fixture(scope="module")
def lib():
    """(The library as such: a question that launches nothing needs no GPU.)"""
    lib = load_library("attention")
    ops._declare("attention", lib)
    return lib


@pytest.mark.parametrize("dtype,H,Hkv,longest,most", [
    (ops.F32, 16, 16, 64, 48), (ops.F32, 16, 16, 128, 48), (ops.F32, 16, 16, 129, None), (ops.F32, 16, 16, 256, None), (ops.F32, 16, 16, 257, 16),
    (ops.F32, 16, 16, 512, 16), (ops.F32, 16, 16, 513, 0), (ops.F32, 16, 4, 64, 24), (ops.F32, 16, 4, 256, 24), (ops.F32, 16, 4, 257, 8),
    (ops.F32, 16, 4, 512, 8), (ops.BF16, 16, 16, 64, 48), (ops.BF16, 16, 4, 65, None), (ops.BF16, 16, 4, 256, None), (ops.BF16, 16, 4, 512, 48),
    (ops.BF16, 16, 4, 513, 0)])
def test_most_rows_that_one_kernel_takes(lib, dtype, H, Hkv, longest, most):
    part = lambda rows, dh=64, ps=16, at=0: lib.dn_attention_rows_part_floats(at, 0, rows, longest, H, Hkv, dh, ps, dtype)
    two = lambda rows, dh=64: rows * H * -(-longest // lib.dn_attention_rows_tile(dh)) * (dh + 2)
    for rows in (1, most or 1, 4096) if most != 0 else ():
        assert part(rows) == (0 if most is None or rows <= most else two(rows))
    if most is not None:
        assert part(most + 1) == two(most + 1)
    # heads of another size, pages that cut a run of four keys, pools that are not aligned: always two kernels
    assert part(1, dh=48) == two(1, 48) and part(1, ps=6) == two(1) and part(1, at=8) == two(1)
