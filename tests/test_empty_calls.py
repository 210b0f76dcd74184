"""Calls with nothing to work on: the host answers them, no kernel is launched.  Where there is no GPU a launch is an error, which
shows it (and nothing can read in front of an empty tensor)."""
import ctypes

import pytest
import torch


@pytest.fixture(scope="module")
def sequence():
    if torch.cuda.is_available():
        pytest.skip("a launch is an error only where there is no GPU")
    from denno_beta_amd.build import load_library
    from denno_beta_amd.kernels import ops
    lib = load_library("sequence")
    ops._declare("sequence", lib)
    return lib


@pytest.mark.parametrize("T,dv,launched", [(0, 64, False), (3, 0, False), (0, 0, False), (3, 64, True)])
@pytest.mark.parametrize("out_dtype", [0, 1])
def test_head_norms_without_columns_or_rows(sequence, T, dv, launched, out_dtype):
    """A kernel that holds its heads reads a head's last column, which heads without columns do not have."""
    here = (ctypes.c_float * (4 * 64 * 2))()
    p = ctypes.addressof(here)
    code = sequence.dn_head_norm(p, 2 * dv, p, 0, 1e-5, p, 2 * dv, 0, 0, None, 0, None, 0, p, out_dtype, 2 * dv, T, 2, dv, None)
    assert (code != 0) == launched
