"""Which form the graph build takes (host arithmetic, no GPU): the rule goes by
the keys, the lists' members per key and the unit that scores the rows."""
import ctypes

import pytest
import torch  # noqa: F401  (binds the library to torch's HIP runtime)

from ssa_amd import _lib


def _form(dtype, d, M, C, R=8, P=3, T=0, mode=_lib.GRAPH_FULL, noalloc=0):
    a = _lib.GraphArgs()
    a.mode, a.B, a.Hq, a.Hkv, a.N, a.M, a.d = mode, 1, 2, 1, M, M, d
    a.q = _lib.Tensor4(0, dtype, 2 * M * d, M * d, d)
    a.k = _lib.Tensor4(256, dtype, M * d, M * d, d)
    a.rand_proj, a.R, a.max_p, a.P, a.T, a.C = 256, R, 12, P, T, C
    a.top_k, a.window, a.causal, a.total_k = max(C // 4, 1), 8, 1, 64
    f = _lib.lib().ssa_graph_form(ctypes.byref(a), noalloc)
    assert f > 0, _lib.lib().ssa_last_error()
    return f


F32, BF16 = _lib.SSA_F32, _lib.SSA_BF16


@pytest.mark.parametrize("dtype,d,line", [(F32, 64, 0.4), (F32, 256, 0.4), (BF16, 64, 1.0),
                                          (BF16, 128, 1.0), (BF16, 136, 0.4), (BF16, 256, 0.4),
                                          (_lib.SSA_F16, 160, 0.4), (BF16, 4, 0.4)])
def test_members_per_key_where_the_dense_form_begins(dtype, d, line):
    """Rows the matrix cores take (16-bit, 8 to 128 wide) from one member per
    key on, rows the vector units score from 0.4 on, both above 1,024 keys."""
    C = int(line * 4096 / 8)
    assert _form(dtype, d, 4096, C + 1) == _lib.FORM_DENSE
    assert _form(dtype, d, 4096, C - 1) == _lib.FORM_LIST


def test_limits_of_the_dense_form():
    assert _form(F32, 64, 4096, 4096) == _lib.FORM_DENSE
    assert _form(F32, 64, 4097, 4097) == _lib.FORM_LIST
    assert _form(F32, 64, 512, 512, R=64, P=1) == _lib.FORM_DENSE
    assert _form(F32, 64, 512, 512, R=65, P=1) == _lib.FORM_LIST
    assert _form(F32, 64, 4096, 4096, mode=_lib.GRAPH_LSH) == _lib.FORM_LIST
    assert _form(BF16, 64, 1024, 32) == _lib.FORM_DENSE
    assert _form(BF16, 64, 1024, 31) == _lib.FORM_LIST
