"""What the gradient entry points take and how much workspace they ask for
(host arithmetic: nothing is launched, this runs without a GPU)."""
import ctypes

import pytest
import torch  # noqa: F401  (binds the library to torch's HIP runtime)

from ssa_amd import _lib


def _args(B, H, kv, N, M, d, K, dtype=_lib.SSA_BF16, q=None, dout=None, det=False):
    """Arguments of one call over contiguous operands (q and dout: other
    strides).  The pointers are never followed."""
    def view(h, L, st=None):
        return _lib.Tensor4(256, dtype, *(st or (h * L * d, L * d, d)))
    a = _lib.ApplyGradArgs()
    f = a.fwd
    f.B, f.Hq, f.Hkv, f.N, f.M, f.d, f.K = B, H, kv, N, M, d, K
    f.q, f.k, f.v = view(H, N, q), view(kv, M), view(kv, M)
    f.neighbors, f.scale, f.out = 256, 1.0, 256
    a.dout, a.dq, a.dk, a.dv = view(H, N, dout), view(H, N), view(kv, M), view(kv, M)
    a.deterministic = int(det)
    return a


def _bytes(a):
    n = _lib.lib().ssa_sparse_gather_attention_grad_workspace_bytes(ctypes.byref(a))
    assert n > 0, _lib.lib().ssa_last_error()
    return n


@pytest.mark.parametrize("det", [False, True])
@pytest.mark.parametrize("N", [32768, 131072, 1 << 20])
def test_workspace_of_one_large_group_is_bounded(N, det):
    """One kv head under 32 query heads of 256 slots: from 2^28 slots on the
    workspace grows with the key rows alone."""
    slots, d = 1 << 28, 128
    fixed = slots * (24 if det else 20) + slots // 4096 * d * (64 if det else 16)
    per_key = (69 if det else 61) + d * (16 if det else 8)
    table = slots // 2 * 4                    # at most two slots per counted key
    assert _bytes(_args(1, 32, 1, N, N, d, 256, det=det)) <= fixed + table + per_key * N + (1 << 20)


def test_workspace_of_many_key_rows_is_bounded():
    """Few query rows over many key rows: launches of at most 2^25 key rows."""
    one = _bytes(_args(512, 1, 1, 2, 65536, 8, 3))
    assert one <= (1 << 25) * 62 + (1 << 20)
    assert _bytes(_args(4096, 1, 1, 2, 65536, 8, 3)) <= one + (1 << 20)


@pytest.mark.parametrize("det", [False, True])
def test_any_strides_of_q_and_dout_are_taken(det):
    """Query rows of a kv head beyond 32-bit offsets from each other, as the
    forward takes them."""
    far, back = (1 << 40, (1 << 32) + 1, 17), (1 << 20, -(1 << 10), 16)
    want = _bytes(_args(1, 2, 1, 4, 8, 16, 3, det=det))
    for kw in (dict(q=far), dict(dout=far), dict(q=back), dict(dout=back)):
        assert _bytes(_args(1, 2, 1, 4, 8, 16, 3, det=det, **kw)) == want
