"""Gradients of the gather attention through the transposed graph
(ssa_sparse_gather_attention_grad) at the sizes where it can go wrong, against
float64 autograd of the same function.

Bar: a gradient element is a sum of terms w x (w = p (dp - sum p dp) scale for
dq and dk, p for dv), where w itself is a difference.  Its error is held
against the sum of the absolute values of everything that enters it, A = sum
p (|dp| + sum p |dp|) scale |x| (sum p |x| for dv), whose rounding in fp32 is a
few eps (6e-8) times the relative error of p, which is that of a score: at
most eps times the sum of |q k| scale over the head dim, about 30 eps at 1,024.
BAR is 1e-5 of the row's largest A in fp32; a 16-bit result is rounded once
more, by at most its type's unit roundoff: 2^-8 (8 significant bits, bf16) or
2^-11 (11 bits, fp16) of itself; fp16 below 2^-14 is rounded to a multiple of
2^-24, off by at most 2^-25 whatever its size."""
import ctypes

import pytest
import torch

from conftest import has_gpu
from test_gpu_parity import GRAD_REL, _check_grad_rows

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a ROCm GPU")]
DEV = "cuda"


def _inputs(B, H, kv, N, M, d, K, dtype, seed, spread=None):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, h, L, d, generator=g).to(dtype).to(DEV)
               for h, L in ((H, N), (kv, M), (kv, M)))
    nb = torch.randint(0, spread or M, (B, H, N, K), generator=g).to(DEV)
    va = (torch.rand(B, H, N, K, generator=g) > 0.25).to(DEV)
    va[..., 0] = True
    dout = torch.randn(B, H, N, d, generator=g).to(dtype).to(DEV)
    return q, k, v, nb, va, dout


BAR = {torch.float32: 1e-5, torch.bfloat16: 1e-5 + 2 ** -8, torch.float16: 1e-5 + 2 ** -11}


def _reference(q, k, v, nb, va, scale, dout):
    """(gradients, their A as above), float64, written out over the slots."""
    B, H, N, K = nb.shape
    kv, M, d = k.shape[1:]
    qr, kr, vr, do = (t.double() for t in (q, k, v, dout))
    flat = (nb + (torch.arange(B, device=DEV).view(B, 1, 1, 1) * kv
                  + torch.arange(H, device=DEV).view(1, H, 1, 1) // (H // kv)) * M).reshape(-1)
    kg, vg = (t.reshape(-1, d).index_select(0, flat).view(B, H, N, K, d) for t in (kr, vr))
    s = ((qr.unsqueeze(3) * kg).sum(-1) * scale).masked_fill(~va, float("-inf"))
    p = torch.softmax(s, -1)
    dp = (do.unsqueeze(3) * vg).sum(-1)
    w = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
    wa = p * (dp.abs() + (p * dp.abs()).sum(-1, keepdim=True)) * scale

    def rows(w, x):
        return (w.unsqueeze(-1) * x).sum(3)

    def keys(w, x):
        t = (w.unsqueeze(-1) * x.unsqueeze(3)).reshape(-1, d)
        return torch.zeros_like(kr).reshape(-1, d).index_add_(0, flat, t).view_as(kr)
    return ((rows(w, kg), keys(w, qr), keys(p, do)),
            (rows(wa, kg.abs()), keys(wa, qr.abs()), keys(p, do.abs())))


def _check(got, exp, dtype):
    for name, a, b, c in zip(("dq", "dk", "dv"), got, *exp):
        assert a.dtype == dtype and a.shape == b.shape
        err = (a.double() - b).abs().amax(-1)
        assert not err[c.amax(-1) == 0].any(), f"{name}: gradient in a row nothing reaches"
        if dtype == torch.float16:
            err = (err - 2 ** -25).clamp_min(0)
        worst = (err / c.amax(-1).clamp_min(1e-300)).max().item()
        print(f"  {name}: worst row error {worst:.2e}", flush=True)
        assert worst <= BAR[dtype], (name, worst)


# (B, H, kv, N, M, d, K, ids below): K over and under a wave's slots and a loop
# step; one key, keys that no row reaches, keys whose lists take several
# segments (ids below a few), key rows beyond one counting range (M > 16,384),
# a block of query rows that ends a group, every head-dim instance
CASES = [(1, 1, 1, 1, 1, 4, 1, None), (1, 2, 1, 3, 2, 8, 5, None), (2, 4, 2, 65, 40, 16, 63, None),
         (1, 8, 1, 130, 300, 32, 65, 3), (2, 6, 3, 257, 129, 64, 17, None),
         (1, 4, 4, 100, 500, 64, 129, None), (3, 4, 2, 33, 70, 80, 31, None),
         (1, 4, 1, 600, 90, 96, 40, 2), (1, 2, 1, 900, 257, 128, 70, 5),
         (1, 2, 2, 40, 20000, 128, 96, None), (1, 1, 1, 700, 40000, 32, 33, None),
         (1, 2, 1, 20, 50, 256, 24, None), (1, 2, 1, 9, 30, 512, 11, None),
         (1, 1, 1, 7, 20, 1024, 9, None), (1, 1, 1, 4, 3500, 64, 3073, None),
         (1, 1, 1, 5, 200, 64, 3072, None)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"N{c[3]}_M{c[4]}_d{c[5]}_K{c[6]}")
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("det", [False, True], ids=["default", "deterministic"])
def test_gradients_match_float64_autograd(case, dtype, det):
    from ssa_amd import _lib
    *shape, spread = case
    q, k, v, nb, va, dout = _inputs(*shape, dtype, 3, spread)
    scale = shape[5] ** -0.5
    exp = _reference(q, k, v, nb, va, scale, dout)
    runs = [_lib.gather_attention_grad(q, k, v, nb, va, scale, False, 0.0, 0, dout, det)
            for _ in range(2)]
    _check(runs[0], exp, dtype)
    if det:
        for a, b in zip(*runs):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gradients_of_other_layouts_and_graph_forms(dtype):
    """Rows at odd element offsets and strides, a projection's transposed
    views, an fp32 upstream gradient, an int32 graph: the same gradients."""
    from ssa_amd import _lib
    B, H, kv, N, M, d, K = 2, 4, 2, 70, 90, 32, 37
    q, k, v, nb, va, dout = _inputs(B, H, kv, N, M, d, K, dtype, 5)
    scale = d ** -0.5
    base = _lib.gather_attention_grad(q, k, v, nb, va, scale, False, 0.0, 0, dout, True)
    _check(base, _reference(q, k, v, nb, va, scale, dout), dtype)

    def odd(t):
        b, h, n, e = t.shape
        w = torch.zeros(b, n, h, e + 3, dtype=t.dtype, device=DEV)
        w[..., 1:e + 1] = t.transpose(1, 2)
        return w[..., 1:e + 1].transpose(1, 2)

    def proj(t):
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    nb32 = torch.where(va, nb, -1).to(torch.int32)
    for name, args in {"odd": (odd(q), odd(k), odd(v), nb, va, odd(dout)),
                       "projection": (proj(q), proj(k), proj(v), nb, va, proj(dout)),
                       "int32 graph": (q, k, v, nb32, None, dout),
                       "fp32 upstream": (q, k, v, nb, va, dout.float())}.items():
        qq, kk, vv, n, m, g = args
        got = _lib.gather_attention_grad(qq, kk, vv, n, m, scale, False, 0.0, 0, g, True)
        for a, b, t in zip(got, base, (qq, kk, vv)):
            assert a.shape == t.shape
            # the key rows' terms keep their grid; fp32 products of an fp32
            # upstream gradient may round the scores' sums differently
            rel = ((a.double() - b.double()).norm() / b.double().norm()).item()
            assert rel <= (2e-6 if dtype == torch.float32 else 4e-3), (name, rel)


def test_gradients_per_launch_of_groups():
    """Three groups of 2^27 slots take two launches: each group's gradients
    equal those of a call on the group alone, bit for bit (deterministic)."""
    from ssa_amd import _lib
    B, N, M, d, K = 3, 131072, 64, 8, 1024
    g = torch.Generator(DEV).manual_seed(9)
    q = torch.randn(B, 1, N, d, generator=g, device=DEV)
    k, v = (torch.randn(B, 1, M, d, generator=g, device=DEV) for _ in range(2))
    dout = torch.randn(B, 1, N, d, generator=g, device=DEV)
    nb = torch.randint(0, M, (B, 1, N, K), generator=g, device=DEV, dtype=torch.int32)
    got = _lib.gather_attention_grad(q, k, v, nb, None, 0.3, False, 0.0, 0, dout, True)
    for b in range(B):
        s = slice(b, b + 1)
        one = _lib.gather_attention_grad(q[s], k[s], v[s], nb[s], None, 0.3, False, 0.0, 0,
                                         dout[s], True)
        for a, c in zip(got, one):
            assert torch.equal(a[s], c)


@pytest.mark.parametrize("det", [False, True])
def test_gradients_of_rows_without_a_finite_softmax(det):
    """A row whose slots are all masked has NaN weights: NaN in its dq and in
    the rows of dk and dv its ids name, as the atomic backward leaves them;
    nothing else is touched."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 2, 1, 40, 50, 64, 12, torch.float32, 8)
    va[0, 1, 7] = False
    nb[0, 1, 7] = torch.arange(12, device=DEV)
    old = _lib.gather_attention_bwd(q, k, v, nb, va, 0.125, False, 0.0, 0, dout)
    new = _lib.gather_attention_grad(q, k, v, nb, va, 0.125, False, 0.0, 0, dout, det)
    for a, b in zip(new, old):
        assert torch.equal(torch.isnan(a), torch.isnan(b))
        fine = ~torch.isnan(b)
        err = (a - b)[fine].abs().max() / b[fine].abs().max()
        assert err <= GRAD_REL[torch.float32]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_backward_c_entries_agree(dtype):
    """ssa_sparse_gather_attention_bwd (atomics, no workspace), _bwd_det and
    _grad on one input with dropout: the same gradients."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(2, 4, 2, 150, 80, 64, 50, dtype, 4)
    a = _lib.gather_attention_bwd(q, k, v, nb, va, 0.125, False, 0.2, 77, dout)
    b = _lib.gather_attention_bwd(q, k, v, nb, va, 0.125, False, 0.2, 77, dout, deterministic=True)
    c = _lib.gather_attention_grad(q, k, v, nb, va, 0.125, False, 0.2, 77, dout, False)
    for x, y, z in zip(a, b, c):
        _check_grad_rows("bwd_det", y, x, torch.float32)
        _check_grad_rows("grad", z, x, dtype)


def test_gradient_workspace_is_checked():
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 2, 1, 8, 9, 16, 4, torch.float32, 1)
    grads = [torch.empty_like(t) for t in (q, k, v)]
    f, keep = _lib._apply_args(q, k, v, nb, va, 1.0, False, 0.0, 0, grads[0])
    a = _lib.ApplyGradArgs()
    a.fwd = f
    a.dout, _ = _lib.view4(dout)
    (a.dq, _), (a.dk, _), (a.dv, _) = (_lib.view4(t) for t in grads)
    L = _lib.lib()
    need = L.ssa_sparse_gather_attention_grad_workspace_bytes(ctypes.byref(a))
    assert need > 0
    ws = torch.empty(int(need), dtype=torch.uint8, device=DEV)
    assert L.ssa_sparse_gather_attention_grad(ctypes.byref(a), ws.data_ptr(), int(need) - 1, 0) != 0
    assert b"workspace" in L.ssa_last_error()
    a.dk.dtype = _lib.SSA_F16
    assert L.ssa_sparse_gather_attention_grad_workspace_bytes(ctypes.byref(a)) < 0


# ---- rows and slots that hold infinities, NaNs or nothing

@pytest.mark.parametrize("K", [65, 3073], ids=["lds", "long"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_dq_takes_nothing_from_a_key_no_slot_names(K, dtype, bad):
    """Key row 0 is named by no slot (K is no multiple of a step, some slots
    are masked, some ids lie out of range): what it holds reaches no gradient,
    bit for bit."""
    from ssa_amd import _lib
    N = 20 if K < 100 else 3
    q, k, v, nb, va, dout = _inputs(2, 4, 2, N, 90, 64, K, dtype, 13)
    nb.clamp_min_(1)
    nb[:, :, ::2, 3], nb[:, :, ::3, 5] = -7, 90
    graphs = {"int64": (nb, va), "int32": (torch.where(va, nb, -1).to(torch.int32), None)}
    for name, (n, m) in graphs.items():
        runs = []
        for x in (1.0, bad):
            k[:, :, 0] = x
            runs.append(_lib.gather_attention_grad(q, k, v, n, m, 0.125, False, 0.0, 0, dout, True))
        for a, b in zip(*runs):
            assert torch.isfinite(a).all() and torch.equal(a, b), name


@pytest.mark.parametrize("K", [12, 3100], ids=["lds", "long"])
@pytest.mark.parametrize("det", [False, True])
def test_gradients_of_rows_without_any_key(K, det):
    """Query rows whose ids all lie out of range (an int32 graph's -1) have no
    key: their dq is zero, as the atomic backward leaves it."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 2, 1, 6, 50, 64, K, torch.float32, 8)
    va[:] = True
    nb[0, 1, 3] = -1
    old = _lib.gather_attention_bwd(q, k, v, nb, va, 0.125, False, 0.0, 0, dout)
    for n, m in ((nb, va), (nb.to(torch.int32), None)):
        new = _lib.gather_attention_grad(q, k, v, n, m, 0.125, False, 0.0, 0, dout, det)
        assert (new[0][0, 1, 3] == 0).all() and (old[0][0, 1, 3] == 0).all()
        for name, a, b in zip(("dq", "dk", "dv"), new, old):
            _check_grad_rows(name, a, b, torch.float32)


@pytest.mark.parametrize("K", [12, 3100], ids=["lds", "long"])
@pytest.mark.parametrize("det", [False, True])
def test_dq_weighs_a_masked_slots_own_row(K, det):
    """A masked slot's weight of 0 times its own key row, as autograd has it:
    NaN in dq where that row is infinite, in no other query row."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 2, 1, 6, 50, 64, K, torch.float32, 8)
    nb %= 40
    nb[0, 1, 2, 4], va[0, 1, 2, 4] = 45, False
    k[0, 0, 45] = float("inf")
    old = _lib.gather_attention_bwd(q, k, v, nb, va, 0.125, False, 0.0, 0, dout)[0]
    new = _lib.gather_attention_grad(q, k, v, nb, va, 0.125, False, 0.0, 0, dout, det)[0]
    assert torch.equal(torch.isnan(new), torch.isnan(old))
    rows = torch.isnan(new).all(-1)
    assert rows[0, 1, 2] and rows.sum() == 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("det", [False, True])
@pytest.mark.parametrize("which", ["q", "dout"])
def test_one_nan_reaches_only_its_key_rows(dtype, det, which):
    """A NaN in one query row's q or dout: NaN in that row's dq and in the key
    rows it names, as the atomic backward leaves them; the other batch's
    gradients keep their bits and unnamed key rows are zero."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(2, 2, 1, 30, 200, 64, 12, dtype, 17)
    args = (k, v, nb, va, 0.125, False, 0.0, 0)
    clean = _lib.gather_attention_grad(q, *args, dout, True)
    (q if which == "q" else dout)[0, 1, 7, 5] = float("nan")
    old = _lib.gather_attention_bwd(q, *args, dout)
    new = _lib.gather_attention_grad(q, *args, dout, det)
    for name, a, b, c in zip(("dq", "dk", "dv"), new, old, clean):
        assert torch.equal(torch.isnan(a), torch.isnan(b)), name
        assert not torch.isnan(a[1]).any()
        if det:
            assert torch.equal(a[1], c[1]), name
    named = torch.zeros(200, dtype=torch.bool, device=DEV)
    named[nb[0].reshape(-1)] = True
    assert (new[1][0, 0, ~named] == 0).all() and (new[2][0, 0, ~named] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("size", [1e8, 1e12])
def test_deterministic_key_rows_ignore_outliers_they_are_not_named_by(dtype, size):
    """One query row's q and dout many orders above the rest: key rows that row
    does not name keep their gradients' bits."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 4, 2, 130, 40, 64, 33, dtype, 19)
    nb.clamp_min_(8)
    nb[0, 0, 5] %= 8
    args = (k, v, nb, va, 0.125, False, 0.0, 0)
    base = _lib.gather_attention_grad(q, *args, dout, True)
    q[0, 0, 5] *= size
    dout[0, 0, 5] *= size
    got = _lib.gather_attention_grad(q, *args, dout, True)
    for a, b in zip(got[1:], base[1:]):
        assert torch.equal(a[:, :, 8:], b[:, :, 8:])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("size", [1e6, 1e10, 1e14])
def test_deterministic_sums_keep_their_bits_beside_an_outlier(dtype, size):
    """One element of one dout row many orders above everything else: the
    other elements of the key rows it reaches are as close to float64 as
    without it.  Bar per element: BAR of the sum of the terms' sizes."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 2, 1, 200, 6, 64, 40, dtype, 23)
    dout[0, 0, 9, 3] = size
    scale = 0.125
    dv = _lib.gather_attention_grad(q, k, v, nb, va, scale, False, 0.0, 0, dout, True)[2]
    exp, absum = (t[2] for t in _reference(q, k, v, nb, va, scale, dout))
    keep = torch.arange(64, device=DEV) != 3
    err = ((dv.double() - exp).abs() / absum)[..., keep].max().item()
    print(f"  outlier {size:.0e}: {err:.2e}", flush=True)
    assert err <= BAR[dtype]


@pytest.mark.parametrize("dtype,det", [(torch.float32, False), (torch.float32, True),
                                       (torch.bfloat16, True)])
def test_gradients_of_a_group_in_parts(dtype, det):
    """One group of more than 2^28 slots goes in two parts of its query rows:
    dq equals that of calls on the parts' rows, dk and dv the sum of theirs."""
    from ssa_amd import _lib
    N, M, d, K = (1 << 18) + 1000, 64, 8, 1024
    g = torch.Generator(DEV).manual_seed(9)
    q, dout = (torch.randn(1, 1, N, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    k, v = (torch.randn(1, 1, M, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    nb = torch.randint(0, M - 1, (1, 1, N, K), generator=g, device=DEV, dtype=torch.int32)
    got = _lib.gather_attention_grad(q, k, v, nb, None, 0.3, False, 0.0, 0, dout, det)
    if det:
        again = _lib.gather_attention_grad(q, k, v, nb, None, 0.3, False, 0.0, 0, dout, det)
        assert all(torch.equal(a, b) for a, b in zip(got, again))
    parts = [_lib.gather_attention_grad(q[:, :, s], k, v, nb[:, :, s].contiguous(), None, 0.3,
                                        False, 0.0, 0, dout[:, :, s], True)
             for s in (slice(0, 100000), slice(100000, N))]
    assert torch.equal(got[0], torch.cat([p[0] for p in parts], 2))
    for a, b, c in zip(got[1:], *(p[1:] for p in parts)):
        exp = b.double() + c.double()
        assert (a[0, 0, M - 1] == 0).all()
        rel = ((a.double() - exp).norm() / exp.norm()).item()
        assert rel <= (2e-6 if dtype == torch.float32 else 4e-3), rel


def test_gradients_of_more_key_rows_than_a_launch_takes():
    """2^26 key rows under two query rows a batch: launches of 2^25 key rows."""
    from ssa_amd import _lib
    B, M, d, K = 1024, 65536, 4, 3
    q, k, v, nb, va, dout = _inputs(B, 1, 1, 2, M, d, K, torch.float32, 29)
    got = _lib.gather_attention_grad(q, k, v, nb, va, 0.5, False, 0.0, 0, dout, False)
    _check(got, _reference(q, k, v, nb, va, 0.5, dout), torch.float32)


@pytest.mark.parametrize("det", [False, True])
@pytest.mark.parametrize("which", ["q", "dout"])
def test_gradients_of_query_rows_far_apart(which, det):
    """Two query heads of one kv head 2^32 + 1 elements apart (an odd stride, so
    no unit fits 32 bits): the gradients of the same rows side by side."""
    from ssa_amd import _lib
    q, k, v, nb, va, dout = _inputs(1, 2, 1, 70, 50, 32, 37, torch.bfloat16, 31)
    base = _lib.gather_attention_grad(q, k, v, nb, va, 0.2, False, 0.0, 0, dout, det)
    far = torch.empty((1 << 32) + 70 * 33 + 64, dtype=torch.bfloat16, device=DEV).as_strided(
        (1, 2, 70, 32), (1 << 33, (1 << 32) + 1, 33, 1))
    far.copy_(q if which == "q" else dout)
    got = _lib.gather_attention_grad(far if which == "q" else q, k, v, nb, va, 0.2, False, 0.0, 0,
                                     far if which == "dout" else dout, det)
    for name, a, b in zip(("dq", "dk", "dv"), got, base):
        if det or name == "dq":
            assert torch.equal(a, b), name
        _check_grad_rows(name, a, b, torch.bfloat16)
