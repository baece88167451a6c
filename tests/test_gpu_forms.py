"""The graph build's two forms (over the lists' members, over every key) on the
same inputs: the rule of a plain build takes one of them, so each test here
builds in both, the list form against the oracle (bit for bit, as the tests it
runs ask) and the dense form against the list form."""
import contextlib
import math

import numpy as np
import pytest
import torch

import oracle
import test_gpu_checked as checked
import test_gpu_dense as dense
import test_gpu_parity as parity
import test_gpu_sweep as sweep
from conftest import has_gpu
from ssa_amd import _lib

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a ROCm GPU")]
DEV = "cuda"
DENSE_KEYS, DENSE_LISTS, DENSE_LDS = 4096, 64, 65536


def _dense_takes(k, kw):
    M, lists = k.shape[2], kw["R"] * (1 + min(kw["T"], kw["P"]))
    return (M <= DENSE_KEYS and lists <= DENSE_LISTS
            and 2 ** kw["P"] * ((M + 63) // 64 * 8 + 4) <= DENSE_LDS)


@contextlib.contextmanager
def both_forms(monkeypatch, seen):
    """Within: FULL-mode builds run in each form that takes the sizes and must
    agree; the list form's graph is returned.  seen: (auto form, forms run)."""
    plain = _lib.build_graph

    def build(q, k, rand_proj, **kw):
        if kw.get("mode", _lib.GRAPH_FULL) != _lib.GRAPH_FULL:
            return plain(q, k, rand_proj, **kw)
        kw["count_ties"] = True
        sizes = {n: kw[n] for n in ("P", "T", "C", "top_k", "window", "causal", "is_cross",
                                    "total_k", "glob")}
        auto = _lib.graph_form(q, k, rand_proj, **sizes)
        out = plain(q, k, rand_proj, form=_lib.FORM_LIST, **kw)
        forms = [_lib.FORM_LIST]
        if _dense_takes(k, dict(kw, R=rand_proj.shape[0])):
            forms.append(_lib.FORM_DENSE)
            got = plain(q, k, rand_proj, form=_lib.FORM_DENSE, **kw)
            assert torch.equal(got[0], out[0])
            if out[1] is not None:
                assert torch.equal(got[1], out[1])
            assert int(got[2].item()) == int(out[2].item())
        else:
            with pytest.raises(RuntimeError, match="dense form"):
                plain(q, k, rand_proj, form=_lib.FORM_DENSE, **kw)
        assert auto in forms
        seen.append((auto, tuple(forms)))
        return out
    with monkeypatch.context() as m:
        m.setattr(_lib, "build_graph", build)
        yield


DTYPES = [torch.float32, torch.bfloat16, torch.float16]


@pytest.mark.parametrize("case", parity.GRAPH_CASES, ids=lambda c: c[0])
@pytest.mark.parametrize("dtype", DTYPES)
def test_exact_tier_in_both_forms(case, dtype, monkeypatch):
    seen = []
    with both_forms(monkeypatch, seen):
        if dtype == torch.float32:
            parity.test_full_graph_exact_tier_matches_oracle(case, 0)
        else:
            parity.test_graph_16bit_inputs_exact_tier(case, dtype)
    assert len(seen) == 1 and (len(seen[0][1]) == 2) == (case[5] <= DENSE_KEYS)


@pytest.mark.parametrize("case", parity.MANY_TIES, ids=lambda c: c[0])
def test_many_tied_rows_in_both_forms(case, monkeypatch):
    seen = []
    with both_forms(monkeypatch, seen):
        parity.test_graph_exact_tier_many_tied_rows(case)
    assert len(seen[0][1]) == 2


def test_huge_k_in_both_forms(monkeypatch):
    """More neighbours than either replay holds in LDS."""
    seen = []
    with both_forms(monkeypatch, seen):
        parity.test_full_graph_exact_tier_huge_k_replay_outside_lds()
        parity.test_full_graph_exact_tier_huge_k_per_wave_replay_workspace()
    assert [len(s[1]) for s in seen] == [2, 2]


@pytest.mark.parametrize("case,dtype", sweep.CASES + sweep.WIDE_CASES,
                         ids=[c[0][0] for c in sweep.CASES + sweep.WIDE_CASES])
def test_sweep_in_both_forms(case, dtype, monkeypatch):
    seen = []
    with both_forms(monkeypatch, seen):
        sweep.test_graph_shape_sweep_matches_oracle(case, dtype)
    assert len(seen) == 1


@pytest.mark.parametrize("case", dense.SIZES,
                         ids=lambda c: f"N{c[3]}_M{c[4]}_d{c[5]}_R{c[6]}_T{c[8]}")
@pytest.mark.parametrize("dtype", DTYPES)
def test_dense_edges_in_both_forms(case, dtype, monkeypatch):
    """What test_gpu_dense says of its sizes: all but the last of a limit (4,097
    keys, 65 lists) are taken by the dense form, and by the rule."""
    seen = []
    with both_forms(monkeypatch, seen):
        dense.test_dense_graph_sizes_match_oracle(case, dtype)
    M, lists = case[4], case[6] * (1 + case[8])
    takes = M <= DENSE_KEYS and lists <= DENSE_LISTS
    assert seen == [(_lib.FORM_DENSE if takes else _lib.FORM_LIST,
                     (_lib.FORM_LIST, _lib.FORM_DENSE)[:1 + takes])]


@pytest.mark.parametrize("edit", [dense._one_sided, dense._zero_rows, dense._copies,
                                  dense._outlier], ids=lambda f: f.__name__.strip("_"))
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_hard_inputs_in_both_forms(edit, causal, dtype, monkeypatch):
    seen = []
    with both_forms(monkeypatch, seen):
        dense.test_dense_graph_hard_inputs_match_oracle(edit, causal, dtype)
    assert seen == [(_lib.FORM_DENSE, (_lib.FORM_LIST, _lib.FORM_DENSE))]


@pytest.mark.parametrize("shape", [(1, 4, 1, 4096, 64, 0, True), (2, 4, 2, 777, 128, 1, True),
                                   (1, 4, 4, 1500, 96, 2, False)],
                         ids=["n4096_d64", "n777_d128_probes", "n1500_d96_two_sided"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_real_scores_in_both_forms(shape, dtype, monkeypatch):
    """Normally distributed rows: scores whose order depends on how they are
    summed, which both forms do alike."""
    B, H, kv, N, d, T, causal = shape
    g = torch.Generator().manual_seed(41)
    q = torch.randn(B, H, N, d, generator=g).to(dtype).to(DEV)
    k = torch.randn(B, kv, N, d, generator=g).to(dtype).to(DEV)
    rp = torch.randn(8, 12, d, generator=g).to(DEV)
    seen = []
    with both_forms(monkeypatch, seen):
        _lib.build_graph(q, k, rp, P=max(1, round(math.log2(N / 368))), T=T, C=368, top_k=92,
                         window=16, causal=causal, is_cross=False, total_k=128,
                         glob=torch.arange(2, device=DEV))
    assert len(seen[0][1]) == 2


@pytest.mark.parametrize("case", checked.INT_CASES, ids=lambda c: c[0])
def test_checked_build_in_both_forms(case, monkeypatch):
    """Every index of either form inside its buffer."""
    seen = []
    with both_forms(monkeypatch, seen):
        checked.test_checked_build_exact_tier(case, _lib.GRAPH_FULL)
    assert len(seen) == 2 and (len(seen[0][1]) == 2) == (case[5] <= DENSE_KEYS)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_dense_form_in_head_chunks(dtype):
    """Four heads whose dense score rows take 35 MB each go through the scratch
    array one at a time (later chunks take their aux pass, scores and scales
    apart from the key phase, and the tied rows of all are replayed at the end):
    the oracle's graph, and the workspace build's, which has one chunk."""
    B, H, kv, N, d, R, P, C, kk, K, w = 1, 4, 2, 4096, 16, 8, 3, 656, 164, 200, 16
    g = torch.Generator().manual_seed(43)
    q, k = parity._ints((B, H, N, d), -6, 6, g), parity._ints((B, kv, N, d), -6, 6, g)
    rp = parity._ints((R, P, d), -6, 6, g)
    args = (q.to(DEV, dtype), k.to(DEV, dtype), rp.to(DEV))
    kw = dict(P=P, T=0, C=C, top_k=kk, window=w, causal=True, is_cross=False, total_k=K,
              glob=torch.arange(2, device=DEV))
    for noalloc in (False, True):
        assert _lib.graph_form(*args, noalloc=noalloc, **kw) == _lib.FORM_DENSE
    got = _lib.build_graph(*args, count_ties=True, noalloc=True, **kw)
    one = _lib.build_graph(*args, count_ties=True, **kw)
    for a, b in zip(got, one):
        assert torch.equal(a, b)
    ref = oracle.lsh_forward(q.reshape(B * H, N, d).numpy(), k.reshape(B * kv, N, d).numpy(),
                             rp.numpy(), kv_rep=H // kv, P=P, T=0, C=C, top_k=kk, causal=True,
                             glob=np.arange(2))
    assert ref["n_ties"] == int(got[2].item()) > 0
    pos = np.arange(N)[:, None]
    win = np.clip(np.minimum(pos + np.arange(-w, w + 1)[None], pos), 0, N - 1)
    rnb, rva = oracle.merge(win, np.arange(2), ref["idx"], has_self=True, total_k=K)
    np.testing.assert_array_equal(got[0].cpu().numpy().reshape(B * H, N, -1), rnb)
    np.testing.assert_array_equal(got[1].cpu().numpy().reshape(B * H, N, -1), rva)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_that_are_not_finite_in_both_forms(causal, dtype, monkeypatch):
    """Infinities and NaNs in query and key rows (and so in norms, codes and
    exact keys): the same graph from both forms, every index of the
    bounds-checked build inside its buffer."""
    g = torch.Generator().manual_seed(47)
    q = torch.randn(1, 2, 500, 32, generator=g)
    k = torch.randn(1, 2, 500, 32, generator=g)
    # the first kv head finite but for two query rows, the second with such keys
    q[0, 0, 70], q[0, 0, 300, 3], q[0, 1, 400, 5] = float("nan"), float("inf"), float("nan")
    k[0, 1, 9], k[0, 1, 33, 2], k[0, 1, 200, 4] = float("nan"), float("inf"), -float("inf")
    rp = torch.randn(6, 12, 32, generator=g).to(DEV)
    seen = []
    with both_forms(monkeypatch, seen), _lib.checked_library() as record:
        record()
        _lib.build_graph(q.to(DEV, dtype), k.to(DEV, dtype), rp, P=3, T=1, C=112, top_k=28,
                         window=4, causal=causal, is_cross=False, total_k=40,
                         glob=torch.arange(2, device=DEV))
        torch.cuda.synchronize()
        assert record() is None
    assert len(seen[0][1]) == 2
