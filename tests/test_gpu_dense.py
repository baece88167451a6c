"""The graph build's dense form (every key scored once, candidates as bucket
bitmaps) at the sizes and inputs where it can go wrong, against the oracle.

q, k and the hyperplanes hold small integers, so projections and scores are
exact in every type and order: neighbours and valid masks must equal the
oracle's bit for bit, tied kk-th scores included."""
import numpy as np
import pytest
import torch

import oracle
from conftest import has_gpu
from test_gpu_parity import _ints, _nowarn

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a ROCm GPU")]
DEV = "cuda"


def _build(B, H, nkv, N, M, d, R, maxP, T, K, w, G, causal, cross, dtype, edit=None, seed=0):
    from ssa_amd import SSAConfig, SparseAttention
    cfg = SSAConfig(d_model=H * d, num_heads=H, num_kv_heads=nkv, num_neighbors=K,
                    max_num_hashes=maxP, num_hash_rounds=R, lsh_num_probes=T, window_size=w,
                    num_global_tokens=G if isinstance(G, int) else 2,
                    global_token_indices=G if isinstance(G, list) else None, causal=causal)
    torch.manual_seed(seed)
    with _nowarn():
        attn = SparseAttention(cfg)
    g = torch.Generator().manual_seed(50 + seed)
    q, k = _ints((B, H, N, d), -6, 6, g), _ints((B, nkv, M, d), -6, 6, g)
    rp = _ints(tuple(attn.lsh_builder.rand_proj.shape), -6, 6, g)
    if edit:
        q, k = edit(q, k)
    attn.lsh_builder.rand_proj.copy_(rp)
    attn = attn.to(DEV)
    lb = attn.lsh_builder
    P = lb.compute_effective_p(M, lb.C, maxP)
    glob = attn.glob_builder(M, "cpu").numpy()
    with torch.no_grad():
        nb, va = attn.build_graph(q.to(DEV, dtype), k.to(DEV, dtype), N, M, B, DEV,
                                  causal and not cross, cross)
    ref = oracle.lsh_forward(q.reshape(B * H, N, d).numpy(), k.reshape(B * nkv, M, d).numpy(),
                             rp.numpy(), kv_rep=H // nkv, P=P, T=T, C=lb.C, top_k=attn.lsh_k,
                             causal=causal and not cross, glob=glob)
    win = np.zeros((N, 0), np.int64) if cross else attn.win_builder(N, M, "cpu").numpy()
    rnb, rva = oracle.merge(win, glob, ref["idx"], has_self=not cross, total_k=K)
    np.testing.assert_array_equal(nb.cpu().numpy().reshape(B * H, N, -1), rnb)
    np.testing.assert_array_equal(va.cpu().numpy().reshape(B * H, N, -1), rva)
    return ref


# (B, H, kv, N, M, d, R, maxP, T, K, w, G, causal, cross): key counts at the edges
# of a 64-key word, a 128-key block, the instances of 4, 8, 16 and 32 blocks and
# the form's limit (4,096; 4,097 takes the list form), score rows padded against
# equal L2 channels (1,024, 2,048), one list, 64 lists and 65 (list form)
SIZES = [(1, 2, 1, 63, 63, 16, 2, 3, 0, 40, 2, 1, True, False),
         (1, 2, 1, 70, 64, 32, 3, 3, 1, 40, 2, 2, False, True),
         (2, 2, 2, 65, 65, 16, 1, 2, 0, 48, 2, 2, True, False),
         (1, 2, 2, 127, 127, 64, 3, 3, 1, 60, 3, 2, False, False),
         (1, 4, 2, 129, 129, 128, 4, 3, 0, 60, 3, 2, True, False),
         (1, 2, 1, 40, 512, 64, 6, 3, 0, 64, 2, 2, False, True),
         (1, 2, 1, 33, 513, 96, 6, 3, 0, 64, 2, 2, False, True),
         (1, 1, 1, 1024, 1024, 64, 8, 3, 0, 128, 8, 2, True, False),
         (1, 1, 1, 1025, 1025, 48, 8, 3, 0, 128, 8, 2, True, False),
         (1, 1, 1, 50, 2048, 32, 8, 3, 1, 128, 2, 2, False, True),
         (1, 1, 1, 50, 2049, 256, 8, 3, 1, 128, 2, 2, False, True),
         (1, 1, 1, 4096, 4096, 16, 16, 4, 0, 128, 16, 2, True, False),
         (1, 1, 1, 30, 4097, 16, 16, 4, 0, 128, 2, 2, False, True),
         (1, 1, 1, 100, 100, 16, 64, 3, 0, 40, 2, 2, True, False),
         (1, 1, 1, 100, 100, 16, 65, 3, 0, 40, 2, 2, True, False)]


@pytest.mark.parametrize("case", SIZES, ids=lambda c: f"N{c[3]}_M{c[4]}_d{c[5]}_R{c[6]}_T{c[8]}")
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_dense_graph_sizes_match_oracle(case, dtype):
    _build(*case, dtype)


def _one_sided(q, k):
    return q, k.abs()                     # whole buckets stay empty


def _zero_rows(q, k):
    q[:, :, ::3] = 0                      # padded positions: every score ties at 0
    return q, k


def _copies(q, k):
    k[:, :, 5::2] = k[:, :, 5:6]          # hundreds of candidates with one score
    return q, k


def _outlier(q, k):
    k[:, :, 7] *= 64                      # one large key: many codes fall together
    return q, k


@pytest.mark.parametrize("edit", [_one_sided, _zero_rows, _copies, _outlier],
                         ids=lambda f: f.__name__.strip("_"))
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_dense_graph_hard_inputs_match_oracle(edit, causal, dtype):
    """Empty buckets (glob ++ 0, globals past a causal query), tied codes in
    LDS and beyond it, tied scores through the replay."""
    ref = _build(1, 2, 1, 900, 900, 16, 8, 4, 0, 100, 4, [0, 5, 450, 899], causal, False, dtype, edit)
    if edit in (_zero_rows, _copies):
        assert ref["n_ties"] > 0
