"""The calls this package's speed is measured on.

Each case is one pass through a public entry point, as a user's program calls
it: inference through ``SparseAttention`` (self- and cross-attention, MHA, GQA
and MQA) and ``SparseTransformer``, a training step through
``SparseAttention``, ``build_graph`` alone, and ``sparse_gather_attention``
over a graph the program already holds (forward, and forward + backward).
``listed()`` names them, ``draw(rng)`` gives others of the same ranges.
"""
import math
import warnings

import torch

from ssa_amd import SSAConfig, SparseAttention, SparseTransformer, sparse_gather_attention

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


# ---------------------------------------------------------------------------- cases
def _attn(kind, dtype, B, N, H, kv, d, K, w, R, *, M=0, T=0, G=2, causal=False, xscale=1.0,
          dropout=0.0, fp32w=False):
    """A case that goes through the module; M: key length of cross-attention (0: self)."""
    return dict(kind=kind, dtype=dtype, B=B, N=N, M=M, H=H, kv=kv, d=d, K=K, w=w, R=R, T=T, G=G,
                causal=causal, xscale=xscale, dropout=dropout, fp32w=fp32w)


def _gather(kind, dtype, B, N, M, H, kv, d, K, w, *, causal=True, fp32w=False,
            deterministic=False):
    """A case over a graph that is there already (one build, many applies)."""
    return dict(kind=kind, dtype=dtype, B=B, N=N, M=M, H=H, kv=kv, d=d, K=K, w=w, causal=causal,
                fp32w=fp32w, deterministic=deterministic)


def listed():
    return [
        # the smallest call: a short prompt through a small fp32 layer, where
        # launches and host work count
        dict(_attn("forward", "f32", 2, 96, 4, 2, 16, 32, 4, 4, causal=True), name="fwd_tiny_f32"),
        # fp32 causal self-attention, 8 heads, two sequences of 1,024
        dict(_attn("forward", "f32", 2, 1024, 8, 8, 64, 128, 8, 8, causal=True),
             name="fwd_f32_n1024"),
        # the benchmark's layer: bf16 GQA prefill of 4,096 tokens, d_model 4096
        dict(_attn("forward", "bf16", 1, 4096, 32, 8, 128, 128, 16, 8, causal=True, xscale=0.02),
             name="fwd_gqa_bf16_n4096"),
        # long-context prefill: bf16 MQA over 32,768 tokens with two probes
        dict(_attn("forward", "bf16", 1, 32768, 32, 1, 128, 256, 32, 8, T=2, G=3, causal=True),
             name="fwd_mqa_bf16_n32768"),
        # decoder queries over encoder states, bf16
        dict(_attn("forward", "bf16", 4, 2048, 16, 16, 64, 64, 4, 6, M=512),
             name="fwd_cross_bf16"),
        # the same in fp32 at lengths that divide by nothing
        dict(_attn("forward", "f32", 3, 1531, 16, 16, 64, 64, 4, 6, M=389, T=1),
             name="fwd_cross_f32_ragged"),
        # a whole model call: six layers over token ids, with the statistics
        dict(kind="model", dtype="bf16", B=2, N=8192, H=16, kv=4, d=64, K=128, w=16, R=8, T=1,
             G=2, layers=6, vocab=32000, causal=True, name="model_bf16_n8192"),
        # the graph alone, for a program that keeps it over layers: fp16, head
        # dim 96, ragged length
        dict(_attn("graph", "f16", 1, 2999, 16, 4, 96, 96, 8, 8, T=1, causal=True),
             name="graph_f16_ragged"),
        # a kept graph applied to a layer's q, k, v at the benchmark's sizes
        dict(_gather("apply", "bf16", 1, 4096, 4096, 32, 8, 128, 128, 16), name="apply_gqa_bf16"),
        # a training step of the fp32 layer: loss gradient in, every gradient out
        dict(_attn("train", "f32", 2, 1024, 8, 8, 64, 128, 8, 8, causal=True),
             name="train_f32_n1024"),
        # a training step of the benchmark's layer
        dict(_attn("train", "bf16", 1, 4096, 32, 8, 128, 128, 16, 8, causal=True, xscale=0.02),
             name="train_gqa_bf16_n4096"),
        # reproducible training over a kept graph (torch's deterministic
        # switch on), fp32 weights, ragged
        dict(_gather("apply_train", "bf16", 2, 1237, 1237, 8, 4, 80, 64, 8, fp32w=True,
                     deterministic=True), name="apply_train_det_ragged"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "cross", "graph", "apply", "train",
                       "train", "apply_train", "model"])
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    d = rng.choice([32, 48, 64, 64, 80, 96, 128, 128])
    kv = rng.choice([1, 2, 4, 8])
    H = kv * rng.choice([1, 2, 4, 8])
    B = rng.choice([1, 1, 2, 3, 4])
    w = rng.randint(2, 32)
    T = rng.choice([0, 0, 1, 2])
    R = rng.randint(4, 8)
    K = min(256, 2 * w + 4 + _log(rng, 16, 192))
    if kind == "model":
        H, kv, d = 8, rng.choice([2, 4, 8]), 64
        return dict(kind="model", dtype=rng.choice(["bf16", "f16"]), B=rng.choice([1, 2]),
                    N=_log(rng, 128, 4096), H=H, kv=kv, d=d, K=K, w=w, R=R, T=T, G=2,
                    layers=rng.randint(2, 4), vocab=rng.choice([1000, 8000, 32000]), causal=True)
    N = _log(rng, 64, 8192)
    while B * H * N > 131072 and N > 64:        # no dearer than the largest listed case
        N = max(64, N // 2)
    N = max(48, N - rng.randint(0, 16))
    if kind in ("apply", "apply_train"):
        return _gather(kind, dtype, B, N, N if rng.random() < 0.6 else _log(rng, 300, 4096), H,
                       kv, d, K, w, causal=False if rng.random() < 0.3 else True,
                       fp32w=rng.random() < 0.3, deterministic=rng.random() < 0.3)
    M = 0
    if kind == "cross":
        kind, M = rng.choice(["forward", "forward", "train"]), _log(rng, 64, 4096)
    return _attn(kind, dtype, B, N, H, kv, d, K, w, R, M=M, T=T,
                 causal=(M == 0 and rng.random() < 0.8), xscale=rng.choice([1.0, 0.02]),
                 dropout=rng.choice([0.0, 0.0, 0.1]) if kind == "train" else 0.0,
                 fp32w=rng.random() < 0.2)


# ---------------------------------------------------------------------------- inputs
def _config(c):
    kw = {}
    if c["G"] == 3:                   # explicit globals: two sinks and a middle token
        kw = dict(global_token_indices=[0, 1, 16384])
    return SSAConfig(d_model=c["H"] * c["d"], num_heads=c["H"], num_kv_heads=c["kv"],
                     num_neighbors=c["K"], window_size=c["w"], num_global_tokens=2,
                     num_hash_rounds=c["R"], max_num_hashes=12, lsh_num_probes=c["T"],
                     causal=c["causal"], dropout=c.get("dropout", 0.0),
                     fp32_attn_weights=c.get("fp32w", False), **kw)


def _module(c, seed):
    """The layer (Xavier projections, as the benchmark draws them) in the
    case's type; the hyperplanes stay fp32."""
    torch.manual_seed(seed)
    with warnings.catch_warnings(), torch.device(DEV):
        warnings.simplefilter("ignore")
        attn = SparseAttention(_config(c))
        for lin in (attn.Wq, attn.Wk, attn.Wv, attn.Wo):
            torch.nn.init.xavier_uniform_(lin.weight)
    for p in attn.parameters():
        p.data = p.data.to(DTYPES[c["dtype"]])
    return attn


def _stream(c, L, g):
    """(B, L, d_model) activations: N(0, 1) or the benchmark's 0.02 N(0, 1)."""
    x = torch.randn(c["B"], L, c["H"] * c["d"], generator=g, device=DEV) * c["xscale"]
    return x.to(DTYPES[c["dtype"]])


def _dense_graph(q, k, c):
    """A graph a program might keep: per query the window, two globals and the
    best-scoring keys, ids ascending, unused slots 0 and marked invalid."""
    B, N, M, H, K, w = c["B"], c["N"], c["M"], c["H"], c["K"], c["w"]
    rep = H // c["kv"]
    kk = min(K, M)
    pos, key = torch.arange(N, device=DEV)[:, None], torch.arange(M, device=DEV)[None]
    future = (key > pos) if c["causal"] else torch.zeros(N, M, dtype=torch.bool, device=DEV)
    always = ((key - pos).abs() <= w) | (key < 2)
    nb = torch.zeros(B, H, N, K, dtype=torch.int64, device=DEV)
    va = torch.zeros(B, H, N, K, dtype=torch.bool, device=DEV)
    for b in range(B):
        for h in range(H):
            s = q[b, h].float() @ k[b, h // rep].float().t()
            s.masked_fill_(always, math.inf).masked_fill_(future, -math.inf)
            top, ids = s.topk(kk, dim=-1)
            ids = torch.where(top > -math.inf, ids, M).sort(-1).values
            ok = ids < M
            nb[b, h, :, :kk] = torch.where(ok, ids, 0)
            va[b, h, :, :kk] = ok
    va[..., 0] = True                 # a query always sees some key
    return nb, va


def _gather_inputs(c, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    dt = DTYPES[c["dtype"]]

    def heads(h, L):
        # as the projections leave them: (B, L, h, d) seen as (B, h, L, d)
        t = torch.randn(c["B"], L, h, c["d"], generator=g, device=DEV).to(dt)
        return t.transpose(1, 2)
    q, k, v = heads(c["H"], c["N"]), heads(c["kv"], c["M"]), heads(c["kv"], c["M"])
    nb, va = _dense_graph(q, k, c)
    dout = torch.randn(c["B"], c["N"], c["H"], c["d"], generator=g, device=DEV).to(dt)
    return q, k, v, nb, va, dout.transpose(1, 2)


def prepare(case, seed):
    c = case
    if c["kind"] in ("apply", "apply_train"):
        q, k, v, nb, va, dout = _gather_inputs(c, seed)
        if c["kind"] == "apply_train":
            q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
        return dict(case=c, q=q, k=k, v=v, nb=nb, va=va, dout=dout)
    if c["kind"] == "model":
        torch.manual_seed(seed)
        with warnings.catch_warnings(), torch.device(DEV):
            warnings.simplefilter("ignore")
            model = SparseTransformer(_config(c), num_layers=c["layers"], vocab_size=c["vocab"])
        for p in model.parameters():
            p.data = p.data.to(DTYPES[c["dtype"]])
        g = torch.Generator(DEV).manual_seed(seed + 1)
        ids = torch.randint(0, c["vocab"], (c["B"], c["N"]), generator=g, device=DEV)
        return dict(case=c, model=model.eval(), ids=ids)
    attn = _module(c, seed)
    g = torch.Generator(DEV).manual_seed(seed + 1)
    x = _stream(c, c["N"], g)
    src = _stream(c, c["M"], g) if c["M"] else None
    s = dict(case=c, attn=attn, x=x, src=src, seed=seed)
    if c["kind"] == "train":
        attn.train()
        s["leaves"] = [x.requires_grad_()] + ([src.requires_grad_()] if src is not None else []) \
            + [m.weight for m in (attn.Wq, attn.Wk, attn.Wv, attn.Wo)]
        s["dout"] = torch.randn(x.shape, generator=g, device=DEV).to(x.dtype)
        return s
    attn.eval()
    if c["kind"] == "graph":
        with torch.no_grad():
            s["q"], s["k"] = attn._split_q(attn.Wq(x)), attn._split_kv_compact(
                attn.Wk(x if src is None else src))
    return s


# ---------------------------------------------------------------------------- the pass
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "forward":
        with torch.no_grad():
            return state["attn"](state["x"], state["src"])[0]
    if kind == "model":
        with torch.no_grad():
            out, stats = state["model"](state["ids"], return_stats=True)
        return [out] + [s["padding_fraction"] for s in stats]
    if kind == "graph":
        M = c["M"] or c["N"]
        with torch.no_grad():
            return state["attn"].build_graph(state["q"], state["k"], c["N"], M, c["B"], DEV,
                                             c["causal"], bool(c["M"]))
    if kind == "train":
        if c["dropout"]:
            torch.manual_seed(state["seed"])
        for t in state["leaves"]:
            t.grad = None
        out, _ = state["attn"](state["x"], state["src"])
        out.backward(state["dout"])
        return [out.detach()] + [t.grad for t in state["leaves"]]
    q, k, v = state["q"], state["k"], state["v"]
    scale = c["d"] ** -0.5
    if kind == "apply":
        with torch.no_grad():
            return sparse_gather_attention(q, k, v, state["nb"], scale, state["va"],
                                           fp32_attn_weights=c["fp32w"])
    q.grad = k.grad = v.grad = None
    torch.use_deterministic_algorithms(c["deterministic"])
    try:
        out = sparse_gather_attention(q, k, v, state["nb"], scale, state["va"], training=True,
                                      fp32_attn_weights=c["fp32w"])
        out.backward(state["dout"])
    finally:
        torch.use_deterministic_algorithms(False)
    return [out.detach(), q.grad, k.grad, v.grad]


# ---------------------------------------------------------------------------- what it takes
def work(case):
    """Inputs and weights read once, outputs written once; the products of the
    projections, the hash, one score per candidate the lists can hold (half
    of them in a causal row on average) and the K weighted rows."""
    c = case
    e = 4 if c["dtype"] == "f32" else 2
    B, N, H, kv, d, K = c["B"], c["N"], c["H"], c["kv"], c["d"], c["K"]
    M = c.get("M") or N
    dm = H * d
    rows = B * H * N
    qkv = (B * N * dm + 2 * B * M * kv * d) * e
    attend = 4 * rows * K * d
    if c["kind"] in ("apply", "apply_train"):
        graph = rows * K * 9
        if c["kind"] == "apply":
            return dict(bytes=qkv + graph + B * N * dm * e, flops=attend)
        return dict(bytes=2 * qkv + graph + 2 * B * N * dm * e, flops=attend * 7 // 2)
    lsh_k = max(K - (2 * c["w"] + 2 + c["G"]), 8)
    C = 4 * lsh_k
    P = max(1, min(12, round(math.log2(max(M, 1) / C))))
    cand = min(C * c["R"] * (1 + min(c["T"], P)), M) * (0.5 if c["causal"] else 1.0)
    graph = 2 * c["R"] * P * d * (rows + B * kv * M) + 2 * rows * cand * d
    if c["kind"] == "graph":
        return dict(bytes=(B * N * dm + B * M * kv * d) * e + rows * K * 9, flops=graph)
    weights = (2 * dm * dm + 2 * kv * d * dm) * e
    proj = 4 * B * N * dm * dm + 4 * B * M * kv * d * dm
    x = (B * N * dm + (B * M * dm if c.get("M") else 0)) * e
    if c["kind"] == "model":
        L = c["layers"]
        return dict(bytes=L * (weights + 8 * dm * dm * e) + B * N * (8 + 2 * dm * e),
                    flops=L * (proj + graph + attend + 16 * B * N * dm * dm))
    if c["kind"] == "train":
        return dict(bytes=2 * (weights + x) + 2 * B * N * dm * e,
                    flops=3 * proj + graph + attend * 7 // 2)
    return dict(bytes=weights + x + B * N * dm * e, flops=proj + graph + attend)


def tolerance(case):
    """Measured on an MI355X, stated at about four times what was seen there.

    Over a kept graph only the sums' order and the outputs' rounding differ:
    against 64 bits 1.6e-3..2.3e-3 in bf16, about an eighth of that in fp16,
    below 2e-6 in fp32.  Through the whole layer a near tie at the last place
    (or a projection within rounding of zero) may pick another neighbour in a
    row: fp32 against 64 bits 2.9e-4, the bf16 layers 9e-3 against 64 bits and
    2e-4 (0.1 at one value) between two orders of the projections' sums.  In
    the whole model such a row travels: 2e-2 (0.17 at one value) between the
    same two orders.  The graph alone came out the same in two orders; against
    a scalar restatement 36 of 1,048,576 rows of the longest one differ."""
    c = case
    if c["kind"] == "graph":
        return dict(differ=max(2e-4, min(1e-2, 2 / (c["B"] * c["H"] * c["N"]))))
    if c["kind"] == "model":
        return dict(rel=3e-2, max=0.7)
    if c["kind"] in ("apply", "apply_train"):
        return dict(rel={"f32": 1e-5, "f16": 1.5e-3, "bf16": 1e-2}[c["dtype"]])
    return dict(rel={"f32": 1.2e-3, "f16": 3e-3, "bf16": 1e-2}[c["dtype"]], max=0.5)


# ---------------------------------------------------------------------------- 64 bits
def _graph64(attn, c, q, k, b, h):
    """The graph of one head as an (N, M) mask: the layer's definition (hash
    signs, bucket lists of C members in the order torch.sort gives on the CPU,
    first occurrences, the best lsh_k by score, window, globals, self) with
    every product in 64 bits."""
    N, M, C, causal = q.shape[0], k.shape[0], attn.lsh_builder.C, c["causal"]
    P = attn.lsh_builder.compute_effective_p(M, C, attn.lsh_builder.max_P)
    planes = attn.lsh_builder.rand_proj[:, :P].double()
    glob = attn.glob_builder(M, DEV)
    pos = torch.arange(N, device=DEV)[:, None]
    pw = 2 ** torch.arange(P, device=DEV)
    filler = torch.cat([glob, torch.zeros(max(0, C - len(glob)), dtype=torch.long,
                                          device=DEV)])[:C]
    cands, oks = [], []
    for r in range(c["R"]):
        qp = q @ planes[r].t()
        kid = ((k @ planes[r].t() > 0).long() * pw).sum(-1)
        qid = ((qp > 0).long() * pw).sum(-1)
        perm = torch.sort(kid.cpu()[None], dim=-1)[1][0].to(DEV)
        size = torch.bincount(kid, minlength=2 ** P)
        start = size.cumsum(0) - size
        flips = qp.abs().argsort(-1)[:, :min(c["T"], P)]
        for ids in [qid] + [qid ^ pw[flips[:, t]] for t in range(flips.shape[1])]:
            at = start[ids][:, None] + torch.arange(C, device=DEV)
            ok = at < (start + size)[ids][:, None]
            cand = perm[torch.where(ok, at, M - 1)]
            if causal:
                cand = torch.where(cand > pos, pos, cand)
            empty = (size[ids] == 0)[:, None]
            cands.append(torch.where(empty, filler, cand))
            oks.append(ok | empty)
    cand, ok = torch.cat(cands, -1), torch.cat(oks, -1)
    slot = torch.arange(cand.shape[1], device=DEV).expand_as(cand)
    first = torch.full((N, M), cand.shape[1], device=DEV).scatter_reduce_(1, cand, slot, "amin")
    ok &= first.gather(1, cand) == slot
    kept = torch.zeros(N, M, dtype=torch.uint8, device=DEV).scatter_reduce_(
        1, cand, ok.to(torch.uint8), "amax").bool()
    s = (q @ k.t()).masked_fill_(~kept, -math.inf)
    kk = min(attn.lsh_k, cand.shape[1])
    top, ids = s.topk(min(kk, M), dim=-1)
    short = top == -math.inf
    pool = torch.zeros(N, M, dtype=torch.bool, device=DEV)
    pool.scatter_(1, torch.where(short, glob[0] if len(glob) else 0, ids), True)
    pool[:, 0] |= (short.any(-1) | (kk > M)) & (kk > len(glob))
    pool[:, glob] = True
    if not c["M"]:
        off = torch.arange(-c["w"], c["w"] + 1, device=DEV)[None]
        win = pos + (off.clamp(max=0) if causal else off)
        pool.scatter_(1, win.clamp(0, M - 1), True)
        pool.scatter_(1, pos, True)
    return pool


class _Attend64(torch.autograd.Function):
    """softmax(q k^T scale over the mask) v and its gradients, head by head,
    keeping nothing but the operands."""

    @staticmethod
    def forward(ctx, q, k, v, scale, mask_of):
        ctx.args = scale, mask_of
        ctx.save_for_backward(q, k, v)
        out = torch.empty_like(q)
        rep = q.shape[1] // k.shape[1]
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                s = (q[b, h] @ k[b, h // rep].t() * scale).masked_fill_(~mask_of(b, h), -math.inf)
                out[b, h] = s.softmax(-1) @ v[b, h // rep]
        return out

    @staticmethod
    def backward(ctx, g):
        q, k, v = ctx.saved_tensors
        scale, mask_of = ctx.args
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
        rep = q.shape[1] // k.shape[1]
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                kh, vh = k[b, h // rep], v[b, h // rep]
                p = (q[b, h] @ kh.t() * scale).masked_fill_(~mask_of(b, h), -math.inf).softmax(-1)
                dp = g[b, h] @ vh.t()
                ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
                dq[b, h] = ds @ kh
                dk[b, h // rep] += ds.t() @ q[b, h]
                dv[b, h // rep] += p.t() @ g[b, h]
        return dq, dk, dv, None, None


def exact(case, seed):
    """The outputs with every product and sum in 64 bits.  The layer's q, k
    and v are rounded to the model's type first, as the layer stores them:
    the hash signs and the ranking are taken from the stored rows, and a graph
    of unrounded rows would be another graph.  None for whole models (a
    layer's rounding moves the next layers' graphs), graphs (whole numbers),
    dropout (its noise is the package's own) and lengths whose dense scores
    take too long."""
    c = case
    if c["kind"] in ("model", "graph") or c.get("dropout") or c["N"] > 8192:
        return None
    if c["kind"] in ("apply", "apply_train"):
        q, k, v, nb, va, dout = _gather_inputs(c, seed)

        def mask_of(b, h):
            m = torch.zeros(c["N"], c["M"], dtype=torch.uint8, device=DEV)
            return m.scatter_reduce_(1, nb[b, h], va[b, h].to(torch.uint8), "amax").bool()
        grad = c["kind"] == "apply_train"
        q, k, v = (t.double().requires_grad_(grad) for t in (q, k, v))
        out = _Attend64.apply(q, k, v, c["d"] ** -0.5, mask_of)
        if not grad:
            return out
        return [out.detach()] + list(torch.autograd.grad(out, (q, k, v), dout.double()))
    if 2 * c["w"] + 2 + c["G"] > c["K"]:
        return None                   # more guaranteed keys than slots: the cut is by id
    s = prepare(c, seed)
    attn, x, src = s["attn"], s["x"], s["src"]
    grad = c["kind"] == "train"
    x = x.detach().double().requires_grad_(grad)
    src = src.detach().double().requires_grad_(grad) if src is not None else None
    ws = [m.weight.detach().double().requires_grad_(grad)
          for m in (attn.Wq, attn.Wk, attn.Wv, attn.Wo)]
    dt = DTYPES[c["dtype"]]

    def heads(t, w):
        y = t @ w.t()
        y = y + (y.to(dt).double() - y).detach()
        return y.view(*y.shape[:2], -1, c["d"]).transpose(1, 2)
    y = x if src is None else src
    q, k, v = heads(x, ws[0]), heads(y, ws[1]), heads(y, ws[2])
    rep = attn.kv_rep
    masks = {}

    def mask_of(b, h):
        if (b, h) not in masks:
            masks[b, h] = _graph64(attn, c, q.detach()[b, h], k.detach()[b, h // rep], b, h)
        return masks[b, h]
    out = _Attend64.apply(q, k, v, attn.scale, mask_of)
    out = out.transpose(1, 2).reshape(*x.shape) @ ws[3].t()
    if not grad:
        return out
    leaves = [x] + ([src] if src is not None else []) + ws
    return [out.detach()] + list(torch.autograd.grad(out, leaves, s["dout"].double()))
