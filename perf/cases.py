"""The workloads this framework's speed is measured on.

One decode step of asynchronous speculative decoding with a diffusion draft,
taken apart into the calls a program makes: proposals drawn from the draft's
logits, the unmasking of a block, the anchors' LM head, block attention over
the paged KV cache, whole block forwards replayed from HIP graphs (as the
engine runs them), the target's acceptance of a block, and the prefill of new
prompts.  Vocabulary 151,936, 16-token blocks, 16-token pages, the
8B-shaped target and the 1.7B-shaped draft: the sizes bench.py, the tests and
``workloads`` use.  The block forwards and the prefill run a few of the
model's layers at full width, with enough weights to exceed every cache.
"""
import math
import random

import torch

VOCAB = 151936
MASK_ID = 151669
PAGE = 16
BLOCK = 16
D = 128
ROPE_THETA = 1_000_000.0
EPS = 1e-6
# hidden, query heads, KV heads, MLP width of the two models.
MODELS = {"target": (4096, 32, 8, 12288), "draft": (2048, 16, 8, 6144)}
DEV = "cuda:0"


def listed():
    return [
        # One request's sampled block checked against the target (K = 15 draft
        # tokens, fp32 logits of both models): the smallest call.
        dict(name="accept_dense_b1", kind="accept", B=1, K=15, V=VOCAB, S=0, T=1.0, dtype="float32"),
        # A serving batch's blocks against the sparse proposals the draft
        # keeps (top 64 tokens per position), bf16 logits as the model leaves them.
        dict(name="accept_sparse_b8", kind="accept", B=8, K=15, V=VOCAB, S=64, T=0.7, dtype="bfloat16"),
        # One denoise step's proposals for four blocks: the sorted top-64
        # support, the nucleus filter over it and a draw.
        dict(name="propose_top64", kind="support", N=64, V=VOCAB, top_k=64, top_p=0.95, T=0.7, dtype="bfloat16"),
        # The same step sampled from the nucleus of the whole vocabulary.
        dict(name="sample_nucleus", kind="sample", N=64, V=VOCAB, top_k=0, top_p=0.9, T=0.8, dtype="bfloat16",
             dense=False),
        # One greedy denoise step: confidences of four blocks, four tokens unmasked in each.
        dict(name="unmask_b4", kind="unmask", B=4, Q=16, V=VOCAB, k=4, T=0.0, dtype="bfloat16"),
        # The recovery's anchors: LM head and top-2 log-probabilities of four blocks.
        dict(name="lmhead_top2", kind="lmhead", N=64, H=2048, V=VOCAB, k=2),
        # Block-verify attention of a serving batch with mixed contexts.
        dict(name="verify_attn_b8", kind="attn", mode="causal", B=8, Q=16, Hq=32, Hkv=8, lo=512, hi=8192, ctx_seed=3),
        # The packed multi-branch prediction's attention: 17 branch blocks per request.
        dict(name="packed_attn_b4", kind="attn", mode="packed", B=4, Q=272, Hq=16, Hkv=8, lo=512, hi=2048,
             ctx_seed=5),
        # The target's verify forward of a single request, logits of every position.
        dict(name="target_block_b1", kind="block", model="target", layers=4, B=1, Q=16, lo=2048, hi=2048, ctx_seed=1),
        # The same for a batch of eight.
        dict(name="target_block_b8", kind="block", model="target", layers=4, B=8, Q=16, lo=512, hi=4096, ctx_seed=7),
        # The draft's packed prediction forward (hidden states and draft K/V).
        dict(name="draft_predict_b4", kind="block", model="draft", layers=4, B=4, Q=272, lo=512, hi=1024, ctx_seed=2),
        # Admission: the ragged prompts of four new requests, the last position's logits.
        dict(name="prefill_b4", kind="prefill", model="target", layers=2, B=4, lo=512, hi=4096, ctx_seed=11),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng):
    # The models' own vocabulary, or any other length (odd ones too).
    return VOCAB if rng.random() < 0.6 else _log(rng, 32000, VOCAB)


def draw(rng):
    kind = rng.choice(["accept", "accept", "support", "support", "sample", "sample", "unmask", "lmhead", "attn",
                       "attn", "block", "block", "block", "prefill"])
    dt = rng.choice(["bfloat16", "float32"])
    if kind == "accept":
        return dict(kind=kind, B=_log(rng, 1, 16), K=15, V=_vocab(rng), S=rng.choice([0, 0, _log(rng, 8, 256)]),
                    T=rng.choice([0.0, 1.0, round(rng.uniform(0.3, 1.2), 3)]), dtype=dt)
    if kind == "support":
        return dict(kind=kind, N=_log(rng, 1, 128), V=_vocab(rng), top_k=_log(rng, 4, 1024),
                    top_p=rng.choice([1.0, round(rng.uniform(0.7, 0.98), 3)]), T=round(rng.uniform(0.4, 1.2), 3),
                    dtype=dt)
    if kind == "sample":
        return dict(kind=kind, N=_log(rng, 1, 128), V=_vocab(rng), top_k=rng.choice([0, _log(rng, 16, 2000)]),
                    top_p=round(rng.uniform(0.6, 0.98), 3), T=round(rng.uniform(0.4, 1.2), 3), dtype=dt,
                    dense=rng.random() < 0.25)
    if kind == "unmask":
        return dict(kind=kind, B=_log(rng, 1, 16), Q=BLOCK, V=_vocab(rng), k=rng.randint(1, 8),
                    T=rng.choice([0.0, round(rng.uniform(0.4, 1.2), 3)]), dtype=dt)
    if kind == "lmhead":
        return dict(kind=kind, N=_log(rng, 1, 128), H=rng.choice([2048, 4096]), V=_vocab(rng), k=rng.randint(1, 8))
    if kind == "attn":
        mode = rng.choice(["causal", "full", "packed"])
        hi = _log(rng, 256, 8192 if mode != "packed" else 2048)
        return dict(kind=kind, mode=mode, B=_log(rng, 1, 16 if mode != "packed" else 4),
                    Q=rng.choice([272, 272, 752]) if mode == "packed" else rng.choice([16, 16, rng.randint(2, 31)]),
                    Hq=32 if mode == "causal" else 16, Hkv=8, lo=max(16, hi // rng.choice([1, 4, 16])), hi=hi,
                    ctx_seed=rng.randrange(1000))
    if kind == "block":
        model = rng.choice(["target", "target", "draft"])
        hi = _log(rng, 128, 4096)
        packed = model == "draft" and rng.random() < 0.3
        return dict(kind=kind, model=model, layers=rng.randint(2, 4), B=_log(rng, 1, 4 if packed else 12),
                    Q=272 if packed else BLOCK, lo=max(16, hi // rng.choice([1, 4])), hi=hi,
                    ctx_seed=rng.randrange(1000))
    hi = _log(rng, 64, 1900)
    return dict(kind="prefill", model=rng.choice(["target", "draft"]), layers=rng.randint(1, 2),
                B=_log(rng, 1, 4), lo=max(8, hi // 4), hi=hi, ctx_seed=rng.randrange(1000))


# ---------------------------------------------------------------- inputs
def _lens(c):
    r = random.Random(c["ctx_seed"])
    return [_log(r, c["lo"], c["hi"]) for _ in range(c["B"])]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _logits(g, rows, V, dtype, peak=0.0):
    """Rows of logits ~ N(0, 2^2); with ``peak`` a few tokens stand out, as a language model's do."""
    x = torch.randn(rows, V, generator=g, device=DEV) * 2.0
    if peak:
        at = torch.randint(0, V, (rows, 32), generator=g, device=DEV)
        x.scatter_add_(1, at, torch.rand(rows, 32, generator=g, device=DEV) * peak)
    return x.to(getattr(torch, dtype))


def _softmax_draw(g, logits, T):
    u = torch.rand(logits.shape, generator=g, device=DEV).clamp_(1e-20, 1 - 1e-7)
    return (logits.float() / max(T, 1e-3) - (-u.log()).log()).argmax(-1)


def _pages(g, lens, extra):
    """A shuffled pool: page tables [B, width] (0 past a request's pages) of ``lens`` + ``extra`` tokens."""
    need = [-(-(n + extra) // PAGE) for n in lens]
    pool = -(-sum(need) // 64) * 64
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(int(g.initial_seed()))).tolist()
    tables, off = [], 0
    for n in need:
        tables.append(perm[off:off + n])
        off += n
    return pool, tables


def _table_tensor(tables):
    w = max(len(t) for t in tables)
    return torch.tensor([t + [0] * (w - len(t)) for t in tables], dtype=torch.int32, device=DEV)


def _branches(Q):
    """Accepted counts of a packed block's branches: 1..15 per anchor, then all 16."""
    A = (Q // BLOCK - 2) // (BLOCK - 1)
    return [n for n in range(1, BLOCK) for _ in range(A)] + [BLOCK]


def _visibility(Q):
    rows = [(i + 1, 0, 0) for i in range(BLOCK)]
    for j, n in enumerate(_branches(Q)):
        off = BLOCK * (j + 1)
        rows += [(n, off, off + BLOCK)] * BLOCK
    return rows


def _weights(c, seed):
    """bf16 weights of ``layers`` layers and the embeddings, ~ N(0, 0.02^2); norm weights near 1."""
    H, Hq, Hkv, mlp = MODELS[c["model"]]
    g = _gen(seed)

    def w(*dims):
        return (torch.randn(*dims, generator=g, device=DEV) * 0.02).to(torch.bfloat16)

    def n(k):
        return (1.0 + 0.1 * torch.randn(k, generator=g, device=DEV)).to(torch.bfloat16)

    top = dict(embed=w(VOCAB, H), lm_head=w(VOCAB, H), norm=n(H))
    layers = [dict(qkv=w((Hq + 2 * Hkv) * D, H), o=w(H, Hq * D), gate_up=w(2 * mlp, H), down=w(H, mlp),
                   ln1=n(H), ln2=n(H), qn=n(D), kn=n(D)) for _ in range(c["layers"])]
    return top, layers


def _model(c, seed):
    from d3d_amd.model import ModelShape, Qwen3PagedModel
    H, Hq, Hkv, mlp = MODELS[c["model"]]
    shape = ModelShape(layers=c["layers"], hidden=H, heads=Hq, kv_heads=Hkv, head_dim=D, mlp=mlp, vocab=VOCAB,
                       rope_theta=ROPE_THETA, eps=EPS)
    m = Qwen3PagedModel(shape, DEV, draft=c["model"] == "draft", seed=0)
    top, layers = _weights(c, seed)
    for k, v in top.items():
        getattr(m, k).data.copy_(v)
    for mine, theirs in zip(m.layers, layers):
        for k, v in theirs.items():
            mine[k].data.copy_(v)
    return m


def _prefix_kv(g, pool, layers, Hkv):
    """K/V of the committed prefixes: K normalised per head, V of unit scale."""
    return [(torch.randn(pool, PAGE, Hkv, D, generator=g, device=DEV).to(torch.bfloat16),
             torch.randn(pool, PAGE, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)) for _ in range(layers)]


def _attn_inputs(c, seed):
    g = _gen(seed)
    lens = _lens(c)  # tokens before the block
    pool, tables = _pages(g, lens, c["Q"])
    q = torch.randn(c["B"], c["Q"], c["Hq"], D, generator=g, device=DEV).to(torch.bfloat16)
    k, v = _prefix_kv(g, pool, 1, c["Hkv"])[0]
    return q, k, v, tables, lens


def _block_inputs(c, seed):
    g = _gen(seed + 1)
    lens = _lens(c)
    pool, tables = _pages(g, lens, c["Q"])
    ids = torch.randint(0, VOCAB, (c["B"], c["Q"]), generator=g, device=DEV)
    kv = _prefix_kv(g, pool, c["layers"], MODELS[c["model"]][2])
    # Branch blocks continue the prefix at their own accepted count.
    rel = list(range(BLOCK))
    if c["Q"] > BLOCK:
        for n in _branches(c["Q"]):
            rel += [n + i for i in range(BLOCK)]
    pos = torch.tensor([[n + r for r in rel] for n in lens], device=DEV)
    slots = torch.tensor([t[p // PAGE] * PAGE + p % PAGE for t, n in zip(tables, lens)
                          for p in range(n, n + c["Q"])], device=DEV)
    return ids, pos, slots, kv, tables, lens


def _prompts(c, seed):
    r = random.Random(seed)
    return [[r.randrange(VOCAB) for _ in range(n)] for n in _lens(c)]


def prepare(case, seed):
    c, k = case, case["kind"]
    if k == "accept":
        g = _gen(seed)
        B, K, V = c["B"], c["K"], c["V"]
        target = _logits(g, B * (K + 1), V, "float32").view(B, K + 1, V)
        draft = target[:, :K] + torch.randn(B, K, V, generator=g, device=DEV) * 0.5
        s = dict(c=c, target=target.to(getattr(torch, c["dtype"])), u=torch.rand(B, K, generator=g, device=DEV),
                 ru=torch.rand(B, generator=g, device=DEV))
        if c["S"]:
            vals, ids = (draft / max(c["T"], 0.5)).topk(c["S"], dim=-1)
            s.update(ids=ids, probs=vals.softmax(-1))
            s["tok"] = ids.gather(-1, _softmax_draw(g, vals, 1.0)[..., None])[..., 0]
        else:
            s.update(draft=draft.to(s["target"].dtype))
            s["tok"] = draft.argmax(-1) if c["T"] == 0 else _softmax_draw(g, draft, c["T"])
        return s
    if k in ("support", "sample"):
        g = _gen(seed)
        return dict(c=c, logits=_logits(g, c["N"], c["V"], c["dtype"], peak=12.0),
                    u=torch.rand(c["N"], generator=g, device=DEV))
    if k == "unmask":
        g = _gen(seed)
        block = torch.randint(0, min(c["V"], 100000), (c["B"], c["Q"]), generator=g, device=DEV)
        block[:, 1:] = MASK_ID
        return dict(c=c, logits=_logits(g, c["B"] * c["Q"], c["V"], c["dtype"], peak=12.0).view(c["B"], c["Q"], -1),
                    block=block)
    if k == "lmhead":
        g = _gen(seed)
        return dict(c=c, h=torch.randn(c["N"], c["H"], generator=g, device=DEV).to(torch.bfloat16),
                    w=(torch.randn(c["V"], c["H"], generator=g, device=DEV) * 0.02).to(torch.bfloat16))
    if k == "attn":
        q, kc, vc, tables, lens = _attn_inputs(c, seed)
        s = dict(c=c, q=q, k=kc, v=vc, table=_table_tensor(tables),
                 lens=torch.tensor([n + c["Q"] for n in lens], dtype=torch.int32, device=DEV))
        if c["mode"] == "packed":
            from d3d_amd.attention import packed_visibility
            s["vis"] = packed_visibility(BLOCK, _branches(c["Q"])).to(DEV)
        return s
    if k == "block":
        from d3d_amd.attention import packed_visibility
        from d3d_amd.model import BlockStep, PagedKV
        m = _model(c, seed)
        ids, pos, slots, kv_init, tables, lens = _block_inputs(c, seed)
        kv = PagedKV(m.shape, kv_init[0][0].shape[0], PAGE, DEV)
        for i, (kc, vc) in enumerate(kv_init):
            kv.k[i].copy_(kc)
            kv.v[i].copy_(vc)
        table = _table_tensor(tables)
        packed = c["Q"] > BLOCK
        # The engine's steps: logits of a verify or recovery block, hidden
        # states of a packed prediction; one graph kept per shape.
        step = BlockStep(m, kv, c["B"], c["Q"], table.shape[1], causal=c["model"] == "target",
                         post=(lambda h, _: h) if packed else (lambda h, _: m.logits(h)),
                         q_vis=packed_visibility(BLOCK, _branches(c["Q"])) if packed else None)
        s = dict(c=c, step=step, kv=kv,
                 args=(ids, pos, table, slots, torch.tensor([n + c["Q"] for n in lens], dtype=torch.int32, device=DEV)))
        step(*s["args"])
        return s
    if k == "prefill":
        from d3d_amd.model import PagedKV, Sequence
        m = _model(c, seed)
        prompts = _prompts(c, seed)
        pages = sum(-(-len(p) // PAGE) for p in prompts) + 8
        return dict(c=c, m=m, kv=PagedKV(m.shape, pages, PAGE, DEV),
                    seqs=[Sequence(i, p) for i, p in enumerate(prompts)])
    raise ValueError(k)


# ---------------------------------------------------------------- one pass
def run(state):
    s, c = state, state["c"]
    k = c["kind"]
    if k == "accept":
        from d3d_amd import speculative_sampling as ss
        if c["T"] == 0.0 and not c["S"]:
            out = ss.accept_fused(s["target"], None, s["tok"], temperature=0.0)
        elif c["S"]:
            out = ss.accept_fused_sparse(s["target"], s["tok"], s["ids"], s["probs"], temperature=max(c["T"], 0.5),
                                         uniforms=s["u"], resample_uniform=s["ru"], input_kind="logits")
        else:
            out = ss.accept_fused(s["target"], s["draft"], s["tok"], temperature=c["T"], uniforms=s["u"],
                                  resample_uniform=s["ru"])
        return dict(accepted=out.accepted, mask=out.accept_mask, token=out.out_token, all=out.all_accepted,
                    posterior=out.posterior)
    if k == "support":
        from d3d_amd import draft
        tok, ids, probs = draft.sample_with_sparse_probs(s["logits"], c["T"], c["top_k"], c["top_p"], uniforms=s["u"])
        return dict(tokens=tok, ids=ids, probs=probs)
    if k == "sample":
        from d3d_amd import draft
        if c["dense"]:
            return dict(probs=draft.sampling_probs(s["logits"], c["T"], c["top_k"], c["top_p"]))
        tok, p = draft.sample_with_prob(s["logits"], c["T"], c["top_k"], c["top_p"], uniforms=s["u"])
        return dict(tokens=tok, probs=p)
    if k == "unmask":
        from d3d_amd import draft
        block = s["block"].clone()  # updated in place
        x0, conf = draft.confidence_topk_unmask(s["logits"], block, MASK_ID, c["k"], c["T"])
        return dict(block=block, x0=x0, conf=conf)
    if k == "lmhead":
        from d3d_amd.lmhead import lmhead_topk
        ids, vals = lmhead_topk(s["h"], s["w"], c["k"], with_values=True, log_softmax=True)
        return dict(ids=ids, vals=vals)
    if k == "attn":
        from d3d_amd import attention as att
        if c["mode"] == "packed":
            return att.packed_block_attn(s["q"], s["k"], s["v"], s["lens"], s["table"], s["vis"])
        return att.flash_attn_with_kvcache(s["q"], s["k"], s["v"], s["lens"], s["table"], causal=c["mode"] == "causal")
    if k == "block":
        out = s["step"](*s["args"])
        return dict(out=out, k=s["kv"].k[-1], v=s["kv"].v[-1])
    if k == "prefill":
        from d3d_amd.model import prefill
        with torch.inference_mode():
            h = prefill(s["m"], s["kv"], s["seqs"], "target")
            return dict(logits=s["m"].logits(h), k=s["kv"].k[-1], v=s["kv"].v[-1])
    raise ValueError(k)


# ---------------------------------------------------------------- what a pass cannot do without
def _row_bytes(c, rows):
    return rows * c["V"] * (4 if c["dtype"] == "float32" else 2)


def _attn_flops(Q, Hq, lens, mode):
    """4 D per visible (query, key) pair and head."""
    pairs = 0
    for n in lens:
        if mode == "causal":
            pairs += Q * n + Q * (Q + 1) // 2
        elif mode == "full":
            pairs += Q * (n + Q)
        else:
            pairs += sum(n + a + (hi - lo) for a, lo, hi in _visibility(Q))
    return 4 * D * Hq * pairs


def _model_work(c, rows, attn_pairs_flops, kv_tokens, out_rows):
    H, Hq, Hkv, mlp = MODELS[c["model"]]
    per = (Hq + 2 * Hkv) * D * H + H * Hq * D + 3 * mlp * H
    by = c["layers"] * (2 * per + kv_tokens * Hkv * D * 4) + 2 * rows * H
    fl = c["layers"] * (2 * rows * per + attn_pairs_flops)
    if out_rows:
        by += 2 * VOCAB * H + 2 * out_rows * VOCAB
        fl += 2 * out_rows * VOCAB * H
    return {"bytes": by, "flops": fl}


def work(case):
    c, k = case, case["kind"]
    if k == "accept":
        B, K = c["B"], c["K"]
        rows = B * (K + 1) + (B * K if c["T"] > 0 and not c["S"] else 0)
        return {"bytes": _row_bytes(c, rows) + B * K * c["S"] * 12, "flops": 4 * rows * c["V"]}
    if k == "support":
        return {"bytes": _row_bytes(c, c["N"]) + c["N"] * c["top_k"] * 12, "flops": 4 * c["N"] * c["V"]}
    if k == "sample":
        return {"bytes": _row_bytes(c, c["N"]) + (c["N"] * c["V"] * 4 if c["dense"] else 0),
                "flops": 4 * c["N"] * c["V"]}
    if k == "unmask":
        return {"bytes": _row_bytes(c, c["B"] * c["Q"]), "flops": 4 * c["B"] * c["Q"] * c["V"]}
    if k == "lmhead":
        return {"bytes": 2 * (c["V"] + c["N"]) * c["H"], "flops": 2 * c["N"] * c["V"] * c["H"]}
    if k == "attn":
        lens = _lens(c)
        return {"bytes": sum((n + c["Q"]) * c["Hkv"] * D * 4 + 2 * c["Q"] * c["Hq"] * D * 2 for n in lens),
                "flops": _attn_flops(c["Q"], c["Hq"], lens, c["mode"])}
    lens = _lens(c)
    Hq = MODELS[c["model"]][1]
    if k == "block":
        mode = "packed" if c["Q"] > BLOCK else "causal" if c["model"] == "target" else "full"
        rows = c["B"] * c["Q"]
        return _model_work(c, rows, _attn_flops(c["Q"], Hq, lens, mode), sum(lens) + rows,
                           0 if c["Q"] > BLOCK else rows)
    pairs = sum(n * (n + 1) // 2 for n in lens)
    return _model_work(c, sum(lens), 4 * D * Hq * pairs, sum(lens), len(lens))


def tolerance(case):
    k = case["kind"]
    if k == "accept":
        return "exact"  # decisions and tokens
    if k in ("support", "sample"):
        # Probabilities from fp32 sums; a draw may fall on a rounding of its cumulative sum.
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.005}
    if k == "unmask":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if k == "lmhead":
        # Logits are bf16 before they are compared: a tie at a rounding may swap two ids.
        return {"rel": 3e-3, "max": 2e-2, "differ": 0.01}
    if k == "attn":
        return {"rel": 1e-2, "max": 0.1}
    # Whole forwards: bf16 rounding of every layer's outputs.
    return {"rel": 0.03, "max": 0.5}


# ---------------------------------------------------------------- 64-bit results
def _kept(z, top_k, top_p):
    """Mask of the entries of z [N, V] the top-k (ties kept) and top-p filters keep."""
    N, V = z.shape
    keep = torch.ones_like(z, dtype=torch.bool)
    if 0 < top_k < V:
        keep &= z >= z.topk(top_k, dim=-1).values[:, -1:]
    if top_p < 1.0:
        zz = z.masked_fill(~keep, -math.inf)
        vals, order = zz.sort(dim=-1, descending=True, stable=True)
        before = vals.softmax(-1).cumsum(-1)
        drop = torch.zeros_like(keep)
        drop[:, 1:] = before[:, :-1] > top_p
        keep &= ~torch.zeros_like(keep).scatter(1, order, drop)
    return keep


def _attend(q, k, v, vis):
    """q [Q, Hq, D], k/v [S, Hkv, D] in fp64, vis [Q, S]: one KV head at a time."""
    G = q.shape[1] // k.shape[1]
    out = torch.empty_like(q)
    for h in range(k.shape[1]):
        s = torch.matmul(q[:, h * G:(h + 1) * G].transpose(0, 1), k[:, h].transpose(0, 1)) / math.sqrt(D)
        p = s.masked_fill(~vis, -math.inf).softmax(-1)
        out[:, h * G:(h + 1) * G] = torch.matmul(p, v[:, h]).transpose(0, 1)
    return out


def _vis_mask(mode, n, Q):
    """[Q, n + Q] visibility of a block of Q after n tokens."""
    t = torch.arange(n + Q, device=DEV)
    if mode == "full":
        return torch.ones(Q, n + Q, dtype=torch.bool, device=DEV)
    if mode == "causal":
        return t[None] <= n + torch.arange(Q, device=DEV)[:, None]
    a, lo, hi = torch.tensor(_visibility(Q), device=DEV).T[..., None]
    return (t < n + a) | ((t >= n + lo) & (t < n + hi))


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    inv = 1.0 / ROPE_THETA ** (torch.arange(0, D // 2, device=DEV, dtype=torch.float64) * 2 / D)
    f = pos.double()[:, None, None] * inv
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * f.cos() - b * f.sin(), b * f.cos() + a * f.sin()], -1)


def _forward64(c, weights, ids, pos, prefix, mode):
    """Hidden states [T, H] of each request: ids / pos lists of [Q], prefix[b][layer] = (k, v) [n, Hkv, D]."""
    top, layers = weights
    H, Hq, Hkv, mlp = MODELS[c["model"]]
    xs = [top["embed"][i].double() for i in ids]
    for li, L in enumerate(layers):
        w = {k: v.double() for k, v in L.items()}
        for b, x in enumerate(xs):
            Q = x.shape[0]
            qkv = (_norm(x, w["ln1"]) @ w["qkv"].T).view(Q, Hq + 2 * Hkv, D)
            q = _rope(_norm(qkv[:, :Hq], w["qn"]), pos[b])
            k = _rope(_norm(qkv[:, Hq:Hq + Hkv], w["kn"]), pos[b])
            pk, pv = prefix[b][li]
            n = pk.shape[0]
            a = _attend(q, torch.cat([pk.double(), k]), torch.cat([pv.double(), qkv[:, Hq + Hkv:]]),
                        _vis_mask(mode, n, Q))
            x = x + a.reshape(Q, Hq * D) @ w["o"].T
            gu = _norm(x, w["ln2"]) @ w["gate_up"].T
            xs[b] = x + (torch.nn.functional.silu(gu[:, :mlp]) * gu[:, mlp:]) @ w["down"].T
    return [_norm(x, top["norm"]) for x in xs]


def _logits64(h, w):
    # The largest matrix a step at a time: its 64-bit copy is not needed whole.
    return torch.cat([h @ p.double().T for p in w.split(16384)], -1)


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "accept":
        return None  # whole numbers
    if k in ("support", "sample"):
        s = prepare(c, seed)
        z = s["logits"].double() / c["T"]
        if k == "support":
            S = min(c["top_k"], c["V"])
            vals = z.sort(dim=-1, descending=True, stable=True).values[:, :S]
            p = vals.softmax(-1)
            if c["top_p"] < 1.0:
                drop = torch.zeros_like(p, dtype=torch.bool)
                drop[:, 1:] = p.cumsum(-1)[:, :-1] > c["top_p"]
                p = vals.masked_fill(drop, -math.inf).softmax(-1)
            return dict(tokens=None, ids=None, probs=p)
        p = z.masked_fill(~_kept(z, c["top_k"], c["top_p"]), -math.inf).softmax(-1)
        if c["dense"]:
            return dict(probs=p)
        cdf = p.cumsum(-1)
        t = torch.searchsorted(cdf, s["u"].double()[:, None] * cdf[:, -1:], right=True).clamp_(max=c["V"] - 1)
        return dict(tokens=None, probs=p.gather(1, t)[:, 0])
    if k == "unmask":
        z = prepare(c, seed)["logits"].double() / (c["T"] if c["T"] > 1e-5 else 1.0)
        return dict(block=None, x0=None, conf=z.softmax(-1).amax(-1))
    if k == "lmhead":
        s = prepare(c, seed)
        x = _logits64(s["h"].double(), s["w"])
        return dict(ids=None, vals=x.log_softmax(-1).topk(c["k"], dim=-1).values)
    if k == "attn":
        q, kc, vc, tables, lens = _attn_inputs(c, seed)
        out = []
        for b, n in enumerate(lens):
            t = torch.tensor(tables[b], device=DEV)
            ks, vs = (x[t].reshape(-1, c["Hkv"], D)[:n + c["Q"]].double() for x in (kc, vc))
            out.append(_attend(q[b].double(), ks, vs, _vis_mask(c["mode"], n, c["Q"])))
        return torch.stack(out)
    if k == "block":
        weights = _weights(c, seed)
        ids, pos, _, kv, tables, lens = _block_inputs(c, seed)
        prefix = []
        for t, n in zip(tables, lens):
            at = torch.tensor(t, device=DEV)
            prefix.append([tuple(x[at].reshape(-1, x.shape[2], D)[:n] for x in layer) for layer in kv])
        packed = c["Q"] > BLOCK
        mode = "packed" if packed else "causal" if c["model"] == "target" else "full"
        h = torch.stack(_forward64(c, weights, ids, pos, prefix, mode))
        return dict(out=h if packed else _logits64(h, weights[0]["lm_head"]), k=None, v=None)
    if k == "prefill":
        weights = _weights(c, seed)
        H, Hq, Hkv, mlp = MODELS[c["model"]]
        ids = [torch.tensor(p, device=DEV) for p in _prompts(c, seed)]
        none = torch.empty(0, Hkv, D, device=DEV)
        h = _forward64(c, weights, ids, [torch.arange(len(i), device=DEV) for i in ids],
                       [[(none, none)] * c["layers"]] * len(ids), "causal")
        return dict(logits=_logits64(torch.stack([x[-1] for x in h]), weights[0]["lm_head"]), k=None, v=None)
    raise ValueError(k)
