"""Performance cases of the multi-future drafting hot path on one MI355X.

A case names one piece of work that a decode loop hands to this package, with its sizes; ``prepare`` makes what
the loop holds before the call (seeded inputs on the GPU), ``run`` makes one pass through the public entry points,
``work`` says what the pass cannot do without, and ``exact`` gives the same outputs from plain torch in float64.

Kinds of work (``case["kind"]``):
  tree_gdn   one tree through one Gated-DeltaNet layer in the Hugging Face form (ancestor matrix, no context)
  verify     a ragged batch of trees: the round's tree context, then ``layers`` GDN layers
  attn       mode attention of one draft step over a flat KV cache (Hugging Face layout)
  paged      mode attention of a continuous batch over a paged KV cache or a per-token slot table (SGLang layout)
  trees      draft logits -> top candidates and log Z -> mixture trees with their visibility
  candidates draft logits -> top candidates and log Z on the device (what the Hugging Face loop's host heap consumes)
  head       draft hidden states -> LM head -> top candidates (the end of a draft step)
  inputs     conv windows of a round's trees, then conv + normalisation and gates of ``layers`` GDN layers
  commit     GDN and conv states of all layers advanced to the accepted node
  plumbing   draft block ids and window slots, verify inputs with the flat mask, the accept walk, the KV moves
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "multi-future-drafting_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ddtree_sglang_ops  # noqa: E402
import mode_attention  # noqa: E402
import paged_mode_attention  # noqa: E402
import tree_gdn_kernel  # noqa: E402
import tree_logits  # noqa: E402

D = 128  # head dim of every configuration
DEPTH = 16  # nodes on the longest root path
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# Context lengths of 16 running requests, uniform over 1024 .. 8192, and their tree sizes, uniform over 16 .. 64.
_CTX16 = "7316,1903,5221,2874,6650,1187,4096,8033,3519,5902,1466,7704,2333,4777,6128,3050"
_NODES16 = "47,22,64,31,58,16,39,53,27,61,35,19,50,44,29,56"


def listed():
    return [
        # One 64-node tree through one layer: the smallest verify call, a single user's decode step, where latency
        # and launches count.
        dict(name="tree_gdn_64", kind="tree_gdn", nodes=64, hk=16, h=32),
        # A verify round of 8 requests with full 128-node trees: the headline batch (4 layers of the stack).
        dict(name="verify_8x128", kind="verify", sizes="128,128,128,128,128,128,128,128", hk=16, h=32, layers=4),
        # Continuous batch: 16 requests with ragged trees, the larger layer shape (48 value heads).
        dict(name="verify_ragged16", kind="verify", sizes=_NODES16, hk=16, h=48, layers=4),
        # The Hugging Face loop's default budget of 256 (257 nodes with the root), four requests.
        dict(name="verify_4x257", kind="verify", sizes="257,257,257,257", hk=16, h=32, layers=2),
        # One request's draft step: 8 modes x 16 tokens over 4096 context tokens, causal inside a mode's block.
        dict(name="attn_ctx4096", kind="attn", ctx=4096, modes=8, block=16, h=32, hkv=8, causal=True),
        # The continuous batch's draft step: 16 requests, 40 heads, 64-token pages.
        dict(name="paged_16", kind="paged", ctx=_CTX16, modes=8, block=16, h=40, hkv=8, page=64),
        # Tree construction of one request: 8 modes x 16 positions, top-8 candidates, 64 nodes.
        dict(name="trees_top8", kind="trees", bs=1, modes=8, block=16, vocab=151936, topk=8, budget=64, dtype="bf16"),
        # The candidates of the Hugging Face loop's default budget: every rank that a 256-node tree can reach.
        dict(name="candidates_top256", kind="candidates", rows=120, vocab=248320, topk=256, dtype="bf16"),
        # The end of one request's draft step with the full vocabulary: 8 modes x 15 drafted rows, hidden 2560.
        dict(name="head_full", kind="head", bs=1, modes=8, block=16, hidden=2560, vocab=151936, budget=8,
             reduced=False),
        # What the layers of a verify round consume, at the headline batch.
        dict(name="inputs_8x128", kind="inputs", sizes="128,128,128,128,128,128,128,128", hk=16, h=32, layers=4),
        # The accepted path of one request committed into all 24 GDN layers of the stack.
        dict(name="commit_24", kind="commit", layers=24, nodes=128, hk=16, h=32, path=13),
        # Everything between the draft and the verify forward of the continuous batch, 36 attention layers.
        dict(name="plumbing_16", kind="plumbing", ctx=_CTX16, nodes=64, block=16, layers=36, hkv=8),
    ]


# ---------------------------------------------------------------------------------------------- drawn cases


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    """One more case of the same ranges, odd and ragged sizes among them."""
    kind = rng.choice(["tree_gdn", "verify", "verify", "verify", "attn", "attn", "paged", "paged", "trees", "trees",
                       "candidates", "candidates", "head", "inputs", "commit", "plumbing"])
    hk, h = rng.choice([(16, 32), (16, 48), (16, 16), (8, 32)])
    if kind == "tree_gdn":
        return dict(kind=kind, nodes=_log_int(rng, 2, 300), hk=hk, h=h)
    if kind in ("verify", "inputs"):
        top = rng.choice([48, 64, 100, 128, 128, 200, 257])
        R = _log_int(rng, 1, 16)
        while R * top > 1100:
            R -= 1
        low = rng.choice([top, max(1, top // 4)])
        sizes = [rng.randint(low, top) for _ in range(R)]
        return dict(kind=kind, sizes=",".join(map(str, sizes)), hk=hk, h=h, layers=rng.randint(1, 4))
    if kind == "attn":
        h, hkv = rng.choice([(32, 8), (40, 8), (32, 4), (16, 8)])
        return dict(kind=kind, ctx=_log_int(rng, 16, 32768), modes=rng.choice([1, 2, 3, 4, 8, 8]),
                    block=rng.choice([7, 8, 16, 16]), h=h, hkv=hkv, causal=rng.random() < 0.5)
    if kind == "paged":
        h, hkv = rng.choice([(32, 8), (40, 8), (32, 4), (16, 8)])
        ctx = [_log_int(rng, 64, 8192) for _ in range(_log_int(rng, 1, 16))]
        return dict(kind=kind, ctx=",".join(map(str, ctx)), modes=rng.choice([1, 3, 4, 8, 8]), block=16, h=h, hkv=hkv,
                    page=rng.choice([1, 1, 64, 64, 16]))
    if kind in ("trees", "candidates"):
        vocab = _log_int(rng, 8192, 248320)
        if rng.random() < 0.6:
            vocab = max(8192, vocab // 64 * 64)
        dtype = rng.choice(["bf16"] * 6 + ["f32", "f16"])
    if kind == "candidates":
        rows = rng.choice([1, 4, 8]) * rng.randint(4, 16)
        return dict(kind=kind, rows=rows, vocab=vocab, topk=rng.choice([1, 8, 16, 31, 64, 128, 256]), dtype=dtype)
    if kind == "trees":
        bs, modes, block = rng.choice([1, 1, 2, 4]), rng.choice([1, 4, 8]), rng.randint(4, 16)
        while bs * modes * block * vocab > 128 * 248320 and bs > 1:
            bs //= 2
        budget = rng.choice([16, 31, 64, 64, 128, 256])
        # every rank the budget can reach, where a request's candidates fit the device heap
        topk = budget if modes * block * budget <= 8192 and modes * budget <= 1024 else 8
        return dict(kind=kind, bs=bs, modes=modes, block=block, vocab=vocab, topk=topk, budget=budget, dtype=dtype)
    if kind == "head":
        vocab = _log_int(rng, 8192, 151936) // 8 * 8
        return dict(kind=kind, bs=rng.choice([1, 1, 1, 2]) if vocab < 65536 else 1, modes=rng.choice([1, 4, 8]),
                    block=rng.choice([8, 16]), hidden=rng.choice([1024, 2048, 2560, 4096] if vocab < 90000 else [1024, 2560]),
                    vocab=vocab, budget=rng.choice([8, 32, 64]), reduced=rng.random() < 0.5)
    if kind == "commit":
        return dict(kind=kind, layers=_log_int(rng, 4, 24), nodes=_log_int(rng, 16, 257), hk=hk, h=min(h, 32),
                    path=rng.randint(1, DEPTH))
    ctx = [_log_int(rng, 64, 8192) for _ in range(_log_int(rng, 1, 16))]
    return dict(kind=kind, ctx=",".join(map(str, ctx)), nodes=rng.choice([17, 32, 64, 128, 257]), block=16,
                layers=rng.choice([24, 36]), hkv=rng.choice([4, 8]))


# ---------------------------------------------------------------------------------------------- inputs


def _ints(text):
    return [int(x) for x in text.split(",")]


def _tree(n, rng):
    """Parents of a random tree: uniform over the earlier nodes whose depth is below the limit (node 0 = root)."""
    parents, depth, ok = [-1], [1], [0]
    for i in range(1, n):
        p = ok[rng.randrange(len(ok))]
        parents.append(p)
        depth.append(depth[p] + 1)
        if depth[i] < DEPTH:
            ok.append(i)
    return parents


def _trees(sizes, seed):
    rng = random.Random(seed)
    return [_tree(n, rng) for n in sizes]


def _anc(parents):
    """Ancestor-or-self matrix of one tree, [n, n] bool on the host."""
    n = len(parents)
    a = torch.zeros(n, n, dtype=torch.bool)
    for i, p in enumerate(parents):
        if p >= 0:
            a[i] = a[p]
        a[i, i] = True
    return a


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _bf16(t):
    return t.to(torch.bfloat16)


def _gdn_layer(g, sizes, ancs, hk, h):
    n = sum(sizes)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    decay = -torch.nn.functional.softplus(_randn(g, n, h)) * 0.1
    g_cum = torch.cat([a.float() @ d for a, d in zip(ancs, decay.split(sizes))])
    return dict(q=_bf16(unit(_randn(g, n, hk, D))), k=_bf16(unit(_randn(g, n, hk, D))), v=_bf16(_randn(g, n, h, D)),
                g_cum=g_cum, beta=torch.sigmoid(_randn(g, n, h)), s0=_randn(g, len(sizes), h, D, D) * 0.02)


def _round(case, seed, sizes):
    """The trees of one verify round on the device: parents, node offsets, ancestor matrices."""
    trees = _trees(sizes, seed)
    cu = torch.tensor([0] + sizes).cumsum(0).to(torch.int32)
    return dict(trees=trees, sizes=sizes, parents=torch.tensor(sum(trees, []), dtype=torch.int32).to(DEV), cu=cu.to(DEV),
                ancs=[_anc(t).to(DEV) for t in trees])


def _prepare_tree_gdn(case, seed):
    g = _gen(seed)
    s = _round(case, seed, [case["nodes"]])
    s["layer"] = _gdn_layer(g, s["sizes"], s["ancs"], case["hk"], case["h"])
    s["anc8"] = s["ancs"][0].to(torch.int8)
    return s


def _prepare_verify(case, seed):
    g = _gen(seed)
    s = _round(case, seed, _ints(case["sizes"]))
    n, h = sum(s["sizes"]), case["h"]
    s["layers"] = [_gdn_layer(g, s["sizes"], s["ancs"], case["hk"], h) for _ in range(case["layers"])]
    # u is kept until the commit, o feeds the layer's output projection: the loop holds one pair per layer
    s["out"] = [(torch.empty(n, h, D, device=DEV), torch.empty(n, h, D, device=DEV)) for _ in range(case["layers"])]
    return s


def _prepare_attn(case, seed):
    g, KL = _gen(seed), case["modes"] * case["block"]
    return dict(q=_bf16(_randn(g, 1, case["h"], KL, D) * 0.5),
                k=_bf16(_randn(g, 1, case["hkv"], case["ctx"] + KL, D) * 0.5),
                v=_bf16(_randn(g, 1, case["hkv"], case["ctx"] + KL, D) * 0.5))


def _prepare_paged(case, seed):
    g = _gen(seed)
    lens, page, hkv = _ints(case["ctx"]), case["page"], case["hkv"]
    T = len(lens) * case["modes"] * case["block"]
    pages = [-(-c // page) for c in lens]
    perm = torch.randperm(sum(pages) + 3, generator=g, device=DEV).to(torch.int32)
    table = torch.zeros(len(lens) + 2, max(pages), dtype=torch.int32, device=DEV)
    off = 0
    for r, n in enumerate(pages):
        table[r + 2, :n] = perm[off:off + n]
        off += n
    slots = perm.numel() * page
    return dict(q=_bf16(_randn(g, T, case["h"], D) * 0.5), k_new=_bf16(_randn(g, T, hkv, D) * 0.5),
                v_new=_bf16(_randn(g, T, hkv, D) * 0.5), k_cache=_bf16(_randn(g, slots, hkv, D) * 0.5),
                v_cache=_bf16(_randn(g, slots, hkv, D) * 0.5), table=table,
                rows=torch.arange(2, len(lens) + 2, dtype=torch.int64, device=DEV),
                lens=torch.tensor(lens, dtype=torch.int64, device=DEV))


def _prepare_trees(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    bs, K, L, V = case["bs"], case["modes"], case["block"], case["vocab"]
    x = _randn(g, bs, K, L, V) * 3
    for b in range(bs):  # one mode is sure of one token at every position
        for pos in range(L):
            x[b, rng.randrange(K), pos, rng.randrange(V)] += 6
    return dict(logits=x.to(DTYPES[case["dtype"]]), prior=torch.log_softmax(_randn(g, bs, K), dim=-1))


def _prepare_candidates(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    x = _randn(g, case["rows"], case["vocab"]) * 3
    for row in x:
        row[rng.randrange(case["vocab"])] += 6
    return dict(logits=x.to(DTYPES[case["dtype"]]))


def _prepare_head(case, seed):
    g = _gen(seed)
    rows = case["bs"] * case["modes"] * case["block"]
    hidden = _bf16(_randn(g, rows, case["hidden"]))
    weight = torch.empty(case["vocab"], case["hidden"], dtype=torch.bfloat16, device=DEV)
    for part in weight.split(16384):
        part.copy_(_randn(g, *part.shape) * 0.02)
    ids = None
    if case["reduced"]:  # a draft vocabulary out of the target's
        ids = torch.randperm(151936, generator=g, device=DEV)[:case["vocab"]].sort().values.to(torch.int32)
    head = ddtree_sglang_ops.DDTreeDraftTopK(weight=weight, block_size=case["block"], num_modes=case["modes"],
                                             budget=case["budget"], max_bs=case["bs"], vocab_ids=ids)
    return dict(hidden=hidden, weight=weight, head=head)


KC = 4  # conv kernel of the GDN layers


def _prepare_inputs(case, seed):
    g = _gen(seed)
    s = _round(case, seed, _ints(case["sizes"]))
    n, R, h = sum(s["sizes"]), len(s["sizes"]), case["h"]
    cd = (2 * case["hk"] + h) * D
    s["layers"] = [dict(x=_bf16(_randn(g, n, cd) * 0.5), conv=_bf16(_randn(g, R, cd, KC) * 0.5),
                        w=_bf16(_randn(g, cd, KC) * 0.5), a=_bf16(_randn(g, n, h)), b=_bf16(_randn(g, n, h)),
                        A_log=torch.rand(h, generator=g, device=DEV).mul(15).add(1).log(), dt=_randn(g, h) * 0.5)
                   for _ in range(case["layers"])]
    return s


def _prepare_commit(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    Lc, n, hk, h = case["layers"], case["nodes"], case["hk"], case["h"]
    cd = (2 * hk + h) * D
    # a tree whose first `path` nodes are the accepted chain, the others hang anywhere below the depth limit
    p = min(case["path"], n)
    parents, depth = list(range(-1, p - 1)), list(range(1, p + 1))
    for i in range(p, n):
        j = rng.randrange(i)
        while depth[j] >= DEPTH:
            j = rng.randrange(i)
        parents.append(j)
        depth.append(depth[j] + 1)
    par = torch.tensor(parents, dtype=torch.int32, device=DEV)
    decay = -torch.nn.functional.softplus(_randn(g, Lc, n, h)) * 0.1
    k = _randn(g, Lc, n, hk, D)
    return dict(state=_randn(g, Lc, h, D, D) * 0.02, u=_randn(g, Lc, n, h, D), k=_bf16(k / k.norm(dim=-1, keepdim=True)),
                g_cum=torch.matmul(_anc(parents).to(DEV).float(), decay), path=torch.arange(p, dtype=torch.int32, device=DEV),
                conv=_bf16(_randn(g, Lc, cd, KC) * 0.5), x=_bf16(_randn(g, Lc, n, cd) * 0.5),
                index=tree_gdn_kernel.conv_index(par, KC))


def _prepare_plumbing(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    lens, W, L = _ints(case["ctx"]), case["nodes"], case["block"]
    bs = len(lens)
    vocab = 151936
    trees, post = [], []
    for _ in range(bs):
        parents = _tree(W, rng)
        depth = [0] * W
        for i in range(1, W):
            depth[i] = depth[parents[i]] + 1
        tokens = [0] + rng.sample(range(vocab), W - 1)
        follow = [rng.randrange(vocab) for _ in range(W)]  # the target's choice at every node
        cur, accepted = 0, 0
        while accepted < 5:  # it agrees with the tree for a few steps
            kids = [i for i in range(cur + 1, W) if parents[i] == cur]
            if not kids:
                break
            cur_next = rng.choice(kids)
            follow[cur] = tokens[cur_next]
            cur, accepted = cur_next, accepted + 1
        trees.append([tokens, depth, parents])
        post.append(follow)
    i64 = lambda v: torch.tensor(v, dtype=torch.int64, device=DEV)
    rows = [W * (c + W) for c in lens]
    slots = 2 * bs * W
    # the verify window's slots of every request, as the allocator handed them out
    perm = torch.randperm(slots, generator=g, device=DEV).to(torch.int32)
    table = torch.zeros(bs + 2, max(lens) + W, dtype=torch.int32, device=DEV)
    for b, c in enumerate(lens):
        table[b + 2, c:c + W] = perm[b * W:(b + 1) * W]
    pool = torch.empty(2 * case["layers"], slots, case["hkv"], D, dtype=torch.bfloat16, device=DEV)
    for part in pool:
        part.copy_(_randn(g, *part.shape))
    out = lambda *shape, dtype=torch.int64: torch.empty(*shape, dtype=dtype, device=DEV)
    return dict(tree=i64(trees), post=i64(post), prefix=i64(lens), offsets=i64([sum(rows[:b]) for b in range(bs)]),
                root=i64([rng.randrange(vocab) for _ in range(bs)]), req=i64(list(range(2, bs + 2))), table=table, pool=pool,
                mover=ddtree_sglang_ops.DDTreeKVCompactor(data_ptrs=i64([t.data_ptr() for t in pool]),
                                                          slot_bytes=case["hkv"] * D * 2, num_slots=slots),
                block=out(bs, L), block_pos=out(bs, L), window=out(bs, W), mask=out(sum(rows), dtype=torch.bool),
                ids=out(bs, W), pos=out(bs, W), accept=out(bs, dtype=torch.int32), commit=out(bs, dtype=torch.int32),
                bonus=out(bs), tokens=out(bs, L), lens=out(bs), src=out(bs, L), tgt=out(bs, L), hidden=out(bs, L))


def prepare(case, seed):
    return dict(globals()["_prepare_" + case["kind"]](case, seed), case=case)


# ---------------------------------------------------------------------------------------------- one pass


def _run_tree_gdn(s, case):
    y = s["layer"]
    return tree_gdn_kernel.tree_gdn(y["q"], y["k"], y["v"], y["g_cum"], y["beta"], y["s0"][0], s["anc8"])


def _run_verify(s, case):
    ctx = tree_gdn_kernel.tree_context(s["parents"], s["cu"], max_nodes=max(s["sizes"]))
    return [tree_gdn_kernel.tree_gdn_varlen(y["q"], y["k"], y["v"], y["g_cum"], y["beta"], y["s0"], None, s["cu"], out=out,
                                            ctx=ctx) for y, out in zip(s["layers"], s["out"])]


def _run_attn(s, case):
    return mode_attention.mode_block_attention(s["q"], s["k"], s["v"], case["modes"], case["block"], D ** -0.5,
                                               causal_in_block=case["causal"])


def _run_paged(s, case):
    return paged_mode_attention.paged_mode_block_attention(
        q=s["q"], k_new=s["k_new"], v_new=s["v_new"], k_cache=s["k_cache"], v_cache=s["v_cache"], req_to_token=s["table"],
        req_pool_indices=s["rows"], ctx_lens=s["lens"], num_modes=case["modes"], block_size=case["block"],
        scaling=D ** -0.5, num_ctx_splits=-1, page_size=case["page"])


def _run_trees(s, case):
    return ddtree_sglang_ops.build_mixture_trees_from_logits(s["logits"], s["prior"], case["budget"], topk=case["topk"])


def _run_candidates(s, case):
    return tree_logits.topk_logz(s["logits"], case["topk"], with_logz=True)


def _run_head(s, case):
    s["head"](s["hidden"])
    return s["head"].outputs(case["bs"])


def _run_inputs(s, case):
    index = tree_gdn_kernel.conv_index(s["parents"], KC, s["cu"])
    out = []
    for y in s["layers"]:
        out.append(tree_gdn_kernel.tree_prep(y["x"], y["conv"], index, y["w"], case["hk"], case["h"], D, cu_nodes=s["cu"]))
        out.append(tree_gdn_kernel.tree_gates(y["a"], y["b"], y["A_log"], y["dt"], s["parents"], s["cu"]))
    return [index, out]


def _run_commit(s, case):
    return tree_gdn_kernel.gdn_commit(s["state"], s["u"], s["k"], s["g_cum"], s["path"], conv=s["conv"], x=s["x"],
                                      conv_index=s["index"])


def _run_plumbing(s, case):
    ops, tree = ddtree_sglang_ops, s["tree"]
    ops.ddtree_prepare(bonus_tokens=s["root"], prefix_lens=s["prefix"], req_pool_indices=s["req"], req_to_token=s["table"],
                       block_ids_out=s["block"], positions_out=s["block_pos"], window_out=s["window"], mask_token_id=151935)
    ops.ddtree_verify_inputs(root_tokens=s["root"], prefix_lens=s["prefix"], tokens=tree[:, 0], depths=tree[:, 1],
                             parents=tree[:, 2], mask_offsets=s["offsets"], ids_out=s["ids"], positions_out=s["pos"],
                             mask_out=s["mask"], max_depth=DEPTH)
    ops.ddtree_follow(posterior=s["post"], verify_ids=s["ids"], parents=tree[:, 2], window=s["window"],
                      prefix_lens=s["prefix"], accept_len_out=s["accept"], commit_lens_out=s["commit"],
                      bonus_out=s["bonus"], out_tokens_out=s["tokens"], new_seq_lens_out=s["lens"], move_src_out=s["src"],
                      move_tgt_out=s["tgt"], hidden_index_out=s["hidden"])
    s["mover"](move_src=s["src"], move_tgt=s["tgt"])
    return {k: s[k] for k in ("block", "block_pos", "window", "mask", "ids", "pos", "accept", "commit", "bonus", "tokens",
                              "lens", "src", "tgt", "hidden", "pool")}


_RUN = {k[5:]: v for k, v in globals().items() if k.startswith("_run_")}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


# ---------------------------------------------------------------------------------------------- what a pass needs


def _gdn_work(n, R, hk, h):
    # states, q / k / v, gates and parents in, u and o out; the S0 products of every node's k and q
    return (R * h * D * D * 4 + n * hk * D * 2 * 2 + n * h * D * 2 + n * h * 4 * 2 + n * 4 + n * h * D * 4 * 2,
            2 * 2 * n * h * D * D)


def work(case):
    kind = case["kind"]
    if kind == "tree_gdn":
        b, f = _gdn_work(case["nodes"], 1, case["hk"], case["h"])
    elif kind == "verify":
        sizes = _ints(case["sizes"])
        b, f = _gdn_work(sum(sizes), len(sizes), case["hk"], case["h"])
        b, f = b * case["layers"], f * case["layers"]
    elif kind in ("attn", "paged"):
        lens = _ints(case["ctx"]) if kind == "paged" else [case["ctx"]]
        KL, h, hkv = case["modes"] * case["block"], case["h"], case["hkv"]
        b = sum(2 * KL * h * D * 2 + 2 * (c + KL) * hkv * D * 2 for c in lens)
        b += sum(-(-c // case["page"]) * 4 for c in lens) if kind == "paged" else 0
        f = sum(4 * h * D * KL * (c + case["block"]) for c in lens)
    elif kind == "trees":
        rows, W = case["bs"] * case["modes"] * case["block"], case["budget"] + 1
        size = 4 if case["dtype"] == "f32" else 2
        b = rows * case["vocab"] * size + rows * case["topk"] * 8 + case["bs"] * (3 * W * 8 + 8 + W * W + case["modes"] * 4)
        f = rows * case["vocab"] * 2
    elif kind == "candidates":
        b = case["rows"] * (case["vocab"] * (4 if case["dtype"] == "f32" else 2) + case["topk"] * 12 + 4)
        f = case["rows"] * case["vocab"] * 2
    elif kind == "head":
        blocks = case["bs"] * case["modes"]
        M = blocks * (case["block"] - 1)
        b = case["vocab"] * case["hidden"] * 2 + M * case["hidden"] * 2 + M * case["budget"] * 8
        b += case["vocab"] * 4 if case["reduced"] else 0
        f = 2 * M * case["vocab"] * case["hidden"]
    elif kind == "inputs":
        sizes = _ints(case["sizes"])
        n, h = sum(sizes), case["h"]
        cd = (2 * case["hk"] + h) * D
        b = case["layers"] * (n * cd * 2 * 2 + (len(sizes) + 1) * cd * KC * 2 + n * KC * 4 + n * h * (2 * 2 + 2 * 4)) + n * 20
        f = case["layers"] * (n * cd * (2 * KC + 8) + n * h * 12)
    elif kind == "commit":
        Lc, p, h = case["layers"], min(case["path"], case["nodes"]), case["h"]
        cd = (2 * case["hk"] + h) * D
        b = Lc * (2 * h * D * D * 4 + p * (h * D * 4 + case["hk"] * D * 2 + h * 4) + 2 * cd * KC * 2 + KC * cd * 2)
        f = Lc * h * D * D * (2 * p + 1)
    else:
        lens, W = _ints(case["ctx"]), case["nodes"]
        bs = len(lens)
        moved = 5 * bs * 2 * case["layers"] * case["hkv"] * D * 2  # the accepted nodes' rows in every K and V buffer
        b = sum(W * (c + W) for c in lens) + bs * W * 8 * 8 + bs * case["block"] * 8 * 6 + 2 * moved
        f = 0
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("tree_gdn", "verify"):
        return {"rel": 2e-3, "max": 2e-2}
    if kind in ("attn", "paged"):
        return {"rel": 4e-3, "max": 4e-2}
    if kind == "candidates":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "trees":
        if case["dtype"] == "bf16":
            return {"rel": 1e-6, "max": 1e-5}
        return {"rel": 1e-6, "max": 1e-5, "differ": 5e-3}
    if kind == "head":
        return {"rel": 2e-3, "max": 2e-2, "differ": 1e-2}
    if kind == "inputs":
        return {"rel": 2e-3, "max": 2e-2}
    if kind == "commit":
        return {"rel": 1e-5, "max": 1e-4}
    return "exact"


# ---------------------------------------------------------------------------------------------- float64 answers


def _exact_gdn(y, sizes, ancs, R):
    """u and o of every node in float64: the dense triangular system of each tree and head."""
    us, os_ = [], []
    h, hk = y["v"].shape[1], y["k"].shape[1]
    parts = [y[name].double().split(sizes) for name in ("q", "k", "v", "g_cum", "beta")]
    for r in range(R):
        q, k, v, G, beta = (p[r].transpose(0, 1) for p in parts)  # heads first
        q, k = q.repeat_interleave(h // hk, 0), k.repeat_interleave(h // hk, 0)
        s0, anc = y["s0"][r].double(), ancs[r]
        n = anc.shape[0]
        decay = torch.where(anc, G[:, :, None] - G[:, None, :], -math.inf).exp()
        strict = decay * (~torch.eye(n, dtype=torch.bool, device=DEV))
        kt = k.transpose(1, 2).contiguous()
        A = beta[:, :, None] * strict * torch.matmul(k, kt)
        rhs = beta[:, :, None] * (v - G.exp()[:, :, None] * torch.matmul(k, s0))
        u = torch.linalg.solve_triangular(A + torch.eye(n, dtype=torch.float64, device=DEV), rhs, upper=False,
                                          unitriangular=True)
        o = G.exp()[:, :, None] * torch.matmul(q, s0) + torch.matmul(decay * torch.matmul(q, kt), u)
        us.append(u.transpose(0, 1))
        os_.append(o.transpose(0, 1))
    return torch.cat(us), torch.cat(os_)


def _exact_tree_gdn(s, case):
    return _exact_gdn(s["layer"], s["sizes"], s["ancs"], 1)


def _exact_verify(s, case):
    return [_exact_gdn(y, s["sizes"], s["ancs"], len(s["sizes"])) for y in s["layers"]]


def _attention(q, kc, vc, kb, vb, modes, block, causal):
    """q [H, KL, D]; kc, vc [Hkv, ctx, D]; kb, vb [Hkv, KL, D] -> [KL, H, D] in float64."""
    rep = q.shape[0] // kb.shape[0]
    KL = modes * block
    row = torch.arange(KL, device=DEV)
    seen = row[:, None] // block == row[None, :] // block
    if causal:
        seen &= row[None, :] <= row[:, None]
    outs = []
    for hk in range(kb.shape[0]):
        qh = q[hk * rep:(hk + 1) * rep].double().reshape(rep * KL, D) * D ** -0.5
        s_ctx = qh @ kc[hk].double().T
        s_blk = (qh @ kb[hk].double().T).masked_fill(~seen.repeat(rep, 1), -math.inf)
        p = torch.softmax(torch.cat([s_ctx, s_blk], -1), -1)
        outs.append((p @ torch.cat([vc[hk], vb[hk]]).double()).reshape(rep, KL, D))
    return torch.cat(outs).transpose(0, 1)


def _exact_attn(s, case):
    c = case["ctx"]
    q, k, v = s["q"][0], s["k"][0], s["v"][0]
    return _attention(q, k[:, :c], v[:, :c], k[:, c:], v[:, c:], case["modes"], case["block"], case["causal"])[None]


def _exact_paged(s, case):
    KL, page = case["modes"] * case["block"], case["page"]
    out = []
    for b, c in enumerate(_ints(case["ctx"])):
        t = torch.arange(c, device=DEV)
        at = s["table"][b + 2][t // page].long() * page + t % page
        rows = slice(b * KL, (b + 1) * KL)
        first = lambda x: x.transpose(0, 1)
        out.append(_attention(first(s["q"][rows]), first(s["k_cache"][at]), first(s["v_cache"][at]), first(s["k_new"][rows]),
                              first(s["v_new"][rows]), case["modes"], case["block"], False))
    return torch.cat(out)


def _exact_trees(s, case):
    x = s["logits"].double()
    logp = torch.topk(x, case["topk"], dim=-1).values - torch.logsumexp(x, -1, keepdim=True)
    return None, None, None, logp, None


def _exact_candidates(s, case):
    x = s["logits"].double()
    logz = torch.logsumexp(x, -1)
    return torch.topk(x, case["topk"], dim=-1).values - logz[:, None], None, logz


def _exact_head(s, case):
    rows = s["hidden"].view(-1, case["block"], case["hidden"])[:, 1:].reshape(-1, case["hidden"]).double()
    x = torch.cat([rows @ w.double().T for w in s["weight"].split(16384)], dim=1)
    logp = torch.topk(x, case["budget"], dim=-1).values - torch.logsumexp(x, -1, keepdim=True)
    return logp.view(case["bs"], case["modes"], case["block"] - 1, case["budget"]), None


def _exact_inputs(s, case):
    hk, h, cu = case["hk"], case["h"], [0]
    for n in s["sizes"]:
        cu.append(cu[-1] + n)
    out = []
    for y in s["layers"]:
        qkv, gates = [], []
        for r, parents in enumerate(s["trees"]):
            x = y["x"][cu[r]:cu[r + 1]].double()
            src = torch.cat([y["conv"][r].double().T, x])  # [cached columns, oldest first ; nodes]
            windows = []
            for i in range(len(parents)):
                win, j = [], i
                while len(win) < KC and j >= 0:
                    win.append(KC + j)
                    j = parents[j]
                win += [KC - 1 - t for t in range(KC - len(win))]
                windows.append(win[::-1])
            acc = (src[torch.tensor(windows, device=DEV)] * y["w"].double().T[None]).sum(1)
            z = acc * torch.sigmoid(acc)
            qk = z[:, :2 * hk * D].reshape(-1, 2 * hk, D)
            qk = qk * torch.rsqrt((qk * qk).sum(-1, keepdim=True) + 1e-6)
            qkv.append((qk[:, :hk] * D ** -0.5, qk[:, hk:], z[:, 2 * hk * D:].reshape(-1, h, D)))
            dec = -y["A_log"].double().exp() * torch.nn.functional.softplus(y["a"][cu[r]:cu[r + 1]].double() + y["dt"].double())
            gates.append((s["ancs"][r].double() @ dec, torch.sigmoid(y["b"][cu[r]:cu[r + 1]].double())))
        out.append(tuple(torch.cat(t) for t in zip(*qkv)))
        out.append(tuple(torch.cat(t) for t in zip(*gates)))
    return [None, out]


def _exact_commit(s, case):
    p = s["path"].long()
    rep = case["h"] // case["hk"]
    G = s["g_cum"].double()[:, p]  # [layers, p, h]
    k = s["k"][:, p].double().repeat_interleave(rep, dim=2) * (G[:, -1:] - G).exp()[..., None]
    u = s["u"][:, p].double()
    new = G[:, -1].exp()[..., None, None] * s["state"].double()
    new = new + torch.matmul(k.permute(0, 2, 3, 1).contiguous(), u.permute(0, 2, 1, 3).contiguous())
    src = torch.cat([s["conv"].double(), s["x"].double().transpose(1, 2)], dim=-1)  # [layers, channels, KC + nodes]
    return new, src[..., s["index"][p[-1]].long()]


_EXACT = {k[7:]: v for k, v in globals().items() if k.startswith("_exact_") and k != "_exact_gdn"}


def exact(case, seed):
    if case["kind"] not in _EXACT:  # whole numbers and copied bytes only
        return None
    return _EXACT[case["kind"]](prepare(case, seed), case)
