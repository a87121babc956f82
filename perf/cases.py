"""The work that a serving runtime has this package do, as measurable cases.

Four kinds of pass, each through the public API:

``decode``   the indexer + cache part of one decode step of a registered flow:
             plan_decode once, then for every sparse layer forward_cache (the
             pages that the newest tokens close) and forward_indexer (page
             scores, top-k, sparse block table).
``attend``   paged decode attention of several layers over a block table: the
             dense table (a full-attention layer) or a sparse one.
``model``    a whole decode step's share of the package: plan_decode, a full
             attention layer (new keys and values stored, dense attention),
             then sparse layers (stored, forward_cache, forward_indexer,
             sparse attention).
``prefill``  the cache side after a chunk of prompt tokens, layer by layer:
             the new keys and values stored, forward_cache over the pages that
             they fill; with "burst" only the reduction, CMean and CMax.

Decode passes are captured once in a HIP graph, as a serving runtime captures
its decode step, and a pass replays it on the runtime's static buffers;
prefill passes are called eagerly, as a runtime does whose chunks differ in
size.  Every layer has its own pools, and pages lie scattered over them.

Request lengths are spread over [min_len, max_len], odd ones among them, and
are a function of the case alone; the seed decides their order, the block
tables and all values.
"""
from __future__ import annotations

import math
import os
import random
import sys
from types import SimpleNamespace

import torch

_PKG = os.path.join(os.getcwd(), "vortex_torch-dev_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

FLOWS = {"block": "block_sparse_attention", "gqa": "gqa_block_sparse_attention",
         "quest": "gqa_quest_sparse_attention"}
BOS = EOS = 1
SOFTMAX_SCALE = 0.09  # of the gqa flow


# ------------------------------------------------------------------- cases
def _decode(name, flow, batch, min_len, max_len, layers, heads=8, group=2, dim=128, topk=30, page=16):
    c = {"kind": "decode", "flow": flow, "batch": batch, "min_len": min_len, "max_len": max_len, "layers": layers,
         "heads": heads, "group": group, "dim": dim, "topk": topk, "page": page}
    return dict(c, name=name) if name else c


def _attend(name, table, batch, min_len, max_len, layers, heads=8, group=2, dim=128, topk=30, page=16):
    c = {"kind": "attend", "table": table, "batch": batch, "min_len": min_len, "max_len": max_len, "layers": layers,
         "heads": heads, "group": group, "dim": dim, "topk": topk, "page": page}
    return dict(c, name=name) if name else c


def _model(name, batch, min_len, max_len, layers, heads=8, group=2, dim=128, topk=30, page=16):
    c = {"kind": "model", "batch": batch, "min_len": min_len, "max_len": max_len, "layers": layers, "heads": heads,
         "group": group, "dim": dim, "topk": topk, "page": page}
    return dict(c, name=name) if name else c


def _prefill(name, tokens, requests, layers, heads=8, dim=128, page=16, burst=False):
    c = {"kind": "prefill", "tokens": tokens, "requests": requests, "layers": layers, "heads": heads, "dim": dim,
         "page": page, "burst": burst}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user, one request of 4096 tokens: the smallest step, latency and launches
        _decode("block_1x4k", "block", 1, 4096, 4096, 8),
        # the ordinary server: 64 requests of 1k to 8k tokens, Qwen3-1.7B head shape
        _decode("block_64x8k", "block", 64, 1024, 8192, 4),
        # few long requests, top-64
        _decode("block_8x32k", "block", 8, 32768, 32768, 4, topk=64),
        # a full server of long requests: the largest decode step
        _decode("block_64x32k", "block", 64, 4096, 32768, 4),
        # MLA latent cache (one latent head of 512 + 64, 16 query heads), top-32
        _decode("mla_32x16k", "block", 32, 4096, 16384, 4, heads=1, group=16, dim=576, topk=32),
        # the flow that scores every query head, a medium batch of ragged requests
        _decode("gqa_16x16k", "gqa", 16, 1024, 16384, 4),
        # the envelope flow on the ordinary server
        _decode("quest_64x8k", "quest", 64, 1024, 8192, 4),
        # sparse attention over the pages that the indexer kept
        _attend("attend_sparse_64x8k", "sparse", 64, 1024, 8192, 4),
        # the full-attention layer (layer 0 of the sparse models, all layers of a dense one)
        _attend("attend_dense_16x16k", "dense", 16, 1024, 16384, 2),
        # the package's share of a decode step: one full-attention layer, three sparse ones
        _model("model_32x8k", 32, 512, 8192, 4),
        # the cache side of a chunked prefill: 8k tokens of three requests
        _prefill("prefill_8k", 8191, 3, 4),
        # page-finish burst: 65,536 pages in shuffled token order, CMean and CMax
        _prefill("burst_65536_pages", 65536 * 16, 128, 1, burst=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "decode", "attend", "attend", "model", "prefill"])
    heads = rng.choice([1, 2, 4, 8, 8])
    page = rng.choice([16, 16, 16, 32])
    if kind == "prefill":
        if rng.random() < 0.3:
            return _prefill(None, _log(rng, 16384, 524288), _log(rng, 4, 64), 1, heads=heads,
                            dim=rng.choice([64, 128]), page=page, burst=True)
        return _prefill(None, _log(rng, 512, 16384) | 1, rng.randint(1, 8), 4, heads=heads,
                        dim=rng.choice([64, 128, 128]), page=page)
    batch = _log(rng, 1, 64)
    max_len = _log(rng, 1024, 32768)
    min_len = max(64, int(max_len * rng.choice([0.05, 0.25, 0.5, 1.0])))
    topk = rng.choice([16, 30, 32, 64])
    if kind == "decode":
        flow = rng.choice(["block", "block", "gqa", "quest"])
        if flow == "block" and rng.random() < 0.25:
            return _decode(None, flow, min(batch, 48), min_len, max_len, 4, heads=1, group=16, dim=576, topk=topk)
        group = rng.choice([1, 2, 2, 4, 8])
        if flow != "block":  # every query head is scored: no dearer than the largest listed case
            batch, group = min(batch, 48), min(group, 4)
        return _decode(None, flow, batch, min_len, max_len, rng.choice([2, 3, 4]), heads=heads, group=group,
                       dim=rng.choice([64, 128, 128]), topk=topk, page=page)
    group = rng.choice([1, 2, 2, 4])
    if kind == "attend":
        table = rng.choice(["sparse", "dense"])
        if table == "dense":
            batch = max(1, min(batch, 262144 // max_len))
        return _attend(None, table, batch, min_len, max_len, 2, heads=heads, group=group,
                       dim=rng.choice([64, 128, 128]), topk=topk, page=page)
    return _model(None, max(1, min(batch, 262144 // max_len)), min_len, max_len, 3, heads=heads, group=group,
                  topk=topk, page=page)


# ------------------------------------------------------------------ inputs
def _lengths(case):
    """The requests' lengths: max_len itself, the rest uniform."""
    r = random.Random(f"{case['batch']} {case['min_len']} {case['max_len']}")
    return [case["max_len"]] + [r.randint(case["min_len"], case["max_len"]) for _ in range(case["batch"] - 1)]


def _closing(lens, page):
    return sum(1 for n in lens if n % page == 0)


def _gen(seed, *what):
    return torch.Generator(device="cuda").manual_seed(random.Random(f"{seed} {what}").randrange(1 << 62))


def _randn(shape, gen, std=1.0):
    t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)
    return t.mul_(std) if std != 1.0 else t


def _requests(case, seed):
    """The batch's block tables: lengths in the seed's order, every request's
    pages drawn from one shuffled pool, req_to_token rows in shuffled order."""
    P, H = case["page"], case["heads"]
    r = random.Random(f"requests {seed}")
    lens = _lengths(case)
    r.shuffle(lens)
    n = [(x + P - 1) // P for x in lens]
    pool = sum(n) + max(64, sum(n) // 8)
    perm = torch.randperm(pool, generator=_gen(seed, "pages"), device="cuda")
    B, T = len(lens), (case["max_len"] + P - 1) // P * P
    rows = list(range(B + 2))
    r.shuffle(rows)
    r2t = torch.zeros((B + 2, T), dtype=torch.int32, device="cuda")
    tok = torch.arange(T, device="cuda")
    pages, at = [], 0
    for b in range(B):
        pg = perm[at:at + n[b]]
        at += n[b]
        pages.append(pg)
        t = tok[:lens[b]]
        r2t[rows[b], :lens[b]] = (pg[t // P] * P + t % P).to(torch.int32)
    loc = torch.stack([pages[b][(lens[b] - 1) // P] * P + (lens[b] - 1) % P for b in range(B)])
    heads = torch.arange(H, device="cuda")
    # segment (b, h): rows page * H + h of the pools, in token order
    segs = [pages[b][None, :] * H + heads[:, None] for b in range(B)]
    return SimpleNamespace(lens=lens, n=n, pool=pool, r2t=r2t, rows=rows[:B], loc=loc, segs=segs)


def _layer(case, rq, seed, i, *want):
    """Layer i's tensors by name, a function of the seed alone."""
    P, H, G, D, B = case["page"], case["heads"], case["group"], case["dim"], case["batch"]
    rows = rq.pool * H
    made = {}
    for w in want:
        g = _gen(seed, "layer", i, w)
        if w in ("k", "v"):
            made[w] = _randn((rows, P, D), g)
        elif w == "q":
            made[w] = _randn((B * H, G, D), g)
        elif w in ("new_k", "new_v"):
            made[w] = _randn((B, H, D), g)
        else:  # a summary row per page: the spread of a mean of keys, or of their extremes
            made[w] = _randn((rows, 1, D), g, 0.25 if w == "centroids" else 0.5)
            if w in ("max", "min"):
                made[w].add_(1.75 if w == "max" else -1.75)
    return made


def _contexts(case, rq):
    from vortex_torch.cache import Context as CacheContext
    from vortex_torch.indexer import Context as IndexerContext

    P, H, G, D, B = case["page"], case["heads"], case["group"], case["dim"], case["batch"]
    i32 = dict(dtype=torch.int32, device="cuda")
    per_request = (case["max_len"] + P - 1) // P
    S = B * H
    parent = SimpleNamespace(
        kv_indices_decode=(torch.zeros(per_request * S, **i32),
                           torch.zeros(min(per_request, case["topk"] + BOS + EOS) * S, **i32)),
        kv_indptr_decode=(torch.zeros(S + 1, **i32), torch.zeros(S + 1, **i32)),
        kv_last_page_len_decode=torch.zeros(S, **i32), group_size=G, num_kv_heads=H, num_qo_heads=G * H, head_dim=D,
        page_size=P, num_pages=rq.pool, head_num=H)
    runner = SimpleNamespace(
        server_args=SimpleNamespace(page_size=P, vortex_max_seq_lens=case["max_len"], vortex_lb_max_chunk_size=64,
                                    vortex_lb_min_chunk_size=16, vortex_topk_val=case["topk"],
                                    vortex_page_reserved_bos=BOS, vortex_page_reserved_eos=EOS,
                                    max_prefill_tokens=16384),
        model_config=SimpleNamespace(context_len=case["max_len"]),
        req_to_token_pool=SimpleNamespace(size=B), device="cuda")
    return IndexerContext().create(parent, runner), CacheContext().create(parent, runner)


def _captured(step):
    """A HIP graph of step(), after a first run outside it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        step()
    torch.cuda.synchronize()
    return graph


def _scores(flow):
    """The score buffers that a flow's ops leave, zeroed where they never write."""
    from vortex_torch.flow.algorithms import BlockSparseAttention, GQABlockSparseAttention

    if isinstance(flow, BlockSparseAttention):
        bufs = [flow.gemv.output_buffer]
    elif isinstance(flow, GQABlockSparseAttention):
        bufs = [flow.gemm.output_buffer, flow.max_op.output_buffer]
    else:
        bufs = [flow.sum.output_buffer, flow.max_op.output_buffer]
    for b in bufs:
        b.zero_()
    return bufs


def _prepare_decode(case, seed):
    from vortex_torch.abs import FORMAT, as_vtensor
    from vortex_torch.cache import set_kv_buffer_launcher
    from vortex_torch.decode_attention import dense_decode_attention, sparse_decode_attention
    from vortex_torch.flow import build_vflow
    from vortex_torch.indexer.utils_sglang import plan_decode

    rq = _requests(case, seed)
    ictx, cctx = _contexts(case, rq)
    model = case["kind"] == "model"
    name = FLOWS[case.get("flow", "block")]
    seq_lens = torch.tensor(rq.lens, dtype=torch.int32, device="cuda")
    req = torch.tensor(rq.rows, dtype=torch.int64, device="cuda")
    o = as_vtensor(ictx.sparse_kv_indices.view(-1, 1, 1), FORMAT.RAGGED)
    ictx.profile()
    cctx.profile()
    layers = []
    for i in range(case["layers"]):
        ly = SimpleNamespace(flow=None, cache=None)
        if not model or i > 0:
            ly.flow = build_vflow(name)
            summaries = sorted(ly.flow.create_cache(case["page"], case["dim"]))
            t = _layer(case, rq, seed, i, "k", "q", *summaries)
            ly.cache = {n: as_vtensor(t[n], FORMAT.PAGED) for n in ["k"] + summaries}
            ly.summaries = [t[n] for n in summaries]
            q = as_vtensor(t["q"], FORMAT.BATCHED)
            ly.q = q
            ly.flow.forward_cache(ly.cache, rq.loc, cctx)
            ly.flow.forward_indexer(q, o, ly.cache, ictx)
            ly.scores = _scores(ly.flow)
        else:
            t = _layer(case, rq, seed, i, "k", "q")
        if model:
            ly.k, ly.plain_q = t["k"], t["q"]
            more = _layer(case, rq, seed, i, "v", "new_k", "new_v")
            ly.v, ly.new_k, ly.new_v = more["v"], more["new_k"], more["new_v"]
            ly.out = torch.zeros_like(ly.plain_q)
        layers.append(ly)
    ictx.execute()
    cctx.execute()

    def step():
        plan_decode(seq_lens, rq.r2t, req, ictx)
        for ly in layers:
            if model:
                set_kv_buffer_launcher(ly.k, ly.v, ly.new_k, ly.new_v, rq.loc, case["page"])
            if ly.flow is not None:
                ly.flow.forward_cache(ly.cache, rq.loc, cctx)
                ly.flow.forward_indexer(ly.q, o, ly.cache, ictx)
            if model:
                attend = dense_decode_attention if ly.flow is None else sparse_decode_attention
                attend(ly.plain_q, ly.k, ly.v, ictx, out=ly.out)

    graph = _captured(step)
    out = {"table": ictx.sparse_kv_indices, "indptr": ictx.sparse_kv_indptr, "dense": ictx.dense_kv_indptr,
           "last": ictx.kv_last_page_len,
           "summaries": [x for ly in layers if ly.flow is not None for x in ly.summaries],
           "scores": [x for ly in layers if ly.flow is not None for x in ly.scores]}
    if model:
        out["attention"] = [ly.out for ly in layers]
    return SimpleNamespace(graph=graph, out=out, keep=(layers, ictx, cctx, rq, seq_lens, req, o))


def _table(case, rq, seed):
    """(indptr, rows, last page lengths, segments' rows) of the block table
    that an attention layer reads; a sparse segment holds its first page, topk
    others in no order, and its last page, or all of a short request's."""
    g, H = _gen(seed, "table"), case["heads"]
    last, segs = [], []
    for b, n in enumerate(rq.n):
        last += [(rq.lens[b] - 1) % case["page"] + 1] * H
        rows = rq.segs[b]
        if case["table"] == "sparse" and n > case["topk"] + BOS + EOS:
            mid = torch.rand((H, n - BOS - EOS), generator=g, device="cuda").argsort(1)[:, :case["topk"]] + BOS
            rows = torch.cat([rows[:, :BOS], rows.gather(1, mid), rows[:, n - EOS:]], 1)
        segs += list(rows)
    indptr = [0]
    for s in segs:
        indptr.append(indptr[-1] + s.numel())
    dev = dict(dtype=torch.int32, device="cuda")
    return torch.tensor(indptr, **dev), torch.cat(segs).to(torch.int32), torch.tensor(last, **dev), segs


def _prepare_attend(case, seed):
    from vortex_torch.decode_attention import paged_decode_attention

    rq = _requests(case, seed)
    indptr, rows, last, _ = _table(case, rq, seed)
    layers = [_layer(case, rq, seed, i, "q", "k", "v") for i in range(case["layers"])]
    outs = [torch.zeros_like(t["q"]) for t in layers]

    def step():
        for t, out in zip(layers, outs):
            paged_decode_attention(t["q"], t["k"], t["v"], indptr, rows, last, case["batch"], case["heads"], out=out)

    return SimpleNamespace(graph=_captured(step), out={"attention": outs}, keep=(layers, indptr, rows, last))


def _chunk(case, seed):
    """(pool pages, loc) of a prefill chunk: the requests' tokens one after
    another, each continuing its own scattered pages from some slot on; of a
    burst, every slot of its pages in shuffled order."""
    P, n = case["page"], case["tokens"]
    g = _gen(seed, "chunk")
    if case["burst"]:
        pages = n // P
        pool = pages + pages // 16 + 64
        pg = torch.randperm(pool, generator=g, device="cuda")[:pages]
        slots = (pg[:, None] * P + torch.arange(P, device="cuda")).reshape(-1)
        return pool, slots[torch.randperm(slots.numel(), generator=g, device="cuda")]
    r = random.Random(f"{n} {case['requests']}")
    cuts = [0] + sorted(r.sample(range(1, n), case["requests"] - 1)) + [n]
    parts, at = [], 0
    pool = n // P + 2 * case["requests"] + 64
    perm = torch.randperm(pool, generator=g, device="cuda")
    for a, b in zip(cuts, cuts[1:]):
        pos = r.randrange(P) + torch.arange(b - a, device="cuda")
        used = (int(pos[-1]) // P) + 1
        parts.append(perm[at:at + used][pos // P] * P + pos % P)
        at += used
    return pool, torch.cat(parts)


def _chunk_layer(case, seed, pool, i):
    P, H, D = case["page"], case["heads"], case["dim"]
    rows = pool * H
    t = {"k": _randn((rows, P, D), _gen(seed, "layer", i, "k"))}
    if not case["burst"]:
        t["v"] = _randn((rows, P, D), _gen(seed, "layer", i, "v"))
        for w in ("new_k", "new_v"):
            t[w] = _randn((case["tokens"], H, D), _gen(seed, "layer", i, w))
    return t


def _prepare_prefill(case, seed):
    from vortex_torch.abs import FORMAT, as_vtensor
    from vortex_torch.cache import Context, MultiReduce
    from vortex_torch.flow import build_vflow
    from vortex_torch.utils import ReduceType

    P, H, D = case["page"], case["heads"], case["dim"]
    pool, loc = _chunk(case, seed)
    ctx = Context().create(
        SimpleNamespace(page_size=P, num_pages=pool, head_num=H, head_dim=D),
        SimpleNamespace(server_args=SimpleNamespace(max_prefill_tokens=16384),
                        req_to_token_pool=SimpleNamespace(size=64)))
    ctx.profile()
    layers = []
    for i in range(case["layers"]):
        t = _chunk_layer(case, seed, pool, i)
        ly = SimpleNamespace(t=t, k=as_vtensor(t["k"], FORMAT.PAGED))
        names = ["mean", "max"] if case["burst"] else ["centroids"]
        ly.outs = [torch.zeros((pool * H, 1, D), dtype=torch.bfloat16, device="cuda") for _ in names]
        tagged = [as_vtensor(x, FORMAT.PAGED) for x in ly.outs]
        if case["burst"]:
            ly.op = MultiReduce([ReduceType.Mean, ReduceType.Max])
            ly.tagged = tagged
            ly.op(ly.k, tagged, loc=loc, ctx=ctx)
        else:
            ly.flow = build_vflow(FLOWS["block"])
            ly.cache = {"k": ly.k, "centroids": tagged[0]}
            ly.flow.forward_cache(ly.cache, loc, ctx)
        layers.append(ly)
    ctx.execute()
    return SimpleNamespace(graph=None, case=case, layers=layers, loc=loc, ctx=ctx)


def prepare(case, seed):
    if case["kind"] == "prefill":
        return _prepare_prefill(case, seed)
    if case["kind"] == "attend":
        return _prepare_attend(case, seed)
    return _prepare_decode(case, seed)


def run(state):
    if state.graph is not None:
        state.graph.replay()
        return state.out
    from vortex_torch.cache import set_kv_buffer_launcher

    out = []
    for ly in state.layers:
        if state.case["burst"]:
            ly.op(ly.k, ly.tagged, loc=state.loc, ctx=state.ctx)
            out += ly.outs
        else:
            t = ly.t
            set_kv_buffer_launcher(t["k"], t["v"], t["new_k"], t["new_v"], state.loc, state.case["page"])
            ly.flow.forward_cache(ly.cache, state.loc, state.ctx)
            out += [t["k"], t["v"]] + ly.outs
    return out


# -------------------------------------------------------------------- work
def work(case):
    P, H, D = case["page"], case["heads"], case["dim"]
    row = 2 * D
    if case["kind"] == "prefill":
        n = case["tokens"]
        pages = n // P - (0 if case["burst"] else case["requests"] // 2)
        reduce = 8 * n + pages * H * row * (P + (2 if case["burst"] else 1))
        store = 0 if case["burst"] else 8 * n + 4 * n * H * row
        # a page's reduction reads what the store before it has just written
        return {"bytes": case["layers"] * (reduce + store), "flops": case["layers"] * 2 * pages * H * P * D}
    G, L, k = case["group"], case["layers"], case["topk"]
    lens = _lengths(case)
    S = len(lens) * H
    n = [(x + P - 1) // P for x in lens]
    budget = k + BOS + EOS
    kept = [min(x, budget) for x in n]
    q = S * G * row

    def attention(table, pages):
        tok = H * sum((m - 1) * P + (x - 1) % P + 1 for m, x in zip(pages, lens))
        return tok * 2 * row + 4 * H * sum(pages) + 2 * q, 4 * tok * G * D

    plan = sum(n) * 4 + H * (sum(n) + sum(kept)) * 4 + 12 * S
    scored = H * sum(m - BOS - EOS for m in n if m - BOS - EOS > k)
    flow = case.get("flow", "block")
    summaries = 2 if flow == "quest" else 1
    outs = 1 if flow == "block" else G + 1
    heads = 1 if flow == "block" else G
    closed = _closing(lens, P) * H
    index = (scored * (summaries * row + 4 + 2 * outs) + q + 4 * k * sum(H for m in n if m - BOS - EOS > k)
             + closed * row * (P + summaries) + 8 * len(lens))
    index_flops = 2 * scored * D * heads * summaries
    if case["kind"] == "decode":
        return {"bytes": plan + L * index, "flops": L * index_flops}
    if case["kind"] == "attend":
        b, f = attention(case["table"], n if case["table"] == "dense" else kept)
        return {"bytes": L * b, "flops": L * f}
    store = len(lens) * (8 + 4 * H * row)
    db, df = attention("dense", n)
    sb, sf = attention("sparse", kept)
    return {"bytes": plan + L * store + db + (L - 1) * (index + sb), "flops": df + (L - 1) * (index_flops + sf)}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    # Outputs are bf16: one rounding of a result (0.0017 against 64 bits), with
    # those of the query mean and the centroid, bf16 between the ops, 0.0025.
    # A page whose score ties with the k-th best may be another one.
    if case["kind"] == "prefill":
        return {"rel": 0.007, "max": 0.02}
    if case["kind"] == "attend":
        return {"rel": 0.007, "max": 0.05}
    return {"rel": 0.01, "max": 0.1, "differ": 0.004}


# ------------------------------------------------------------------- exact
def _exact_attention(t, segs, last, case):
    G, D, P = case["group"], case["dim"], case["page"]
    out = torch.zeros((len(segs), G, D), dtype=torch.float64, device="cuda")
    for s, rows in enumerate(segs):
        tok = (rows.numel() - 1) * P + last[s]
        k = t["k"][rows].view(-1, D)[:tok].double()
        v = t["v"][rows].view(-1, D)[:tok].double()
        p = torch.softmax((k @ t["q"][s].double().t().contiguous()) / math.sqrt(D), 0)
        out[s] = p.t().contiguous() @ v
    return out


def _exact_scores(case, flow, t, summaries, seg_rows, at, total):
    """The flow's score outputs in 64 bits (zeros where no page is scored)."""
    G, S = case["group"], len(seg_rows)
    width = [1] if flow == "block" else [G, 1]
    outs = [torch.zeros((total, w), dtype=torch.float64, device="cuda") for w in width]
    q = t["q"].double()
    for s in range(S):
        rows = seg_rows[s][BOS:seg_rows[s].numel() - EOS]
        if rows.numel() <= case["topk"]:
            continue
        p0 = at[s] + BOS
        span = slice(p0, p0 + rows.numel())
        if flow == "block":
            outs[0][span, 0] = summaries["centroids"][rows, 0] @ q[s].mean(0)
            continue
        if flow == "gqa":
            x = (summaries["centroids"][rows, 0] @ q[s].t().contiguous()) * SOFTMAX_SCALE
            x = torch.softmax(x, 0)
        else:
            hi, lo = summaries["max"][rows, 0], summaries["min"][rows, 0]
            x = torch.stack([torch.maximum(hi * q[s, g], lo * q[s, g]).sum(1) for g in range(G)], 1)
        outs[0][span] = x
        outs[1][span, 0] = x.amax(1)
    if flow == "block":
        return [outs[0].view(total, 1, 1)]
    return [outs[0].view(total, 1, G) if flow == "gqa" else outs[0].view(total, G, 1), outs[1].view(total, 1, 1)]


def exact(case, seed):
    P, H = case["page"], case["heads"]
    if case["kind"] == "prefill":
        pool, loc = _chunk(case, seed)
        out = []
        pages = loc[(loc + 1) % P == 0] // P
        rows = (pages[:, None] * H + torch.arange(H, device="cuda")).reshape(-1)
        for i in range(case["layers"]):
            t = _chunk_layer(case, seed, pool, i)
            if not case["burst"]:
                for w in ("k", "v"):
                    t[w].view(pool, H, P, -1).permute(0, 2, 1, 3)[loc // P, loc % P] = t["new_" + w]
                out += [t["k"].double(), t["v"].double()]
            for op in ("mean", "max") if case["burst"] else ("mean",):
                o = torch.zeros((pool * H, 1, case["dim"]), dtype=torch.float64, device="cuda")
                for part in rows.split(1 << 16):
                    x = t["k"][part].double()
                    o[part] = x.mean(1, keepdim=True) if op == "mean" else x.amax(1, keepdim=True)
                out.append(o)
        return out
    rq = _requests(case, seed)
    if case["kind"] == "attend":
        _, _, last, segs = _table(case, rq, seed)
        last = last.tolist()
        return {"attention": [_exact_attention(_layer(case, rq, seed, i, "q", "k", "v"), segs, last, case)
                              for i in range(case["layers"])]}
    flow, model = case.get("flow", "block"), case["kind"] == "model"
    names = ["max", "min"] if flow == "quest" else ["centroids"]
    seg_rows = [r for rows in rq.segs for r in rows]
    at = [0]
    for r in seg_rows:
        at.append(at[-1] + r.numel())
    total = (case["max_len"] + P - 1) // P * case["batch"] * H
    pages = rq.loc[(rq.loc + 1) % P == 0] // P
    closed = (pages[:, None] * H + torch.arange(H, device="cuda")).reshape(-1)
    last = [(x - 1) % P + 1 for x in rq.lens for _ in range(H)]
    out = {"table": None, "indptr": None, "dense": None, "last": None, "summaries": [], "scores": []}
    attention = []
    for i in range(case["layers"]):
        sparse = not model or i > 0
        t = _layer(case, rq, seed, i, "k", "q", *(names if sparse else []))
        if model:
            t.update(_layer(case, rq, seed, i, "v", "new_k", "new_v"))
            for w in ("k", "v"):
                t[w].view(rq.pool, H, P, -1).permute(0, 2, 1, 3)[rq.loc // P, rq.loc % P] = t["new_" + w]
            # the pages that a sparse layer attends to depend on its scores' rounding
            attention.append(None if sparse else _exact_attention(t, seg_rows, last, case))
        if not sparse:
            continue
        x = t["k"][closed].double()
        summaries = {n: t[n].double() for n in names}
        for n in names:
            summaries[n][closed] = (x.mean(1, keepdim=True) if n == "centroids" else
                                    x.amax(1, keepdim=True) if n == "max" else x.amin(1, keepdim=True))
        out["summaries"] += [summaries[n] for n in names]
        out["scores"] += _exact_scores(case, flow, t, summaries, seg_rows, at, total)
    if model:
        out["attention"] = attention
    return out
