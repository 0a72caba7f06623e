"""Performance cases: the calls a LeanSelect user's program makes on one GPU.

Five families, each called through the package's public entry points:

* ``layer``   one attention layer of LeanSelect sparse prefill on packed sequences
  (``prefill.leanselect_sparse_prefill``: compressed keys, page selection, attention);
* ``nosa``    the same layer with the NOSA two-stage selection and CIS-biased attention
  (``prefill.nosa_sparse_prefill``);
* ``decode``  one decode step of one attention layer over a KV cache: append with compressed
  keys, stage-1 page plans, attention over the plan's pages (``ops.kvcache_append``,
  ``ops.decode_topk_idx``, ``ops.sparse_attention_kvcache``), or attention over every cached
  page (``infllm_v2.infllmv2_attn_with_kvcache`` without a plan);
* ``block``   the decode attention block of a MiniCPM4.1-8B-shaped layer, projections included
  (``minicpm.MiniCPMLeanSelect.attention_decode``);
* ``model``   the prefill of a MiniCPM4.1-8B-shaped model of a few layers, to its last-token
  logits (``minicpm.MiniCPMLeanSelect.prefill``).

All use the MiniCPM4.1-8B attention shape (32 query heads, 2 KV heads, head dimension 128).
Budgets: 64 pages with 4 local blocks (the benchmark's), 96 pages with 32 local blocks (the
reference's published setting), NOSA's 96 pages with 16 local blocks and 24 selected ones.
"""
import math

import torch

from leanselect_amd import minicpm, workloads
from leanselect_amd.infllm_v2 import infllmv2_attn_with_kvcache
from leanselect_amd.ops import decode_topk_idx, kvcache_append, sparse_attention_kvcache
from leanselect_amd.prefill import leanselect_sparse_prefill, nosa_sparse_prefill

DEV = "cuda"
H, G, D = 32, 2, 128
GS = H // G
PAGE, SINK = 64, 1
HIDDEN, INTER, VOCAB = 4096, 16384, 73448
ROUTER = 128  # 4 router heads of 32
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # The benchmark's layer: one 128K prompt whose neighbouring rows choose many pages in common.
        dict(name="layer_128k", kind="layer", lens="131072", dtype="bf16", topics="planted",
             budget=64, local=4),
        # A 32K prompt without shared topics (rows share few pages), the published 96-page setting.
        dict(name="layer_32k_scattered", kind="layer", lens="32768", dtype="bf16", topics="none",
             budget=96, local=32),
        # A batch of prompts of odd lengths, one shorter than a page budget, in fp16.
        dict(name="layer_ragged_fp16", kind="layer", lens="8191,517,3001,12345", dtype="fp16",
             topics="unit", budget=64, local=4),
        # An ordinary 4K prompt.
        dict(name="layer_4k", kind="layer", lens="4096", dtype="bf16", topics="unit", budget=64,
             local=4),
        # A short prompt of odd length: latency and launches count.
        dict(name="layer_1337", kind="layer", lens="1337", dtype="bf16", topics="unit", budget=64,
             local=4),
        # The NOSA layer on a 32K prompt.
        dict(name="nosa_32k", kind="nosa", lens="32768", dtype="bf16", topics="unit", budget=96,
             local=16),
        # The NOSA layer on a small ragged batch.
        dict(name="nosa_ragged", kind="nosa", lens="777,2500,5001", dtype="bf16", topics="unit",
             budget=96, local=16),
        # One decode step of a single 128K conversation.
        dict(name="decode_128k_b1", kind="decode", lens="131071", dtype="bf16", plan="select",
             budget=64, local=4),
        # One decode step of a served batch of 16 conversations of 2K to 64K tokens.
        dict(name="decode_ragged_b16", kind="decode",
             lens="2047,2500,3333,4095,5000,6144,8191,9999,12287,16000,20001,24576,32767,40000,"
                  "50001,65535",
             dtype="bf16", plan="select", budget=64, local=4),
        # Dense decoding (no plan) of four conversations, as below a model's sparse threshold.
        dict(name="decode_dense_b4", kind="decode", lens="4097,9001,16383,30000", dtype="bf16",
             plan="all", budget=0, local=0),
        # The decode attention block of one layer with its projections, eight conversations.
        dict(name="block_decode_b8", kind="block",
             lens="1023,3000,4095,6001,8191,12000,16383,24001", dtype="bf16", budget=64, local=4),
        # Two decoder layers and the head on a packed batch of two prompts, to the logits.
        dict(name="model_prefill_5k", kind="model", lens="3100,2020", dtype="bf16", layers=2,
             budget=64, local=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "nosa", "nosa", "decode", "decode", "decode",
                       "block", "model"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind in ("layer", "nosa"):
        n_seq = rng.choice((1, 1, 2, 3, 4))
        total = _log_int(rng, 600, 65536 if kind == "layer" else 40000)
        cuts = sorted(rng.random() for _ in range(n_seq - 1))
        lens = [max(40, int(total * (b - a))) for a, b in zip([0.0] + cuts, cuts + [1.0])]
        budget, local = rng.choice(((64, 4), (64, 4), (96, 32))) if kind == "layer" else (96, 16)
        return dict(kind=kind, lens=",".join(map(str, lens)), dtype=dtype,
                    topics=rng.choice(("planted", "unit", "none")), budget=budget, local=local)
    if kind == "decode":
        batch = _log_int(rng, 1, 24)
        plan = rng.choice(("select", "select", "all"))
        top = 131000 if batch <= 4 and plan == "select" else 48000
        lens = [_log_int(rng, 700, top) for _ in range(batch)]
        budget, local = rng.choice(((64, 4), (96, 32))) if plan == "select" else (0, 0)
        return dict(kind=kind, lens=",".join(map(str, lens)), dtype=dtype, plan=plan,
                    budget=budget, local=local)
    if kind == "block":
        lens = [_log_int(rng, 700, 40000) for _ in range(_log_int(rng, 1, 16))]
        return dict(kind=kind, lens=",".join(map(str, lens)), dtype=dtype, budget=64, local=4)
    lens = [_log_int(rng, 100, 4000) for _ in range(rng.choice((1, 2, 3)))]
    return dict(kind=kind, lens=",".join(map(str, lens)), dtype=dtype, layers=2, budget=64, local=4)


def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _cu(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


def _n_windows(n):
    return (n - 32) // 16 + 1 if n >= 32 else 0


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _prepare_layer(case, seed):
    more = {"planted": {}, "unit": workloads.UNIT_SCALE, "none": {"topic_amp": 0.0}}[case["topics"]]
    # The topics are added with index_add_, whose order of sums must not vary between calls.
    before = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        c = workloads.hidden_space_layer(
            _lens(case), device=DEV, seed=seed, dtype=DTYPES[case["dtype"]], topk=case["budget"],
            local_blocks=case["local"], init_blocks=SINK, **more)
    finally:
        torch.use_deterministic_algorithms(before)
    state = dict(kind=case["kind"], case=c)
    if case["kind"] == "nosa":
        g = torch.Generator(device=DEV).manual_seed(seed + 7)
        state["cis"] = torch.randn(c.cu_host[-1], G, generator=g, device=DEV).to(c.q.dtype)
    return state


def _window_means(k):
    """Means of the 32-token windows at stride 16 of ``k [n, G, D]``."""
    if k.shape[0] < 32:
        return k.new_empty((0,) + tuple(k.shape[1:]))
    return k.float().unfold(0, 32, 16).mean(-1).to(k.dtype)


def _fill_sequences(lens, dtype, gen, k, v, kc):
    """Fills the caches: keys and values ~ N(0, 1), and in each sequence a share of the pages
    carries a direction that the returned vectors ``[B, G, D]`` point to (what a query of that
    sequence looks for)."""
    dirs = []
    for b, n in enumerate(lens):
        u = torch.randn(G, D, generator=gen, device=DEV)
        u = u / u.norm(dim=-1, keepdim=True)
        kk = torch.randn(n, G, D, generator=gen, device=DEV)
        hot = (torch.rand(-(-n // PAGE), generator=gen, device=DEV) < 0.03).float()
        kk += 3.0 * hot.repeat_interleave(PAGE)[:n, None, None] * u
        k[b, :n] = kk.to(dtype)
        v[b, :n] = torch.randn(n, G, D, generator=gen, device=DEV).to(dtype)
        kc[b, :_n_windows(n)] = _window_means(k[b, :n])
        dirs.append(u)
    return torch.stack(dirs)


def _prepare_decode(case, seed):
    lens, dtype = _lens(case), DTYPES[case["dtype"]]
    B = len(lens)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    cap = -(-(max(lens) + 1) // PAGE) * PAGE
    k = torch.zeros(B, cap, G, D, dtype=dtype, device=DEV)
    v = torch.zeros_like(k)
    kc = torch.zeros(B, _n_windows(cap), G, D, dtype=dtype, device=DEV)
    dirs = _fill_sequences(lens, dtype, gen, k, v, kc)
    q = torch.randn(B, G, GS, D, generator=gen, device=DEV) + 4.0 * dirs[:, :, None]
    after = [n + 1 for n in lens]
    cu = list(range(B + 1))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    return dict(kind="decode", plan=case["plan"], budget=case["budget"], local=case["local"], k=k,
                v=v, kc=kc, q=q.reshape(B, H, D).to(dtype),
                k_new=torch.randn(B, G, D, generator=gen, device=DEV).to(dtype),
                v_new=torch.randn(B, G, D, generator=gen, device=DEV).to(dtype), lens=lens,
                after=after, lens_t=i32(lens), after_t=i32(after), cu=cu, cu_t=i32(cu))


def _config(case):
    return minicpm.MiniCPMConfig(hidden_size=HIDDEN, num_hidden_layers=case.get("layers", 1),
                                 num_attention_heads=H, num_key_value_heads=G,
                                 intermediate_size=INTER, vocab_size=VOCAB, topk=case["budget"],
                                 init_blocks=SINK, local_blocks=case["local"])


def _prepare_block(case, seed):
    lens, dtype = _lens(case), DTYPES[case["dtype"]]
    B = len(lens)
    cfg = _config(case)
    cfg.intermediate_size, cfg.vocab_size = 64, 64  # the block uses neither the FFN nor the head
    model = minicpm.MiniCPMLeanSelect(cfg, device=DEV, dtype=dtype, seed=seed)
    gen = torch.Generator(device=DEV).manual_seed(seed + 1)
    cache = model.new_cache(B, max(lens) + 1)
    for t in (cache.k, cache.v, cache.kc):
        t.zero_()
    _fill_sequences(lens, dtype, gen, cache.k[0], cache.v[0], cache.kc[0])
    cache.lengths = list(lens)
    cache.seqlens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    cache.begin([1] * B)
    h = torch.randn(B, HIDDEN, generator=gen, device=DEV).to(dtype)
    cu = list(range(B + 1))
    model.rope_tables(max(lens) + 1)
    return dict(kind="block", model=model, cache=cache, h=h, lens=lens,
                pos=torch.tensor(lens, dtype=torch.int32, device=DEV), cu=cu,
                cu_t=torch.tensor(cu, dtype=torch.int32, device=DEV))


def _prepare_model(case, seed):
    lens = _lens(case)
    model = minicpm.MiniCPMLeanSelect(_config(case), device=DEV, dtype=DTYPES[case["dtype"]],
                                      seed=seed)
    gen = torch.Generator(device=DEV).manual_seed(seed + 1)
    ids = torch.randint(0, VOCAB, (sum(lens),), generator=gen, device=DEV, dtype=torch.int32)
    model.rope_tables(max(lens))
    return dict(kind="model", model=model, ids=ids, cu=_cu(lens))


def prepare(case, seed):
    make = {"layer": _prepare_layer, "nosa": _prepare_layer, "decode": _prepare_decode,
            "block": _prepare_block, "model": _prepare_model}
    with torch.no_grad():
        return make[case["kind"]](case, seed)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "layer":
        c = state["case"]
        out, ids = leanselect_sparse_prefill(
            c.q, c.k, c.v, c.cu_seqlens, c.selector, topk=c.topk, local_blocks=c.local_blocks,
            init_blocks=c.init_blocks, cu_seqlens_host=c.cu_host, return_topk_idx=True)
        return {"out": out, "topk_idx": ids}
    if kind == "nosa":
        c = state["case"]
        out, ids = nosa_sparse_prefill(
            c.q, c.k, c.v, state["cis"], c.cu_seqlens, c.selector, topk=c.topk,
            init_blocks=c.init_blocks, local_blocks=c.local_blocks, select_blocks=24,
            cu_seqlens_host=c.cu_host, return_topk_idx=True)
        return {"out": out, "topk_idx": ids}
    if kind == "decode":
        s = state
        if s["plan"] == "all":
            B = len(s["lens"])
            out = infllmv2_attn_with_kvcache(
                s["q"].view(B, 1, H, D), s["k"], s["v"], s["k_new"].view(B, 1, G, D),
                s["v_new"].view(B, 1, G, D), cache_seqlens=s["lens_t"], causal=True)
            return {"out": out, "k": s["k"], "v": s["v"]}
        kvcache_append(s["k"], s["v"], s["lens_t"], s["k_new"], s["v_new"], s["cu_t"],
                       kc_cache=s["kc"], cache_seqlens_host=s["lens"],
                       cu_seqlens_new_host=s["cu"])
        ids = decode_topk_idx(s["q"], s["kc"], s["after_t"], s["cu_t"], topk=s["budget"],
                              init_blocks=SINK, local_blocks=s["local"],
                              cache_seqlens_host=s["after"], cu_seqlens_q_host=s["cu"])
        out = sparse_attention_kvcache(s["q"], s["k"], s["v"], s["after_t"], ids, s["cu_t"])
        return {"out": out, "topk_idx": ids, "k": s["k"], "v": s["v"], "kc": s["kc"]}
    if kind == "block":
        c = state["cache"]
        o = state["model"].attention_decode(0, state["h"], state["pos"], c, state["cu_t"],
                                            state["cu"])
        return {"o": o, "k": c.k, "v": c.v, "kc": c.kc}
    seen = []
    logits = state["model"].prefill(state["ids"], state["cu"],
                                    layer_hook=lambda li, x: seen.append(x))
    return {"logits": logits, "hidden": seen[-1]}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _prefill_work(lens, budget, local, all_pages):
    """Operations of one prefill layer: attention over the budget, router projections, page scores."""
    n, keys, atoms, dots = sum(lens), 0, 0, 0
    for ln in lens:
        a = _n_windows(ln)
        atoms += a
        if a == 0:
            continue
        for qb in range(-(-ln // PAGE)):
            rows = min(PAGE, ln - PAGE * qb)
            pages = min(budget, qb + 1)
            # Whole pages but the row's own, of which row i sees i + 1 keys.
            keys += rows * (pages - 1) * PAGE + rows * (rows + 1) // 2
            if all_pages:
                dots += rows * a
            elif qb + 1 > budget:
                dots += rows * max(0, min(4 * (qb - local) - 1, a - 1) - (4 * SINK - 1) + 1)
    flops = 4.0 * D * H * keys + 2.0 * n * H * D * ROUTER + 2.0 * atoms * G * D * ROUTER
    return flops + 2.0 * G * ROUTER * dots


def work(case):
    lens = _lens(case)
    B, n = len(lens), sum(lens)
    if case["kind"] in ("layer", "nosa"):
        take = min(case["budget"], -(-max(lens) // PAGE))
        flops = _prefill_work(lens, case["budget"], case["local"], case["kind"] == "nosa")
        nbytes = 2 * (2 * n * H * D + 2 * n * G * D) + 4 * G * n * take
        return {"bytes": nbytes + (2 * n * G if case["kind"] == "nosa" else 0), "flops": flops}
    if case["kind"] == "model":
        flops = _prefill_work(lens, case["budget"], case["local"], False)
        weights = (H * D + 2 * G * D) * HIDDEN + H * D * HIDDEN + 3 * INTER * HIDDEN
        return {"bytes": (2 * (case["layers"] * weights + VOCAB * HIDDEN + 2 * n * HIDDEN)
                          + 4 * B * VOCAB),
                "flops": case["layers"] * (flops + 2.0 * n * weights) + 2.0 * B * VOCAB * HIDDEN}
    pages = [min(case["budget"] or 1 << 30, -(-(x + 1) // PAGE)) for x in lens]
    keys = sum(min(PAGE * p, x + 1) for p, x in zip(pages, lens))
    nbytes = 2 * (2 * G * D * keys + 2 * B * H * D + 4 * B * G * D)
    flops = 4.0 * D * H * keys
    if case.get("plan", "select") == "select":
        windows = sum(_n_windows(x + 1) for x in lens)
        nbytes += 2 * windows * G * D + 4 * G * B * case["budget"]
        flops += 2.0 * D * H * windows
    if case["kind"] == "block":
        weights = (H * D + 2 * G * D) * HIDDEN + H * D * HIDDEN
        nbytes += 2 * (weights + 2 * B * HIDDEN)
        flops += 2.0 * B * weights
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times the error against ``exact`` (the rounding of the 16-bit outputs).  A page at a
    budget's edge whose score ties within a rounding may be another one: that row's ids shift and
    single outputs of it move by their own size, so the largest difference says little where
    plans are formed."""
    half = case["dtype"] == "fp16"
    if case["kind"] in ("layer", "nosa"):
        return {"rel": 3e-3 if half else 8e-3, "max": 0.9, "differ": 5e-4}
    if case["kind"] == "decode":
        select = case["plan"] == "select"
        return {"rel": 1e-3 if half else 7e-3, "max": 0.5 if select else 0.02,
                "differ": 1e-2 if select else 0.0}
    if case["kind"] == "block":  # projections in 16 bits before and after
        return {"rel": 2e-3 if half else 1e-2, "max": 0.5}
    # Two whole layers: each layer's 16-bit roundings travel through what follows.
    return {"rel": 1e-2 if half else 3e-2, "max": 0.9}


# ---------------------------------------------------------------------------
# The same results in 64 bits (plain torch).  Where the path's contract is a 16-bit tensor (the
# router's folded weights, projections and scores, the stage-1 scores, the rotated projections)
# the 64-bit value is rounded to it; attention itself is 64 bits throughout.
# ---------------------------------------------------------------------------
def _order16(x):
    """bf16/fp16 values as integers that sort like them."""
    i = x.contiguous().view(torch.int16).to(torch.int64)
    return torch.where(i < 0, -(i & 0x7FFF), i)


def _top_pages(scores16, k):
    """The k best columns of each row (ties to the lower column)."""
    n = scores16.shape[-1]
    key = _order16(scores16) * 65536 + (n - 1 - torch.arange(n, device=scores16.device))
    return torch.topk(key, min(k, n), dim=-1).indices


def _attend(q, k, v, ids, limit, bias=None):
    """q [R, G, GS, D] over the pages ids [G, R, T] (-1: none) of k, v [n, G, D] (64 bits); row r
    sees the keys below limit[r]."""
    R, T = q.shape[0], ids.shape[2]
    out = torch.empty(R, G, GS, D, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 20) // max(1, T * PAGE))
    lane = torch.arange(PAGE, device=q.device)
    for g in range(G):
        kg, vg = k[:, g].contiguous(), v[:, g].contiguous()
        for r0 in range(0, R, step):
            i = ids[g, r0:r0 + step].long()
            j = (i[:, :, None] * PAGE + lane).reshape(i.shape[0], -1)
            seen = (i >= 0).repeat_interleave(PAGE, 1) & (j < limit[r0:r0 + step, None])
            j = j.clamp(0, k.shape[0] - 1)
            s = torch.matmul(q[r0:r0 + step, g].double(), kg[j].transpose(1, 2).contiguous())
            s = s / math.sqrt(D)
            if bias is not None:
                s = s + bias[:, g][j][:, None]
            s = s.masked_fill(~seen[:, None], float("-inf"))
            m = s.amax(-1, keepdim=True)
            p = torch.exp(s - torch.where(torch.isfinite(m), m, torch.zeros_like(m)))
            out[r0:r0 + step, g] = torch.matmul(p, vg[j]) / p.sum(-1, keepdim=True).clamp_min(1e-300)
    return out.reshape(R, H, D)


def _page_max(x):
    """Page maxima of atom columns x [R, A] (-inf padded): page p pools atoms 4p-1 .. 4p+3."""
    R, A = x.shape
    P = A // 4 + 1
    pad = x.new_full((R, 4 * P + 4), float("-inf"))
    pad[:, 1:A + 1] = x
    return pad[:, :4 * P + 1].unfold(1, 5, 4).amax(-1)


def _router(sel, dtype):
    """The folded router weights, [G, GS*D, F] and [G, D, F]."""
    qw = (sel.head_mix.float()[:, :, None, None] * sel.q_proj.float()[None]).to(dtype)
    kw = (sel.kv_head_mix.float()[:, :, None, None] * sel.k_proj.float()[None]).to(dtype)
    # [heads, R, D, RD] -> [heads, D, R*RD]
    qw = qw.permute(0, 2, 1, 3).reshape(G, GS * D, ROUTER).double()
    return qw, kw.permute(0, 2, 1, 3).reshape(G, D, ROUTER).double()


def _exact_layer_seq(q, k, v, sel, budget, local, take, cis=None, max_len=0):
    """One sequence of a prefill layer (cis given: the NOSA selection and bias)."""
    n, dtype, dev = q.shape[0], q.dtype, q.device
    A = _n_windows(n)
    if A == 0:
        return torch.zeros(n, H, D, dtype=torch.float64, device=dev)
    kc = (k.double().unfold(0, 32, 16).mean(-1)).to(dtype)
    qw, kw = _router(sel, dtype)
    kt = torch.stack([kc[:, g].double() @ kw[g] for g in range(G)]).to(dtype).double()
    n_pages = -(-n // PAGE)
    ids = torch.full((G, n, take), -1, dtype=torch.int32, device=dev)
    inf = float("inf")
    for g in range(G):
        for r0 in range(0, n, 4096):
            rows = torch.arange(r0, min(n, r0 + 4096), device=dev)
            qt = (q[rows, g * GS:(g + 1) * GS].reshape(rows.numel(), -1).double() @ qw[g]).to(dtype)
            pooled = _page_max((qt.double() @ kt[g].t()))  # rounding is monotone: round the maxima
            own = rows // PAGE
            if cis is None:
                cols = torch.arange(n_pages, device=dev)
                s = torch.full((rows.numel(), n_pages), -inf, dtype=torch.float64, device=dev)
                m = min(n_pages, pooled.shape[1])
                s[:, :m] = pooled[:, :m]
                forced = (cols < SINK) | ((cols >= own[:, None] - local) & (cols <= own[:, None]))
                s = s.masked_fill(forced, inf).masked_fill(cols > own[:, None], -inf)
                top = _top_pages(s.to(dtype), take)
                top = torch.where(top > own[:, None], torch.full_like(top, -1), top)
                ids[g, rows, :top.shape[1]] = top.int()
            else:
                cols = torch.arange(-(-max_len // PAGE), device=dev)
                q_idx = (rows + max_len - n) // PAGE
                forced = (cols < SINK) | ((cols >= own[:, None] - local) & (cols <= own[:, None]))
                m = min(cols.numel(), pooled.shape[1])
                s = torch.full((rows.numel(), cols.numel()), -inf, dtype=torch.float64, device=dev)
                s[:, :m] = pooled[:, :m]
                first = _top_pages(s.masked_fill(forced, inf).to(dtype), SINK + local + 24)
                c = cis[:, g].double()
                cp = _page_max(c.unfold(0, 32, 16).mean(-1).to(cis.dtype).double()[None])[0]
                s = torch.full((rows.numel(), cols.numel()), -inf, dtype=torch.float64, device=dev)
                s[:, :m] = cp[:m]
                s = s.masked_fill(cols > q_idx[:, None], -inf).masked_fill(forced, inf)
                s.scatter_(1, first, inf)
                top = _top_pages(s.to(cis.dtype), take)
                top = torch.where(top > q_idx[:, None], torch.full_like(top, -1), top)
                ids[g, rows, :top.shape[1]] = top.int()
    limit = torch.arange(1, n + 1, device=dev)
    return _attend(q.view(n, G, GS, D), k.double(), v.double(), ids, limit,
                   None if cis is None else cis.double())


def _exact_layer(q, k, v, cu, sel, budget, local, cis=None):
    max_len = max(b - a for a, b in zip(cu, cu[1:]))
    take = min(budget, -(-max_len // PAGE))
    return torch.cat([
        _exact_layer_seq(q[a:b], k[a:b], v[a:b], sel, budget, local, take,
                         None if cis is None else cis[a:b], max_len)
        for a, b in zip(cu, cu[1:])])


def _exact_decode_rows(q, k, v, kc, after, budget, local):
    """Decode attention [B, H, D] of q [B, H, D] over caches that hold `after` tokens."""
    outs = []
    for b, n in enumerate(after):
        n_pages = -(-n // PAGE)
        take = min(budget, n_pages) if budget else n_pages
        ids = torch.arange(n_pages, device=q.device).expand(G, 1, n_pages)
        if take < n_pages:
            own = (n - 1) // PAGE
            cols = torch.arange(n_pages, device=q.device)
            forced = (cols < SINK) | ((cols >= own - local) & (cols <= own))
            plan = []
            for g in range(G):
                x = q[b].view(G, GS, D)[g].double() @ kc[b, :_n_windows(n), g].double().t()
                p = torch.softmax(x / math.sqrt(D), -1).sum(0).to(q.dtype).to(torch.bfloat16)
                s = torch.full((1, n_pages), float("-inf"), dtype=torch.float64, device=q.device)
                pm = _page_max(p.double()[None])
                m = min(n_pages, pm.shape[1])
                s[:, :m] = pm[:, :m]
                plan.append(_top_pages(s.masked_fill(forced, float("inf")).to(torch.bfloat16), take))
            ids = torch.stack(plan)
        outs.append(_attend(q[b:b + 1].view(1, G, GS, D), k[b, :n].double(), v[b, :n].double(),
                            ids, torch.tensor([n], device=q.device)))
    return torch.cat(outs)


def _rope(x, pos, cos, sin):
    """x [n, heads, D] 16-bit rotated at pos, products and sum in 32 bits."""
    f = x.float()
    half = torch.cat((-f[..., D // 2:], f[..., :D // 2]), -1)
    return (f * cos[pos][:, None] + half * sin[pos][:, None]).to(x.dtype)


def _norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _exact_block(st):
    m, cache, lens = st["model"], st["cache"], st["lens"]
    L = m.layers[0]
    qkv = (st["h"].double() @ L.w_qkv.double().t()).to(st["h"].dtype)
    pos = st["pos"].long()
    cos, sin = m.rope_tables(max(lens) + 1)
    q = _rope(qkv[:, :H * D].view(-1, H, D), pos, cos, sin)
    k1 = _rope(qkv[:, H * D:(H + G) * D].view(-1, G, D), pos, cos, sin)
    k, v, kc = cache.k[0].clone(), cache.v[0].clone(), cache.kc[0].clone()
    for b, n in enumerate(lens):
        k[b, n], v[b, n] = k1[b], qkv[b, (H + G) * D:].view(G, D)
        kc[b, :_n_windows(n + 1)] = _window_means(k[b, :n + 1])
    out = _exact_decode_rows(q, k, v, kc, [n + 1 for n in lens], m.cfg.topk, m.cfg.local_blocks)
    return out.reshape(len(lens), H * D) @ L.w_o.double().t()


def _exact_model(st):
    m, cu = st["model"], st["cu"]
    cfg, dtype = m.cfg, m.dtype
    lens = [b - a for a, b in zip(cu, cu[1:])]
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    cos, sin = m.rope_tables(max(lens))
    x = m.embed[st["ids"].long()].double() * cfg.scale_emb
    c = cfg.scale_depth / math.sqrt(cfg.num_hidden_layers)
    for L in m.layers:
        h = _norm(x, L.input_norm, cfg.rms_norm_eps)
        qkv = (h @ L.w_qkv.double().t()).to(dtype)
        q = _rope(qkv[:, :H * D].view(-1, H, D), pos, cos, sin)
        k = _rope(qkv[:, H * D:(H + G) * D].view(-1, G, D), pos, cos, sin)
        v = qkv[:, (H + G) * D:].view(-1, G, D)
        a = _exact_layer(q, k, v, cu, L.selector, cfg.topk, cfg.local_blocks)
        x = x + c * (a.reshape(-1, H * D) @ L.w_o.double().t())
        h = _norm(x, L.post_norm, cfg.rms_norm_eps)
        gu = h @ L.w_gate_up.double().t()
        act = torch.nn.functional.silu(gu[:, :INTER]) * gu[:, INTER:]
        x = x + c * (act @ L.w_down.double().t())
    last = torch.tensor([b - 1 for b in cu[1:]], device=DEV)
    h = _norm(x[last], m.final_norm, cfg.rms_norm_eps) / (cfg.hidden_size / cfg.dim_model_base)
    return {"logits": h @ m.lm_head.double().t(), "hidden": x}


@torch.no_grad()
def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind in ("layer", "nosa"):
        c = st["case"]
        return {"out": _exact_layer(c.q, c.k, c.v, c.cu_host, c.selector, c.topk, c.local_blocks,
                                    st.get("cis")), "topk_idx": None}
    if kind == "decode":
        for b, n in enumerate(st["lens"]):
            st["k"][b, n], st["v"][b, n] = st["k_new"][b], st["v_new"][b]
            if case["plan"] == "select":
                st["kc"][b, :_n_windows(n + 1)] = _window_means(st["k"][b, :n + 1])
        out = _exact_decode_rows(st["q"], st["k"], st["v"], st["kc"], st["after"], case["budget"],
                                 case["local"])
        if case["plan"] == "all":
            return {"out": out[:, None], "k": None, "v": None}
        return {"out": out, "topk_idx": None, "k": None, "v": None, "kc": None}
    if kind == "block":
        return {"o": _exact_block(st), "k": None, "v": None, "kc": None}
    return _exact_model(st)
