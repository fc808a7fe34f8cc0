"""The workloads this library's speed is measured on.

A case is a dict of plain values; ``prepare`` makes what a user's program has in hand (weights, page
tables, caches, inputs) from a seed, ``run`` is one pass through the public entry points.  Six kinds:

* ``step``    the attention path of one decode step of one sequence, through ``InferenceController``
              and the operators a model's attention layers call: selection layers (full attention,
              logits, top-k) at layers 0 and 2, sparse attention over the persisted tokens elsewhere,
              RoPE and the cache append of the new token inside each layer;
* ``batch``   the same for several sequences of different lengths in lock step
              (``BatchInferenceController``);
* ``select``  the top-k alone, from logits whose values are given: every row of every sequence;
* ``prompt``  one layer's attention over new prompt tokens: RoPE, append, causal attention; a fresh
              prompt (``past`` = 0) or a further turn on top of a cached conversation;
* ``prefill`` a decoder's whole forward over a prompt (``TidalLlama.prefill``);
* ``token``   one decode step of a whole decoder (``TidalLlama.decode_step``).

Values are N(0, 1) as a normalised model has them, pages are scattered over the pool, contexts are
rarely multiples of anything.
"""
import math

import numpy as np
import torch

from tidaldecode_amd import _kernels
from tidaldecode_amd import utils as ops
from tidaldecode_amd.llama import TidalLlama, TidalLlamaConfig
from tidaldecode_amd.utils import BatchInferenceController, InferenceController

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
_DEV = "cuda:0"
_SELECT_AT = (0, 2)   # selection layers of the attention-path cases
_GROW = 4096          # tokens a `token` case has room to grow by: every pass appends one


def listed():
    step = dict(kind="step", head_dim=128, page=16, layout="NHD", mode="per_head")
    return [
        # an assistant's short context with the page size of the reference: launches are all there is
        dict(step, name="step short", layers=4, heads=32, kv_heads=32, page=1, ctx=777, budget=256, dtype="fp16"),
        # the benchmark's decode step: Llama-2-7B shape at 32K tokens, 2048 selected
        dict(step, name="step 7b 32k", layers=32, heads=32, kv_heads=32, ctx=32768, budget=2048, dtype="bf16"),
        # grouped-query decoder (Llama-3-8B shape) deep in a document, lists per KV head
        dict(step, name="step gqa 100k", layers=32, heads=32, kv_heads=8, ctx=102391, budget=4096, dtype="bf16",
             mode="group_sum"),
        # serving a ragged batch: the benchmark's eight sequences of 8K to 64K tokens, fp16
        dict(kind="batch", name="batch 8 ragged", layers=3, heads=32, kv_heads=32, head_dim=128, page=16, batch=8,
             lo=8192, hi=65536, budget=1024, dtype="fp16", mode="per_head"),
        # serving many short grouped-query chats
        dict(kind="batch", name="batch 16 chats", layers=8, heads=32, kv_heads=8, head_dim=128, page=16, batch=16,
             lo=500, hi=8192, budget=512, dtype="bf16", mode="per_head"),
        # token selection of that ragged batch by itself, and the exactness of it
        dict(kind="select", name="select 8 ragged", heads=32, batch=8, lo=14000, hi=63000, budget=1024, page=16,
             dtype="bf16"),
        # a short question as a fresh prompt
        dict(kind="prompt", name="prompt 300", heads=32, kv_heads=8, head_dim=128, page=16, past=0, n=300,
             dtype="bf16", layout="NHD"),
        # the next turn of a long conversation
        dict(kind="prompt", name="prompt turn at 32k", heads=32, kv_heads=32, head_dim=128, page=16, past=32768,
             n=500, dtype="bf16", layout="NHD"),
        # a whole document as a prompt, the benchmark's prefill layer
        dict(kind="prompt", name="prompt 32k", heads=32, kv_heads=32, head_dim=128, page=16, past=0, n=32768,
             dtype="bf16", layout="NHD"),
        # a decoder's prefill (time to the first token), a quarter of the 7B shape's layers
        dict(kind="prefill", name="prefill 7b", shape="llama2_7b", layers=8, n=2900),
        # the next token of the 7B decoder at 32K tokens
        dict(kind="token", name="token 7b 32k", shape="llama2_7b", attn="tidal", layers=32, ctx=32768, budget=2048),
        # the same with the page-estimate attention that TidalDecode is compared with
        dict(kind="token", name="token quest 10k", shape="llama2_7b", attn="quest", layers=16, ctx=10240, budget=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "batch", "select", "prompt", "prompt", "prompt", "prefill",
                       "token", "token"])
    if kind in ("step", "batch", "prompt"):
        heads, kv = rng.choice([(32, 32), (32, 8), (40, 40), (28, 4), (32, 8), (16, 16)])
        case = dict(kind=kind, heads=heads, kv_heads=kv, head_dim=rng.choice([128, 128, 128, 128, 64]),
                    page=rng.choice([1, 16, 16, 16, 32]), dtype=rng.choice(["bf16", "bf16", "fp16"]))
        mode = "per_head" if heads == kv else rng.choice(["per_head", "group_sum"])
        if kind == "step":
            ctx = _log(rng, 700, 102400)
            return dict(case, layers=rng.randint(4, 32), ctx=ctx, budget=min(_log(rng, 64, 4096), ctx), mode=mode,
                        layout=rng.choice(["NHD", "NHD", "HND"]))
        if kind == "batch":
            hi = _log(rng, 2000, 65536)
            return dict(case, layers=rng.randint(3, 8) if hi < 16384 else 3, batch=rng.randint(2, 16 if hi < 16384 else 8),
                        lo=max(1, int(hi * rng.uniform(0.05, 0.9))), hi=hi, budget=_log(rng, 64, 2048), mode=mode)
        past = rng.choice([0, _log(rng, 500, 65536)])
        n = _log(rng, 16, 32768) if past == 0 else _log(rng, 16, 4096)
        return dict(case, past=past, n=n, layout=rng.choice(["NHD", "NHD", "HND"]))
    if kind == "select":
        hi = _log(rng, 1000, 102400)
        return dict(kind=kind, heads=rng.choice([8, 32, 32, 40]), batch=rng.choice([1, 1, rng.randint(2, 8)]),
                    lo=max(1, int(hi * rng.uniform(0.2, 0.95))), hi=hi, budget=_log(rng, 64, 4096), page=16,
                    dtype=rng.choice(["bf16", "fp16"]))
    shape = rng.choice(["llama2_7b", "llama3_8b"])
    if kind == "prefill":
        return dict(kind=kind, shape=shape, layers=rng.randint(2, 8), n=_log(rng, 64, 4096))
    return dict(kind=kind, shape=shape, attn=rng.choice(["tidal", "tidal", "full", "quest"]), layers=rng.randint(8, 20),
                ctx=_log(rng, 4096, 65536), budget=_log(rng, 128, 4096))


# ---------------------------------------------------------------------------------------------
def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device=_DEV, dtype=torch.float32).to(dtype)


def _lengths(case, seed):
    # the set of lengths belongs to the case (every seed does the same work), their order to the seed
    r = np.random.RandomState(case["batch"] * 1000003 + case["hi"])
    lens = r.randint(case["lo"], case["hi"] + 1, case["batch"])
    lens[0] = case["hi"]
    return [int(x) for x in np.random.RandomState(seed).permutation(lens)]


def prepare(case, seed):
    g = torch.Generator(device=_DEV).manual_seed(seed)
    return {"step": _prepare_step, "batch": _prepare_batch, "select": _prepare_select, "prompt": _prepare_prompt,
            "prefill": _prepare_model, "token": _prepare_model}[case["kind"]](case, seed, g)


def run(state):
    return state["run"](state)


def _prepare_step(case, seed, g):
    dtype, heads, kv, d = _DTYPES[case["dtype"]], case["heads"], case["kv_heads"], case["head_dim"]
    c = InferenceController(case["layers"], heads, d, case["page"], case["budget"], case["ctx"] + 1, dtype,
                            torch.device(_DEV), num_kv_heads=kv, select_mode=case["mode"], kv_layout=case["layout"],
                            page_order_seed=seed)
    c.kv_cache.pool.buf.normal_(generator=g)
    c.prepare_metadata(case["ctx"])     # what is cached
    c.prepare_metadata(1)               # the token being decoded
    c.begin_forward(1)
    pos = c.kv_cache.seqlen - 1
    page = c.kv_cache.indicies[pos // c.page_size]
    i32 = dict(dtype=torch.int32, device=_DEV)
    return dict(run=_run_step, c=c, layers=case["layers"], d=d, page=page,
                positions=torch.tensor([pos], **i32),
                slot=torch.tensor([page * c.page_size + pos % c.page_size], **i32),
                q=_normal(g, (case["layers"], 1, heads, d), dtype), k=_normal(g, (case["layers"], 1, kv, d), dtype),
                v=_normal(g, (case["layers"], 1, kv, d), dtype))


def _run_step(s):
    c, out = s["c"], []
    cos, sin = _kernels.rope_table(s["positions"], s["d"])
    for layer in range(s["layers"]):
        fresh = (s["k"][layer], s["v"][layer], cos, sin, s["slot"])
        select = layer in _SELECT_AT
        pages = c.kv_indices_without_last if select else c.topk_dindices_buffer
        out.append(ops.decode_sparse_attn(s["q"][layer], c, layer, pages, select, fresh=fresh))
        if select:
            ops.decode_topk(c)
    # the page the new token went to, in every layer
    return dict(o=out, logits=c.qk_product, lse=c.lse, written=c.kv_cache.pool.buf[:, s["page"]])


def _prepare_batch(case, seed, g):
    dtype, heads, kv, d, b = (_DTYPES[case["dtype"]], case["heads"], case["kv_heads"], case["head_dim"], case["batch"])
    c = BatchInferenceController(case["layers"], heads, d, case["page"], case["budget"], case["hi"] + 1, b, dtype,
                                 torch.device(_DEV), num_kv_heads=kv, select_mode=case["mode"], page_order_seed=seed)
    c.pool.buf.normal_(generator=g)
    c.add_sequences(_lengths(case, seed))
    c.begin_step()                      # room for the tokens being decoded
    return dict(run=_run_batch, c=c, layers=case["layers"], q=_normal(g, (case["layers"], b, heads, d), dtype),
                k=_normal(g, (case["layers"], b, kv, d), dtype), v=_normal(g, (case["layers"], b, kv, d), dtype))


def _run_batch(s):
    c, out = s["c"], []
    cos, sin = c.rope_table()
    for layer in range(s["layers"]):
        q, k, v, fresh = s["q"][layer], s["k"][layer], s["v"][layer], None
        if c.fused_step_ok:
            fresh = (k, v, cos, sin)
        else:                           # pools of 4 GiB a layer and more
            q = q.clone()
            c.rope_append(q, k, v, layer)
        if layer in _SELECT_AT:
            out.append(c.attend_full(q, layer, output_qk_product=True, fresh=fresh))
            c.select()
        else:
            out.append(c.attend_sparse(q, layer, fresh=fresh))
    return dict(o=out, logits=c.qk_product, lse=c.lse)


def _prepare_select(case, seed, g):
    # one small KV head: the cache is not read, its page tables are
    c = BatchInferenceController(1, case["heads"], 64, case["page"], case["budget"], case["hi"], case["batch"],
                                 _DTYPES[case["dtype"]], torch.device(_DEV), num_kv_heads=1, page_order_seed=seed)
    lens = _lengths(case, seed)
    c.add_sequences(lens)
    rows = c.qk_product.view(case["batch"], case["heads"], -1)
    for b, n in enumerate(lens):        # logits as a selection layer leaves them, q.k / sqrt(D)
        rows[b, :, :n] = torch.randn((case["heads"], n), generator=g, device=_DEV)
        c.lse[b] = torch.logsumexp(rows[b, :, :n], dim=1)
    return dict(run=_run_select, c=c)


def _run_select(s):
    s["c"].select()
    return s["c"].topk_dindices_buffer


def _prepare_prompt(case, seed, g):
    dtype, heads, kv, d = _DTYPES[case["dtype"]], case["heads"], case["kv_heads"], case["head_dim"]
    past, n = case["past"], case["n"]
    c = InferenceController(1, heads, d, case["page"], 256, past + n, dtype, torch.device(_DEV), num_kv_heads=kv,
                            kv_layout=case["layout"], page_order_seed=seed)
    c.kv_cache.pool.buf.normal_(generator=g)
    if past:
        c.prepare_metadata(past)
    c.prepare_metadata(n)
    c.begin_forward(n)
    return dict(run=_run_prompt, c=c, past=past, q=_normal(g, (n, heads, d), dtype), k=_normal(g, (n, kv, d), dtype),
                v=_normal(g, (n, kv, d), dtype))


def _run_prompt(s):
    c, q, k, v = s["c"], s["q"], s["k"], s["v"]
    # in place, as a model does with its fresh projections (here the same tensors turn once more
    # with every pass)
    ops.apply_rope_in_place(q, k, s["past"])
    ops.append_kv(k, v, c, 0)
    return dict(o=ops.prefill_forward(q, c, 0), q=q, k=k, cache=c.kv_cache.buf_layer(0))


def _config(case):
    cfg = getattr(TidalLlamaConfig, case["shape"])(
        top_k=case.get("budget", 256), sparse_layer_start=0, correction_layer=2, attn_type=case.get("attn", "tidal"))
    cfg.num_layers = case["layers"]
    return cfg


def _prepare_model(case, seed, g):
    model = TidalLlama(_config(case), _DEV, seed=seed)
    if case["kind"] == "prefill":
        model.tidal_init(16, case["n"], page_order_seed=seed)
        model.iController.kv_cache.pool.buf.zero_()
        return dict(run=_run_prefill, model=model,
                    ids=torch.randint(0, model.config.vocab_size, (case["n"],), generator=g, device=_DEV))
    model.tidal_init(16, case["ctx"] + _GROW, page_order_seed=seed, with_metadata=case["attn"] == "quest")
    torch.manual_seed(seed)             # what synthetic_prefill fills the cache from
    model.synthetic_prefill(case["ctx"])
    return dict(run=_run_token, model=model,
                token=torch.randint(0, model.config.vocab_size, (1,), generator=g, device=_DEV))


def _run_prefill(s):
    model = s["model"]
    model.tidal_clear()
    return dict(logits=model.prefill(s["ids"]), cache=model.iController.kv_cache.pool.buf)


def _run_token(s):
    cache = s["model"].iController.kv_cache
    logits = s["model"].decode_step(s["token"])
    return dict(logits=logits, written=cache.pool.buf[:, cache.indicies[-1]])


# ---------------------------------------------------------------------------------------------
def _attention(case, lens, layers, n_select, el=2):
    """bytes and flops of `layers` decode-attention layers over sequences of `lens` tokens"""
    heads, kv, d = case["heads"], case["kv_heads"], case["head_dim"]
    rows = {"per_head": heads, "group_sum": kv, "head_sum": 1}[case["mode"]]
    full = sum(lens)
    few = sum(min(case["budget"], n) for n in lens)
    # a list per query head reads its own rows, however few KV heads there are (but no row twice)
    sparse_rows = sum(min(rows if rows > kv else kv, heads) * min(case["budget"], n) if rows <= kv
                      else min(heads * min(case["budget"], n), kv * n) for n in lens)
    per = 2 * len(lens) * (heads + kv) * d * el
    nbytes = n_select * (full * kv * d * 2 * el + full * heads * 4 * 2 + rows * few * 4 + per)
    nbytes += (layers - n_select) * (sparse_rows * d * 2 * el + rows * few * 4 + per)
    flops = 4 * heads * d * (n_select * full + (layers - n_select) * few)
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind in ("step", "batch"):
        lens = [case["ctx"] + 1] if kind == "step" else [n + 1 for n in _lengths(case, 0)]
        n_select = sum(1 for x in _SELECT_AT if x < case["layers"])
        nbytes, flops = _attention(case, lens, case["layers"], n_select)
        return {"bytes": nbytes, "flops": flops}
    if kind == "select":
        lens = _lengths(case, 0)
        return {"bytes": case["heads"] * sum(4 * n + 4 * min(n, case["budget"]) for n in lens), "flops": 0}
    if kind == "prompt":
        heads, kv, d, past, n = case["heads"], case["kv_heads"], case["head_dim"], case["past"], case["n"]
        # q and k turned in place, v read, the cache rows written and all of the cache read, o written
        nbytes = 2 * d * (2 * n * heads + 2 * n * kv + n * kv + 2 * n * kv + 2 * (past + n) * kv + n * heads)
        return {"bytes": nbytes, "flops": 4 * heads * d * (n * past + n * (n + 1) // 2)}
    cfg = _config(case)
    hid, heads, kv, d = cfg.hidden_size, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    layer_weights = hid * (heads + 2 * kv) * d + heads * d * hid + 3 * hid * cfg.intermediate_size
    head = hid * cfg.vocab_size
    weights = cfg.num_layers * layer_weights + head
    if kind == "prefill":
        n = case["n"]
        flops = 2 * (n * cfg.num_layers * layer_weights + head) + cfg.num_layers * 4 * heads * d * n * (n + 1) // 2
        return {"bytes": 2 * (weights + n * hid + cfg.num_layers * n * 2 * kv * d), "flops": flops}
    n = case["ctx"] + 1
    geo = dict(heads=heads, kv_heads=kv, head_dim=d, mode="per_head", budget=case["budget"])
    if case["attn"] == "tidal":
        nbytes, flops = _attention(geo, [n], cfg.num_layers, 2)
    elif case["attn"] == "full":
        nbytes, flops = _attention(geo, [n], cfg.num_layers, cfg.num_layers)
    else:
        nbytes, flops = _attention(geo, [n], cfg.num_layers, 2)
        nbytes += (cfg.num_layers - 2) * (n // 16) * kv * d * 2 * 2     # the page bounds
    return {"bytes": nbytes + 2 * weights, "flops": flops + 2 * weights}


def tolerance(case):
    if case["kind"] == "select":
        return "exact"
    if case["kind"] in ("prefill", "token"):
        # the roundings of many bf16 layers with random weights: the same decoder with its sums in
        # another order is 0.01 - 0.05 away
        return {"rel": 0.03, "max": 0.3}
    # against attention in 64 bits: 2.0e-3 - 2.3e-3 (largest 0.028) in bf16, 2.9e-4 (1.4e-3) in fp16
    return {"rel": 0.01, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 0.0012, "max": 0.02}
