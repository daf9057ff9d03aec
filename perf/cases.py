"""Workloads of the OMMX KV-cache path that performance work is measured on.

Three kinds of call, each through the entry point a program uses:

* ``decode``    one attention layer of one decode step over packed planes
                (``ommx_paged_decode_attention_canonical``);
* ``store``     a prompt's K/V rows quantized into planes, either as a block of its own
                (``ommx_pack_kv_canonical_block``) or into a request slot of a pool
                (``MultiSeqKVPool.append_block``);
* ``generate``  requests served through the attention-backend classes: one full-prefill step and
                then one-token steps, ``build`` -> per layer ``do_kv_cache_update`` -> ``forward``.

``listed()`` holds the fixed cases, ``draw(rng)`` gives further ones of the same ranges.
"""
import math
import os
from types import SimpleNamespace

import torch

from open_ommx_serve_amd.attention import MultiSeqKVPool, WindowSpec
from open_ommx_serve_amd.attention.pack import alloc_planes, ommx_pack_kv_canonical_block, store_pack_into
from open_ommx_serve_amd.attention.paged_decode import ommx_paged_decode_attention_canonical
from open_ommx_serve_amd.integration.vllm import backend

DEV = "cuda"
PAGE = 16

# The recipes a cache is packed with: the serving default, the same with position streams, and the
# two longer-group recipes ("low-bit lever": base-shared outliers; "paper-kv": 10 outliers of 128).
RECIPES = {
    "bitmap": dict(outlier_repr="bitmap", outliers_per_vector=6, group_tokens=32, group_channels=32,
                   kv_outlier_map=True),
    "relidx7": dict(outlier_repr="relidx7", outliers_per_vector=6, group_tokens=32, group_channels=32,
                    kv_outlier_map=True),
    "lever": dict(outlier_repr="relidx7", outliers_per_vector=6, group_tokens=64, group_channels=64,
                  kv_outlier_map=False),
    "paper-kv": dict(outlier_repr="relidx7", outliers_per_vector=10, group_tokens=128, group_channels=128,
                     kv_outlier_map=True),
}

# Attention shapes (q heads, kv heads, head_dim): the 8B layer, the 70B layer, one of two and one of
# eight tensor-parallel shards of them, and a 64-channel layer.
SHAPES = ((32, 8, 128), (64, 8, 128), (16, 4, 128), (8, 1, 128), (32, 8, 64))


def listed():
    def case(name, kind, shape, **kw):
        q_heads, kv_heads, head_dim = shape
        return dict(name=name, kind=kind, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, **kw)

    b8, b70 = SHAPES[0], SHAPES[1]
    return [
        # one short chat turn: launch latency and host time are everything
        case("decode-1k", "decode", b8, batch=1, ctx_min=1024, ctx_max=1024, recipe="bitmap"),
        # one long document, the headline benchmark step
        case("decode-64k", "decode", b8, batch=1, ctx_min=65536, ctx_max=65536, recipe="bitmap"),
        # a serving batch of requests of very different length
        case("decode-ragged-b32", "decode", b8, batch=32, ctx_min=1024, ctx_max=16384, recipe="bitmap"),
        # eight long requests on the wide-GQA layer: the largest decode step
        case("decode-gqa8-b8-32k", "decode", b70, batch=8, ctx_min=32768, ctx_max=32768, recipe="bitmap"),
        # one of eight tensor-parallel shards (a single kv head), position-stream planes, odd lengths
        case("decode-shard-b3", "decode", SHAPES[3], batch=3, ctx_min=701, ctx_max=9001, recipe="relidx7"),
        # 64-channel heads, two requests of odd length
        case("decode-d64-b2", "decode", SHAPES[4], batch=2, ctx_min=12345, ctx_max=12345, recipe="bitmap"),
        # the lowest-bit recipe: long groups, ten outliers
        case("decode-paper-b4", "decode", b8, batch=4, ctx_min=2003, ctx_max=20011, recipe="paper-kv"),
        # a 4096-token block packed on its own
        case("store-4k", "store", b8, tokens=4096, into="block", recipe="bitmap"),
        # a long prompt quantized into its pool slot
        case("store-pool-32k", "store", b8, tokens=32768, into="pool", recipe="bitmap"),
        # a block in a longer-group recipe
        case("store-lever-8k", "store", b8, tokens=8128, into="block", recipe="lever"),
        # time to the second token of one long prompt
        case("prompt-4k", "generate", b8, batch=1, prompt_min=4096, prompt_max=4096, new_tokens=1, layers=1),
        # a batch of short prompts answered with 40 tokens each, group boundaries on the way
        case("generate-b8", "generate", b8, batch=8, prompt_min=97, prompt_max=701, new_tokens=40, layers=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "store", "store", "generate", "generate"))
    if kind == "generate":
        q_heads, kv_heads, head_dim = SHAPES[rng.choice((0, 0, 2, 3))]
        batch, layers = _log_int(rng, 1, 16), rng.randint(1, 2)
        top = _log_int(rng, 33, int(4096 / math.sqrt(batch * layers)))
        low = top if batch == 1 else max(17, int(top * rng.uniform(0.2, 1.0)))
        # no more tokens than the listed batch of eight takes, in steps and in planes read
        new = _log_int(rng, 1, max(1, min(80 // layers, 250000 // (batch * layers * top))))
        return dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, batch=batch,
                    prompt_min=low, prompt_max=top, new_tokens=new, layers=layers)
    recipe = rng.choice(("bitmap", "bitmap", "bitmap", "relidx7", "lever", "paper-kv"))
    q_heads, kv_heads, head_dim = SHAPES[rng.choice((0, 0, 1, 2, 3, 4))]
    if kind == "store":
        unit = RECIPES[recipe]["group_tokens"]
        into = rng.choice(("block", "pool"))
        tokens = _log_int(rng, 160, 32768)
        if into == "block":
            tokens = max(unit, tokens // unit * unit)
        return dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, tokens=tokens,
                    into=into, recipe=recipe)
    batch = _log_int(rng, 1, 48)
    top = _log_int(rng, 300, min(65536, 262144 // batch))
    low = top if batch == 1 or rng.random() < 0.3 else max(100, int(top * rng.uniform(0.05, 0.9)))
    return dict(kind=kind, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, batch=batch,
                ctx_min=low, ctx_max=top, recipe=recipe)


# ── geometry ─────────────────────────────────────────────────────────────────────────────────

def _spread(lo, hi, n):
    """``n`` lengths from ``lo`` to ``hi`` in scattered order, both ends among them."""
    return [lo + round((hi - lo) * ((i * 5) % n if math.gcd(5, n) == 1 else i) / max(1, n - 1)) for i in range(n)]


def _recipe(case):
    r = dict(RECIPES[case["recipe"]])
    r["group_channels"] = min(r["group_channels"], case["head_dim"])
    return r


def _window(recipe):
    return WindowSpec(page_size=PAGE, group_tokens=recipe["group_tokens"])


def _packed_bytes(recipe, head_dim, tokens):
    """Plane bytes of ``tokens`` packed tokens of one kv head."""
    gt, gc, k = recipe["group_tokens"], recipe["group_channels"], recipe["outliers_per_vector"]
    index = gt // 8 if recipe["outlier_repr"] == "bitmap" else (7 * k + 7) // 8
    per_vector = 1 + 2 + index + (k + 1) // 2 + (4 if recipe["kv_outlier_map"] else 0)
    return tokens * (head_dim // 2 + 3 * (head_dim // gc)) + tokens // gt * head_dim * per_vector


# ── inputs ───────────────────────────────────────────────────────────────────────────────────

def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV, dtype=torch.bfloat16)


def _kv(gen, tokens, kv_heads, head_dim):
    """bf16 K and V ~ N(0,1) with K's outliers: four fixed channels of every head x12 and 0.5 % of
    all elements x8."""
    K, V = _normal(gen, tokens, kv_heads, head_dim), _normal(gen, tokens, kv_heads, head_dim)
    loud = torch.rand(kv_heads, head_dim, generator=gen, device=DEV).argsort(-1) < 4
    K *= torch.where(loud, 12.0, 1.0).to(torch.bfloat16)
    K *= 1 + 7 * (torch.rand(K.shape, generator=gen, device=DEV, dtype=torch.float16) < 0.005).to(torch.bfloat16)
    return K, V


def _prepare_decode(case, gen):
    recipe = _recipe(case)
    win, gt = _window(recipe), recipe["group_tokens"]
    B, Hq, H, D = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"]
    lens = _spread(case["ctx_min"], case["ctx_max"], B)
    packed = [win.packed_len(n) for n in lens]
    pages, groups = max(gt // PAGE, sum(packed) // PAGE), max(1, sum(packed) // gt)
    planes = alloc_planes(pages, groups, H, D, page_size=PAGE, device=DEV,
                          outliers_per_vector=recipe["outliers_per_vector"], outlier_repr=recipe["outlier_repr"],
                          kv_outlier_map=recipe["kv_outlier_map"], group_tokens=gt,
                          group_channels=recipe["group_channels"])
    page_ids = torch.randperm(pages, generator=gen, device=DEV).to(torch.int32)
    group_ids = torch.randperm(groups, generator=gen, device=DEV).to(torch.int32)
    req_to_token = torch.zeros(B, max(1, max(packed) // PAGE), dtype=torch.int32, device=DEV)
    req_to_group = torch.zeros(B, max(1, max(packed) // gt), dtype=torch.int32, device=DEV)
    p0 = g0 = 0
    for b, n in enumerate(packed):
        if n == 0:
            continue
        K, V = _kv(gen, n, H, D)
        dst_pages, dst_groups = page_ids[p0:p0 + n // PAGE], group_ids[g0:g0 + n // gt]
        store_pack_into(K, V, planes, outliers_per_vector=recipe["outliers_per_vector"], page_size=PAGE,
                        dst_pages=dst_pages, dst_groups=dst_groups, outlier_repr=recipe["outlier_repr"],
                        group_tokens=gt, group_channels=recipe["group_channels"])
        req_to_token[b, :n // PAGE] = dst_pages
        req_to_group[b, :n // gt] = dst_groups
        p0, g0 = p0 + n // PAGE, g0 + n // gt
    T = win.max_tail_len()
    k_tail, v_tail = _kv(gen, B * T, H, D)
    o = torch.empty(B, Hq, D, dtype=torch.float32, device=DEV)
    lse = torch.empty(B, Hq, dtype=torch.float32, device=DEV)
    tails = [len(win.tail_indices(n)) for n in lens]
    args = (_normal(gen, B, Hq, D), planes["k_base"], planes["k_scale"], planes["k_zp"], planes["k_oidx"],
            planes["k_oval"], planes["v_main"], planes["v_scale"], planes["v_zp"],
            k_tail.view(B, T, H, D), v_tail.view(B, T, H, D),
            torch.tensor(tails, dtype=torch.int32, device=DEV), o, lse, req_to_token, req_to_group,
            torch.tensor(packed, dtype=torch.int32, device=DEV))
    kwargs = dict(sm_scale=D ** -0.5, page_size=PAGE, k_outliers_per_vector=recipe["outliers_per_vector"],
                  bitmap_read=recipe["outlier_repr"] == "bitmap", k_obmp=planes["k_obmp"],
                  k_fp4_mapscale=planes["k_fp4_mapscale"], k_fp4_mapcenter=planes["k_fp4_mapcenter"],
                  kv_outlier_map=recipe["kv_outlier_map"], kv_int8_scale=True,
                  max_seq_len=max(1, max(packed)), max_tail_len=T)
    return dict(kind="decode", args=args, kwargs=kwargs, out=(o, lse))


def _prepare_store(case, gen):
    recipe = _recipe(case)
    H, D, T = case["kv_heads"], case["head_dim"], case["tokens"]
    K, V = _kv(gen, T, H, D)
    how = dict(outliers_per_vector=recipe["outliers_per_vector"], outlier_repr=recipe["outlier_repr"],
               outlier_select="signed", use_pow2=True, kv_outlier_map=recipe["kv_outlier_map"],
               group_channels=recipe["group_channels"])
    if case["into"] == "pool":
        pool = MultiSeqKVPool(D, H, 1, T, window=_window(recipe), device=DEV, kv_ring=True, **how)
        return dict(kind="pool", K=K, V=V, pool=pool)
    return dict(kind="block", K=K, V=V, how=dict(how, page_size=PAGE, device=DEV,
                                                 group_tokens=recipe["group_tokens"]))


_engine_now = (None, None)


def _engine(case):
    """The worker of a serving process: one set of layers, kept while the model and its limits stay
    the same, whatever requests come."""
    global _engine_now
    key = tuple(case[k] for k in ("q_heads", "kv_heads", "head_dim", "batch", "prompt_max", "new_tokens", "layers"))
    if _engine_now[0] != key:
        os.environ["OMMX_ATTN_MAXCTX"] = str(case["prompt_max"] + case["new_tokens"])
        backend.reset_worker_state(graph=False, batched=case["batch"] > 1, batched_graph=False,
                                   max_num_seqs=case["batch"])
        D = case["head_dim"]
        _engine_now = (key, SimpleNamespace(
            builder=backend.OMMXCanonicalMetadataBuilder(),
            layers=[SimpleNamespace() for _ in range(case["layers"])],
            impls=[backend.OMMXCanonicalImpl(case["q_heads"], D, D ** -0.5, case["kv_heads"])
                   for _ in range(case["layers"])]))
    return _engine_now[1]


def _prepare_generate(case, gen, seed):
    B, Hq, H, D = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"]
    lens = _spread(case["prompt_min"], case["prompt_max"], B)
    table = torch.tensor([[1 + (seed % 1000003) * 64 + b, 0] for b in range(B)], dtype=torch.int64)
    steps = []
    for s in range(1 + case["new_tokens"]):
        counts = lens if s == 0 else [1] * B
        starts = [0]
        for c in counts:
            starts.append(starts[-1] + c)
        meta = SimpleNamespace(seq_lens_cpu=torch.tensor([n + s for n in lens], dtype=torch.int32),
                               query_start_loc_cpu=torch.tensor(starts, dtype=torch.int32),
                               block_table_tensor=table)
        rows = []
        for _ in range(case["layers"]):
            K, V = _kv(gen, starts[-1], H, D)
            q = _normal(gen, starts[-1], Hq, D)
            rows.append((q, K, V, torch.empty_like(q)))
        steps.append((meta, rows))
    prompt_out = [r[3] for r in steps[0][1]]
    token_out = [torch.empty(case["new_tokens"], B, Hq, D, dtype=torch.bfloat16, device=DEV)
                 for _ in range(case["layers"])]
    for s in range(case["new_tokens"]):
        steps[1 + s] = (steps[1 + s][0], [(q, K, V, token_out[i][s])
                                          for i, (q, K, V, _) in enumerate(steps[1 + s][1])])
    return dict(kind="generate", engine=_engine(case), steps=steps, out=prompt_out + token_out)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    if case["kind"] == "decode":
        return _prepare_decode(case, gen)
    if case["kind"] == "store":
        return _prepare_store(case, gen)
    return _prepare_generate(case, gen, int(seed))


# ── the calls ────────────────────────────────────────────────────────────────────────────────

def run(state):
    kind = state["kind"]
    if kind == "decode":
        ommx_paged_decode_attention_canonical(*state["args"], **state["kwargs"])
        return state["out"]
    if kind == "block":
        planes = ommx_pack_kv_canonical_block(state["K"], state["V"], **state["how"])
        return {k: v for k, v in planes.items() if torch.is_tensor(v)}
    if kind == "pool":
        pool = state["pool"]
        pool.reset_slot(0)
        pool.append_block(0, state["K"], state["V"])
        planes = {k: v for k, v in pool.pool_planes().items() if torch.is_tensor(v)}
        return dict(planes, k_hist=pool.k_hist, v_hist=pool.v_hist)
    engine = state["engine"]
    for meta, rows in state["steps"]:
        engine.builder.build(0, meta)
        for layer, impl, (q, K, V, out) in zip(engine.layers, engine.impls, rows):
            impl.do_kv_cache_update(layer, K, V)
            impl.forward(layer, q, K, V, None, meta, out)
    return state["out"]


# ── what a pass cannot do without ────────────────────────────────────────────────────────────

def _decode_work(recipe, lens, q_heads, kv_heads, head_dim):
    win = _window(recipe)
    nbytes = flops = 0
    for n in lens:
        packed, tail = win.packed_len(n), len(win.tail_indices(n))
        nbytes += kv_heads * (_packed_bytes(recipe, head_dim, packed) + tail * head_dim * 4)
        nbytes += q_heads * (head_dim * 6 + 4) + 4 * (packed // PAGE + packed // recipe["group_tokens"])
        flops += 4 * q_heads * head_dim * (packed + tail)
    return nbytes, flops


def work(case):
    Hq, H, D = case["q_heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "decode":
        lens = _spread(case["ctx_min"], case["ctx_max"], case["batch"])
        nbytes, flops = _decode_work(_recipe(case), lens, Hq, H, D)
        return {"bytes": nbytes, "flops": flops}
    if case["kind"] == "store":
        recipe, T = _recipe(case), case["tokens"]
        packed = T if case["into"] == "block" else _window(recipe).packed_len(T)
        kept = 0 if case["into"] == "block" else min(T, recipe["group_tokens"] * 2 + 40)
        return {"bytes": H * (T * D * 4 + _packed_bytes(recipe, D, packed) + kept * D * 4), "flops": 0}
    recipe = RECIPES["bitmap"]
    win = _window(recipe)
    lens = _spread(case["prompt_min"], case["prompt_max"], case["batch"])
    nbytes = flops = 0
    for n in lens:
        # the prompt: q, K, V read, the output, the row history and the planes written
        nbytes += n * D * (4 * Hq + 8 * H) + H * _packed_bytes(recipe, D, win.packed_len(n))
        flops += 2 * Hq * D * n * (n + 1)
    for s in range(1, 1 + case["new_tokens"]):
        b, f = _decode_work(recipe, [n + s for n in lens], Hq, H, D)
        nbytes, flops = nbytes + b + case["batch"] * D * 8 * H, flops + f
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    if case["kind"] == "store":
        return "exact"                     # codes, exponents, positions and bf16 side planes
    if case["kind"] == "decode":
        return {"rel": 2e-3}               # fp32 results of f16 softmax weights and operands
    return {"rel": 1e-2}                   # bf16 results
