"""Performance cases: the work a serving program has this package do, one pass at a time.

Five kinds, each called the way the engine calls it:

* ``step``    a whole captured decode step of a few layers (``LMBackend.decode_steps``), with the
              logits it computed: every small launch of a step at its real batch size;
* ``ffn``     the second half of a block and the norm after it (add + RMSNorm, SwiGLU FFN, add +
              RMSNorm), where a decode step spends its weight traffic;
* ``decode``  one layer's decode attention with the token's RoPE and KV append fused in: all pages
              of a row (a full layer) or the selected ones (a subset layer);
* ``plan``    the planner layer: full attention, page scores, page selection;
* ``prefill`` one layer's RoPE + KV append + causal attention of a prompt step, including steps in
              which a new prompt joins rows that are already decoding.

Shapes are the model shapes and benchmark configurations of this repository (Llama-3-8B, Qwen2.5-7B,
Qwen2.5-14B, DeepSeek-R1-Distill-Qwen-1.5B; contexts of 1 k to 64 k tokens, batches of 1 to 128 rows).
"""
import math
import random

import torch

from delta_amd import kernels as K
from delta_amd import ops
from delta_amd.backend import LMBackend
from delta_amd.model import ModelArgs

DEV = "cuda:0"
PAGE = 16
D = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
THETA = 500000.0
BIAS = 1e-7  # the selector's position bias


def listed():
    return [
        # A small batch at a long context (Qwen2.5-7B shape, 4 rows of 64 k tokens, 4096-token
        # budget): launches of a few microseconds each, streaming weights for 4 rows.
        {"name": "step_b4_64k", "kind": "step", "model": "Qwen2.5-7b", "layers": 4, "full": "0,1", "batch": 4,
         "ctx": 65536, "k": 256, "dtype": "bf16"},
        # The speed recipe's step (DeepSeek-R1-Distill-Qwen-1.5B shape, 64 rows, 64-page budget) with
        # two planner layers, mid-generation.
        {"name": "step_b64_8k", "kind": "step", "model": "DeepSeek-R1-Distill-Qwen-1.5B", "layers": 6,
         "full": "0,1,4", "batch": 64, "ctx": 8192, "k": 64, "dtype": "bf16"},
        # FFN of one interactive request, of a Llama-3-8B batch of 32 and of a Qwen2.5-14B batch of 128.
        {"name": "ffn_1", "kind": "ffn", "model": "llama-3-8b", "rows": 1, "dtype": "bf16"},
        {"name": "ffn_32", "kind": "ffn", "model": "llama-3-8b", "rows": 32, "dtype": "bf16"},
        {"name": "ffn_128", "kind": "ffn", "model": "Qwen2.5-14b", "rows": 128, "dtype": "bf16"},
        # Subset attention of 128 ragged rows (1 k - 32 k tokens), budget max(512, len / 8) tokens.
        {"name": "subset_b128", "kind": "decode", "batch": 128, "hq": 40, "hkv": 8, "lo": 1024, "hi": 32768,
         "min_tokens": 512, "divisor": 8, "lens": 0, "dtype": "bf16"},
        # Full attention of a full-cache layer, 32 rows of 8 k tokens.
        {"name": "full_b32", "kind": "decode", "batch": 32, "hq": 32, "hkv": 8, "lo": 8192, "hi": 8192,
         "min_tokens": 0, "divisor": 0, "lens": 0, "dtype": "fp16"},
        # The planner layer at a short uniform batch and at the ragged large one.
        {"name": "plan_b8_16k", "kind": "plan", "batch": 8, "hq": 32, "hkv": 8, "lo": 16384, "hi": 16384, "k": 128,
         "lens": 0, "dtype": "fp16"},
        {"name": "plan_b128", "kind": "plan", "batch": 128, "hq": 40, "hkv": 8, "lo": 1024, "hi": 32768, "k": 256,
         "lens": 0, "dtype": "bf16"},
        # One long prompt; several short ragged prompts; a prompt joining 31 decoding rows.
        {"name": "prefill_8k", "kind": "prefill", "hq": 32, "hkv": 8, "prompts": 1, "qlo": 8192, "qhi": 8192,
         "past": 0, "decoding": 0, "lo": 0, "hi": 0, "lens": 0, "dtype": "bf16"},
        {"name": "prefill_ragged", "kind": "prefill", "hq": 28, "hkv": 4, "prompts": 8, "qlo": 37, "qhi": 1500,
         "past": 0, "decoding": 0, "lo": 0, "hi": 0, "lens": 1, "dtype": "fp16"},
        {"name": "prefill_joins", "kind": "prefill", "hq": 32, "hkv": 8, "prompts": 1, "qlo": 777, "qhi": 777,
         "past": 0, "decoding": 31, "lo": 1024, "hi": 8192, "lens": 2, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (q heads, kv heads) of the model table: group sizes 4, 5, 6 and 7.
HEADS = [(32, 8), (40, 8), (12, 2), (28, 4)]


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "decode", "decode", "plan", "prefill", "prefill", "step"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "ffn":
        return {"kind": "ffn", "model": rng.choice(["llama-3-8b", "Qwen2.5-7b", "Qwen2.5-14b",
                                                    "DeepSeek-R1-Distill-Qwen-1.5B"]),
                "rows": _log(rng, 1, 128), "dtype": dtype}
    if kind == "step":
        batch = _log(rng, 1, 64)
        return {"kind": "step", "model": rng.choice(["Qwen2.5-7b", "DeepSeek-R1-Distill-Qwen-1.5B"]), "layers": 4,
                "full": "0,1", "batch": batch, "ctx": min(_log(rng, 2000, 65536), 262144 // batch),
                "k": rng.choice([32, 64, 100]), "dtype": "bf16"}
    hq, hkv = rng.choice(HEADS)
    if kind in ("decode", "plan"):
        batch = _log(rng, 1, 128)
        hi = min(_log(rng, 1024, 65536), 2000000 // (batch * hkv) * 4)
        lo = rng.choice([hi, max(64, hi // 8)])
        if kind == "plan":
            return {"kind": "plan", "batch": batch, "hq": hq, "hkv": hkv, "lo": lo, "hi": hi,
                    "k": max(1, min(rng.choice([32, 64, 128, 256]), hi // 32)), "lens": rng.randrange(1000),
                    "dtype": dtype}
        subset = rng.random() < 0.6
        return {"kind": "decode", "batch": batch, "hq": hq, "hkv": hkv, "lo": lo, "hi": hi,
                "min_tokens": rng.choice([512, 1024, 2048]) if subset else 0,
                "divisor": rng.choice([8, 16, 1 << 30]) if subset else 0, "lens": rng.randrange(1000),
                "dtype": dtype}
    qhi = _log(rng, 32, 4096)
    prompts = max(1, min(rng.choice([1, 2, 4, 8]), 8192 // qhi))
    return {"kind": "prefill", "hq": hq, "hkv": hkv, "prompts": prompts, "qlo": rng.choice([qhi, max(1, qhi // 8)]),
            "qhi": qhi, "past": rng.choice([0, 0, 1000]), "decoding": rng.choice([0, 0, 5, 30]),
            "lo": 500, "hi": _log(rng, 1000, 16384), "lens": rng.randrange(1000), "dtype": dtype}


# ------------------------------------------------------------------ row lengths (the case alone)
def _lens(rng, n, lo, hi):
    return [rng.randint(lo, hi) for _ in range(n)]


def _decode_lens(case):
    """Tokens of each row, the step's own token included."""
    return _lens(random.Random(case["lens"]), case["batch"], case["lo"], case["hi"])


def _budgets(case, lens):
    """Selected pages per row of a subset layer, or every page of a full one."""
    pages = [n // PAGE + 1 for n in lens]
    if not case["min_tokens"]:
        return pages
    return [min(p, max(1, max(case["min_tokens"], n // case["divisor"]) // PAGE)) for p, n in zip(pages, lens)]


def _prefill_rows(case):
    """(new tokens, tokens after the step) per row: the prompts, then the decoding rows."""
    rng = random.Random(case["lens"])
    q = _lens(rng, case["prompts"], case["qlo"], case["qhi"])
    rows = [(n, n + case["past"]) for n in q]
    return rows + [(1, n) for n in _lens(rng, case["decoding"], case["lo"], case["hi"])]


# ------------------------------------------------------------------ paged inputs
def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _pages(lens, seed):
    """Page tables of rows of ``lens`` tokens over a shuffled pool, in the scheduler's convention
    (a full page is followed by an empty one): (indptr, ids per row, last page lengths, total)."""
    counts = [n // PAGE + 1 for n in lens]
    total = sum(counts)
    perm = list(range(total))
    random.Random(seed).shuffle(perm)
    rows, at = [], 0
    for c in counts:
        rows.append(perm[at:at + c])
        at += c
    return counts, rows, [n % PAGE for n in lens], total


def _csr(rows):
    indptr = [0]
    for r in rows:
        indptr.append(indptr[-1] + len(r))
    return _i32(indptr), _i32([p for r in rows for p in r])


def _normal(shape, dtype, gen, std=1.0):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=gen)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _qkv(n, hq, hkv, dtype, gen):
    """q, k, v as the model hands them over: slices of one projection output."""
    x = _normal((n, (hq + 2 * hkv) * D), dtype, gen)
    q, k, v = x.split([hq * D, hkv * D, hkv * D], dim=-1)
    return q.view(n, hq, D), k.view(n, hkv, D), v.view(n, hkv, D)


# ------------------------------------------------------------------ engines
def _engine(model, layers, dtype, seed, batch, max_len, full=(), k=64, **shape):
    be = LMBackend(dtype=DTYPES[dtype], device=DEV, cuda_graph_decode=True)
    be.is_main_process = False
    be.load_model(f"random:{model}", n_layer=layers, seed=seed, **shape)
    gen = _gen(seed + 1)
    with torch.no_grad():  # norms and biases of a trained model are not ones and zeros
        for name, p in be.model.named_parameters():
            if name.endswith("norm.weight"):
                p.normal_(1.0, 0.1, generator=gen)
            elif name.endswith("bias"):
                p.normal_(0.0, 0.1, generator=gen)
    cfg = be.model.config
    cfg.enable_selective_cache = bool(full)
    cfg.full_cache_layers = list(full)
    cfg.subset_cache_size = k
    cfg.compression_ratio = 1.0
    cfg.L = 8
    be.setup_caches(max_batch_size=batch, max_seq_length=max_len)
    return be


def _full_layers(case):
    return [int(x) for x in case["full"].split(",")]


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    with torch.inference_mode():  # as the engine runs its steps
        return globals()["_run_" + state["kind"]](state)


def _prepare_step(case, seed):
    be = _engine(case["model"], case["layers"], case["dtype"], seed, case["batch"], case["ctx"] + 64,
                 full=_full_layers(case), k=case["k"])
    be.prepare_synthetic_decode(case["ctx"], decode_budget=32, seed=seed)
    st = {"kind": "step", "be": be, "tokens": be.static_tokens.clone(), "lens": be.cachelens.clone(),
          "ctx": case["ctx"]}
    finalize = be.model._finalize_logits

    def keep(logits):  # the program samples from the logits: the captured step leaves them here
        st["logits"] = logits
        return finalize(logits)

    be.model._finalize_logits = keep
    run(st)  # captures the step, as a server does before it takes requests
    return st


def _run_step(st):
    be = st["be"]
    ops.set_active_backend(be)
    be.static_tokens.copy_(st["tokens"])
    be.cachelens.copy_(st["lens"])
    be._host_lens = [st["ctx"]] * be.batch_size
    be.decode_steps(1)
    return {"logits": st["logits"], "kv": [layer.attention.kv_cache.kv_cache for layer in be.model.layers]}


def _prepare_ffn(case, seed):
    # One block of the engine, so the weights are laid out as the engine lays them out for this batch.
    be = _engine(case["model"], 1, case["dtype"], seed, case["rows"], 64, vocab_size=64)
    gen = _gen(seed + 2)
    dim = be.model.config.dim
    shape, dtype = (1, case["rows"], dim), DTYPES[case["dtype"]]
    return {"kind": "ffn", "be": be, "x": _normal(shape, dtype, gen), "attn": _normal(shape, dtype, gen, 0.3)}


def _run_ffn(st):
    model = st["be"].model
    blk = model.layers[0]
    h, y = K.add_rmsnorm(st["x"], st["attn"], blk.ffn_norm.weight, blk.ffn_norm.eps)
    f = blk.feed_forward.forward_fused(y)
    h, y = K.add_rmsnorm(h, f, model.norm.weight, model.norm.eps)
    return {"h": h, "y": y}


def _prepare_decode(case, seed):
    lens = _decode_lens(case)
    dtype, hq, hkv, B = DTYPES[case["dtype"]], case["hq"], case["hkv"], case["batch"]
    counts, rows, last, total = _pages(lens, seed)
    rng = random.Random(seed + 1)
    budgets = _budgets(case, lens)
    picked = []
    for r, c, k in zip(rows, counts, budgets):  # the last 8 pages, the rest anywhere, ascending
        tail = min(8, k)
        head = sorted(rng.sample(range(c - tail), k - tail))
        picked.append([r[j] for j in head] + r[c - tail:])
    gen = _gen(seed)
    kv = _normal((total, 2, PAGE, hkv, D), dtype, gen)
    q, k, v = _qkv(B, hq, hkv, dtype, gen)
    full_ptr, full_ids = _csr(rows)
    ptr, ids = _csr(picked)
    ap = K.DecodeAppend(k, v, _i32([n - 1 for n in lens]), full_ptr, full_ids, rope_theta=THETA)
    max_pages = max(budgets)
    return {"kind": "decode", "q": q, "kv": kv, "ptr": ptr, "ids": ids, "last": _i32(last), "ap": ap,
            "max_pages": max_pages, "subset": bool(case["min_tokens"]), "rows": picked, "full_rows": rows,
            "ws": torch.empty(max(256, K.decode_workspace_bytes(B, hq, hkv, max_pages)), dtype=torch.uint8,
                              device=DEV)}


def _run_decode(st):
    o = K.paged_decode(st["q"], st["kv"], st["ptr"], st["ids"], st["last"], max_pages_per_row=st["max_pages"],
                       workspace=st["ws"], subset=st["subset"], append=st["ap"])
    return {"o": o, "kv": st["kv"]}


def _prepare_plan(case, seed):
    lens = _decode_lens(case)
    dtype, hq, hkv, B = DTYPES[case["dtype"]], case["hq"], case["hkv"], case["batch"]
    counts, rows, last, total = _pages(lens, seed)
    gen = _gen(seed)
    kv = _normal((total, 2, PAGE, hkv, D), dtype, gen)
    q, k, v = _qkv(B, hq, hkv, dtype, gen)
    ptr, ids = _csr(rows)
    ap = K.DecodeAppend(k, v, _i32([n - 1 for n in lens]), ptr, ids, rope_theta=THETA)
    n = max(counts)
    table = torch.zeros((B, n), dtype=torch.int32)
    for b, r in enumerate(rows):
        table[b, :len(r)] = torch.tensor(r, dtype=torch.int32)
    on_chip = K.paged_decode_scores_supported(B, hq, hkv, n, True)
    ws = max(256, K.decode_workspace_bytes(B, hq, hkv, n), K.paged_decode_scores_workspace_bytes(B, hkv, n))
    return {"kind": "plan", "q": q, "kv": kv, "ptr": ptr, "ids": ids, "last": _i32(last), "ap": ap, "n": n,
            "k": case["k"], "table": table.to(DEV), "on_chip": on_chip, "rows": rows,
            "lse": torch.zeros((B, hq), dtype=torch.float32, device=DEV),
            "scores": torch.zeros((B, n), dtype=torch.float32, device=DEV),
            "dump": None if on_chip else torch.full((B, hq, n * PAGE), float("-inf"), device=DEV),
            "sel": torch.zeros(B * n, dtype=torch.int32, device=DEV),
            "sel_ptr": torch.zeros(B + 1, dtype=torch.int32, device=DEV),
            "ws": torch.empty(ws, dtype=torch.uint8, device=DEV)}


def _run_plan(st):
    common = dict(max_pages_per_row=st["n"], lse=st["lse"], workspace=st["ws"], append=st["ap"])
    if st["on_chip"]:
        o, _ = K.paged_decode_scores(st["q"], st["kv"], st["ptr"], st["ids"], st["last"], scores=st["scores"], **common)
    else:
        o = K.paged_decode(st["q"], st["kv"], st["ptr"], st["ids"], st["last"], logits_dump=st["dump"], **common)
        K.page_scores_from_logits(st["dump"], st["ptr"], st["last"], st["n"], lse=st["lse"], scores=st["scores"],
                                  workspace=st["ws"])
    K.select_pages(st["scores"], st["ptr"], st["table"], st["k"], 8, pos_bias_scale=BIAS, out_indices=st["sel"],
                   out_indptr=st["sel_ptr"])
    return {"o": o, "lse": st["lse"], "scores": st["scores"], "pages": st["sel"], "indptr": st["sel_ptr"]}


def _prepare_prefill(case, seed):
    rows_len = _prefill_rows(case)
    dtype, hq, hkv = DTYPES[case["dtype"]], case["hq"], case["hkv"]
    lens = [n for _, n in rows_len]
    _, rows, last, total = _pages(lens, seed)
    gen = _gen(seed)
    kv = _normal((total, 2, PAGE, hkv, D), dtype, gen)
    qo = [0]
    for n, _ in rows_len:
        qo.append(qo[-1] + n)
    q, k, v = _qkv(qo[-1], hq, hkv, dtype, gen)
    ptr, ids = _csr(rows)
    return {"kind": "prefill", "q": q, "k": k, "v": v, "kv": kv, "qo": _i32(qo), "ptr": ptr, "ids": ids,
            "last": _i32(last), "offsets": _i32([n - m for m, n in rows_len]), "max_qo": max(m for m, _ in rows_len),
            "rows": rows}


def _run_prefill(st):
    q = K.rope_append(st["q"], st["k"], st["v"], st["qo"], st["offsets"], st["kv"], st["ids"], st["ptr"], st["last"],
                      rope_theta=THETA)
    o = K.paged_prefill(q, st["kv"], st["qo"], st["ptr"], st["ids"], st["last"], max_qo_len=st["max_qo"])
    return {"o": o, "kv": st["kv"]}


# ------------------------------------------------------------------ work
def work(case):
    kind = case["kind"]
    if kind in ("step", "ffn"):
        cfg = ModelArgs.from_name(case["model"])
        dim, inter = cfg.dim, cfg.intermediate_size
        if kind == "ffn":
            n = case["rows"]
            return {"bytes": 2 * (3 * dim * inter + 4 * n * dim + 2 * dim), "flops": 6 * n * dim * inter}
        B, layers, full = case["batch"], case["layers"], _full_layers(case)
        weights = layers * (dim * (cfg.n_head + 2 * cfg.n_local_heads) * D + dim * dim + 3 * dim * inter)
        weights += dim * cfg.vocab_size
        n = case["ctx"] + 1
        sub = min(n, case["k"] * PAGE)
        tokens = B * sum(n if i in full else sub for i in range(layers))
        kv = tokens * cfg.n_local_heads * D * 2 * 2
        return {"bytes": 2 * weights + kv + 2 * B * cfg.vocab_size,
                "flops": 2 * B * weights + 4 * tokens * cfg.n_head * D}
    hq, hkv = case["hq"], case["hkv"]
    if kind == "prefill":
        rows = _prefill_rows(case)
        nnz = sum(m for m, _ in rows)
        pairs = sum(m * (n - m) + m * (m + 1) // 2 for m, n in rows)
        past = sum(n - m for m, n in rows)
        # q, k, v in, o out, the new K and V into the cache, the earlier ones out of it
        return {"bytes": 2 * D * (nnz * (2 * hq + 4 * hkv) + past * 2 * hkv), "flops": 4 * D * hq * pairs}
    lens = _decode_lens(case)
    B = case["batch"]
    if kind == "plan":
        n = max(lens) // PAGE + 1
        tokens, extra = sum(lens), 4 * (2 * B * n + B * case["k"] + B * hq)
    else:
        budgets = _budgets(case, lens)
        tokens = sum(min(n, (k - 1) * PAGE + n % PAGE) for n, k in zip(lens, budgets))
        extra = 4 * sum(budgets)
    return {"bytes": tokens * hkv * D * 2 * 2 + 2 * D * B * (2 * hq + 4 * hkv) + extra,
            "flops": 4 * tokens * hq * D}


def tolerance(case):
    """About four times what two correct orders of the same sums were measured to differ by: the
    projections on this package's kernels against fp32 products rounded once, the attention under
    another split plan or against fp64 from the same rotated queries."""
    bf16 = case["dtype"] == "bf16"
    kind = case["kind"]
    if kind == "step":  # measured 0.012 / 0.11: roundings travel through the layers and the selection
        return {"rel": 3e-2, "max": 0.45}
    if kind == "ffn":  # measured 6e-4 / 0.02 in bf16, 1.8e-4 / 0.0028 in fp16
        return {"rel": 2.5e-3, "max": 0.08} if bf16 else {"rel": 7e-4, "max": 0.011}
    # measured 2.6e-3 / 0.023 in bf16, 3.5e-4 / 0.0026 in fp16
    t = {"rel": 1e-2, "max": 0.09} if bf16 else {"rel": 1.4e-3, "max": 0.011}
    if kind == "plan":  # pages whose scores are equal to fp32 rounding
        t["differ"] = 5e-3
    return t


# ------------------------------------------------------------------ exact results in 64 bits
def exact(case, seed):
    with torch.no_grad():
        return globals()["_exact_" + case["kind"]](case, prepare(case, seed))


def _rope64(x, pos, theta, scale=1.0):
    """Interleaved RoPE of x [n, heads, 128] at positions pos [n]."""
    j = torch.arange(D // 2, dtype=torch.float64, device=x.device)
    ang = pos.double()[:, None] * (theta ** (-2.0 * j / D) / scale)
    cs, sn = ang.cos()[:, None], ang.sin()[:, None]
    x = x.double()
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cs - b * sn, b * cs + a * sn], dim=-1).flatten(-2)


def _row_kv(kv, pages, n):
    """K and V [n, hkv, 128] of a row's first n tokens, in 64 bits."""
    x = kv[torch.tensor(pages, device=DEV)].double()
    return tuple(x[:, i].reshape(-1, *x.shape[3:])[:n] for i in (0, 1))


def _attend64(q, k, v, causal_from=None):
    """q [m, hq, 128] over k, v [n, hkv, 128] -> (o, logits per head [hq, m, n], lse [hq, m])."""
    m, hq, _ = q.shape
    hkv = k.shape[1]
    qh = q.view(m, hkv, hq // hkv, D).permute(1, 2, 0, 3).reshape(hkv, -1, D)  # [hkv, G m, D]
    s = torch.matmul(qh, k.permute(1, 2, 0).contiguous()) / math.sqrt(D)
    s = s.view(hq, m, -1)
    if causal_from is not None:
        pos = causal_from + torch.arange(m, device=DEV)
        s = s.masked_fill(torch.arange(k.shape[0], device=DEV)[None] > pos[:, None], float("-inf"))
    lse = torch.logsumexp(s, dim=-1)
    p = (s - lse[..., None]).exp().view(hkv, -1, k.shape[0])
    o = torch.matmul(p, v.permute(1, 0, 2).contiguous()).view(hkv, hq // hkv, m, D)
    return o.permute(2, 0, 1, 3).reshape(m, hq, D), s, lse


def _exact_decode(case, st):
    lens = _decode_lens(case)
    ap = st["ap"]
    pos = torch.tensor([n - 1 for n in lens], device=DEV)
    q, k_new = _rope64(st["q"], pos, THETA), _rope64(ap.k, pos, THETA)
    out = []
    for b, n in enumerate(lens):
        pages = st["rows"][b]
        m = (len(pages) - 1) * PAGE + n % PAGE
        k, v = _row_kv(st["kv"], pages, m)
        k[m - 1], v[m - 1] = k_new[b], ap.v[b].double()
        out.append(_attend64(q[b:b + 1], k, v)[0])
    return {"o": torch.cat(out), "kv": None}


def _scores64(s, lse, n_pages):
    """Page scores of one row from its logits [hq, 1, n]: per token the largest head's probability."""
    p = (s - lse[..., None]).exp().amax(dim=0)[0]
    t = torch.zeros(n_pages * PAGE, dtype=torch.float64, device=DEV)
    t[:p.numel()] = p
    return t.view(n_pages, PAGE).sum(-1)


def _exact_plan(case, st):
    lens = _decode_lens(case)
    ap = st["ap"]
    pos = torch.tensor([n - 1 for n in lens], device=DEV)
    q, k_new = _rope64(st["q"], pos, THETA), _rope64(ap.k, pos, THETA)
    out, lses, scores = [], [], []
    for b, n in enumerate(lens):
        k, v = _row_kv(st["kv"], st["rows"][b], n)
        k[n - 1], v[n - 1] = k_new[b], ap.v[b].double()
        o, s, lse = _attend64(q[b:b + 1], k, v)
        out.append(o)
        lses.append(lse[:, 0])
        scores.append(_scores64(s, lse, st["n"]))
    return {"o": torch.cat(out), "lse": torch.stack(lses), "scores": torch.stack(scores), "pages": None,
            "indptr": None}


def _exact_prefill(case, st):
    rows_len = _prefill_rows(case)
    pos = torch.cat([torch.arange(n - m, n, device=DEV) for m, n in rows_len])
    q, k_new = _rope64(st["q"], pos, THETA), _rope64(st["k"], pos, THETA)
    out, at = [], 0
    for b, (m, n) in enumerate(rows_len):
        k, v = _row_kv(st["kv"], st["rows"][b], n)
        k[n - m:], v[n - m:] = k_new[at:at + m], st["v"][at:at + m].double()
        for c in range(0, m, 512):
            e = min(m, c + 512)
            out.append(_attend64(q[at + c:at + e], k[:n - m + e], v[:n - m + e], causal_from=n - m + c)[0])
        at += m
    return {"o": torch.cat(out), "kv": None}


def _norm64(x, norm):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + norm.eps) * norm.weight.double()


def _ffn64(ff, y):
    w13 = ff.w13 if hasattr(ff, "w13") else ff.w13_t.t()
    g, u = (y @ w13.double().t()).split(ff.inter, dim=-1)
    return (g * torch.sigmoid(g) * u) @ ff.w2.weight.double().t()


def _exact_ffn(case, st):
    model = st["be"].model
    blk = model.layers[0]
    h = st["x"].double() + st["attn"].double()
    h = h + _ffn64(blk.feed_forward, _norm64(h, blk.ffn_norm))
    return {"h": h, "y": _norm64(h, model.norm)}


def _exact_step(case, st):
    be = st["be"]
    model, cfg = be.model, be.model.config
    hq, hkv, n = cfg.n_head, cfg.n_local_heads, case["ctx"] + 1
    tp = n // PAGE + 1
    table = be.slot_block_table.tolist()
    pos = torch.full((case["batch"],), n - 1, device=DEV)
    full = _full_layers(case)
    x = model.tok_embeddings.weight[st["tokens"][0]].double()
    picked = None
    for i, blk in enumerate(model.layers):
        att = blk.attention
        qkv = _norm64(x, blk.attention_norm) @ att.wqkv.weight.double().t()
        if att.wqkv.bias is not None:
            qkv = qkv + att.wqkv.bias.double()
        q, k_new, v_new = qkv.split([hq * D, hkv * D, hkv * D], dim=-1)
        q = _rope64(q.reshape(-1, hq, D), pos, cfg.rope_base, cfg.scaling_factor)
        k_new = _rope64(k_new.reshape(-1, hkv, D), pos, cfg.rope_base, cfg.scaling_factor)
        v_new = v_new.reshape(-1, hkv, D)
        plans = i in full and i + 1 < case["layers"] and i + 1 not in full
        out, chosen = [], []
        for b in range(case["batch"]):
            pages = table[b][:tp] if i in full else picked[b]
            m = (len(pages) - 1) * PAGE + n % PAGE
            k, v = _row_kv(att.kv_cache.kv_cache, pages, m)
            k[m - 1], v[m - 1] = k_new[b], v_new[b]
            o, s, lse = _attend64(q[b:b + 1], k, v)
            out.append(o)
            if plans:
                key = _scores64(s, lse, tp) - torch.arange(tp, device=DEV).double() * BIAS
                key[tp - cfg.L:] = float("inf")
                top = key.topk(case["k"]).indices.sort().values.tolist()
                chosen.append([table[b][j] for j in top])
        if plans:
            picked = chosen
        x = x + torch.cat(out).reshape(case["batch"], -1) @ att.wo.weight.double().t()
        x = x + _ffn64(blk.feed_forward, _norm64(x, blk.ffn_norm))
    logits = _norm64(x, model.norm) @ model.output.weight.double().t()
    return {"logits": logits[None], "kv": [None] * case["layers"]}
