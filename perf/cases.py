"""Performance cases of the paged-KV framework, through its public entry points.

Six kinds of work, each over the range a serving engine meets it in:

* ``decode``   one layer's ``page16_decode_attention`` of a decode batch;
* ``step``     one decode step's attention of every layer, the token append fused in
               (``page16_decode_append_attention``);
* ``prefill``  one layer's ``chunked_prefill``: a chunk's K/V into its pages, then causal attention;
* ``scores``   ``score_layer_blocks``: SnapKV block scores of one layer from its dense K;
* ``final``    the last prefill chunk of a group of layers with SnapKV statistics, then
               ``score_blocks`` from them;
* ``compact``  retain-set selection and compaction into new pages (``select_blocks``,
               ``retained_pages``, ``compact``).

Head shapes are Llama-3-8B's (32 q heads, 8 KV heads, 128 dims), Qwen2.5-7B's (28, 4, 128), their
per-GPU shards and the 64-dim shape of smaller models. A case is a dict of plain values; sequence
lengths follow from its ``mix`` (the generator's seed for the layout), so that ``work`` knows them,
and the values and page placements from ``prepare``'s seed.
"""
import math

import numpy as np
import torch

from unifiedkv_amd import compaction, page16_native, prefill, snapkv
from unifiedkv_amd.pool import PagedKVPool

PAGE = 16
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


# ------------------------------------------------------------------------------------- cases
def listed():
    llama = dict(kv_heads=8, n_rep=4, dim=128)
    qwen = dict(kv_heads=4, n_rep=7, dim=128)
    return [
        # The smallest decode call: four chats of a few hundred to two thousand tokens. Launches
        # and latency count.
        dict(name="decode_tiny", kind="decode", dtype="fp16", batch=4, lens="uniform", lo=256, hi=2048, mix=1, **llama),
        # The framework's headline: 16 sequences at 32K context.
        dict(name="decode_long", kind="decode", dtype="bf16", batch=16, lens="uniform", lo=32768, hi=32768, mix=2,
             **llama),
        # A mixed batch: 64 sequences, lognormal lengths with median 2048.
        dict(name="decode_ragged", kind="decode", dtype="bf16", batch=64, lens="lognormal", lo=128, hi=32768, mix=3,
             **llama),
        # One GPU's share of the 32K batch when the heads are split over eight GPUs.
        dict(name="decode_shard", kind="decode", dtype="bf16", batch=16, lens="uniform", lo=32768, hi=32768, mix=4,
             kv_heads=1, n_rep=4, dim=128),
        # A whole decode step over 28 layers of sequences compressed to a 2048-token budget, some
        # hundred tokens generated since.
        dict(name="step_budget", kind="step", dtype="fp16", batch=8, lens="uniform", lo=2049, hi=2600, mix=5, layers=28,
             **qwen),
        # Chunked prefill at long prefixes, the largest attention call.
        dict(name="prefill_long", kind="prefill", dtype="bf16", batch=4, prefix_lo=16384, prefix_hi=16384,
             chunk_lo=2048, chunk_hi=2048, mix=6, **llama),
        # The online scheduler's chunk: four sequences, 512 tokens each, somewhere in their prompts.
        dict(name="prefill_chunk", kind="prefill", dtype="fp16", batch=4, prefix_lo=500, prefix_hi=8000,
             chunk_lo=512, chunk_hi=512, mix=7, **qwen),
        # The last, ragged chunk of one long prompt.
        dict(name="prefill_tail", kind="prefill", dtype="bf16", batch=1, prefix_lo=32256, prefix_hi=32256,
             chunk_lo=389, chunk_hi=389, mix=8, **llama),
        # A group of short prompts prefilled at once, no prefix, 64-dim heads.
        dict(name="prefill_prompts", kind="prefill", dtype="fp16", batch=12, prefix_lo=0, prefix_hi=0,
             chunk_lo=16, chunk_hi=700, mix=9, kv_heads=8, n_rep=4, dim=64),
        # Scoring one layer of one sequence after its prefill, as the unchanged scheduler does per layer.
        dict(name="scores_layer", kind="scores", dtype="fp16", seq_len=16500, sink=64, obs=64, **qwen),
        # The final chunk of two 16K sequences over four layers, and their scores.
        dict(name="final_scores", kind="final", dtype="bf16", batch=2, layers=4, seq_len=16384, chunk=512, sink=64,
             obs=128, **llama),
        # Fixed-ratio compression of four 32K sequences over eight layers.
        dict(name="compact_ratio", kind="compact", dtype="bf16", batch=4, layers=8, seq_len=32768, sink=64, obs=128,
             ratio_pct=20, **llama),
    ]


# No drawn case moves more bytes or computes more than these (the long decode and prefill above; head
# shapes other than the large power-of-two ones up to a chunk call's work).
MAX_BYTES = 2.2e9
MAX_FLOPS = 2.4e12
MAX_FLOPS_OTHER = 2.0e11


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(["decode", "decode", "step", "prefill", "prefill", "scores", "final", "compact"])
    heads, n_rep = rng.choice([(8, 4), (8, 4), (4, 7), (4, 7), (1, 4), (2, 4), (1, 7), (2, 7), (8, 1), (4, 8)])
    case = dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), kv_heads=heads, n_rep=n_rep,
                dim=rng.choice([128, 128, 64]))
    if kind in ("decode", "step"):
        case.update(batch=_log_int(rng, 1, 64), lens=rng.choice(["uniform", "lognormal"]), mix=rng.randrange(1 << 30))
        case["lo"] = _log_int(rng, 17, 8192)
        case["hi"] = max(case["lo"], _log_int(rng, 17, 32768))
        if kind == "step":
            case["layers"] = _log_int(rng, 2, 32)
    elif kind == "prefill":
        case.update(batch=_log_int(rng, 1, 16), mix=rng.randrange(1 << 30))
        case["prefix_lo"] = 0 if rng.random() < 0.3 else _log_int(rng, 16, 16384)
        case["prefix_hi"] = 0 if case["prefix_lo"] == 0 else max(case["prefix_lo"], _log_int(rng, 16, 32768))
        case["chunk_lo"] = _log_int(rng, 16, 1024)
        case["chunk_hi"] = max(case["chunk_lo"], _log_int(rng, 16, 2048))
    elif kind == "scores":
        case.update(obs=rng.choice([16, 32, 64, 128]), sink=rng.choice([0, 4, 16, 64]), seq_len=_log_int(rng, 300, 32768))
    elif kind == "final":
        case.update(dim=128, obs=rng.choice([16, 32, 64, 128]), sink=rng.choice([4, 16, 64]), batch=_log_int(rng, 1, 8),
                    layers=_log_int(rng, 1, 8), chunk=_log_int(rng, 128, 1024))
        case["seq_len"] = case["chunk"] + _log_int(rng, 200, 24000)
    else:
        case.update(batch=_log_int(rng, 1, 8), layers=_log_int(rng, 2, 32), sink=rng.choice([16, 64]),
                    obs=rng.choice([16, 64, 128]), ratio_pct=rng.choice([10, 20, 35, 50]),
                    seq_len=PAGE * _log_int(rng, 32, 2048))
    return case


def draw(rng):
    while True:
        case = _draw_once(rng)
        w = work(case)
        cap = MAX_FLOPS if case["dim"] == 128 and case["n_rep"] != 7 else MAX_FLOPS_OTHER
        if w["bytes"] <= MAX_BYTES and w["flops"] <= cap and _pool_bytes(case) <= 6e9:
            return case


# ------------------------------------------------------------------------------------ layouts
def _lens(case):
    rng = np.random.default_rng(case["mix"])
    if case["lens"] == "uniform":
        return [int(x) for x in rng.integers(case["lo"], case["hi"], size=case["batch"], endpoint=True)]
    median = math.sqrt(case["lo"] * case["hi"])
    raw = rng.lognormal(mean=math.log(median), sigma=1.0, size=case["batch"])
    return [int(x) for x in np.clip(np.round(raw), case["lo"], case["hi"])]


def _chunks(case):
    """(prefix lengths, chunk lengths) of a prefill case."""
    if case["kind"] == "final":
        return [case["seq_len"] - case["chunk"]] * case["batch"], [case["chunk"]] * case["batch"]
    rng = np.random.default_rng(case["mix"])
    pre = rng.integers(case["prefix_lo"], case["prefix_hi"], size=case["batch"], endpoint=True)
    chk = rng.integers(case["chunk_lo"], case["chunk_hi"], size=case["batch"], endpoint=True)
    return [int(x) for x in pre], [int(x) for x in chk]


def _pages(n_tokens):
    return -(-n_tokens // PAGE)


def _keep(case):
    """Pages a compacted sequence keeps, and its middle blocks kept."""
    k, eff, _ = compaction.selection_budget_blocks(case["seq_len"], sink_len=case["sink"], obs_len=case["obs"],
                                                   retain_ratio=case["ratio_pct"] / 100.0)
    return eff // PAGE, k


def _pool_pages(case):
    kind = case["kind"]
    if kind in ("decode", "step"):
        used = sum(_pages(n) for n in _lens(case))
    elif kind in ("prefill", "final"):
        used = sum(_pages(p + c) for p, c in zip(*_chunks(case)))
    elif kind == "compact":
        return case["batch"] * (_pages(case["seq_len"]) + _keep(case)[0])
    else:
        return 0
    return used + max(8, used // 10)  # a pool is never quite full


def _pool_bytes(case):
    return 2 * 2 * case.get("layers", 1) * _pool_pages(case) * PAGE * case["kv_heads"] * case["dim"]


def _normal(shape, dtype, gen):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=gen)


def _tables(page_counts, pool_pages, seed):
    """Each sequence's pages scattered over the pool, and the zero-padded device table."""
    perm = np.random.default_rng(seed).permutation(pool_pages)
    lists, at = [], 0
    for n in page_counts:
        lists.append([int(x) for x in perm[at:at + n]])
        at += n
    table = np.zeros((len(lists), max(page_counts)), dtype=np.int32)
    for row, ids in zip(table, lists):
        row[:len(ids)] = ids
    return lists, torch.from_numpy(table).cuda()


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


# ------------------------------------------------------------------------------------ prepare
def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    H, R, D = case["kv_heads"], case["n_rep"], case["dim"]
    state = dict(case=case, scale=1.0 / math.sqrt(D))
    kind, layers, n = case["kind"], case.get("layers", 1), _pool_pages(case)

    if kind == "scores":
        state["k"] = _normal((H, case["seq_len"], D), dt, gen)
        state["q"] = _normal((H * R, case["obs"], D), dt, gen)
        return state

    if kind == "compact":
        keep, _ = _keep(case)
        per = _pages(case["seq_len"])
        pool = PagedKVPool(PAGE, layers, H, D, dt, num_blocks=n, device="cuda:0")
        ids = pool.allocate_blocks(case["batch"] * per)  # the free list left: the compacted pages exactly
        perm = np.random.default_rng(seed).permutation(ids)
        state["lists"] = [[int(x) for x in perm[b * per:(b + 1) * per]] for b in range(case["batch"])]
        pool.k_cache.normal_(generator=gen)
        pool.v_cache.normal_(generator=gen)
        mid = per - (case["sink"] + case["obs"]) // PAGE
        state["scores"] = torch.rand((case["batch"] * layers, mid), generator=gen, device="cuda")
        state["pool"] = pool
        return state

    k = _normal((layers, n, PAGE, H, D), dt, gen)
    v = _normal((layers, n, PAGE, H, D), dt, gen)
    if kind in ("decode", "step"):
        lens = _lens(case)
        _, state["table"] = _tables([_pages(x) for x in lens], n, seed)
        state["lens"] = _i32(lens)
        state["q"] = _normal((layers, len(lens), H * R, D), dt, gen)
        if kind == "step":
            state["k_new"] = _normal((layers, len(lens), H, D), dt, gen)
            state["v_new"] = _normal((layers, len(lens), H, D), dt, gen)
    else:
        pre, chk = _chunks(case)
        kv = [p + c for p, c in zip(pre, chk)]
        _, state["table"] = _tables([_pages(x) for x in kv], n, seed)
        state["cu"] = _i32([0] + [int(x) for x in np.cumsum(chk)])
        state["kv_lens"] = _i32(kv)
        state["max_chunk"] = max(chk)
        state["q"] = _normal((layers, sum(chk), H * R, D), dt, gen)
        state["k_new"] = _normal((layers, sum(chk), H, D), dt, gen)
        state["v_new"] = _normal((layers, sum(chk), H, D), dt, gen)
        if kind == "final":
            # The engine keeps each layer's window queries from its attention hook.
            q = state["q"].view(layers, case["batch"], case["chunk"], H * R, D)[:, :, -case["obs"]:]
            state["q_obs"] = q.permute(1, 0, 3, 2, 4).contiguous()
            state["host_lens"] = (chk, kv)
            state["stats"] = snapkv.ObsStats(case["batch"], layers, H * R, sink_len=case["sink"], obs_len=case["obs"],
                                             softmax_scale=state["scale"], device="cuda")
    state["k"], state["v"] = k, v
    return state


# ---------------------------------------------------------------------------------------- run
def run(state):
    case, scale = state["case"], state["scale"]
    kind, R = case["kind"], case["n_rep"]
    if kind == "decode":
        return page16_native.page16_decode_attention(state["q"][0], state["k"][0], state["v"][0], state["table"],
                                                     state["lens"], softmax_scale=scale, n_rep=R)
    if kind == "step":
        outs = [page16_native.page16_decode_append_attention(
            state["q"][l], state["k"][l], state["v"][l], state["table"], state["lens"], state["k_new"][l],
            state["v_new"][l], softmax_scale=scale, n_rep=R) for l in range(case["layers"])]
        return outs, state["k"], state["v"]
    if kind == "prefill":
        out = prefill.chunked_prefill(state["q"][0], state["k_new"][0], state["v_new"][0], state["k"][0], state["v"][0],
                                      state["table"], state["cu"], state["kv_lens"], softmax_scale=scale, n_rep=R,
                                      max_chunk=state["max_chunk"])
        return out, state["k"], state["v"]
    if kind == "scores":
        return snapkv.score_layer_blocks(state["k"], state["q"], sink_len=case["sink"], obs_len=case["obs"], n_rep=R)
    if kind == "final":
        outs = []
        for l in range(case["layers"]):
            prefill.write_chunk_kv(state["k"][l], state["v"][l], state["k_new"][l], state["v_new"][l], state["table"],
                                   state["cu"], state["kv_lens"], state["max_chunk"])
            outs.append(prefill.paged_prefill_attention(
                state["q"][l], state["k"][l], state["v"][l], state["table"], state["cu"], state["kv_lens"],
                softmax_scale=scale, n_rep=R, max_chunk=state["max_chunk"], obs_stats=state["stats"], layer_id=l,
                host_lens=state["host_lens"]))
        scores = snapkv.score_blocks(state["q_obs"], state["k"], state["table"], seq_len=case["seq_len"],
                                     sink_len=case["sink"], obs_len=case["obs"], n_rep=R, obs_stats=state["stats"])
        return outs, scores, state["k"], state["v"]
    layers, pool = case["layers"], state["pool"]
    keep, k_mid = _keep(case)
    sel = compaction.select_blocks(state["scores"], k_mid)
    retained = [compaction.retained_pages(case["seq_len"], sel[b * layers:(b + 1) * layers], sink_len=case["sink"],
                                          obs_len=case["obs"]) for b in range(case["batch"])]
    res = compaction.compact(pool, state["lists"], retained, [keep * PAGE] * case["batch"])
    for ids in res.page_lists:  # given back in order, so that the next pass is handed the same pages
        pool.free_blocks_by_ids(ids)
    return sel, res.block_table, pool.k_cache, pool.v_cache


# --------------------------------------------------------------------------------------- work
def work(case):
    kind, L = case["kind"], case.get("layers", 1)
    H, R, D = case["kv_heads"], case["n_rep"], case["dim"]
    row = H * D * 2  # one token's K (or V) row of one layer
    if kind in ("decode", "step"):
        lens = _lens(case)
        tokens, B = sum(lens), len(lens)
        table = 4 * sum(_pages(x) for x in lens) + 4 * B
        per_layer = 2 * tokens * row + 2 * B * R * row
        if kind == "step":
            per_layer += 2 * B * row  # the new rows are read in place of old ones, and written
        return {"bytes": L * (per_layer + table), "flops": L * 4 * tokens * H * R * D}
    if kind in ("prefill", "final"):
        pre, chk = _chunks(case)
        keys = sum(p + c for p, c in zip(pre, chk))
        pairs = sum(c * p + c * (c + 1) // 2 for p, c in zip(pre, chk))
        total = sum(chk)
        size = 2 * keys * row + 2 * total * row + 2 * total * R * row + 4 * _pages(keys)
        flops = 4 * pairs * H * R * D
        if kind == "final":
            s = _score_work(case)
            # the scores' queries are the chunk's; K is read again, after every layer's attention
            return {"bytes": L * (size + case["batch"] * s["bytes"]), "flops": L * (flops + case["batch"] * s["flops"])}
        return {"bytes": size, "flops": flops}
    if kind == "scores":
        return _score_work(case)
    keep, k_mid = _keep(case)
    mid = _pages(case["seq_len"]) - (case["sink"] + case["obs"]) // PAGE
    rows = case["batch"] * L
    return {"bytes": rows * (2 * 2 * keep * PAGE * row + 4 * mid + 4 * k_mid), "flops": 0}


def _score_work(case):
    """One layer of one sequence: Q K^T over the middle keys, their K and the window's queries read once."""
    H, R, D = case["kv_heads"], case["n_rep"], case["dim"]
    mid = case["seq_len"] - case["sink"] - case["obs"]
    if mid < PAGE:
        return {"bytes": 0, "flops": 0}
    return {"bytes": mid * H * D * 2 + H * R * case["obs"] * D * 2 + 4 * _pages(mid),
            "flops": 2 * H * R * case["obs"] * mid * D}


# ---------------------------------------------------------------------------------- tolerance
# Four times the distance measured from ``exact`` (2-norm), the larger of the kinds' cases.
TOLERANCE = {
    ("decode", "bf16"): 7e-3, ("decode", "fp16"): 9e-4,
    ("step", "bf16"): 7e-3, ("step", "fp16"): 9e-4,
    ("prefill", "bf16"): 7e-3, ("prefill", "fp16"): 1.2e-3,
    ("scores", "bf16"): 1.2e-4, ("scores", "fp16"): 1.2e-4,
    ("final", "bf16"): 7e-3, ("final", "fp16"): 1.2e-3,
}


def tolerance(case):
    if case["kind"] == "compact":
        return "exact"
    return {"rel": TOLERANCE[case["kind"], case["dtype"]]}


# -------------------------------------------------------------------------------------- exact
def _rows(pool_layer, table_row, n_tokens):
    """[H, n_tokens, D] in 64 bits: one sequence's rows of one layer."""
    x = pool_layer[table_row[:_pages(n_tokens)].long()]
    return x.reshape(-1, x.shape[2], x.shape[3])[:n_tokens].double().permute(1, 0, 2).contiguous()


def _attend(q, keys, values, scale, first_pos):
    """Causal attention of q [R, C, D] (query i at position first_pos + i) over [T, D] keys, in slabs of queries."""
    out = torch.empty_like(q)
    kt = keys.t().contiguous()
    pos = torch.arange(keys.shape[0], device=q.device)
    for i0 in range(0, q.shape[1], 512):
        qs = q[:, i0:i0 + 512]
        s = torch.matmul(qs.reshape(-1, q.shape[2]), kt).view(qs.shape[0], qs.shape[1], -1) * scale
        limit = torch.arange(first_pos + i0, first_pos + i0 + qs.shape[1], device=q.device)
        s.masked_fill_(pos[None, None, :] > limit[None, :, None], -math.inf)
        p = torch.softmax(s, dim=-1)
        out[:, i0:i0 + 512] = torch.matmul(p.view(-1, keys.shape[0]), values).view(qs.shape)
    return out


def _exact_scores(q, keys, case):
    """Block scores of one layer of one sequence: q [Hq, obs, D], keys [H, T, D], in 64 bits."""
    H, R, D = case["kv_heads"], case["n_rep"], case["dim"]
    mid = keys[:, case["sink"]:keys.shape[1] - case["obs"]]
    n = _pages(mid.shape[1])
    mid = torch.nn.functional.pad(mid, (0, 0, 0, n * PAGE - mid.shape[1]))
    best = torch.zeros(n * PAGE, dtype=torch.float64, device=q.device)
    for h in range(H):
        kt = mid[h].t().contiguous()
        for r in range(R):
            w = torch.softmax(torch.matmul(q[h * R + r], kt) / math.sqrt(D), dim=-1)
            best = torch.maximum(best, w.mean(dim=0))
    block = best.view(n, PAGE).sum(dim=1)
    if n >= 3:
        block = torch.nn.functional.max_pool1d(block[None, None], 3, stride=1, padding=1)[0, 0]
    return block


def _exact_prefill(state, layer, case):
    """The layer's attention outputs, its pools updated in place first."""
    pre, chk = _chunks(case)
    H, R, D = case["kv_heads"], case["n_rep"], case["dim"]
    out = torch.empty(state["q"][layer].shape, dtype=torch.float64, device="cuda")
    at = 0
    for b, (p, c) in enumerate(zip(pre, chk)):
        pos = torch.arange(p, p + c, device="cuda")
        page = state["table"][b][pos // PAGE].long()
        for pool, new in ((state["k"][layer], state["k_new"][layer]), (state["v"][layer], state["v_new"][layer])):
            pool[page, pos % PAGE] = new[at:at + c]
        keys = _rows(state["k"][layer], state["table"][b], p + c)
        values = _rows(state["v"][layer], state["table"][b], p + c)
        q = state["q"][layer][at:at + c].double().permute(1, 0, 2).contiguous()
        for h in range(H):
            o = _attend(q[h * R:(h + 1) * R], keys[h], values[h], state["scale"], p)
            out[at:at + c, h * R:(h + 1) * R] = o.permute(1, 0, 2)
        at += c
    return out


def exact(case, seed):
    state = prepare(case, seed)
    kind, layers = case["kind"], case.get("layers", 1)
    H, R = case["kv_heads"], case["n_rep"]
    if kind == "scores":
        return _exact_scores(state["q"].double(), state["k"].double(), case)
    if kind == "compact":
        keep, k_mid = _keep(case)
        order = torch.sort(state["scores"].double(), dim=1, descending=True, stable=True).indices[:, :k_mid]
        return torch.sort(order, dim=1).values, None, None, None  # the rest are copies
    if kind in ("prefill", "final"):
        outs = [_exact_prefill(state, l, case) for l in range(layers)]
        if kind == "prefill":
            return outs[0], state["k"].double(), state["v"].double()
        scores = torch.stack([_exact_scores(state["q_obs"][b, l].double(),
                                            _rows(state["k"][l], state["table"][b], case["seq_len"]), case)
                              for b in range(case["batch"]) for l in range(layers)])
        return outs, scores, state["k"].double(), state["v"].double()
    lens = _lens(case)
    outs = []
    for l in range(layers):
        out = torch.empty(state["q"][l].shape, dtype=torch.float64, device="cuda")
        for b, n in enumerate(lens):
            if kind == "step":
                page = int(state["table"][b, (n - 1) // PAGE])
                state["k"][l][page, (n - 1) % PAGE] = state["k_new"][l][b]
                state["v"][l][page, (n - 1) % PAGE] = state["v_new"][l][b]
            keys = _rows(state["k"][l], state["table"][b], n)
            values = _rows(state["v"][l], state["table"][b], n)
            q = state["q"][l][b].double()
            for h in range(H):
                w = torch.softmax(torch.matmul(q[h * R:(h + 1) * R], keys[h].t().contiguous()) * state["scale"], dim=-1)
                out[b, h * R:(h + 1) * R] = torch.matmul(w, values[h])
        outs.append(out)
    if kind == "decode":
        return outs[0]
    return outs, state["k"].double(), state["v"].double()
