"""The work that users of this library have it do, as cases that can be timed and checked.

Each case is one call pattern on the public entry points: the C-ABI launches
of include/kimkv_hip.h (through the Python binding `device`), the engine of
include/kimkv_host.h (through `host`) and the model runner on top of it.
Operations:

  decode   one layer's paged decode attention of a batch of lanes
  prefill  one layer's causal attention of a batch of prompt chunks
  append   one token of every lane written to its tail page, all layers, and
           the tail pages read back
  prompt   prompts written to micro pages, promoted to extent pages and read
           back contiguous (ingest and hand-off of a prefix), all layers
  gather   one sequence's pages copied to a contiguous tensor, all layers
  mlp      the MLP half (RMSNorm, gate|up, SwiGLU, down + residual) of a few
           model layers for a batch of rows
  engine   token steps of forked requests through the engine: reserve, per
           layer write + attend, commit
  forward  one iteration of the TinyLlama-shaped runner over decode lanes and
           prompt chunks, with logits

Lengths of ragged batches follow from the case alone (`mix`), contents from
the seed.
"""
import importlib
import math
import random

import numpy as np
import torch

from _loader import load_package

_package = load_package()
device = _package.device
host = importlib.import_module(_package.__name__ + ".host")

MICRO, EXTENT = 8, 64

# TinyLlama-1.1B dimensions (the library's end-to-end configuration).
MODEL = {"hidden": 2048, "inter": 5632, "layers": 22, "qh": 32, "kvh": 4, "dim": 64, "vocab": 32000, "positions": 2048,
         "eps": 1e-5, "theta": 10000.0}


def listed():
    return [
        # A single user's few chats: the smallest decode launch, one layer.
        {"name": "decode_few", "op": "decode", "lanes": 4, "min": 18, "max": 1001, "kvh": 4, "group": 8, "dim": 64, "mix": 1},
        # A serving batch of ordinary, ragged contexts.
        {"name": "decode_batch", "op": "decode", "lanes": 48, "min": 200, "max": 6000, "kvh": 4, "group": 8, "dim": 64, "mix": 2},
        # Long contexts, the HBM-bound end of the range.
        {"name": "decode_long", "op": "decode", "lanes": 96, "min": 32769, "max": 32769, "kvh": 4, "group": 8, "dim": 64, "mix": 3},
        # 128-wide heads, eight KV heads.
        {"name": "decode_wide", "op": "decode", "lanes": 16, "min": 500, "max": 4000, "kvh": 8, "group": 4, "dim": 128, "mix": 4},
        # Chunked prefill as the scheduler hands it out: 512-token chunks on unequal contexts.
        {"name": "prefill_chunks", "op": "prefill", "chunks": 4, "new": 512, "ragged": 0, "min": 256, "max": 2048, "kvh": 4, "group": 8, "dim": 64, "mix": 5},
        # Shorter ragged chunks of 128-wide heads.
        {"name": "prefill_wide", "op": "prefill", "chunks": 2, "new": 256, "ragged": 1, "min": 100, "max": 1500, "kvh": 8, "group": 4, "dim": 128, "mix": 6},
        # The ragged one-token append of a decode batch outside the fused path, some tails copied on write.
        {"name": "append_step", "op": "append", "lanes": 64, "layers": 22, "kvh": 4, "dim": 64, "mix": 7},
        # Four prompts ingested, promoted and handed on.
        {"name": "prompt_ingest", "op": "prompt", "prompts": 4, "min": 256, "max": 2048, "layers": 22, "kvh": 4, "dim": 64, "mix": 8},
        # The long-sequence gather.
        {"name": "gather_long", "op": "gather", "tokens": 16384, "layers": 22, "kvh": 4, "dim": 64, "mix": 9},
        # The MLP of a decode step: few rows, so the weights' bytes count.
        {"name": "mlp_decode", "op": "mlp", "rows": 60, "layers": 4, "mix": 10},
        # Token steps of requests that share prompt prefixes, through the engine.
        {"name": "engine_shared", "op": "engine", "groups": 8, "per_group": 4, "prefix": 2048, "min": 128, "max": 8192, "steps": 2, "mix": 11},
        # One scheduler iteration's model call: prompt chunks beside decode lanes.
        {"name": "forward_mixed", "op": "forward", "lanes": 28, "chunks": 2, "new": 512, "min": 256, "max": 1500, "mix": 12},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "append", "prompt", "gather", "mlp", "engine", "forward"])
    mix = rng.randrange(1 << 20)
    heads = rng.choice([(4, 8, 64), (4, 8, 64), (4, 8, 64), (8, 4, 64), (2, 16, 64), (8, 4, 128), (4, 4, 128)])
    kvh, group, dim = heads
    if op == "decode":
        hi = _log_uniform(rng, 32, 32768)
        # At most the listed long case's K/V bytes.
        most = max(1, min(256, 3_000_000 * 256 // (hi * kvh * dim)))
        return {"op": op, "lanes": _log_uniform(rng, 1, most), "min": max(1, int(hi * rng.uniform(0.1, 1.0))), "max": hi,
                "kvh": kvh, "group": group, "dim": dim, "mix": mix}
    if op == "prefill":
        new = _log_uniform(rng, 3, 700)
        return {"op": op, "chunks": rng.randint(1, 4), "new": new, "ragged": rng.randint(0, 1), "min": rng.randint(0, 200),
                "max": _log_uniform(rng, 200, 2048), "kvh": kvh, "group": group, "dim": dim, "mix": mix}
    if op == "append":
        return {"op": op, "lanes": _log_uniform(rng, 1, 256), "layers": rng.choice([2, 16, 22]), "kvh": kvh, "dim": dim, "mix": mix}
    if op == "prompt":
        return {"op": op, "prompts": rng.randint(1, 6), "min": rng.randint(9, 256), "max": _log_uniform(rng, 256, 2048),
                "layers": rng.choice([2, 16, 22]), "kvh": kvh, "dim": dim, "mix": mix}
    if op == "gather":
        return {"op": op, "tokens": _log_uniform(rng, 50, 16000), "layers": rng.choice([2, 16, 22]), "kvh": kvh, "dim": dim, "mix": mix}
    if op == "mlp":
        return {"op": op, "rows": _log_uniform(rng, 1, 2108), "layers": 4, "mix": mix}
    if op == "engine":
        return {"op": op, "groups": rng.randint(1, 8), "per_group": rng.randint(1, 4), "prefix": rng.randint(40, 2048),
                "min": 64, "max": _log_uniform(rng, 500, 6000), "steps": 2, "mix": mix}
    return {"op": op, "lanes": rng.randint(1, 28), "chunks": rng.randint(0, 2), "new": rng.randint(30, 512), "min": 64,
            "max": rng.randint(200, 1400), "mix": mix}


# ---- what a case holds -------------------------------------------------------


def _lengths(case, count, key=0, spread="uniform"):
    rng = random.Random(case["mix"] * 1009 + key)
    lo, hi = min(case["min"], case["max"]), case["max"]
    if spread == "log":
        return [max(1, _log_uniform(rng, max(1, lo), hi)) for _ in range(count)]
    return [rng.randint(lo, hi) for _ in range(count)]


def _chunks(case):
    """(context tokens, new tokens) of each prompt chunk."""
    rng = random.Random(case["mix"] * 1013)
    contexts = _lengths(case, case["chunks"])
    return [(t, rng.randint(max(1, case["new"] // 3), case["new"]) if case.get("ragged") else case["new"]) for t in contexts]


def _engine_lengths(case):
    """(prefix of each group, length of each lane): a prefix ends in a partial page, a lane goes past its prefix."""
    rng = random.Random(case["mix"] * 1019)
    prefixes = [case["prefix"] + rng.randint(1, 7) for _ in range(case["groups"])]
    lanes = _lengths(case, case["groups"] * case["per_group"], 1, "log")
    return prefixes, [max(n, prefixes[i // case["per_group"]] + 8) for i, n in enumerate(lanes)]


def _normal(seed, tag, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1_000_003 + tag * 7919 + 17) & 0x7FFFFFFFFFFFFFFF)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)


def _on_gpu(array):
    """A numpy (structured) array as bytes on the GPU."""
    return torch.from_numpy(np.ascontiguousarray(array).view(np.uint8).reshape(-1).copy()).cuda()


class _Slots:
    """Page slots in a scattered order, as a long-running server's free lists hand them out."""

    def __init__(self, micro, extent, mix):
        rng = np.random.RandomState(mix % (1 << 31))
        self.free = [list(rng.permutation(micro)), list(rng.permutation(extent))]

    def table(self, tokens):
        """floor(T / 64) extent pages, then micro pages."""
        full, rest = divmod(tokens, EXTENT)
        pages = [(self.free[1].pop(), 1, i * EXTENT, EXTENT, EXTENT, 1) for i in range(full)]
        pages += [(self.free[0].pop(), 1, full * EXTENT + b, min(MICRO, rest - b), MICRO, 0) for b in range(0, rest, MICRO)]
        return np.array(pages, dtype=device.BLOCK_DESC)

    def micro_table(self, tokens):
        return np.array([(self.free[0].pop(), 1, b, min(MICRO, tokens - b), MICRO, 0) for b in range(0, tokens, MICRO)],
                        dtype=device.BLOCK_DESC)


def _pages(token_counts):
    """(micro, extent) capacities for tables of these token counts."""
    return sum((t % EXTENT + MICRO - 1) // MICRO for t in token_counts) + 8, sum(t // EXTENT for t in token_counts) + 4


def _page_jobs(table, kv):
    """Append jobs that write kv ([L][2][T][H][D]) into the pages of its table."""
    layers, _, tokens, heads, dim = kv.shape
    row = heads * dim
    jobs = np.zeros(len(table), dtype=device.APPEND_JOB)
    begin = table["logical_token_begin"].astype(np.uint64)
    jobs["src_key"] = np.uint64(kv.data_ptr()) + begin * np.uint64(2 * row)
    jobs["src_value"] = jobs["src_key"] + np.uint64(2 * tokens * row)
    jobs["src_layer_stride"] = 2 * tokens * row
    jobs["src_token_stride"] = row
    jobs["layer_count"] = layers
    jobs["token_count"] = table["valid_tokens"]
    jobs["dst_slot"], jobs["dst_kind"] = table["slot"], table["kind"]
    return jobs


def _write(storage, jobs, layers):
    """The jobs' launch; the returned bytes are the launch's jobs."""
    dev_jobs = _on_gpu(jobs)
    _check(device.lib().kimkv_append_batch(storage.h, dev_jobs.data_ptr(), len(jobs), layers, None))
    return dev_jobs


def _check(status):
    if status != 0:
        raise RuntimeError("status %d" % status)


# ---- decode ------------------------------------------------------------------


def _prepare_decode(case, seed):
    counts = _lengths(case, case["lanes"])
    heads, dim, qh = case["kvh"], case["dim"], case["kvh"] * case["group"]
    micro, extent = _pages(counts)
    storage = device.Storage(1, heads, dim, micro, extent)
    slots = _Slots(micro, extent, case["mix"])
    chunk, prefix, total = storage.decode_plan(counts, qh)
    items = np.zeros(len(counts), dtype=device.DECODE_ITEM)
    query = _normal(seed, 1, len(counts), qh, dim)
    out = torch.zeros_like(query)
    need = [device.workspace_bytes(t, chunk, qh, dim) for t in counts]
    work = torch.zeros(max(1, sum(need) // 4), dtype=torch.float32, device="cuda")
    tables, at = [], 0
    for i, t in enumerate(counts):
        table = slots.table(t)
        kv = _normal(seed, 1000 + i, 1, 2, t, heads, dim)
        _write(storage, _page_jobs(table, kv), 1)
        tables.append(_on_gpu(table))
        items[i] = (tables[-1].data_ptr(), len(table), t, 0, query[i].data_ptr(), work.data_ptr() + at if need[i] else 0,
                    out[i].data_ptr(), 1.0 / math.sqrt(dim))
        at += need[i]
    return {"storage": storage, "items": _on_gpu(items), "prefix": _on_gpu(prefix), "plan": (len(counts), total, chunk, qh), "out": out,
            "held": (tables, query, work)}


def _run_decode(s):
    lanes, total, chunk, qh = s["plan"]
    s["storage"].decode_launch(s["items"].data_ptr(), s["prefix"].data_ptr(), lanes, total, chunk, qh)
    return s["out"]


def _attention(q, k, v, causal_from=None):
    """float64 attention of q ([n][QH][D]) over k, v ([T][H][D]); row i of a causal one sees keys [0, causal_from + i]."""
    n, qh, dim = q.shape
    tokens, heads, _ = k.shape
    group = qh // heads
    out = torch.empty(n, qh, dim, dtype=torch.float64, device=q.device)
    for h in range(heads):
        qq = q[:, h * group:(h + 1) * group].double().reshape(n * group, dim)
        s = qq @ k[:, h].double().t().contiguous() / math.sqrt(dim)
        if causal_from is not None:
            limit = causal_from + torch.arange(n, device=q.device).repeat_interleave(group)
            s.masked_fill_(torch.arange(tokens, device=q.device)[None, :] > limit[:, None], -math.inf)
        out[:, h * group:(h + 1) * group] = (torch.softmax(s, 1) @ v[:, h].double().contiguous()).reshape(n, group, dim)
    return out


def _exact_decode(case, seed):
    counts = _lengths(case, case["lanes"])
    heads, dim, qh = case["kvh"], case["dim"], case["kvh"] * case["group"]
    query = _normal(seed, 1, len(counts), qh, dim)
    out = torch.empty(len(counts), qh, dim, dtype=torch.float64, device="cuda")
    for i, t in enumerate(counts):
        kv = _normal(seed, 1000 + i, 1, 2, t, heads, dim)
        out[i] = _attention(query[i:i + 1], kv[0, 0], kv[0, 1])[0]
    return out


def _work_decode(case):
    tokens, qh = sum(_lengths(case, case["lanes"])), case["kvh"] * case["group"]
    return {"bytes": tokens * 4 * case["kvh"] * case["dim"] + case["lanes"] * 4 * qh * case["dim"], "flops": 4 * qh * case["dim"] * tokens}


# ---- prefill -----------------------------------------------------------------


def _prepare_prefill(case, seed):
    chunks = _chunks(case)
    heads, dim, qh = case["kvh"], case["dim"], case["kvh"] * case["group"]
    counts = [t + n for t, n in chunks]
    micro, extent = _pages(counts)
    storage = device.Storage(1, heads, dim, micro, extent)
    slots = _Slots(micro, extent, case["mix"])
    items = np.zeros(len(chunks), dtype=device.PREFILL_ITEM)
    tables, queries, outs = [], [], []
    for i, (t, n) in enumerate(chunks):
        table = slots.table(t + n)
        kv = _normal(seed, 1000 + i, 1, 2, t + n, heads, dim)
        _write(storage, _page_jobs(table, kv), 1)
        tables.append(_on_gpu(table))
        queries.append(_normal(seed, 2000 + i, n, qh, dim))
        outs.append(torch.zeros_like(queries[-1]))
        items[i] = (tables[-1].data_ptr(), len(table), t + n, n, 0, queries[-1].data_ptr(), outs[-1].data_ptr(), 1.0 / math.sqrt(dim))
    order = device.prefill_order(heads, dim, qh, storage.info().compute_units, counts, [n for _, n in chunks])
    return {"storage": storage, "items": _on_gpu(items), "order": _on_gpu(order), "plan": (len(chunks), len(order), qh), "out": outs,
            "held": (tables, queries)}


def _run_prefill(s):
    count, order, qh = s["plan"]
    s["storage"].prefill_ordered_launch(s["items"].data_ptr(), count, s["order"].data_ptr(), order, qh)
    return s["out"]


def _exact_prefill(case, seed):
    heads, dim, qh = case["kvh"], case["dim"], case["kvh"] * case["group"]
    out = []
    for i, (t, n) in enumerate(_chunks(case)):
        kv = _normal(seed, 1000 + i, 1, 2, t + n, heads, dim)
        out.append(_attention(_normal(seed, 2000 + i, n, qh, dim), kv[0, 0], kv[0, 1], t))
    return out


def _work_prefill(case):
    heads, dim, qh = case["kvh"], case["dim"], case["kvh"] * case["group"]
    chunks = _chunks(case)
    pairs = sum(n * t + n * (n + 1) // 2 for t, n in chunks)
    return {"bytes": sum((t + n) * 4 * heads * dim + n * 4 * qh * dim for t, n in chunks), "flops": 4 * qh * dim * pairs}


# ---- pages: append, prompt, gather -------------------------------------------


def _prepare_append(case, seed):
    lanes, layers, heads, dim = case["lanes"], case["layers"], case["kvh"], case["dim"]
    rng = random.Random(case["mix"] * 1021)
    storage = device.Storage(layers, heads, dim, 2 * lanes + 8, 4)
    slots = _Slots(2 * lanes + 8, 4, case["mix"])
    # Every lane's tail page holds 0..7 tokens; one in four partial tails is shared and is copied before the write.
    tails = slots.micro_table(MICRO * lanes)
    kv = _normal(seed, 1, layers, 2, MICRO * lanes, heads, dim)
    _write(storage, _page_jobs(tails, kv), layers)
    new = _normal(seed, 2, lanes, layers, 2, heads, dim)
    jobs = np.zeros(lanes, dtype=device.APPEND_JOB)
    out_table = tails.copy()
    row = heads * dim
    for i in range(lanes):
        held = rng.randint(0, MICRO - 1)
        copied = held > 0 and rng.random() < 0.25
        dst = slots.free[0].pop() if copied else int(tails["slot"][i])
        out_table["slot"][i] = dst
        jobs[i] = (new[i, 0, 0].data_ptr(), new[i, 0, 1].data_ptr(), 2 * row, row, 0, layers, 1, dst, int(tails["slot"][i]), held,
                   held if copied else 0, 0, 0)
    out = torch.zeros(layers, 2, MICRO * lanes, heads, dim, dtype=torch.int16, device="cuda")
    return {"storage": storage, "jobs": _on_gpu(jobs), "table": _on_gpu(out_table), "plan": (lanes, layers), "out": out, "held": new}


def _run_append(s):
    lanes, layers = s["plan"]
    lib, h = device.lib(), s["storage"].h
    _check(lib.kimkv_append_batch(h, s["jobs"].data_ptr(), lanes, layers, None))
    _check(lib.kimkv_gather(h, s["table"].data_ptr(), lanes, MICRO * lanes, s["out"].data_ptr(), None))
    return s["out"]


def _work_append(case):
    row = 2 * case["kvh"] * case["dim"]
    # The new rows read and written; the tail pages read and written by the copy out.
    return {"bytes": case["lanes"] * case["layers"] * 2 * row * (2 + 2 * MICRO), "flops": 0}


def _prepare_prompt(case, seed):
    layers, heads, dim = case["layers"], case["kvh"], case["dim"]
    counts = _lengths(case, case["prompts"])
    micro = sum((t + MICRO - 1) // MICRO for t in counts) + 8
    extent = sum(t // EXTENT for t in counts) + 4
    storage = device.Storage(layers, heads, dim, micro, extent)
    slots = _Slots(micro, extent, case["mix"])
    inputs, jobs, promotions, tables, outs = [], [], [], [], []
    for i, t in enumerate(counts):
        kv = _normal(seed, 1000 + i, layers, 2, t, heads, dim)
        table = slots.micro_table(t)
        inputs.append(kv)
        jobs.append(_page_jobs(table, kv))
        full = t // EXTENT
        final = [table[full * EXTENT // MICRO:]]
        for e in range(full):
            job = np.zeros(1, dtype=device.PROMOTION_JOB)
            job["micro_slots"][0] = table["slot"][e * 8:(e + 1) * 8]
            job["extent_slot"] = slots.free[1].pop()
            promotions.append(job)
            final.insert(e, np.array([(int(job["extent_slot"][0]), 1, e * EXTENT, EXTENT, EXTENT, 1)], dtype=device.BLOCK_DESC))
        final = [np.frombuffer(np.ascontiguousarray(f).tobytes(), dtype=device.BLOCK_DESC) for f in final]
        whole = np.zeros(sum(map(len, final)), dtype=device.BLOCK_DESC)
        at = 0
        for f in final:
            whole[at:at + len(f)] = f
            at += len(f)
        tables.append((_on_gpu(whole), len(whole), t))
        outs.append(torch.zeros(layers, 2, t, heads, dim, dtype=torch.int16, device="cuda"))
    n_jobs, n_promotions = sum(map(len, jobs)), len(promotions)
    return {"storage": storage, "jobs": _on_gpu(np.concatenate([j.view(np.uint8).reshape(-1) for j in jobs])),
            "promotions": _on_gpu(np.concatenate([p.view(np.uint8).reshape(-1) for p in promotions])) if promotions else None,
            "plan": (n_jobs, n_promotions, layers), "tables": tables, "out": outs, "held": inputs}


def _run_prompt(s):
    n_jobs, n_promotions, layers = s["plan"]
    lib, h = device.lib(), s["storage"].h
    _check(lib.kimkv_append_batch(h, s["jobs"].data_ptr(), n_jobs, layers, None))
    if n_promotions:
        _check(lib.kimkv_promote_batch(h, s["promotions"].data_ptr(), n_promotions, None))
    for (table, entries, tokens), out in zip(s["tables"], s["out"]):
        _check(lib.kimkv_gather(h, table.data_ptr(), entries, tokens, out.data_ptr(), None))
    return s["out"]


def _work_prompt(case):
    row = case["layers"] * 4 * case["kvh"] * case["dim"]
    counts = _lengths(case, case["prompts"])
    # Ingest and copy out read and write every token, promotion those of whole extents.
    return {"bytes": row * (4 * sum(counts) + 2 * sum(t // EXTENT * EXTENT for t in counts)), "flops": 0}


def _prepare_gather(case, seed):
    layers, heads, dim, t = case["layers"], case["kvh"], case["dim"], case["tokens"]
    micro, extent = _pages([t])
    storage = device.Storage(layers, heads, dim, micro, extent)
    table = _Slots(micro, extent, case["mix"]).table(t)
    _write(storage, _page_jobs(table, _normal(seed, 1, layers, 2, t, heads, dim)), layers)
    out = torch.zeros(layers, 2, t, heads, dim, dtype=torch.int16, device="cuda")
    return {"storage": storage, "table": _on_gpu(table), "plan": (len(table), t), "out": out}


def _run_gather(s):
    entries, tokens = s["plan"]
    _check(device.lib().kimkv_gather(s["storage"].h, s["table"].data_ptr(), entries, tokens, s["out"].data_ptr(), None))
    return s["out"]


def _work_gather(case):
    return {"bytes": 2 * case["layers"] * case["tokens"] * 4 * case["kvh"] * case["dim"], "flops": 0}


# ---- MLP ---------------------------------------------------------------------


def _prepare_mlp(case, seed):
    rows, hidden, inter, n = case["rows"], MODEL["hidden"], MODEL["inter"], case["layers"]
    weights = []
    for i in range(n):
        norm = (_normal(seed, 10 * i + 3, hidden) * 0.1 + 1.0).half()
        weights.append((norm, (_normal(seed, 10 * i + 1, 2 * inter, hidden) * 0.02).half(), (_normal(seed, 10 * i + 2, hidden, inter) * 0.02).half()))
    s = {"x0": _normal(seed, 9, rows, hidden), "weights": weights, "rows": rows}
    s["x"], s["h"] = torch.zeros_like(s["x0"]), torch.zeros_like(s["x0"])
    s["gu"] = torch.zeros(rows, 2 * inter, dtype=torch.float16, device="cuda")
    s["act"] = torch.zeros(rows, inter, dtype=torch.float16, device="cuda")
    # A program that repeats a product tunes it once, as the model runner does.
    device.linear_tune(s["h"].data_ptr(), rows, hidden, [w[1].data_ptr() for w in weights], 2 * inter, s["gu"].data_ptr(), False, 0.0)
    device.linear_tune(s["act"].data_ptr(), rows, inter, [w[2].data_ptr() for w in weights], hidden, s["x"].data_ptr(), False, 1.0)
    return s


def _run_mlp(s):
    lib, rows, hidden, inter = device.lib(), s["rows"], MODEL["hidden"], MODEL["inter"]
    p = {k: _pointer(s[k]) for k in ("x0", "x", "h", "gu", "act")}
    _check(lib.kimkv_memcpy_d2d_async(p["x"], p["x0"], rows * hidden * 2, None))
    for norm, gate_up, down in s["weights"]:
        _check(lib.kimkv_model_rmsnorm(p["x"], None, rows, _pointer(norm), hidden, _float(MODEL["eps"]), p["h"], None))
        _check(lib.kimkv_linear(p["h"], rows, hidden, _pointer(gate_up), 2 * inter, p["gu"], 0, 0.0, None))
        _check(lib.kimkv_model_swiglu(p["gu"], rows, inter, p["act"], None))
        _check(lib.kimkv_linear(p["act"], rows, inter, _pointer(down), hidden, p["x"], 0, 1.0, None))
    return s["x"]


def _pointer(tensor):
    return device.ctypes.c_void_p(tensor.data_ptr())


def _float(value):
    return device.ctypes.c_float(value)


def _exact_mlp(case, seed):
    rows, hidden, inter = case["rows"], MODEL["hidden"], MODEL["inter"]
    x = _normal(seed, 9, rows, hidden).double()
    for i in range(case["layers"]):
        norm = (_normal(seed, 10 * i + 3, hidden) * 0.1 + 1.0).half().double()
        gate_up = (_normal(seed, 10 * i + 1, 2 * inter, hidden) * 0.02).half().double()
        down = (_normal(seed, 10 * i + 2, hidden, inter) * 0.02).half().double()
        x = x + _swiglu(_rms(x, norm) @ gate_up.t().contiguous(), inter) @ down.t().contiguous()
    return x


def _rms(x, weight):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + MODEL["eps"]) * weight


def _swiglu(gate_up, inter):
    return torch.nn.functional.silu(gate_up[:, :inter]) * gate_up[:, inter:]


def _work_mlp(case):
    hidden, inter, n, rows = MODEL["hidden"], MODEL["inter"], case["layers"], case["rows"]
    return {"bytes": n * 6 * hidden * inter + 4 * rows * hidden, "flops": n * 6 * rows * hidden * inter}


# ---- engine ------------------------------------------------------------------


def _append_context(engine, rid, kv):
    """kv ([L][2][T][H][D]) appended to a request and promoted."""
    rc, _ = engine.append_prefill(rid, kv.shape[2], kv.data_ptr(), None, promote=True)
    _check(rc)


def _engine_kv(case, seed):
    """Each group's prefix K/V and each lane's own: functions of the group and the lane."""
    layers, heads, dim = MODEL["layers"], MODEL["kvh"], MODEL["dim"]
    prefixes, lengths = _engine_lengths(case)
    return (lambda g: _normal(seed, 100 + g, layers, 2, prefixes[g], heads, dim),
            lambda i: _normal(seed, 200 + i, layers, 2, lengths[i] - prefixes[i // case["per_group"]], heads, dim))


def _prepare_engine(case, seed):
    layers, heads, dim, qh = MODEL["layers"], MODEL["kvh"], MODEL["dim"], MODEL["qh"]
    prefixes, lengths = _engine_lengths(case)
    lanes, steps, row = len(lengths), case["steps"], heads * dim
    extents = sum(p // EXTENT for p in prefixes) + sum(t // EXTENT for t in lengths) + 16
    micros = max(prefixes + lengths) // MICRO + 24 * lanes + 64
    ws = max(device.workspace_bytes(max(lengths) + steps, 64, qh, dim), 256)
    engine = host.Engine(layers, heads, dim, qh, ws, micros, extents)
    _check(engine.permute_free_slots(0, case["mix"] + 1))
    _check(engine.permute_free_slots(1, case["mix"] + 2))
    group_kv, lane_kv = _engine_kv(case, seed)
    for g in range(case["groups"]):
        _check(engine.create_request(10_000 + g))
        _append_context(engine, 10_000 + g, group_kv(g))
    for i in range(lanes):
        _check(engine.fork_request(10_000 + i // case["per_group"], 1 + i))
        _append_context(engine, 1 + i, lane_kv(i))
    query = _normal(seed, 1, steps, layers, lanes, qh, dim)
    new = _normal(seed, 2, steps, layers, lanes, 2, heads, dim)
    out = torch.zeros_like(query)
    work = torch.zeros(lanes * ws // 4, dtype=torch.float32, device="cuda")
    lane = np.arange(lanes, dtype=np.uint64)
    batches = []
    for t in range(steps):
        b = host.LaneBatch(engine, 20_001 + lane, work.data_ptr() + lane * np.uint64(ws), ws, 1.0 / math.sqrt(dim))
        for l in range(layers):
            b.keys[l] = new[t, l].data_ptr() + lane * np.uint64(4 * row)
            b.values[l] = b.keys[l] + np.uint64(2 * row)
            b.queries[l] = query[t, l].data_ptr() + lane * np.uint64(2 * qh * dim)
            b.outputs[l] = out[t, l].data_ptr() + lane * np.uint64(2 * qh * dim)
        batches.append((b, np.array(lengths, dtype=np.uint32) + np.uint32(t)))
    return {"engine": engine, "batches": batches, "lanes": lanes, "layers": layers, "out": out, "held": (query, new, work)}


def _run_engine(s):
    engine = s["engine"]
    for i in range(s["lanes"]):
        _check(engine.fork_request(1 + i, 20_001 + i))
    for batch, expected in s["batches"]:
        batch.reserve(expected)
        for layer in range(s["layers"]):
            batch.write(layer)
            batch.attend(layer)
        batch.commit()
        if batch.failed():
            raise RuntimeError("a lane failed")
    for i in range(s["lanes"]):
        _check(engine.release_request(20_001 + i))
    return s["out"]


def _exact_engine(case, seed):
    layers, heads, dim, qh = MODEL["layers"], MODEL["kvh"], MODEL["dim"], MODEL["qh"]
    _, lengths = _engine_lengths(case)
    lanes, steps = len(lengths), case["steps"]
    group_kv, lane_kv = _engine_kv(case, seed)
    query = _normal(seed, 1, steps, layers, lanes, qh, dim)
    new = _normal(seed, 2, steps, layers, lanes, 2, heads, dim)
    out = torch.empty(query.shape, dtype=torch.float64, device="cuda")
    for i in range(lanes):
        kv = torch.cat([group_kv(i // case["per_group"]), lane_kv(i)] + [new[t, :, i][:, :, None] for t in range(steps)], 2).double()
        for t in range(steps):
            n = lengths[i] + t + 1
            for h in range(heads):
                g = qh // heads
                q = query[t, :, i, h * g:(h + 1) * g].double()
                p = torch.softmax(torch.matmul(q, kv[:, 0, :n, h].transpose(1, 2).contiguous()) / math.sqrt(dim), 2)
                out[t, :, i, h * g:(h + 1) * g] = torch.matmul(p, kv[:, 1, :n, h].contiguous())
    return out


def _work_engine(case):
    prefixes, lengths = _engine_lengths(case)
    row = MODEL["layers"] * 4 * MODEL["kvh"] * MODEL["dim"]
    unique = sum(prefixes) + sum(n - prefixes[i // case["per_group"]] for i, n in enumerate(lengths))
    qrow = MODEL["layers"] * 4 * MODEL["qh"] * MODEL["dim"]
    return {"bytes": case["steps"] * (unique * row + len(lengths) * (qrow + 2 * row)),
            "flops": case["steps"] * sum(lengths) * MODEL["layers"] * 4 * MODEL["qh"] * MODEL["dim"]}


# ---- model runner ------------------------------------------------------------


def _spans(case):
    """(context, new tokens) of each request: decode lanes, then prompt chunks."""
    lanes = _lengths(case, case["lanes"])
    chunks = _lengths(case, case["chunks"], 1)
    room = MODEL["positions"]
    return [(t, 1) for t in lanes] + [(min(t, room - case["new"]), case["new"]) for t in chunks]


def _ids(case, seed):
    rng = np.random.RandomState((int(seed) * 31 + 7) % (1 << 31))
    return [rng.randint(3, MODEL["vocab"], n).astype(np.uint32) for _, n in _spans(case)]


def _prepare_forward(case, seed):
    layers, heads, dim, qh = MODEL["layers"], MODEL["kvh"], MODEL["dim"], MODEL["qh"]
    spans = _spans(case)
    engine = host.Engine(layers, heads, dim, qh, 1 << 20, sum(t // MICRO + n // MICRO + 12 for t, n in spans) + 300,
                         sum((t + n) // EXTENT + 1 for t, n in spans) + 16)
    _check(engine.permute_free_slots(0, case["mix"] + 1))
    _check(engine.permute_free_slots(1, case["mix"] + 2))
    positions = sum(n for _, n in spans)
    model = host.ModelConfig(MODEL["hidden"], MODEL["inter"], layers, qh, heads, dim, MODEL["vocab"], MODEL["positions"], 1, 2,
                             MODEL["eps"], MODEL["theta"])
    runner = host.Runner(engine, model, int(seed), positions, len(spans))
    for i, (t, _) in enumerate(spans):
        _check(engine.create_request(1 + i))
        if t:
            _append_context(engine, 1 + i, _normal(seed, 100 + i, layers, 2, t, heads, dim))
    return {"engine": engine, "runner": runner, "spans": [(10_001 + i, t, ids) for i, ((t, _), ids) in enumerate(zip(spans, _ids(case, seed)))]}


def _run_forward(s):
    engine = s["engine"]
    for i in range(len(s["spans"])):
        _check(engine.fork_request(1 + i, 10_001 + i))
    _, ok, logits = s["runner"].forward(s["spans"], want_logits=True)
    if not ok.all():
        raise RuntimeError("a span failed")
    for i in range(len(s["spans"])):
        _check(engine.release_request(10_001 + i))
    return logits


def _weights(seed, row, rows, cols):
    """The runner's seeded weights, rows [row, row + rows) of cols columns: fp16(N(0, 0.02)) from a splitmix64 hash."""

    def signed(c):
        return c - (1 << 64) if c >= 1 << 63 else c

    def mix(z):
        for shift, factor in ((30, 0xBF58476D1CE4E5B9), (27, 0x94D049BB133111EB)):
            z = (z ^ ((z >> shift) & ((1 << (64 - shift)) - 1))) * signed(factor)
        return z ^ ((z >> 31) & ((1 << 33) - 1))

    r = torch.arange(rows, device="cuda", dtype=torch.int64) + row
    h = mix(mix(r * signed(0x9E3779B97F4A7C15) + signed(int(seed) & ((1 << 64) - 1)))[:, None]
            + torch.arange(cols, device="cuda", dtype=torch.int64)[None, :])
    v = sum((h >> s) & 0xFFFF for s in (0, 16, 32, 48)) - 131070
    return ((v.float() * (1.0 / 32768.0)).half().float() * 0.017320508).half().double()


def _rope(x, positions):
    """x ([n][heads][D]) rotated by its rows' positions, pairs (d, d + D / 2)."""
    half = x.shape[2] // 2
    freq = MODEL["theta"] ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / x.shape[2])
    angle = positions.double()[:, None] * freq[None, :]
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    return torch.cat([x[:, :, :half] * c - x[:, :, half:] * s, x[:, :, half:] * c + x[:, :, :half] * s], 2)


def _exact_forward(case, seed):
    hidden, inter, layers, heads, dim, qh = (MODEL[k] for k in ("hidden", "inter", "layers", "kvh", "dim", "qh"))
    spans, ids = _spans(case), _ids(case, seed)
    tokens = torch.from_numpy(np.concatenate(ids).astype(np.int64)).cuda()
    positions = torch.cat([torch.arange(t, t + n, device="cuda") for t, n in spans])
    ends = np.cumsum([n for _, n in spans])

    def tensor(layer, kind, rows, cols):
        return _weights(seed, ((layer + 1) << 40) | (kind << 32), rows, cols)

    one = torch.ones(hidden, dtype=torch.float64, device="cuda")
    x = tensor(layers, 8, MODEL["vocab"], hidden)[tokens]
    context = [_normal(seed, 100 + i, layers, 2, t, heads, dim) for i, (t, _) in enumerate(spans)]
    for l in range(layers):
        a = _rms(x, one)
        q = _rope((a @ tensor(l, 1, qh * dim, hidden).t().contiguous()).reshape(-1, qh, dim), positions)
        k = _rope((a @ tensor(l, 2, heads * dim, hidden).t().contiguous()).reshape(-1, heads, dim), positions)
        v = (a @ tensor(l, 3, heads * dim, hidden).t().contiguous()).reshape(-1, heads, dim)
        o = torch.empty_like(q)
        for i, (t, n) in enumerate(spans):
            rows = slice(ends[i] - n, ends[i])
            o[rows] = _attention(q[rows], torch.cat([context[i][l, 0].double(), k[rows]]), torch.cat([context[i][l, 1].double(), v[rows]]), t)
        x = x + o.reshape(-1, qh * dim) @ tensor(l, 4, hidden, qh * dim).t().contiguous()
        a = _rms(x, one)
        gate_up = torch.cat([a @ tensor(l, 5, inter, hidden).t().contiguous(), a @ tensor(l, 6, inter, hidden).t().contiguous()], 1)
        x = x + _swiglu(gate_up, inter) @ tensor(l, 7, hidden, inter).t().contiguous()
    last = torch.from_numpy(ends - 1).cuda()
    return (_rms(x[last], one) @ tensor(layers, 9, MODEL["vocab"], hidden).t().contiguous()).cpu()


def _work_forward(case):
    hidden, inter, layers, heads, dim, qh, vocab = (MODEL[k] for k in ("hidden", "inter", "layers", "kvh", "dim", "qh", "vocab"))
    spans = _spans(case)
    per_layer = hidden * (2 * qh * dim + 2 * heads * dim) + 3 * hidden * inter
    positions = sum(n for _, n in spans)
    pairs = sum(n * t + n * (n + 1) // 2 for t, n in spans)
    return {"bytes": 2 * (layers * per_layer + vocab * hidden) + layers * 4 * heads * dim * sum(t + 2 * n for t, n in spans) + 4 * vocab * len(spans),
            "flops": 2 * positions * layers * per_layer + layers * 4 * qh * dim * pairs + 2 * len(spans) * vocab * hidden}


# ---- the functions a measurement calls -----------------------------------------


def prepare(case, seed):
    return {**_OPS[case["op"]][0](case, seed), "op": case["op"]}


def run(state):
    return _OPS[state["op"]][1](state)


def work(case):
    return _OPS[case["op"]][2](case)


def exact(case, seed):
    compute = _OPS[case["op"]][3]
    return None if compute is None else compute(case, seed)


def tolerance(case):
    return _OPS[case["op"]][4]


_OPS = {
    # op: (prepare, run, work, exact, tolerance)
    # Tolerances: about four times the distance to exact() that was measured.
    # fp16 outputs of fp32 sums (2.1e-4 off: the rounding to 11 bits).
    "decode": (_prepare_decode, _run_decode, _work_decode, _exact_decode, {"rel": 8e-4, "max": 4e-3}),
    "engine": (_prepare_engine, _run_engine, _work_engine, _exact_engine, {"rel": 8e-4, "max": 4e-3}),
    # Softmax weights of a prompt chunk go to the matrix cores in fp16 (3.0e-4 off).
    "prefill": (_prepare_prefill, _run_prefill, _work_prefill, _exact_prefill, {"rel": 1.2e-3, "max": 8e-3}),
    # Copies.
    "append": (_prepare_append, _run_append, _work_append, None, "exact"),
    "prompt": (_prepare_prompt, _run_prompt, _work_prompt, None, "exact"),
    "gather": (_prepare_gather, _run_gather, _work_gather, None, "exact"),
    # Activations are rounded to fp16 between the kernels: four layers' MLPs (7.6e-4 off), 22 whole layers (4.2e-3 off).
    "mlp": (_prepare_mlp, _run_mlp, _work_mlp, _exact_mlp, {"rel": 3e-3, "max": 2e-2}),
    "forward": (_prepare_forward, _run_forward, _work_forward, _exact_forward, {"rel": 1.7e-2, "max": 1.2e-1}),
}
