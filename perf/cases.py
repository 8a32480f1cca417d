"""The work that a user of this framework has it do, as cases that can be timed.

A pass of every case is a step of a model's full-attention layers through the public entry points (``tinytitan_amd.engine``),
called as the host runner calls them: per layer the QKV epilogue with its cache write, the attention over the cached keys with
the output gate, and the output projection over affine weights; a sparse layer also runs its block indexer (pooling, scores,
selection) in front.  The caches hold what earlier tokens of the sequences left there, every layer its own; the indexer's
query rows are given, with the new tokens' raw keys in its cache, where a layer's own projections would have left them: a
selection follows from them to the last bit, and a last bit of a query is another selection.

kind            a pass is
``rows``        ``rows`` query tokens for each of ``seqs`` sequences: a decode step (1 row) or a draft's verify rows
``chunk``       one prefill chunk of ``rows`` tokens of one sequence behind ``lo`` cached keys, with ``window`` > 0 over a ring
``sparse_rows`` a decode step of one sequence whose layers keep a selection of the keys
``sparse_chunk``  a prefill chunk whose rows each keep a selection of the keys

A sequence's cached keys number ``lo`` .. ``hi`` (spread evenly over the logarithm by a fixed stream where the two differ).
"""
import math

import torch

from tinytitan_amd import synthetic
from tinytitan_amd.engine import (AffineProjection, Attention, HIPContext, KVCacheManager, PrefillAttention,
                                  PrefillAttentionParams, QKVEpilogue, QSAIndexer)

HIDDEN = 2048           # rows of the output projection
ROTARY_DIM, THETA, EPS = 64, 1.0e7, 1.0e-6
INDEX_HEADS, INDEX_DIM, INDEX_RATIO, INDEX_BUDGET = 4, 128, 4, 2048
DEVICE = torch.device("cuda", 0)

_context = None


def _case(kind, heads, kv_heads, dim, lo, hi=None, seqs=1, rows=1, layers=1, kv_bits=16, w_bits=4, window=0, name=None):
    case = {"kind": kind, "heads": heads, "kv_heads": kv_heads, "dim": dim, "lo": lo, "hi": hi or lo, "seqs": seqs, "rows": rows,
            "layers": layers, "kv_bits": kv_bits, "w_bits": w_bits, "window": window}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a short chat on a small model: one decode token, where launches and host work count most
        _case("rows", 8, 2, 256, 2047, layers=4, name="decode_2k"),
        # one user's decode token late in a long document, fp16 cache
        _case("rows", 16, 2, 256, 32767, layers=4, name="decode_32k"),
        # the same over the runtime's default cache precision, at a length nothing is tuned to
        _case("rows", 16, 2, 256, 20010, layers=4, kv_bits=8, name="decode_20k_8bit"),
        # a serving batch's decode token, sequences of all ages
        _case("rows", 16, 2, 256, 511, 16383, seqs=32, name="decode_batch32"),
        # a smaller batch on a memory-saving 4-bit cache
        _case("rows", 16, 2, 256, 300, 9000, seqs=7, layers=2, kv_bits=4, name="decode_batch7_4bit"),
        # speculative decoding for one user: four draft rows checked at once, default cache precision
        _case("rows", 16, 2, 256, 8190, rows=4, layers=4, kv_bits=8, name="verify_8k_8bit"),
        # the same for a batch of very long contexts
        _case("rows", 16, 2, 256, 65536, seqs=8, rows=4, name="verify_batch8_64k"),
        # the first, long chunk of a prompt
        _case("chunk", 16, 2, 256, 0, rows=4096, name="prefill_4096"),
        # the default prefill chunk deep in a long prompt, default cache precision
        _case("chunk", 16, 2, 256, 32640, rows=128, layers=2, kv_bits=8, name="chunk128_32k_8bit"),
        # a ragged chunk of a sliding-window model with many KV heads, over its ring
        _case("chunk", 32, 8, 128, 5003, rows=777, window=4096, name="chunk777_window"),
        # a sparse layer's decode token at a context where the selection pays
        _case("sparse_rows", 16, 2, 256, 131071, layers=2, name="sparse_decode_128k"),
        # ... and its default prefill chunk
        _case("sparse_chunk", 16, 2, 256, 130944, rows=128, name="sparse_chunk128_128k"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case: kinds in the listed ones' proportions, sizes spread over their logarithm."""
    top = [work(c) for c in listed()]
    most_bytes, most_flops = max(w["bytes"] for w in top), max(w["flops"] for w in top)
    while True:
        kind = rng.choice(["rows"] * 7 + ["chunk"] * 3 + ["sparse_rows", "sparse_chunk"])
        heads, kv_heads, dim = rng.choice([(8, 2, 256), (16, 2, 256), (16, 2, 256), (24, 2, 256), (32, 8, 128), (16, 4, 64)])
        case = _case(kind, heads, kv_heads, dim, 1, layers=rng.choice([1, 2, 4]), kv_bits=rng.choice([16, 16, 8, 8, 4]),
                     w_bits=rng.choice([4, 4, 8]))
        if kind == "rows":
            case["seqs"], case["rows"] = rng.choice([1, 1, 1, _log_int(rng, 2, 40)]), rng.choice([1, 1, 1, 2, 3, 4, 6, 8])
            case["lo"] = _log_int(rng, 20, 131072)
            case["hi"] = _log_int(rng, case["lo"], 131072) if case["seqs"] > 1 else case["lo"]
        elif kind == "chunk":
            case["rows"], case["lo"] = _log_int(rng, 10, 4096), rng.choice([0, _log_int(rng, 20, 131072)])
            if case["lo"] > 1024 and rng.random() < 0.25:
                case["window"] = rng.choice([1024, 4096])
            case["layers"] = 1
        else:
            case["lo"] = _log_int(rng, 4000, 262000)
            if kind == "sparse_chunk":
                case["rows"], case["layers"] = _log_int(rng, 16, 512), 1
        if kind != "rows":
            case["hi"] = case["lo"]
        need = work(case)
        # no more than the largest listed cases, and memory for a batch padded to its longest sequence
        padded = case["layers"] * case["seqs"] * (case["hi"] + case["rows"]) * kv_heads * dim * 4
        if need["bytes"] <= most_bytes and need["flops"] <= most_flops and padded <= 8 << 30:
            return case


def _lengths(case):
    """Cached keys of each sequence in front of the pass's own rows."""
    if case["lo"] == case["hi"]:
        return [case["lo"]] * case["seqs"]
    stream = synthetic.uniform(7, "lengths", case["seqs"], math.log(case["lo"]), math.log(case["hi"] + 1))
    return [max(case["lo"], min(case["hi"], int(math.exp(float(u))))) for u in stream]


def _context_of_the_program():
    global _context
    if _context is None:
        _context = HIPContext(0)
    _context.use_torch_stream()
    return _context


class State:
    """What a runner keeps between steps: the context, caches, weights and the buffers a step writes."""


def _weights(gen, rows, columns, bits):
    levels = torch.randint(0, 256, (rows, columns * bits // 8), generator=gen, device=DEVICE, dtype=torch.uint8)
    span = 0.02 + 0.08 * torch.rand(rows, columns // 64, generator=gen, device=DEVICE)
    return levels, (span / ((1 << bits) - 1)).to(torch.bfloat16), (-0.5 * span).to(torch.bfloat16)


def prepare(case, seed):
    ctx = _context_of_the_program()
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float16)

    def norm_weight(n):
        return (1.0 + 0.1 * torch.randn(n, generator=gen, device=DEVICE)).to(torch.bfloat16)

    s = State()
    s.case, s.ctx = case, ctx
    heads, kv_heads, dim, rows, layers = (case[k] for k in ("heads", "kv_heads", "dim", "rows", "layers"))
    width, tokens = heads * dim, case["seqs"] * rows
    s.lengths, s.slots, s.scale = _lengths(case), list(range(case["seqs"])), dim ** -0.5
    total = max(s.lengths) + rows
    ring = 0
    if case["window"]:
        # room for the window, the chunk and the partial block in front; a chunk's rows do not wrap
        ring = -(-(case["window"] + rows + 32) // 32) * 32
        while s.lengths[0] % ring + rows > ring:
            ring += 32
    s.kv = KVCacheManager(ctx, layers, kv_heads, dim, slots=case["seqs"], max_context=total, initial_capacity=total,
                          precision_bits=case["kv_bits"], ring_capacity=ring)
    for layer in range(layers):
        for slot, length in enumerate(s.lengths):
            at = max(0, length - case["window"] - 32) if ring else 0
            while at < length:
                n = min(length - at, 65536, ring - at % ring if ring else 65536)
                s.kv.append(layer, slot, at, randn(n, kv_heads * dim), randn(n, kv_heads * dim))
                at += n
    for slot, length in enumerate(s.lengths):
        s.kv.advance(slot, length)
    # a step's projections, as the layers in front of the attention leave them
    s.packed = [randn(tokens, 2 * width) for _ in range(layers)]
    s.k = [randn(tokens, kv_heads * dim) for _ in range(layers)]
    s.v = [randn(tokens, kv_heads * dim) for _ in range(layers)]
    s.q_norm, s.k_norm = [norm_weight(dim) for _ in range(layers)], [norm_weight(dim) for _ in range(layers)]
    s.o_proj = [_weights(gen, HIDDEN, width, case["w_bits"]) for _ in range(layers)]
    s.q, s.gate = torch.empty(tokens, width, dtype=torch.float16, device=DEVICE), torch.empty(tokens, width, dtype=torch.float16, device=DEVICE)
    s.attended = [torch.zeros(tokens, width, dtype=torch.float16, device=DEVICE) for _ in range(layers)]
    s.y = [torch.zeros(tokens, HIDDEN, dtype=torch.float16, device=DEVICE) for _ in range(layers)]
    s.epilogue, s.attention, s.prefill, s.projection = QKVEpilogue(ctx), Attention(ctx), PrefillAttention(ctx), AffineProjection(ctx)
    if case["kind"].startswith("sparse"):
        s.indexer = QSAIndexer(ctx, INDEX_HEADS, INDEX_DIM, INDEX_RATIO, INDEX_BUDGET, THETA, capacity=total)
        s.index_rows = [randn(tokens, INDEX_HEADS * INDEX_DIM) for _ in range(layers)]
        s.index_q = torch.empty(tokens, INDEX_HEADS * INDEX_DIM, dtype=torch.float16, device=DEVICE)
        s.index_q_norm, s.index_k_norm = [norm_weight(INDEX_DIM) for _ in range(layers)], [norm_weight(INDEX_DIM) for _ in range(layers)]
        for layer in range(layers):
            s.indexer.raw_key_destination(layer, 0, total).copy_(randn(total, INDEX_DIM))
            s.indexer.encode_pool_prefill(layer, 0, s.lengths[0], s.index_k_norm[layer], EPS)
    return s


def run(s):
    case = s.case
    heads, rows, seqs = case["heads"], case["rows"], case["seqs"]
    width, start, tokens = heads * case["dim"], s.lengths[0], seqs * rows
    outputs = []
    for layer in range(case["layers"]):
        q, gate, attended = s.q, s.gate, s.attended[layer]
        s.epilogue.encode(s.kv, layer, s.packed[layer], s.k[layer], s.v[layer], s.q_norm[layer], s.k_norm[layer], q, gate, heads,
                          s.lengths, rows, EPS, ROTARY_DIM, THETA, slots=s.slots)
        if case["kind"] == "rows" and rows == 1:
            s.attention.encode_full(s.kv, layer, q, attended, heads, [n + 1 for n in s.lengths], s.scale, slot=s.slots, gate=gate)
        elif case["kind"] == "rows":
            s.attention.encode_verify_rows(s.kv, layer, q, attended, heads, s.lengths, rows, s.scale, s.slots, gate=gate)
        elif case["kind"] == "chunk":
            params = PrefillAttentionParams(start, rows, start + rows, heads, s.scale, width, width, width, sliding_window=case["window"])
            s.prefill.encode_causal(s.kv, layer, 0, q, attended, params, gate=gate)
        elif case["kind"] == "sparse_rows":
            s.indexer.encode_decode_step(layer, start, s.index_rows[layer], s.index_k_norm[layer], s.index_q_norm[layer], EPS)
            mask = s.indexer.select_keys(start + 1)
            s.attention.encode_full_keep(s.kv, layer, q, attended, heads, start + 1, mask, s.scale, gate=gate)
        else:
            s.indexer.encode_pool_prefill(layer, start, rows, s.index_k_norm[layer], EPS)
            s.index_q.copy_(s.index_rows[layer])  # (they are normed and rotated in place; the projection would write them here)
            s.indexer.encode_scores(layer, s.index_q, s.index_q_norm[layer], start, rows, EPS)
            chosen = s.indexer.select_keys_prefill(start, rows, mask=False)
            params = PrefillAttentionParams(start, rows, start + rows, heads, s.scale, width, width, width)
            s.prefill.encode_causal(s.kv, layer, 0, q, attended, params, gate=gate, keep_indices=chosen.indices,
                                    keep_index_stride=chosen.index_stride, keep_counts=chosen.counts)
        s.projection.encode(case["w_bits"], *s.o_proj[layer], attended, s.y[layer], HIDDEN, width, tokens)
        outputs += [attended, s.y[layer]]
    if case["kind"] == "sparse_rows":
        outputs.append(mask)
    elif case["kind"] == "sparse_chunk":
        outputs += [chosen.indices, chosen.counts]
    return outputs


def work(case):
    heads, kv_heads, dim, rows, layers, seqs = (case[k] for k in ("heads", "kv_heads", "dim", "rows", "layers", "seqs"))
    width, kv_width, tokens, sparse = heads * dim, kv_heads * dim, seqs * rows, case["kind"].startswith("sparse")
    row_bytes = 2 * kv_width * case["kv_bits"] // 8 + (0 if case["kv_bits"] == 16 else 2 * kv_width // 64 * 4)  # a token's K and V
    budget = INDEX_BUDGET + INDEX_RATIO - 1

    def weight_bytes(m, n):
        return m * n * case["w_bits"] // 8 + m * (n // 64) * 4

    keys = pairs = 0
    for length in _lengths(case):
        if sparse:
            # a row's selection; over a chunk every row may keep other keys, and the keys there are bound what is read
            keys += min(length + rows, rows * budget) if rows > 1 else min(length + 1, budget)
            pairs += rows * min(length + 1, budget)
        elif case["window"]:
            keys += min(length + rows, case["window"] + rows - 1)
            pairs += sum(min(length + r + 1, case["window"]) for r in range(rows))
        else:
            keys += length + rows
            pairs += rows * length + rows * (rows + 1) // 2
    moved = keys * row_bytes + weight_bytes(HIDDEN, width)
    # projections in and the cache rows out; the attention's rows and the layer's output
    moved += tokens * (2 * width + 2 * kv_width) * 2 + tokens * row_bytes + tokens * (width + HIDDEN) * 2
    flops = 4 * dim * heads * pairs + 2 * tokens * width * HIDDEN
    if sparse:
        blocks = (case["lo"] + rows - 1) // INDEX_RATIO + 1
        moved += tokens * INDEX_HEADS * INDEX_DIM * 2 + blocks * INDEX_DIM * 2
        moved += (case["lo"] + 1 if rows == 1 else rows * budget * 4)  # the mask, or the lists
        flops += 2 * tokens * INDEX_HEADS * INDEX_DIM * blocks
    return {"bytes": layers * moved, "flops": layers * flops}


def tolerance(case):
    # Against the same pass in float64 over the rows as stored: fp16 caches 3-4.6e-4 (the layer's fp16 roundings), quantised ones
    # 5-7.2e-4 (a probability times a group's scale is an fp16 operand, too); the largest single difference 1.1e-2, where a first
    # row of a prompt sees few keys.  About four times that.  The selections came out the same over float64 scores; a tie that
    # a last bit decides moves a block of four cells, and the list's entries between the two places with it.
    t = {"rel": 2e-3 if case["kv_bits"] == 16 else 3e-3, "max": 4e-2}
    if case["kind"].startswith("sparse"):
        t["differ"] = 2e-3
    return t
