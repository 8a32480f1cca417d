"""tt_hip_attn_prefill at the edges of its routes.

The entry point serves a chunk by one of several kernels, chosen from the chunk's rows, the keys before it, the
cache's precision and the head shape (the chunk kernel whole or over key ranges, the split-K kernel with one-head or
GQA-packed tiles).  Same semantics and the same bar (max-abs 2e-3, mean-abs 2e-4 against the CPU oracle) whichever
serves: the cases sit on both sides of every threshold -- 31 / 32, 63 / 64 rows, 2559 / 2560, 4095 / 4096,
32767 / 32768 keys, 786,432 / rows keys (where the key ranges take over from the split-K tiles), and the keys up to
which the split-K tiles are 16 rows high -- over fp16 and over 8-bit pages, for head groups the chunk kernel takes and
one it does not."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_attention_api import _check, _dev, _prefill

pytestmark = pytest.mark.gpu


def _chunk(gpu_ctx, bits, H, KH, D, rows, kv_valid):
    from tinytitan_amd.engine import KVCacheManager
    import torch
    start = kv_valid - rows
    r = np.random.default_rng(rows * 1000003 + kv_valid * 7 + bits)
    k = r.standard_normal((kv_valid, KH, D)).astype(np.float16)
    v = r.standard_normal((kv_valid, KH, D)).astype(np.float16)
    q = r.standard_normal((rows, H * D)).astype(np.float16)
    g = r.standard_normal((rows, H * D)).astype(np.float16)
    kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=kv_valid, initial_capacity=kv_valid, precision_bits=bits)
    kd, vd = _dev(k), _dev(v)
    torch.cuda.synchronize()
    kv.append(0, 0, 0, kd, vd)
    gpu_ctx.synchronize()
    if bits == 16:
        k32, v32 = k.astype(np.float32), v.astype(np.float32)
    else:  # what the oracle's loader reads back from the oracle's quantiser
        k32 = oracle.kv_dequantize_rows(oracle.kv_quantize_rows(k.reshape(kv_valid, -1).astype(np.float32), bits), KH * D, bits)
        v32 = oracle.kv_dequantize_rows(oracle.kv_quantize_rows(v.reshape(kv_valid, -1).astype(np.float32), bits), KH * D, bits)
    scale = float(D) ** -0.5
    got = _prefill(gpu_ctx, kv, q, start, rows, kv_valid, H, scale, gate=g)
    want = oracle.attention_batch(q.astype(np.float32), k32.reshape(kv_valid, -1), v32.reshape(kv_valid, -1), rows, start, H, KH, D,
                                  scale, threads=4)
    want = want.reshape(rows, -1) / (1 + np.exp(-g.astype(np.float64)))
    _check(got, want, f"{rows} rows behind {start} keys, {H}q/{KH}kv/{D}, {bits} bits")
    kv.close()


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("rows,kv_valid", [(8, 2560), (9, 2559), (9, 2560), (31, 32768), (32, 32767), (32, 32768), (63, 4096),
                                           (64, 4095), (64, 4096), (65, 8200), (130, 2047), (130, 2049), (257, 300),
                                           (1030, 1030), (520, 1600), (64, 12287), (64, 12288), (128, 6143), (128, 6144),
                                           (200, 4095), (200, 4096), (310, 2559), (310, 2560), (32, 20480), (32, 20481),
                                           (48, 16384), (96, 1700), (96, 1720)])
def test_rows_and_keys_on_both_sides_of_every_threshold(gpu_ctx, bits, rows, kv_valid):
    _chunk(gpu_ctx, bits, 8, 2, 128, rows, kv_valid)


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("H,KH,D,rows,kv_valid", [(6, 2, 128, 5, 9000), (6, 2, 128, 300, 5000), (6, 2, 64, 1100, 1100),
                                                   (4, 4, 128, 40, 20000), (16, 2, 256, 3, 33000)])
def test_head_groups_the_chunk_kernel_does_not_take_and_few_rows(gpu_ctx, bits, H, KH, D, rows, kv_valid):
    _chunk(gpu_ctx, bits, H, KH, D, rows, kv_valid)


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize("H,KH,D,rows,kv_valid", [(24, 2, 256, 300, 2040), (24, 2, 256, 300, 2060), (24, 2, 256, 96, 4090), (24, 2, 256, 96, 4100),
                                                   (24, 2, 256, 300, 3300), (12, 1, 64, 200, 9000), (40, 8, 128, 130, 3020), (40, 8, 128, 130, 3030)])
def test_heads_that_leave_a_tiles_rows_empty_on_both_sides_of_the_ranges(gpu_ctx, bits, H, KH, D, rows, kv_valid):
    _chunk(gpu_ctx, bits, H, KH, D, rows, kv_valid)


@pytest.mark.parametrize("bits", [16, 8])
def test_ranges_that_would_have_to_grow_their_stores_inside_a_capture(gpu_ctx, bits):
    # 300 rows of 24/2 heads behind 2,200 keys go over key ranges, whose partial results (and over 8 bits dequantised pages) a context that has run
    # nothing yet has no room for: captured then, the split-K tiles, which need neither; run eagerly afterwards, the ranges.
    import torch
    from tinytitan_amd.engine import HIPContext, KVCacheManager, PrefillAttention, PrefillAttentionParams
    H, KH, D, T, rows = 24, 2, 256, 2500, 300
    r = np.random.default_rng(bits)
    ctx = HIPContext(gpu_ctx.device)
    kv = KVCacheManager(ctx, 1, KH, D, slots=1, max_context=T, initial_capacity=T, precision_bits=bits)
    k, v, q = (_dev(r.standard_normal((n, w)).astype(np.float16)) for n, w in ((T, KH * D), (T, KH * D), (rows, H * D)))
    out, again = torch.zeros_like(q), torch.zeros_like(q)
    torch.cuda.synchronize()
    kv.append(0, 0, 0, k, v)
    ctx.synchronize()
    params, pre = PrefillAttentionParams(T - rows, rows, T, H, D ** -0.5, H * D, H * D, H * D), PrefillAttention(ctx)
    def captured(into):
        ctx.graph_begin()
        try:
            pre.encode_causal(kv, 0, 0, q, into, params)
        finally:  # (no capture is left open)
            graph = ctx.graph_end()
        return graph

    graph = captured(out)
    replays = []
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.launch()
        ctx.synchronize()
        replays.append(out.float().cpu().numpy())
    graph.close()
    # with the stores there, a capture takes the ranges: the eager call's bits
    pre.encode_causal(kv, 0, 0, q, out, params)
    ctx.synchronize()
    graph = captured(again)
    graph.launch()
    ctx.synchronize()
    eager, replayed = out.float().cpu().numpy(), again.float().cpu().numpy()
    graph.close()
    kv.close()
    ctx.close()
    assert np.isfinite(eager).all() and np.abs(eager).max() > 0 and np.array_equal(eager, replayed)
    for got in replays:
        assert np.abs(got - eager).max() <= 2e-3 and not np.array_equal(got, eager)


@pytest.mark.parametrize("H,KH,D,rows,start,window,ring", [
    (24, 2, 256, 777, 150, 500, 0),       # three head sets per KV head, ragged last tile, some windows clipped, some not
    (32, 8, 128, 1029, 1237, 400, 1856),  # eight KV heads (one XCD each), over a ring
    (24, 2, 256, 300, 5001, 3000, 0),     # a window cut into key ranges, its lower edge inside the first one's blocks
    (32, 8, 128, 291, 4100, 3001, 3520),  # ... over a ring: 4,100 % 3,520 + 291 rows do not wrap
    (16, 2, 256, 270, 1900, 4096, 0),     # a window that clips no row is none: the dense routes
    (24, 2, 256, 256, 300, 33, 0),        # a short window: the split-K tiles all at work at once
    (24, 2, 256, 257, 300, 33, 0),        # ... and two tiles more
    (32, 8, 128, 512, 600, 128, 0), (32, 8, 128, 513, 600, 128, 0),
    (16, 2, 256, 1030, 40, 0, 0),         # no window: the causal triangle, the longest tile first
    (12, 1, 64, 2100, 3, 0, 0)])          # one KV head, 66 tiles of three head sets: a second round of workgroups
def test_whole_chunks_in_single_tiles(gpu_ctx, H, KH, D, rows, start, window, ring):
    import torch
    from tinytitan_amd.engine import KVCacheManager, PrefillAttention, PrefillAttentionParams
    total, scale = start + rows, float(D) ** -0.5
    r = np.random.default_rng(rows + start)
    k, v = (r.standard_normal((total, KH * D)).astype(np.float16) for _ in range(2))
    q, g = (r.standard_normal((rows, H * D)).astype(np.float16) for _ in range(2))
    kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=total, initial_capacity=total, ring_capacity=ring)
    first = max(0, start - window - 32) if ring else 0
    at = first
    while at < total:  # (a ring takes ranges that do not wrap)
        n = min(total - at, ring - at % ring) if ring else total - at
        kd, vd = _dev(k[at:at + n]), _dev(v[at:at + n])
        torch.cuda.synchronize()
        kv.append(0, 0, at, kd, vd)
        gpu_ctx.synchronize()
        at += n
    qd, gd = _dev(q), _dev(g)
    out = torch.full(qd.shape, float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    PrefillAttention(gpu_ctx).encode_causal(kv, 0, 0, qd, out, PrefillAttentionParams(start, rows, total, H, scale, H * D, H * D, H * D,
                                                                                     sliding_window=window), gate=gd)
    gpu_ctx.synchronize()
    want = oracle.prefill_ref(q.astype(np.float32), k.astype(np.float32), v.astype(np.float32), H * D, KH * D, D, H, KH, start, rows,
                              total, window, scale).reshape(rows, -1) / (1 + np.exp(-g.astype(np.float64)))
    _check(out.float().cpu().numpy(), want, f"{rows} rows behind {start} keys, {H}q/{KH}kv/{D}, window {window}, ring {ring}")
    kv.close()


@pytest.mark.parametrize("H,KH,D,rows,start,window", [(16, 2, 256, 650, 3980, 4096), (16, 2, 256, 513, 3617, 4096), (32, 8, 128, 257, 3873, 4096),
                                                      (24, 2, 256, 577, 8159, 8192)])
def test_key_ranges_of_a_window_that_begins_to_clip_inside_the_chunk(gpu_ctx, H, KH, D, rows, start, window):
    # The first tile's window still reaches over key 0 and the last tile is ragged: the tiles between them walk a block more, and
    # a tile's last row, whose own key lies in that block, shows whether it is walked.  The oracle on those rows.
    import torch
    from tinytitan_amd.engine import KVCacheManager, PrefillAttention, PrefillAttentionParams
    total, scale = start + rows, float(D) ** -0.5
    r = np.random.default_rng(rows + start)
    k, v = (r.standard_normal((total, KH * D)).astype(np.float16) for _ in range(2))
    q = r.standard_normal((rows, H * D)).astype(np.float16)
    for head in range(KH):  # a row's own key along its group's first query head: a row without it is off by far more than the bar
        k[start:, head * D:(head + 1) * D] = q[:, head * (H // KH) * D:][:, :D] * np.float16(0.5 * 16 * scale)
    kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=total, initial_capacity=total)
    kd, vd, qd = _dev(k), _dev(v), _dev(q)
    out = torch.full(qd.shape, float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    kv.append(0, 0, 0, kd, vd)
    PrefillAttention(gpu_ctx).encode_causal(kv, 0, 0, qd, out, PrefillAttentionParams(start, rows, total, H, scale, H * D, H * D, H * D,
                                                                                     sliding_window=window))
    gpu_ctx.synchronize()
    got = out.float().cpu().numpy()
    kv.close()
    assert np.isfinite(got).all()
    k32, v32 = k.astype(np.float32), v.astype(np.float32)
    for row in [0, *range(31, rows, 32), rows - 1]:
        want = oracle.prefill_ref(q[row:row + 1].astype(np.float32), k32, v32, H * D, KH * D, D, H, KH, start + row, 1, start + row + 1,
                                  window, scale).reshape(1, -1)
        _check(got[row:row + 1], want, f"row {row} of {rows} behind {start} keys, {H}q/{KH}kv/{D}, window {window}")


@pytest.mark.parametrize("H,KH,rows,start,window", [(16, 2, 3989, 0, 0), (16, 2, 4000, 33, 0), (16, 2, 4031, 0, 0), (8, 2, 70, 20003, 0), (32, 8, 777, 5003, 4096)])
def test_heads_of_128_in_steps_of_two_blocks(gpu_ctx, H, KH, rows, start, window):
    # Two key blocks a step: tiles, pairs of tiles (the second one's first blocks copied in behind the first one's last) and key ranges of odd and
    # even numbers of blocks.  Rows on both sides of the tiles' edges, against the oracle over each row's own keys.
    import torch
    from tinytitan_amd.engine import KVCacheManager, PrefillAttention, PrefillAttentionParams
    D = 128
    total, scale = start + rows, float(D) ** -0.5
    r = np.random.default_rng(rows + start)
    k, v = (r.standard_normal((total, KH * D)).astype(np.float16) for _ in range(2))
    q, g = (r.standard_normal((rows, H * D)).astype(np.float16) for _ in range(2))
    kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=total, initial_capacity=total)
    kd, vd, qd, gd = _dev(k), _dev(v), _dev(q), _dev(g)
    out = torch.full(qd.shape, float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    kv.append(0, 0, 0, kd, vd)
    PrefillAttention(gpu_ctx).encode_causal(kv, 0, 0, qd, out, PrefillAttentionParams(start, rows, total, H, scale, H * D, H * D, H * D,
                                                                                     sliding_window=window), gate=gd)
    gpu_ctx.synchronize()
    got = out.float().cpu().numpy()
    kv.close()
    assert np.isfinite(got).all()
    k32, v32 = k.astype(np.float32), v.astype(np.float32)
    edges = {e + o for e in range(0, rows, 32) for o in (-1, 0)}
    some = sorted(e for e in edges | {rows - 1} if 0 <= e < rows)
    for row in some[::max(1, len(some) // 60)] + [rows - 1]:
        want = oracle.prefill_ref(q[row:row + 1].astype(np.float32), k32, v32, H * D, KH * D, D, H, KH, start + row, 1, start + row + 1,
                                  window, scale).reshape(1, -1) / (1 + np.exp(-g[row:row + 1].astype(np.float64)))
        _check(got[row:row + 1], want, f"row {row} of {rows} behind {start} keys, {H}q/{KH}kv/{D}, window {window}")


@pytest.mark.parametrize("rows,kv_valid,first", [(128, 6200, 0), (128, 6300, 0), (160, 6400, 0), (160, 7300, 0), (545, 545, 0), (545, 577, 0)])
def test_infinite_values_reach_the_output_as_they_are(gpu_ctx, rows, kv_valid, first):
    # Key ranges of 13, 11, 17 and 18 blocks, and a whole tile of one row and 18 or 19 blocks: an infinite value in a visible key's
    # dim makes that dim infinite, whichever block it lies in -- the step that has one block left must not add it again with
    # probabilities of zero.  Every block from `first` on that all of the checked rows see has an infinity, in one of the dims
    # 0 .. 95 each; the other dims against the oracle.
    import torch
    from tinytitan_amd.engine import KVCacheManager
    H, KH, D = 8, 2, 128
    start, scale = kv_valid - rows, float(D) ** -0.5
    r = np.random.default_rng(kv_valid + rows)
    k, v = (r.standard_normal((kv_valid, KH, D)).astype(np.float16) for _ in range(2))
    q = (0.05 * r.standard_normal((rows, H * D))).astype(np.float16)
    checked = slice(rows - 1, rows) if rows > 512 else slice(0, rows)  # (a last tile of one row)
    seen = start + checked.start + 1
    infinite = v.copy()
    dims = np.zeros(D, bool)
    for block in range(first, (seen + 31) // 32 if rows > 512 else seen // 32):
        infinite[min(32 * block + 31, seen - 1), :, block % 96] = np.inf
        dims[block % 96] = True
    kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=kv_valid, initial_capacity=kv_valid)
    kd, vd = _dev(k), _dev(infinite)
    torch.cuda.synchronize()
    kv.append(0, 0, 0, kd, vd)
    gpu_ctx.synchronize()
    got = _prefill(gpu_ctx, kv, q, start, rows, kv_valid, H, scale)[checked].reshape(-1, H, D)
    kv.close()
    assert (got[:, :, dims] == np.inf).all(), f"dims {sorted(set(np.argwhere(dims[None, None] & (got != np.inf))[:, 2].tolist()))}"
    want = oracle.attention_batch(q.astype(np.float32), k.reshape(kv_valid, -1).astype(np.float32), v.reshape(kv_valid, -1).astype(np.float32),
                                  rows, start, H, KH, D, scale, threads=4).reshape(rows, H, D)[checked]
    _check(got[:, :, ~dims], want[:, :, ~dims], f"{rows} rows, {kv_valid} keys")


@pytest.mark.parametrize("H,KH,D,rows,kv_valid", [
    (24, 2, 256, 146, 2690), (24, 2, 256, 146, 2694),  # heads that leave rows of a tile empty, in front of the ranges' line and behind it: five
    (24, 2, 256, 294, 2342), (24, 2, 256, 450, 2498), (24, 2, 256, 98, 4146), (24, 2, 256, 64, 6212),  # three, two, seven and thirteen
    (64, 8, 256, 162, 4840), (64, 8, 256, 162, 4910), (64, 8, 256, 130, 6078),  # split-K tiles, two ranges and three
    (64, 16, 128, 130, 6040), (64, 16, 128, 130, 6078), (64, 16, 128, 66, 12014), (16, 2, 256, 162, 4910)])  # ... three, five and seven
def test_infinite_values_through_any_number_of_ranges(gpu_ctx, H, KH, D, rows, kv_valid):
    # As above, over ranges that do not fill the places of a combine pass: every block that all rows see has an infinity, in one of the dims 0 .. 47
    # each, and the other dims come out as they do without.
    import torch
    from tinytitan_amd.engine import KVCacheManager
    start, scale = kv_valid - rows, float(D) ** -0.5
    r = np.random.default_rng(kv_valid + rows)
    k, v = (r.standard_normal((kv_valid, KH, D)).astype(np.float16) for _ in range(2))
    q = (0.05 * r.standard_normal((rows, H * D))).astype(np.float16)
    infinite = v.copy()
    for block in range((start + 1) // 32):
        infinite[32 * block + block % 32, :, block % 48] = np.inf
    got = []
    for values in (v, infinite):
        kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=kv_valid, initial_capacity=kv_valid)
        kd, vd = _dev(k), _dev(values)
        torch.cuda.synchronize()
        kv.append(0, 0, 0, kd, vd)
        gpu_ctx.synchronize()
        got.append(_prefill(gpu_ctx, kv, q, start, rows, kv_valid, H, scale).reshape(rows, H, D))
        kv.close()
    assert np.isfinite(got[0]).all()
    assert (got[1][:, :, :48] == np.inf).all(), f"{np.isnan(got[1]).sum()} NaN"
    assert np.array_equal(got[1][:, :, 48:], got[0][:, :, 48:])


@pytest.mark.parametrize("H,KH,rows,start,window,ring", [
    (64, 8, 2048, 5000, 33, 0), (64, 8, 2048, 5000, 64, 0), (64, 8, 2048, 5000, 99, 0),  # three, four and five blocks a tile, tiles in pairs
    (64, 8, 2047, 3001, 130, 2400),                                                       # pairs over a ring that wraps inside a tile's range
    (8, 2, 4096, 50, 256, 0), (8, 2, 4096, 50, 288, 0),                                   # ten and eleven, in one round
    (8, 2, 33, 40000, 0, 0)])                                                             # key ranges of one full tile and one of one row
def test_heads_of_128_by_halves_of_the_keys(gpu_ctx, H, KH, rows, start, window, ring):
    # On both sides of the lines between the two kernels over heads of 128, rows at the tiles' edges against the oracle over each row's keys.
    import torch
    from tinytitan_amd.engine import KVCacheManager, PrefillAttention, PrefillAttentionParams
    D = 128
    total, scale = start + rows, float(D) ** -0.5
    r = np.random.default_rng(rows + start + window)
    k, v = (r.standard_normal((total, KH * D)).astype(np.float16) for _ in range(2))
    q, g = (r.standard_normal((rows, H * D)).astype(np.float16) for _ in range(2))
    kv = KVCacheManager(gpu_ctx, 1, KH, D, slots=1, max_context=total, initial_capacity=total, ring_capacity=ring)
    at = max(0, start - window - 32) if ring else 0
    while at < total:  # (a ring takes ranges that do not wrap)
        n = min(total - at, ring - at % ring) if ring else total - at
        kd, vd = _dev(k[at:at + n]), _dev(v[at:at + n])
        torch.cuda.synchronize()
        kv.append(0, 0, at, kd, vd)
        gpu_ctx.synchronize()
        at += n
    qd, gd = _dev(q), _dev(g)
    out = torch.full(qd.shape, float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    PrefillAttention(gpu_ctx).encode_causal(kv, 0, 0, qd, out, PrefillAttentionParams(start, rows, total, H, scale, H * D, H * D, H * D,
                                                                                     sliding_window=window), gate=gd)
    gpu_ctx.synchronize()
    got = out.float().cpu().numpy()
    kv.close()
    assert np.isfinite(got).all()
    edges = sorted(e + o for e in range(0, rows, 32) for o in (-1, 0) if 0 <= e + o < rows)
    for row in sorted({*edges[::max(1, len(edges) // 40)], rows - 1}):
        last = start + row + 1
        lo = max(0, last - window) if window else 0
        want = oracle.prefill_ref(q[row:row + 1].astype(np.float32), k[lo:last].astype(np.float32), v[lo:last].astype(np.float32), H * D, KH * D, D,
                                  H, KH, last - lo - 1, 1, last - lo, 0, scale).reshape(1, -1) / (1 + np.exp(-g[row:row + 1].astype(np.float64)))
        _check(got[row:row + 1], want, f"row {row} of {rows} behind {start} keys, {H}q/{KH}kv, window {window}, ring {ring}")
