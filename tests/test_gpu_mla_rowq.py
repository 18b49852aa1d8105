"""GPU parity of MLA window attention over row-quantized latent rows
(ifattn_mla_window_attention_rowq): int8 or int4 codes with one fp32 scale per
row, as if_cache_quantize writes them (native/kernels/cache_quantization.cpp:12-38),
dequantized in registers. The reference dequantizes the whole cache to bf16
(if_cache_dequantize, token_executor.h:806-822) and attends over that
(:863-906); the expected values here are exactly that: the oracle's window
attention over oracle_dequant_legacy's bf16 rows. bf16 outputs within 1e-2
abs + 1e-2 rel. Codes and scales come from oracle_quant_legacy (the reference
kernel's arithmetic, pinned in tests/test_oracle.py); the attention-state test
writes them with the product's if_cache_quantize instead."""
import math
import os

import numpy as np
import pytest

import oracle
from helpers import assert_close, bf16_host, to_dev
from ironpangu_amd import workloads as W

pytestmark = pytest.mark.gpu
f32 = np.float32
SCALE = 1.0 / math.sqrt(192.0)


def bf(x):
    return W.bf16_bits(np.asarray(x, np.float32))


def quantize_pool(lat_bits, bits):
    rows = lat_bits.shape[0]
    packed = np.zeros((rows, 576 * bits // 8), np.uint8)
    scales = np.zeros(rows, np.float32)
    for r in range(rows):
        packed[r], scales[r] = oracle.quant_legacy(lat_bits[r], bits)
    deq = oracle.dequant_legacy(packed.reshape(-1), scales, rows - 1, 576, bits).reshape(rows, 576)
    return packed, scales, deq


def batch(seed, counts, kv, bs, heads, bits, std=0.5):
    rng = np.random.default_rng(seed)
    kv = np.asarray(kv, np.int32)
    need = (kv.astype(np.int64) + bs - 1) // bs
    pool = int(need.sum()) + 8
    stride = int(need.max()) + 2
    table = W.block_tables_for(rng, kv, bs, pool, stride)
    rows = int(sum(counts))
    cu = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    q = bf(rng.standard_normal((rows, heads, 576)).astype(f32) * f32(0.5))
    lat = bf(rng.standard_normal((pool * bs, 576)).astype(f32) * f32(std))
    # rows of very different magnitude, and an all-zero row (scale 1)
    lat[3] = bf(rng.standard_normal(576).astype(f32) * f32(20))
    lat[5] = 0
    packed, scales, deq = quantize_pool(lat, bits)
    return q, packed.reshape(pool, bs, -1), scales, deq, table, kv, cu, stride * bs


def sinks(n, seed):
    rng = np.random.default_rng(seed)
    return (bf(rng.standard_normal((n, 576)).astype(f32) * f32(0.5)),
            bf(rng.standard_normal((n, 512)).astype(f32) * f32(0.5)))


def run(q, packed, scales, bits, table, kv, maxc, cu=None, window=0, sk=None, sv=None):
    import torch
    from ironpangu_amd import ops
    out = ops.mla_attention(to_dev(q), to_dev(packed), to_dev(np.asarray(table, np.int32)),
                            to_dev(np.asarray(kv, np.int32)), maxc,
                            cu_seqlens=None if cu is None else to_dev(cu), window=window,
                            sink_keys=None if sk is None else to_dev(sk),
                            sink_values=None if sv is None else to_dev(sv),
                            row_scales=to_dev(scales), bits=bits)
    torch.cuda.synchronize()
    return bf16_host(out)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("window,bs,with_sinks", [(0, 16, False), (0, 64, True), (37, 16, True),
                                                  (2048, 32, False), (512, 128, True)])
def test_rowq_window_batches(bits, window, bs, with_sinks):
    print(f"rowq bits={bits} window={window} bs={bs} sinks={with_sinks}", flush=True)
    counts = [1, 7, 1, 33, 2]
    kv = [5000, 300, 1, 2100, 40]
    q, packed, scales, deq, table, kv, cu, maxc = batch(5 + bits, counts, kv, bs, 12, bits)
    sk, sv = sinks(128, 6) if with_sinks else (None, None)
    got = run(q, packed, scales, bits, table, kv, maxc, cu=cu, window=window, sk=sk, sv=sv)
    exp = oracle.mla_attention(q, deq, table, kv, 12, bs, SCALE, cu_seqlens=cu, window=window,
                               sink_k=sk, sink_v=sv)
    assert_close(got, exp)


@pytest.mark.parametrize("bits", [8, 4])
def test_rowq_decode_rows_long_context(bits):
    # one row per sequence over long ragged contexts (several shares per row)
    print(f"rowq decode bits={bits}", flush=True)
    kv = [16384, 3, 777, 9000, 12000, 64]
    q, packed, scales, deq, table, kv, _, maxc = batch(21, [1] * 6, kv, 16, 16, bits)
    got = run(q, packed, scales, bits, table, kv, maxc)
    exp = oracle.mla_attention(q, deq, table, kv, 16, 16, SCALE)
    assert_close(got, exp)


def test_rowq_rejects_bad_calls():
    import torch
    from ironpangu_amd import ops
    q, packed, scales, deq, table, kv, cu, maxc = batch(3, [1], [100], 16, 4, 8)
    with pytest.raises(ValueError):  # C8-style index lists are not for row-quantized rows
        ops.mla_attention(to_dev(q), to_dev(packed), to_dev(table), to_dev(kv), maxc,
                          indices=to_dev(np.zeros((1, 8), np.int32)), row_scales=to_dev(scales))
    lib = __import__("ironpangu_amd._native", fromlist=["lib"]).lib()
    st = lib.ifattn_mla_window_attention_rowq(None, None, None, 6, None, 1, None, None, 1, 1, 0,
                                              None, None, 0, None, 4, 16, 1, 16, 0.1, None, 0, None)
    assert st == -1 and b"bits 8 or 4" in lib.ifattn_last_error()
    torch.cuda.synchronize()


@pytest.mark.parametrize("bits", [8, 4])
def test_state_attend_row_quantized(bits):
    """AttentionState(bits 8/4): rows written with the product's if_cache_quantize at
    append() rows, attend() equals the direct call bit for bit and the oracle over
    if_cache_dequantize'd rows (the reference's path) within tolerance."""
    import torch
    from ironpangu_amd import ops
    from ironpangu_amd.host import AttentionState
    from test_gpu_attention_state import view
    print(f"state rowq bits={bits}", flush=True)
    heads, cap = 6, 2048
    s = AttentionState(bits, cap, False, 1, False, 0, heads)
    g = s.geometry
    page, entries = g["page_tokens"], g["table_entries"]
    b = s.buffers()
    rng = np.random.default_rng(30 + bits)
    kv_len = 1500
    rows = bf(rng.standard_normal((kv_len, 576)).astype(f32) * f32(0.5))
    packed = view(b["cache"], (cap * 576 * bits // 8,), torch.uint8)
    scales = view(b["scales"], (cap,), torch.float32)
    dev_rows = to_dev(rows)
    pos = torch.zeros(1, dtype=torch.int64, device="cuda")
    for p in range(kv_len):
        pos.fill_(s.append(p))
        ops.cache_quantize(dev_rows[p], packed, scales, pos, bits=bits)
    q = bf(rng.standard_normal((1, heads, 576)).astype(f32) * f32(0.5))
    view(b["query"], (1, heads, 576), torch.int16).copy_(to_dev(q).view(torch.int16))
    sk, sv = sinks(128, 40)
    view(b["sink_keys"], (128, 576), torch.int16).copy_(to_dev(sk).view(torch.int16))
    view(b["sink_values"], (128, 512), torch.int16).copy_(to_dev(sv).view(torch.int16))
    stream = torch.cuda.current_stream().cuda_stream
    s.upload_table(stream)
    s.set_length(kv_len, stream)
    s.attend(window=1024, sinks=True, stream=stream)
    torch.cuda.synchronize()
    out = view(b["out"], (1, heads, 512), torch.int16).view(torch.bfloat16).clone()
    table = view(b["table"], (1, entries), torch.int32)
    kv = view(b["kv_len"], (1,), torch.int32)
    direct = ops.mla_attention(to_dev(q), packed.view(cap // page, page, -1), table, kv, entries * page,
                               window=1024, sink_keys=to_dev(sk), sink_values=to_dev(sv),
                               row_scales=scales, bits=bits)
    torch.cuda.synchronize()
    assert torch.equal(out, direct)
    # the reference's path: if_cache_dequantize to bf16 rows, then attention
    deq = torch.zeros(cap * 576, dtype=torch.bfloat16, device="cuda")
    last = torch.tensor([kv_len - 1], dtype=torch.int64, device="cuda")
    ops.cache_dequantize(packed, scales, deq, last, 576, bits=bits)
    torch.cuda.synchronize()
    deq_host = deq.view(torch.int16).cpu().numpy().view(np.uint16).reshape(cap, 576)
    host_packed = packed.cpu().numpy()
    host_scales = scales.cpu().numpy()
    assert np.array_equal(deq_host, oracle.dequant_legacy(host_packed, host_scales, kv_len - 1, 576,
                                                          bits).reshape(cap, 576))
    exp = oracle.mla_attention(q, deq_host, s.blocks()[None, :], np.array([kv_len], np.int32), heads,
                               page, SCALE, window=1024, sink_k=sk, sink_v=sv)
    assert_close(bf16_host(out), exp)


def test_state_allocation_failure_cleans_up(monkeypatch):
    """A failed device allocation part way through leaves no half-built state:
    the call fails, and the next one allocates everything (forced from the host
    with the library's IFATTN_STATE_FAIL_ALLOCATION hook)."""
    from ironpangu_amd.host import AttentionState, MetadataError
    s = AttentionState(8, 512, False, 1, False, 0, 6)
    monkeypatch.setenv("IFATTN_STATE_FAIL_ALLOCATION", "5")
    with pytest.raises(MetadataError):
        s.buffers()
    monkeypatch.delenv("IFATTN_STATE_FAIL_ALLOCATION")
    b = s.buffers()
    assert all(b[k] for k in ("cache", "table", "scales", "query", "out", "indices", "kv_len",
                              "sink_keys", "sink_values"))
    assert os.environ.get("IFATTN_STATE_FAIL_ALLOCATION") is None


@pytest.mark.parametrize("bits", [8, 4])
def test_rowq_step_edges(bits):
    # lengths around the wave (16 keys), step (64 keys) and buffer (128 keys) edges
    kv = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 193, 640]
    q, packed, scales, deq, table, kv, _, maxc = batch(31, [1] * len(kv), kv, 16, 6, bits)
    for window in (0, 20, 100):
        got = run(q, packed, scales, bits, table, kv, maxc, window=window)
        exp = oracle.mla_attention(q, deq, table, kv, 6, 16, SCALE, window=window)
        assert_close(got, exp)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("at", [70, 150, 290])
def test_rowq_scores_jump_beyond_the_running_max(bits, at):
    # From position `at` on, keys whose scores exceed all earlier ones by more
    # than 2^64: the step that meets them takes a new base before P is used
    # (and a later, smaller jump moves it after PV).
    q, packed, scales, deq, table, kv, _, maxc = batch(33, [1], [300], 16, 6, bits)
    rng = np.random.default_rng(34)
    d = rng.choice([-1.0, 1.0], 576).astype(f32)
    q[0] = bf(np.tile(d, (6, 1)) * f32(1.5))
    pool = packed.reshape(-1, packed.shape[2])
    pos = np.arange(at, 300)
    slots = table[0, pos // 16].astype(np.int64) * 16 + pos % 16
    rows = bf(d[None] * (2.0 + 0.01 * np.arange(pos.size))[:, None].astype(f32)
              + rng.standard_normal((pos.size, 576)).astype(f32) * f32(0.5))
    pool[slots], scales[slots], deq[slots] = quantize_pool(rows, bits)
    got = run(q, packed, scales, bits, table, kv, maxc)
    exp = oracle.mla_attention(q, deq, table, kv, 6, 16, SCALE)
    x = (W.bf16_to_f32(q[0, 0]) @ W.bf16_to_f32(deq[slots[0]])) * SCALE * 1.4427
    assert x > 80
    assert_close(got, exp)
