"""More rows with sinks than the work split has workers: every row writes its
sink partial and at least one key partial, so the workspace holds two per row."""
import math

import numpy as np
import pytest

import oracle
from helpers import assert_close, bf16_host, to_dev
from ironpangu_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_window_rows_with_sinks_beyond_the_workers():
    from ironpangu_amd import ops
    import torch
    rows, heads, bs, window = 2100, 4, 16, 40
    rng = np.random.default_rng(11)
    kv = rng.integers(1, 90, rows).astype(np.int32)
    need = (kv.astype(np.int64) + bs - 1) // bs
    pool = int(need.sum()) + 3
    table = W.block_tables_for(rng, kv, bs, pool, int(need.max()))
    q = W.bf16_randn(rng, (rows, heads, 576), 0.5)
    cache = W.bf16_randn(rng, (pool * bs, 576), 0.5)
    sk, sv = W.bf16_randn(rng, (17, 576), 0.5), W.bf16_randn(rng, (17, 512), 0.5)
    out = ops.mla_attention(to_dev(q), to_dev(cache).view(pool, bs, 576), to_dev(table), to_dev(kv),
                            int(kv.max()), window=window, sink_keys=to_dev(sk), sink_values=to_dev(sv))
    torch.cuda.synchronize()
    exp = oracle.mla_attention(q, cache, table, kv, heads, bs, 1 / math.sqrt(192.0), window=window,
                               sink_k=sk, sink_v=sv)
    assert_close(bf16_host(out), exp)
