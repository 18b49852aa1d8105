"""MLA merge: one row split over many shares (96 units each: 32-key tiles plus
the row's start and sink cost), on both sides of the all-in-one path (8
partials), one batch of partial loads (32) and one wave of (m, l) pairs (64),
with and without the sink partial."""
import math

import numpy as np
import pytest

import oracle
from helpers import assert_close, bf16_host, to_dev
from ironpangu_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,n_sinks", [(16, 0), (5, 40)])
def test_merge_many_partials(heads, n_sinks):
    import torch
    from ironpangu_amd import ops
    rng = np.random.default_rng(3)
    bs, most = 64, 16384
    pool = most // bs
    cache = W.bf16_randn(rng, (pool * bs, 576), 0.5)
    table = rng.permutation(pool).astype(np.int32)[None]
    dev, dtab = to_dev(cache).view(pool, bs, 576), to_dev(table)
    sk = W.bf16_randn(rng, (n_sinks, 576), 0.5) if n_sinks else None
    sv = W.bf16_randn(rng, (n_sinks, 512), 0.5) if n_sinks else None
    for kv in (500, 600, 700, 800, 900, 1000, 2700, 2900, 3000, 3100, 3300, 5800, 6000, 6100, 6300, 16384):
        q = W.bf16_randn(rng, (1, heads, 576), 0.5)
        lens = np.array([kv], np.int32)
        out = ops.mla_attention(to_dev(q), dev, dtab, to_dev(lens), most,
                                sink_keys=None if sk is None else to_dev(sk),
                                sink_values=None if sv is None else to_dev(sv))
        torch.cuda.synchronize()
        exp = oracle.mla_attention(q, cache, table, lens, heads, bs, 1 / math.sqrt(192.0), sink_k=sk,
                                   sink_v=sv)
        assert_close(bf16_host(out), exp, what=f"kv {kv}")
