"""GPU parity for varlen prefill calls with fewer (query tile, kv head) items than
compute units, whose tiles' keys are cut into pieces and merged (bf16 outputs within
1e-2 abs + 1e-2 rel of the fp32 oracle, as for whole tiles: pieces are kept in fp32)."""
import numpy as np
import pytest

import oracle
from helpers import assert_close, bf16_host, to_dev
from ironpangu_amd import workloads as W

pytestmark = pytest.mark.gpu


# Pieces hold at least 256 keys and are made only if the longest walk shrinks by 512.
@pytest.mark.parametrize("hq,hkv,hd,bs,chunks,rows,prior,decodes,padding", [
    (16, 2, 128, 128, 1, (2, 2), (767, 767), 0, 0),     # 769 keys: the least that is cut
    (16, 2, 128, 32, 1, (2, 2), (766, 766), 0, 0),      # 768 keys: whole
    (16, 2, 128, 128, 1, (70, 70), (9000, 9000), 0, 0),  # tens of pieces per tile
    (16, 2, 128, 64, 3, (33, 1800), (0, 3000), 5, 0),   # cut and whole tiles, decode rows
    (16, 2, 128, 64, 2, (33, 700), (500, 3000), 2, 3000),  # more rows declared than packed
    (16, 1, 256, 64, 2, (9, 60), (100, 4000), 0, 0),    # 8-row tiles
    (8, 2, 256, 32, 1, (130, 130), (2500, 2500), 1, 0),
    (8, 8, 64, 32, 2, (100, 400), (0, 2500), 0, 0),     # 256-row tiles
    (16, 16, 128, 64, 1, (300, 300), (1500, 1500), 0, 0),
    (8, 1, 64, 128, 1, (40, 40), (20000, 20000), 0, 0),
])
def test_prefill_cut_tiles(hq, hkv, hd, bs, chunks, rows, prior, decodes, padding):
    import torch
    from ironpangu_amd import ops
    case = W.mixed_host_case(11, n_chunks=chunks, chunk_lo=rows[0], chunk_hi=rows[1],
                             prior_lo=prior[0], prior_hi=prior[1], n_decode=decodes, dec_lo=1,
                             dec_hi=900, q_heads=hq, kv_heads=hkv, head_dim=hd, block_size=bs)
    h, nb = case.host, case.pool_blocks
    k_ref, v_ref = h["k_pool"].copy(), h["v_pool"].copy()
    oracle.kv_write(h["k_new"], k_ref, case.slot_mapping)
    oracle.kv_write(h["v_new"], v_ref, case.slot_mapping)
    exp = oracle.varlen_prefill(h["q"], k_ref, v_ref, case.block_tables, case.cu_seqlens,
                                case.kv_lens, hq, hkv, hd, bs, case.scale)
    q = to_dev(h["q"])
    q = torch.cat([q, q.new_zeros((padding,) + tuple(q.shape[1:]))])
    out = torch.full_like(q, 7.0)
    ops.varlen_prefill(q, to_dev(k_ref).view(nb, bs, hkv, hd), to_dev(v_ref).view(nb, bs, hkv, hd),
                       to_dev(case.block_tables), to_dev(case.cu_seqlens), to_dev(case.kv_lens),
                       case.max_q_len, case.max_kv_len, case.scale, out=out)
    torch.cuda.synchronize()
    n = int(case.cu_seqlens[-1])
    assert_close(bf16_host(out[:n].contiguous()), exp)
    assert bool((out[n:] == 7.0).all())
