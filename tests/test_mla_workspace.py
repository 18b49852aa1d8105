"""The MLA workspace holds every partial that the work split can write: with
sinks each row writes one sink partial and one per share its keys touch."""
import numpy as np
import pytest

from ironpangu_amd import lib

TILE, SINK_START, ROW_COST, MIN_SHARE, SPARSE_SHARE = 32, 64, 64, 96, 960


def slots_of_plan(keys, n_sinks, workers_most, cap=1 << 31):
    """Partial slots of rows with `keys` keys each, cut into equal shares."""
    sink = TILE * -(-n_sinks // TILE) + SINK_START if n_sinks else 0
    tiles = -(-keys // TILE)
    weight = np.where(tiles > 0, ROW_COST + TILE * tiles, 0) + sink
    pos = np.cumsum(weight) - weight
    total = int(weight.sum())
    workers = max(min(-(-total // MIN_SHARE), workers_most), -(-total // cap))
    share = -(-total // workers)
    first = pos + sink + ROW_COST
    wa, wb = first // share, (first + TILE * np.maximum(tiles - 1, 0)) // share
    spread = np.where((tiles > 0) & ((n_sinks > 0) | (wb > wa)), wb - wa + 1, 0)
    return int(spread.sum()) + (len(keys) if n_sinks else 0)


@pytest.mark.parametrize("rows,keys,topk", [(700, 2048, 0), (1293, 2048, 0), (2118, 2048, 0),
                                            (4096, 512, 0), (900, 512, 512), (2118, 2048, 2048)])
@pytest.mark.parametrize("n_sinks", [0, 1, 128])
def test_workspace_holds_every_partial(rows, keys, topk, n_sinks):
    heads = 16
    size = lib().ifattn_mla_attention_workspace_size(rows, heads, 65536, 0 if topk else keys, topk,
                                                     n_sinks, 64)
    need = slots_of_plan(np.full(rows, keys), n_sinks, 2 * 256, SPARSE_SHARE if topk else 1 << 31)
    assert size >= need * heads * (512 * 2 + 16 * 4), (size, need)
