"""GPU: tiles and persistent grid of a batch, set by hand and reported.

A width of 16 set by hand is a tile of 16 x 16 in both precisions (as many work items); FP32 batches also take
16 x 8, their own tile until tuned or set.  The grid counts workgroups of 512 threads: a batch's own grid is one
per CU whatever its tile.  What info() reports can be set again; every tile and grids of one, three and more
workgroups than items give the same outputs bit for bit.
"""
import numpy as np
import pytest
import torch

import tianxin_amd as txa
from test_gpu_batch import Item, run_batch

pytestmark = pytest.mark.gpu
SHAPES = [(txa.HEX8, 17, 20, 12, 0.0), (txa.TET4, 9, 18, 11, 0.05)]


@pytest.mark.parametrize("jitter", [0.0, 0.1])
@pytest.mark.parametrize("precision", [txa.FP64, txa.FP32])
def test_tiles_and_grid(engine, precision, jitter):
    its = [Item(engine, 90 + i, *s[:4], s[4] + jitter) for i, s in enumerate(SHAPES)]
    b = txa.Batch(engine, [it.m for it in its], precision=precision)
    try:
        own = b.info()
        assert (own["tile_x"], own["tile_y"]) == (16, 8 if precision == txa.FP32 else 16)
        assert own["grid"] == torch.cuda.get_device_properties(0).multi_processor_count
        xs = [it.state(800 + i) for i, it in enumerate(its)]
        ref = None
        for tile in [(16, 0), (16, 16), (32, 0), (32, 8)] + [(16, 8)] * (precision == txa.FP32):
            for grid in (own["grid"], 1, 3, 1 << 30):
                b.shape(tile_x=tile[0], slab=6, grid=grid, tile_y=tile[1])
                i = b.info()
                assert (i["tile_x"], i["tile_y"], i["grid"]) == (tile[0], tile[1] or 256 // tile[0], grid)
                # one column recomputed each way; 13 and 12 vertex layers in slabs of 6
                tiles = [-(-(s[1] + 1) // (i["tile_x"] - 1)) * -(-(s[2] + 1) // (i["tile_y"] - 1)) for s in SHAPES]
                assert i["items"] == 3 * tiles[0] + 2 * tiles[1]
                got = [a for fv in run_batch(b, its, xs, False, 0.0, use_graph=True) for a in fv]
                ref = ref or got
                assert all(np.array_equal(p, q) for p, q in zip(got, ref))
        for bad in [(16, 32), (32, 16), (8, 16), (16, -8)] + [(16, 8)] * (precision == txa.FP64):
            with pytest.raises(txa.TxaError) as e:
                b.shape(tile_x=bad[0], tile_y=bad[1])
            assert e.value.code == txa.TXA_ERR_INVALID
    finally:
        b.destroy()
        for it in its:
            it.m.destroy()
