"""The queue of a batch's large tiles. Several waves of a block, and three
kernels, read the same entry: once the composite has filled the queue, nothing
may write to it (a wave that reads an entry after such a write has another tile
than its block: an access out of range, or a block of which some waves miss a
barrier)."""
import glob
import os
import re

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "vk_order_independent_transparency_amd", "csrc")


def test_queue_entries_are_written_once():
    """Only the two places that put an entry at a place drawn from the queue's
    length store to the queue."""
    stores = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.hpp"))):
        for line in open(path):
            code = line.split("//")[0]
            if re.search(r"\bdeep\[[^;]*\]\s*[|&^+-]?=[^=]", code):
                stores.append((os.path.basename(path), code.strip()))
    assert [f for f, _ in stores] == ["oit_tiles.hpp"] * 2, stores
    assert "tb.deep_base + at + lane_id()" in stores[0][1], stores  # TileQueue::flush
    assert "atomicAdd(&tb.ctl[tb.ctl_index], 1u)" in stores[1][1], stores  # end_share


@pytest.mark.gpu
@pytest.mark.parametrize("layers,tail", [(4, 1), (16, 1), (32, 0)])
@pytest.mark.parametrize("W,H,tiles", [(800, 680, 300), (160, 136, 60)], ids=["unshared", "shared"])
def test_many_deep_tiles(oracle, W, H, tiles, layers, tail):
    """8500 tiles in the group, where a wave takes whole tiles and an entry is
    a tile's number, and 340, which several waves share, where it also
    holds the shares that were left; some of them have 30 to 2500 runs of one
    fragment, on both sides of what the binning sorts (2048). Bit-exact: the
    image is a function of integer keys and of the oracle's float expressions."""
    from vk_order_independent_transparency_amd import Batch, BatchFrame, DeviceBuffer, Stream

    rng = np.random.default_rng(layers)
    runs = rng.choice([30, 300, 1023, 1025, 1400, 2047, 2048, 2049, 2500], tiles)
    which = rng.permutation(W * H // 64)[:tiles]
    # round r: one fragment on every tile that still has one, so each is a run of its own
    tile = np.concatenate([which[runs > r] for r in range(int(runs.max()))])
    assert (tile[1:] != tile[:-1]).all()
    tg = (tile * 64 + rng.integers(0, 64, len(tile))).astype(np.uint32)
    F = len(tg)
    d = rng.random(F, dtype=np.float32)
    a = rng.uniform(0.02, 0.4, F).astype(np.float32)
    c = np.ascontiguousarray(np.concatenate([rng.random((F, 3), dtype=np.float32) * a[:, None], a[:, None]], axis=1))
    want = oracle.run(oracle.make_config(oracle.LINKEDLIST, layers, tail, W, H, ll_capacity=F + 1), tg, d, c)["out"]
    st = Stream()
    t_d, d_d, c_d = (DeviceBuffer.from_numpy(x) for x in (tg, d, c))
    out = DeviceBuffer((W * H, 4), "float32")
    frame = BatchFrame(width=W, height=H, layers=layers, tail_blend=bool(tail), target=t_d, depth=d_d, rgba=c_d,
                       count=F, out=out)
    with Batch(0) as b:
        for rep in range(3):  # the later runs meet the structures that the first one left
            out.upload(np.full((W * H, 4), np.nan, np.float32), st)
            print("deep tiles", layers, tail, F, rep, flush=True)
            b.run([frame], st)
            st.synchronize()
            assert np.array_equal(out.numpy().view(np.uint32), want.view(np.uint32)), rep
