"""The tile path (Loop64, Loop32 and batched Linked List frames) at the sizes
where it changes course, against the CPU oracle.

A stream is built from 64-fragment chunks: the first `length` fragments of a
chunk lie on consecutive targets of one tile of 64 targets, the others on a
filler tile, so the tile receives exactly `runs` runs of `length` fragments.

Bar: bit-exact. Keys, ids, packed colours and counts are integers, and the
composite evaluates the oracle's float expressions in the oracle's order.
"""
import numpy as np
import pytest

from gpu_run import run_gpu

pytestmark = pytest.mark.gpu

LOOP32, LOOP64 = 2, 3
TILES = 7  # the last of them ragged

# (runs, length, depths): depths 0 = all different, else that many values
SHAPES = {
    "few": (3, 5, 0),
    "lds_full": (12, 58, 0),          # 696 fragments: one wave's LDS
    "lds_over": (17, 41, 0),          # 697
    "own_slots": (64, 10, 0),         # as many runs as the tile's own slots
    "lists": (65, 10, 0),             # one more
    "sorted_runs": (512, 3, 0),       # as many runs as a wave sorts
    "over_sorted_runs": (513, 3, 0),
    "all_positions": (64, 64, 0),     # 4096
    "over_positions": (80, 64, 0),
    "bin_runs": (1024, 2, 0),         # as many as the binning sorts
    "over_bin_runs": (1025, 2, 0),
    "one_target": (300, 1, 0),        # nothing on the neighbours
    "ties": (40, 33, 2),
    "deep_ties": (200, 50, 3),
}


def _stream(name, seed, swap=False):
    runs, length, depths = SHAPES[name]
    rng = np.random.default_rng(seed)
    width, height = 23, 19  # 437 targets: six tiles and 53 targets
    T = width * height
    assert (T + 63) // 64 == TILES
    tile = TILES - 2
    target = np.empty((runs, 64), np.uint32)
    for r in range(runs):
        start = 40 if length == 1 else int(rng.integers(0, 64 - length + 1))
        target[r, :length] = tile * 64 + start + np.arange(length)
        filler = r % (TILES - 2)
        target[r, length:] = filler * 64 + np.arange(64 - length)
    target = np.concatenate([target.reshape(-1), np.arange(T - 53, T, dtype=np.uint32)])  # and the ragged tile
    F = len(target)
    depth = rng.random(F, dtype=np.float32) if depths == 0 else \
        (rng.integers(0, depths, F).astype(np.float32) + 1) / np.float32(depths + 1)
    alpha = rng.uniform(0.02, 0.4, F).astype(np.float32)
    rgba = np.concatenate([rng.random((F, 3), dtype=np.float32) * alpha[:, None], alpha[:, None]], axis=1)
    if depths:
        rgba = rgba[rng.integers(0, 4, F)]  # equal colours at equal depths too
    if swap:  # not a raster order: single-fragment runs
        order = rng.permutation(F)
        target, depth, rgba = target[order], depth[order], rgba[order]
    return width, height, target, depth, np.ascontiguousarray(rgba)


@pytest.mark.parametrize("algorithm,layers", [(LOOP64, 1), (LOOP64, 8), (LOOP64, 32), (LOOP32, 4), (LOOP32, 16)])
@pytest.mark.parametrize("tail", [0, 1])
def test_tiled_frames_match_oracle(oracle, algorithm, layers, tail):
    for i, name in enumerate(SHAPES):
        for swap in (False, True):
            w, h, tg, d, c = _stream(name, 11 + i, swap)
            print(algorithm, layers, tail, name, swap, len(tg), flush=True)
            cfg = oracle.make_config(algorithm, layers, tail, w, h)
            want = oracle.run(cfg, tg, d, c)
            got = run_gpu(algorithm, layers, tail, w, h, tg, d, c, splits=1 if i % 2 else 3, max_fragments=len(tg))
            for field in ("count", "frontk_key", "frontk_val", "out"):
                assert np.array_equal(got[field].view(np.uint32), want[field].view(np.uint32)), (name, swap, field)


@pytest.mark.parametrize("large", [False, True])
def test_batched_tiles_match_oracle(oracle, large):
    """`large`: a frame of its own group too big for shared tiles, so that
    whole waves take its tiles."""
    from vk_order_independent_transparency_amd import Batch, BatchFrame, DeviceBuffer, Stream

    specs = []
    for i, name in enumerate(SHAPES):
        for j, (layers, tail) in enumerate([(1, 1), (4, 1), (8, 0), (32, 1)]):
            w, h, tg, d, c = _stream(name, 101 + 7 * i + j, swap=(i + j) % 5 == 4)
            specs.append((w, h, tg, d, c, layers, tail))
    if large:
        rng = np.random.default_rng(5)
        for layers in (2, 16):
            parts = [_stream(name, 307 + i)[2:] for i, name in enumerate(SHAPES)]
            tg = np.concatenate([p[0] + 64 * 350 * i for i, p in enumerate(parts)]).astype(np.uint32)
            d = np.concatenate([p[1] for p in parts])
            c = np.concatenate([p[2] for p in parts])
            specs.append((640, 500, tg, d, c, layers, int(rng.integers(0, 2))))
    st = Stream()
    frames, outs, keep = [], [], []
    for w, h, tg, d, c, layers, tail in specs:
        bufs = [DeviceBuffer.from_numpy(np.ascontiguousarray(a)) for a in (tg, d, c)]
        out = DeviceBuffer((w * h, 4), "float32")
        frames.append(BatchFrame(width=w, height=h, samples=1, layers=layers, tail_blend=bool(tail), target=bufs[0],
                                 depth=bufs[1], rgba=bufs[2], count=len(tg), out=out))
        outs.append(out)
        keep.append(bufs)
    with Batch(0) as b:
        for rep in range(2):  # the second run meets the structures the first one left
            b.run(frames, st)
            st.synchronize()
            print("batch run", rep, flush=True)
    for i, (w, h, tg, d, c, layers, tail) in enumerate(specs):
        cfg = oracle.make_config(oracle.LINKEDLIST, layers, tail, w, h, ll_capacity=len(tg) + 1)
        want = oracle.run(cfg, tg, d, c)["out"]
        got = outs[i].numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (i, layers, tail)
