"""Streams that are not in raster order, through the tile path: quads and
other orders in which a chunk of 64 fragments goes back and forth between
tiles (runs with gaps), shuffled fragments (runs that the tiles' lists hold
uncounted), tiles of many runs and of many fragments, and fragments without
a valid target among them.

Bar: bit-exact against the CPU oracle, as for any other order: keys, packed
colours and counts are integers, and the composite evaluates the oracle's
float expressions in the oracle's order."""
import numpy as np
import pytest

from gpu_run import run_gpu
from vk_order_independent_transparency_amd import Batch, BatchFrame, DeviceBuffer, FrameConfig, Renderer, Stream

pytestmark = pytest.mark.gpu

LOOP32, LOOP64 = 2, 3
W, H = 100, 83  # 8300 targets: 129 tiles and 44 targets
T = W * H


def _spans(rng, n, order):
    """Targets of n spans of a pixel row or two, their fragments in `order` (of a span's two rows)."""
    out = []
    for _ in range(n):
        y, x, w = rng.integers(0, H - 1), rng.integers(0, W - 8), rng.integers(4, 60)
        x1 = min(x + w, W)
        out.append(order(int(x), int(x1), int(y)))
    return np.concatenate(out)


def _quads(size):
    def order(x0, x1, y):
        r = []
        for x in range(x0, x1, size):
            for row in (y, y + 1):
                r += [row * W + k for k in range(x, min(x + size, x1))]
        return np.array(r)
    return order


def _alternate(period):
    """One fragment of tile 3, then period - 1 of others, over and over: gaps of `period` lanes."""
    def make(rng):
        k = np.arange(5000)
        tile = np.where(k % period == 0, 3, 10 + k % period)
        return tile * 64 + rng.integers(0, 64, len(k))
    return make


def _shuffled(tiles, n):
    return lambda rng: rng.permutation(np.repeat(rng.permutation(129)[:tiles], n)) * 64 + rng.integers(0, 64, tiles * n)


def _mixed(rng):
    """Raster spans, quads and shuffled chunks in turn, on the same tiles."""
    parts = []
    for i in range(40):
        parts.append(_spans(rng, 12, _quads(2)) if i % 4 == 0 else
                     _spans(rng, 8, lambda a, b, y: np.arange(a, b) + y * W) if i % 4 == 1 else
                     rng.integers(0, T, 1500))
    return np.concatenate(parts)


STREAMS = {
    "quads2": lambda rng: _spans(rng, 700, _quads(2)),
    "quads4": lambda rng: _spans(rng, 700, _quads(4)),
    "gap_8": _alternate(8),    # as long as a gap may be
    "gap_9": _alternate(9),    # one more
    "shuffled": _shuffled(129, 200),
    "shuffled_1023": _shuffled(60, 1023),  # as many runs as a wave sorts, but for joined ones
    "shuffled_1500": _shuffled(60, 1500),
    "shuffled_few_tiles": _shuffled(9, 600),  # few enough that most lanes join
    "mixed": _mixed,
    "deep_raster": lambda rng: np.concatenate([np.arange(a, a + 40) for a in rng.integers(64 * 40, 64 * 42, 700)]),
}


def _stream(name, seed, invalid=False):
    rng = np.random.default_rng(seed)
    tg = STREAMS[name](rng).astype(np.uint32)
    F = len(tg)
    if invalid:
        bad = rng.random(F) < 0.03
        tg[bad] = rng.choice(np.array([T, T + 1, T + 19, 0x80000000, 0xFFFFFFFE, 0xFFFFFFFF], np.uint32), bad.sum())
    d = rng.integers(1, 4000, F).astype(np.float32) / np.float32(4001)  # some equal depths
    a = rng.uniform(0.02, 0.4, F).astype(np.float32)
    c = np.ascontiguousarray(np.concatenate([rng.random((F, 3), dtype=np.float32) * a[:, None], a[:, None]], axis=1))
    c[F // 2:] = c[rng.integers(0, 5, F - F // 2)]  # and equal colours
    return tg, d, c


def _plain(algorithm, K, tail, tg, d, c, width=W, height=H, samples=1, twice=False):
    """The image without debug outputs, one append; with `twice`, of the context's second frame."""
    bufs = [DeviceBuffer.from_numpy(np.ascontiguousarray(x)) for x in (tg, d, c)]
    out = DeviceBuffer((width * height * samples, 4), "float32")
    with Renderer(0) as r:
        r.configure(FrameConfig(algorithm=algorithm, layers=K, tail_blend=bool(tail), width=width, height=height,
                                samples=samples, max_fragments=len(tg)))
        for _ in range(2 if twice else 1):
            r.render(*bufs, out)
        return out.numpy(), int(r.stats().tail_fragments)


def _same(got, want, what):
    assert np.array_equal(np.ascontiguousarray(got).view(np.uint32), np.ascontiguousarray(want).view(np.uint32)), what


@pytest.mark.parametrize("algorithm,layers,tail", [(LOOP64, 1, 1), (LOOP64, 8, 1), (LOOP64, 16, 1), (LOOP64, 32, 0),
                                                   (LOOP32, 2, 1), (LOOP32, 8, 1), (LOOP32, 16, 0), (LOOP32, 32, 1)])
@pytest.mark.parametrize("name", STREAMS)
def test_streams_match_oracle(oracle, algorithm, layers, tail, name):
    tg, d, c = _stream(name, 3 + layers)
    print(algorithm, layers, tail, name, len(tg), flush=True)
    want = oracle.run(oracle.make_config(algorithm, layers, tail, W, H), tg, d, c)
    out, tails = _plain(algorithm, layers, tail, tg, d, c, twice=True)
    _same(out, want["out"], "out")
    got = run_gpu(algorithm, layers, tail, W, H, tg, d, c, splits=3, max_fragments=len(tg))
    for field in ("out", "count", "frontk_key", "frontk_val"):
        _same(got[field], want[field], field)
    assert tails == got["tail_fragments"]


@pytest.mark.parametrize("algorithm", [LOOP64, LOOP32])
@pytest.mark.parametrize("name", ["quads2", "shuffled", "mixed"])
def test_invalid_targets_are_dropped(oracle, algorithm, name):
    tg, d, c = _stream(name, 29, invalid=True)
    ok = tg < T
    assert 0 < (~ok).sum() < len(tg) // 10
    print(algorithm, name, int((~ok).sum()), flush=True)
    want = oracle.run(oracle.make_config(algorithm, 8, 1, W, H), tg[ok], d[ok], c[ok])
    got, tails = _plain(algorithm, 8, 1, tg, d, c)
    _same(got, want["out"], "out")
    assert tails == _plain(algorithm, 8, 1, tg[ok], d[ok], c[ok])[1]


@pytest.mark.parametrize("algorithm", [LOOP64, LOOP32])
@pytest.mark.parametrize("name", ["quads4", "shuffled", "mixed"])
def test_streams_with_samples_and_an_opaque_draw(oracle, algorithm, name):
    rng = np.random.default_rng(41)
    tg, d, c = _stream(name, 31)
    print(algorithm, name, len(tg), flush=True)
    want = oracle.run(oracle.make_config(algorithm, 8, 1, W // 2, H, samples=2), tg, d, c)
    _same(_plain(algorithm, 8, 1, tg, d, c, width=W // 2, samples=2)[0], want["out"], "samples")
    n = 6000
    otg = rng.integers(0, T, n).astype(np.uint32)
    od = rng.uniform(0.3, 1.0, n).astype(np.float32)
    oc = np.ascontiguousarray(np.concatenate([rng.random((n, 3), dtype=np.float32), np.ones((n, 1), np.float32)], 1))
    opq = oracle.opaque_pass(oracle.make_config(algorithm, 8, 1, W, H), otg, od, oc)
    want = oracle.run(oracle.make_config(algorithm, 8, 1, W, H, opaque=opq), tg, d, c)
    got = run_gpu(algorithm, 8, 1, W, H, tg, d, c, max_fragments=len(tg), opaque=(otg, od, oc, None))
    for field in ("out", "count", "frontk_key", "frontk_val"):
        _same(got[field], want[field], field)


def test_batched_streams_match_oracle(oracle):
    st = Stream()
    frames, wants, keep = [], [], []
    for i, name in enumerate(STREAMS):
        tg, d, c = _stream(name, 51 + i, invalid=name == "quads2")
        K, tail = ((4, 1), (8, 1), (16, 0), (32, 1))[i % 4]
        ok = tg < T
        wants.append(oracle.run(oracle.make_config(oracle.LINKEDLIST, K, tail, W, H, ll_capacity=len(tg) + 1), tg[ok],
                                d[ok], c[ok])["out"])
        bufs = [DeviceBuffer.from_numpy(x) for x in (tg, d, c)]
        out = DeviceBuffer((T, 4), "float32")
        frames.append(BatchFrame(width=W, height=H, layers=K, tail_blend=bool(tail), target=bufs[0], depth=bufs[1],
                                 rgba=bufs[2], count=len(tg), out=out))
        keep.append(bufs)
    with Batch(0) as b:
        for rep in range(2):
            print("batch", rep, flush=True)
            b.run(frames, st)
            st.synchronize()
    for name, f, want in zip(STREAMS, frames, wants):
        _same(f.out.numpy(), want, name)


@pytest.mark.parametrize("algorithm,layers", [(LOOP64, 8), (LOOP32, 8)])
def test_streams_of_an_unshared_frame(oracle, algorithm, layers):
    """Over 8192 tiles, so that a wave takes whole tiles: shuffled fragments, a few per tile and up to
    1500 on some, and quads."""
    w, h = 1100, 500  # 8594 tiles
    rng = np.random.default_rng(layers)
    n = np.zeros(8593, np.int64)
    n[rng.permutation(8593)[:90]] = rng.choice([70, 400, 700, 1023, 1500], 90)
    n += rng.integers(0, 4, 8593)
    tg = rng.permutation(np.repeat(np.arange(8593), n)) * 64
    tg = tg + rng.integers(0, 64, len(tg))
    x, y = rng.integers(0, w - 40, 300), rng.integers(0, h - 1, 300)
    quads = [(yy + r) * w + xx + k for xx, yy in zip(x, y) for b in range(0, 40, 2) for r in (0, 1) for k in (b, b + 1)]
    tg = np.concatenate([tg, np.array(quads)]).astype(np.uint32)
    F = len(tg)
    d = rng.integers(1, 4000, F).astype(np.float32) / np.float32(4001)
    a = rng.uniform(0.02, 0.4, F).astype(np.float32)
    c = np.ascontiguousarray(np.concatenate([rng.random((F, 3), dtype=np.float32) * a[:, None], a[:, None]], axis=1))
    print(algorithm, F, flush=True)
    want = oracle.run(oracle.make_config(algorithm, layers, 1, w, h), tg, d, c)
    _same(_plain(algorithm, layers, 1, tg, d, c, width=w, height=h, twice=True)[0], want["out"], "out")
