"""The lists of a batch, asked for by name (OIT_VARIANT_BATCH_LISTS): the
images of the tile path and of the single-frame Linked List bit for bit, in
every launch mode, and a choice that holds where the tuning is read and set
again."""
import numpy as np
import pytest

from test_gpu_batch import MIXED, _assert_images, _Frames, _single_frame_images, _with_density
from vk_order_independent_transparency_amd import Batch, Stream, _abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mixed():
    st = Stream()
    fr = _Frames(MIXED, st)
    return st, fr, _single_frame_images(fr, st)


def _name_lists(b, k=3, tail=1):
    t = b.tuning
    t.resolve_variant[k][tail] |= _abi.VARIANT_BATCH_LISTS
    b.tuning = t


def _list_bytes(sz):
    return 12 * sz.pool_nodes + 12 * sz.head_entries + sz.head_entries // 256 * 4


def _tile_bytes(sz):
    return 20 * (sz.pool_nodes - 1) + sz.head_entries // 64 * 776


def _run(b, st, fr, want):
    for o in fr.outs:
        o.upload(np.full(o.shape, np.nan, np.float32), st)
    b.run(fr.frames, st)
    _assert_images(fr.images(st), want)


@pytest.mark.parametrize("concurrent,graph,frame_order", [(False, False, False), (True, False, False),
                                                          (False, True, False), (True, True, False),
                                                          (False, False, True), (True, True, True)])
def test_lists_equal_single_frame(mixed, concurrent, graph, frame_order):
    st, fr, want = mixed
    print("lists", concurrent, graph, frame_order, flush=True)
    with Batch(0, concurrent=concurrent, graph=graph, frame_order=frame_order) as b:
        assert b.query(fr.frames).bytes == _tile_bytes(b.query(fr.frames))
        _name_lists(b)
        for rep in range(3):
            _run(b, st, fr, want)
        assert b.query(fr.frames).bytes == _list_bytes(b.query(fr.frames))
        b.tuning = b.tuning
        assert b.query(fr.frames).bytes == _list_bytes(b.query(fr.frames))
        _with_density(b, 0.0)  # binned, on the same pool, and back
        _run(b, st, fr, want)
        _with_density(b, 3.0e38)
        assert b.query(fr.frames).bytes == _list_bytes(b.query(fr.frames))
        _run(b, st, fr, want)
        t = b.tuning
        t.resolve_variant[3][1] = 0  # the defaults: tiles
        b.tuning = t
        assert b.query(fr.frames).bytes == _tile_bytes(b.query(fr.frames))
        _run(b, st, fr, want)


def test_tuned_path_survives_get_and_set(mixed):
    """Whichever path the tuner takes, another batch given its tuning takes the same."""
    st, fr, want = mixed
    with Batch(0) as b, Batch(0) as other:
        b.tune(fr.frames, st)
        t = b.tuning
        other.tuning = t
        assert other.query(fr.frames).bytes == b.query(fr.frames).bytes
        lists = any(v & _abi.VARIANT_BATCH_LISTS for k in t.resolve_variant for v in k)
        assert b.query(fr.frames).bytes == (_list_bytes if lists else _tile_bytes)(b.query(fr.frames))
        for x in (b, other, b):
            _run(x, st, fr, want)
        b.tune(fr.frames, st)  # the path that was given up is built again
        _run(b, st, fr, want)


def test_unknown_variant_is_still_refused():
    with Batch(0) as b:
        t = b.tuning
        t.resolve_variant[0][0] = 0x80
        with pytest.raises(_abi.OitError):
            b.tuning = t
