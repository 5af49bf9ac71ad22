"""Device memory of Loop32 and Loop64 frames: what oit_configure reserves
(so that a frame can be captured at once), and what a served request is
granted, with and without tail blending."""
import numpy as np
import pytest

from conftest import deep_scene
from vk_order_independent_transparency_amd import DeviceBuffer, FrameConfig, Renderer, _abi, scene, serve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algorithm", [_abi.OIT_LOOP, _abi.OIT_LOOP64])
@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("sized", [True, False])
def test_appends_allocate_nothing(oracle, algorithm, tail, sized):
    """A frame of up to max_fragments, in three appends. Without max_fragments: Loop32 without a
    tail, of up to 1.5 fragments a slot (no other frame without it was free of allocation)."""
    if not sized and (tail or algorithm != _abi.OIT_LOOP):
        pytest.skip("grows on demand")
    K = 4
    p, tg, d, c = deep_scene(seed=5, spheres=30)
    F, T = len(tg), p.targets
    assert sized or F <= 1.5 * K * T
    bt, bd, bc = DeviceBuffer.from_numpy(tg), DeviceBuffer.from_numpy(d), DeviceBuffer.from_numpy(c)
    out = DeviceBuffer((T, 4), "float32")
    with Renderer(0) as r:
        r.configure(FrameConfig(algorithm=algorithm, layers=K, tail_blend=tail, width=p.width, height=p.height,
                                max_fragments=F if sized else 0))
        before = r.sizes().resident_bytes
        r.clear()
        for a, b in ((0, F // 3), (F // 3, F // 2), (F // 2, F)):
            r.append(bt.view(a, b - a), bd.view(a, b - a), bc.view(a, b - a), count=b - a)
        r.resolve(out)
        assert r.sizes().resident_bytes == before
    want = oracle.run(oracle.make_config(algorithm, K, int(tail), p.width, p.height), tg, d, c)["out"]
    assert np.array_equal(out.numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("algorithm", [_abi.OIT_LOOP, _abi.OIT_LOOP64])
@pytest.mark.parametrize("spheres", [2, 300])
def test_budget_holds_without_a_tail(algorithm, spheres):
    """One request on a budget of its own bytes: the tiles' structures (776 bytes per 64 targets,
    8 a fragment, 35 KB), or what the slots would take where that is more, and the stream."""
    p = scene.SceneParams(seed=7, width=200, height=150, spheres=spheres, radius=(0.03, 0.1), alpha=(0.1, 0.5))
    F, T = scene.count(p), p.targets
    own = max(-(-T // 64) * 776 + 8 * F + 4 * (128 + 8192) + 64 * 32,
              12 * T if algorithm == _abi.OIT_LOOP else 12 * T + 8 * -(-F // 64))
    budget = own + (24 * F + 16 * T) * 5 // 4 + 64
    with serve.Server(0, slots=1, budget_bytes=budget) as s:
        done = s.replay([serve.Request(p, algorithm, 1, tail_blend=False)], np.zeros(1))
        st = s.stats()
    assert done[0].status == 0
    assert st.peak_held_bytes <= budget, (st.peak_held_bytes, budget, F, T)
