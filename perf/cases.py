"""The workloads this framework is timed on, through its public entry points.

A case is a dict of plain values. Three kinds:

- ``frame``: one frame of one algorithm on a kept ``Renderer`` (clear, the
  opaque draw where there is one, append, resolve, and the display image
  where the mode has an MSAA resolve);
- ``batch``: many Linked List frames of different size and K in one
  ``Batch.run``;
- ``serve``: a burst of requests through ``Server.replay``.

Fragment streams are the synthetic sphere scenes of ``scene.py``, resident on
the GPU before the pass, as a rasteriser leaves them. torch owns the buffers;
everything runs on the null stream, which is torch's default stream too.
"""
from __future__ import annotations

import dataclasses
import math

import torch

from vk_order_independent_transparency_amd import Batch, BatchFrame, FrameConfig, Renderer, Request, Server, scene
from vk_order_independent_transparency_amd import _abi
from vk_order_independent_transparency_amd.serve import served_workload

ALG = {"simple": _abi.OIT_SIMPLE, "linkedlist": _abi.OIT_LINKEDLIST, "loop32": _abi.OIT_LOOP,
       "loop64": _abi.OIT_LOOP64, "spinlock": _abi.OIT_SPINLOCK, "interlock": _abi.OIT_INTERLOCK,
       "weighted": _abi.OIT_WEIGHTED}
BACKGROUND = 0.5
SERVED_RESOLUTIONS = ((1280, 720), (1920, 1080))


def _frame(name, alg, layers, width, height, spheres, r=(0.01, 0.05), a=(0.1, 0.5), samples=1, coverage=0, opaque=0,
           tail=True):
    c = {"kind": "frame", "alg": alg, "layers": layers, "width": width, "height": height, "spheres": spheres,
         "r0": r[0], "r1": r[1], "a0": a[0], "a1": a[1], "samples": samples, "coverage": coverage, "opaque": opaque,
         "tail": tail}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a thumbnail or a probe face: launches and latency are most of it
        _frame("ll_256_k8", "linkedlist", 8, 256, 256, 64, (0.02, 0.08), (0.2, 0.6)),
        # the headline workload: a full-HD frame through the Linked List
        _frame("ll_1080p_k16", "linkedlist", 16, 1920, 1080, 1000),
        # the same stream through the bounded buffers; the Spinlock at 8 layers is the State's default
        _frame("loop64_1080p_k8", "loop64", 8, 1920, 1080, 1000),
        _frame("spinlock_1080p_k8", "spinlock", 8, 1920, 1080, 1000),
        # a resized window: odd width and height
        _frame("simple_odd_k16", "simple", 16, 1283, 717, 700),
        # two geometry passes, deeper buffer
        _frame("loop32_900p_k16", "loop32", 16, 1600, 900, 1200),
        # ordered critical sections at a laptop's resolution
        _frame("interlock_768p_k8", "interlock", 8, 1366, 768, 800),
        # MSAA with coverage masks over an opaque scene, and the display image
        _frame("msaa4_opaque_1080p_k8", "spinlock", 8, 1920, 1080, 600, coverage=4, opaque=80),
        # 4K with four samples per pixel: the weighted blend, and the exact list at its deepest buffer
        _frame("weighted_4k_4x", "weighted", 1, 3840, 2160, 4000, (0.005, 0.03), (0.05, 0.4), samples=4),
        _frame("ll_4k_4x_k32", "linkedlist", 32, 3840, 2160, 4000, (0.005, 0.03), (0.05, 0.4), samples=4),
        # offline or multi-view rendering: frames of mixed size and K, a fifth of the spheres clustered
        {"name": "batch_24_mixed", "kind": "batch", "frames": 24, "mix": 1, "res": 2048},
        # a burst of requests to the render server
        {"name": "serve_12_burst", "kind": "serve", "requests": 12, "mix": 3, "spheres": 2000, "slots": 4},
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    pick = rng.random()
    if pick < 0.14:
        return {"kind": "batch", "frames": rng.randint(3, 16), "mix": rng.randint(1, 1 << 20),
                "res": rng.choice((256, 512, 1024))}
    if pick < 0.22:
        return {"kind": "serve", "requests": rng.randint(2, 10), "mix": rng.randint(1, 1 << 20),
                "spheres": logu(300, 1500), "slots": rng.choice((1, 2, 4))}
    alg = rng.choice(("simple", "linkedlist", "linkedlist", "loop32", "loop64", "loop64", "spinlock", "spinlock",
                      "interlock", "weighted"))
    layers = rng.choice((4, 8, 8, 16, 16, 32))
    samples, coverage, opaque = 1, 0, 0
    aa = rng.random()
    if aa < 0.2:
        samples = rng.choice((4, 8))
    elif aa < 0.35 and alg in ("linkedlist", "spinlock"):
        coverage = rng.choice((4, 8))
    if rng.random() < 0.25:
        opaque = logu(10, 100)
    width = logu(100, 2600)
    height = max(33, int(width * rng.uniform(0.45, 1.0)))
    if samples > 1 and width > 1000:
        width, height = width // 2, height // 2
    r = rng.choice(((0.01, 0.05), (0.005, 0.03), (0.02, 0.08)))
    # sphere count for a mean of 1 to 12 layers per pixel
    spheres = max(1, int(math.exp(rng.uniform(0.0, math.log(12.0))) / (2.0 * _sphere_area(r[0], r[1]))))
    return _frame("", alg, 1 if alg == "weighted" else layers, width, height, spheres, r,
                  rng.choice(((0.1, 0.5), (0.2, 0.6), (0.05, 0.4))), samples, coverage, opaque, rng.random() < 0.85)


# ---- inputs ---------------------------------------------------------------


def _sphere_area(r0, r1):
    """Expected covered fraction of the image per sphere, the part beyond the borders taken off."""
    m2 = (r0 * r0 + r0 * r1 + r1 * r1) / 3.0
    m3 = (r0 ** 3 + r0 * r0 * r1 + r0 * r1 * r1 + r1 ** 3) / 4.0
    return math.pi * m2 - 4.0 * (2.0 / 3.0) * m3


def _mix64(seed, i):
    s = scene._SplitMix64((int(seed) << 20) ^ (0x9E37 * (i + 1)))
    return s.next()


def _stream(p):
    """The scene's fragments in draw order, in torch tensors on the GPU."""
    ds = scene.DeviceScene(p)
    n = ds.fragments
    t = torch.empty(max(n, 1), dtype=torch.int32, device="cuda")
    d = torch.empty(max(n, 1), dtype=torch.float32, device="cuda")
    c = torch.empty((max(n, 1), 4), dtype=torch.float32, device="cuda")
    ds.emit(t.data_ptr(), d.data_ptr(), c.data_ptr())
    torch.cuda.synchronize()
    ds.close()
    return {"target": t[:n], "depth": d[:n], "rgba": c[:n], "count": n}


def _edge_masks(target, samples, seed):
    """Full sample masks inside a sphere's rows, partial ones at its silhouette."""
    n = target.numel()
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    full = (1 << samples) - 1
    m = torch.randint(1, full + 1, (n,), dtype=torch.int32, device="cuda", generator=g)
    inside = torch.zeros(n, dtype=torch.bool, device="cuda")
    if n > 4:
        inside[2:-2] = (target[:-4] == target[2:-2] - 1) & (target[4:] == target[2:-2] + 1)
    return torch.where(inside, torch.full_like(m, full), m)


def _scene_of(case, seed, salt, spheres, alpha):
    return scene.SceneParams(seed=_mix64(seed, salt), width=case["width"], height=case["height"], spheres=spheres,
                             radius=(case["r0"], case["r1"]), alpha=alpha, samples=case["samples"])


def _frame_inputs(case, seed):
    f = _stream(_scene_of(case, seed, 0, case["spheres"], (case["a0"], case["a1"])))
    if case["coverage"]:
        f["mask"] = _edge_masks(f["target"], case["coverage"], _mix64(seed, 2))
    if case["opaque"]:
        o = _stream(_scene_of(case, seed, 1, case["opaque"], (1.0, 1.0)))
        if case["coverage"]:
            o["mask"] = _edge_masks(o["target"], case["coverage"], _mix64(seed, 3))
        f["opaque"] = o
    return f


def _batch_scenes(case, seed):
    res = tuple(x for x in (256, 512, 1024, 2048) if x <= case["res"])
    frames = scene.batch_workload(seed=case["mix"], frames=case["frames"], resolutions=res)
    return [(dataclasses.replace(b.scene, seed=_mix64(seed, i)), b.layers) for i, b in enumerate(frames)]


def _serve_requests(case, seed):
    reqs, _ = served_workload(case["mix"], case["requests"], 1000.0, resolutions=SERVED_RESOLUTIONS,
                              spheres=(200, case["spheres"]))
    return [dataclasses.replace(q, scene=dataclasses.replace(q.scene, seed=_mix64(seed, i)))
            for i, q in enumerate(reqs)]


def prepare(case, seed):
    if case["kind"] == "batch":
        frames, outs, keep = [], [], []
        for p, layers in _batch_scenes(case, seed):
            s = _stream(p)
            out = torch.empty((p.targets, 4), dtype=torch.float32, device="cuda")
            frames.append(BatchFrame(p.width, p.height, layers, s["target"].data_ptr(), s["depth"].data_ptr(),
                                     s["rgba"].data_ptr(), s["count"], out.data_ptr()))
            outs.append(out)
            keep.append(s)
        return {"kind": "batch", "batch": Batch(0), "frames": frames, "outs": outs, "keep": keep}
    if case["kind"] == "serve":
        reqs = _serve_requests(case, seed)
        outs = [torch.empty((q.scene.targets, 4), dtype=torch.float32, device="cuda") for q in reqs]
        return {"kind": "serve", "server": Server(0, slots=case["slots"]), "reqs": reqs, "outs": outs,
                "ptrs": [o.data_ptr() for o in outs], "arrivals": [0.0] * len(reqs)}
    f = _frame_inputs(case, seed)
    n = f["count"]
    T = case["width"] * case["height"] * case["samples"]
    r = Renderer(0)
    r.configure(FrameConfig(algorithm=ALG[case["alg"]], layers=case["layers"], tail_blend=case["tail"],
                            width=case["width"], height=case["height"], samples=case["samples"],
                            coverage_samples=case["coverage"], ll_pool_nodes=n + n // 2 + 1, max_fragments=max(n, 1)))
    st = {"kind": "frame", "renderer": r, "case": dict(case), "f": f,
          "out": torch.empty((T, 4), dtype=torch.float32, device="cuda")}
    if case["coverage"]:
        st["image"] = torch.empty((case["height"], case["width"], 4), dtype=torch.uint8, device="cuda")
    return st


def _frags(f):
    return (f["target"].data_ptr(), f["depth"].data_ptr(), f["rgba"].data_ptr(), None, f["count"],
            f["mask"].data_ptr() if "mask" in f else None)


def run(state):
    if state["kind"] == "batch":
        state["batch"].run(state["frames"])
        return state["outs"]
    if state["kind"] == "serve":
        state["server"].replay(state["reqs"], state["arrivals"], state["ptrs"])
        return state["outs"]
    r, f, out = state["renderer"], state["f"], state["out"]
    r.clear()
    if "opaque" in f:
        r.draw_opaque(*_frags(f["opaque"]))
    r.append(*_frags(f))
    r.resolve(out.data_ptr())
    if "image" not in state:
        return out
    c = state["case"]
    r.finalize_srgb8(out.data_ptr(), state["image"].data_ptr(), c["width"], c["height"])
    return {"rgba": out, "image": state["image"]}


def _fragments(p):
    return 2.0 * p.spheres * _sphere_area(*p.radius) * p.targets


def work(case):
    """Every fragment (24 B, its mask 4 B) read once and every target (16 B) written once, at the expected number of
    fragments; per fragment about 40 operations to unpremultiply, encode, decode and blend."""
    if case["kind"] == "frame":
        p = _scene_of(case, 0, 0, case["spheres"], (0.0, 1.0))
        n = _fragments(p) + (_fragments(_scene_of(case, 0, 1, case["opaque"], (1.0, 1.0))) if case["opaque"] else 0.0)
        b = n * (28 if case["coverage"] else 24) + p.targets * (20 if case["coverage"] else 16)
        return {"bytes": b, "flops": 40.0 * n}
    if case["kind"] == "batch":
        ps = [p for p, _ in _batch_scenes(case, 0)]
        n = sum(_fragments(p) for p in ps)
        return {"bytes": 24.0 * n + 16.0 * sum(p.targets for p in ps), "flops": 40.0 * n}
    # the server makes its fragments itself: only the images have to be written
    ps = [q.scene for q in _serve_requests(case, 0)]
    return {"bytes": 16.0 * sum(p.targets for p in ps), "flops": 60.0 * sum(_fragments(p) for p in ps)}


# ---- the same images in 64 bits, in torch ----------------------------------


def _key(depth):
    b = depth.view(torch.int32).to(torch.int64)
    return torch.where(b < 0, -(b + 1), b + (1 << 31))


def _encode(rgba):
    """sRGB8 codes [n, 4] of premultiplied colours: the stored colour is 8 bits a channel by definition."""
    a = rgba[:, 3:]
    c = torch.where(a > 0, rgba[:, :3] / torch.where(a > 0, a, torch.ones_like(a)), torch.zeros_like(rgba[:, :3]))
    c = c.double()
    s = torch.where(c < 0.0031308, c * 12.92, 1.055 * c.clamp(min=1e-9) ** (1 / 2.4) - 0.055).clamp(0, 1)
    qa = torch.floor(a.clamp(0, 1) * 255.0 + 0.5)
    return torch.cat([torch.floor(s * 255.0 + 0.5), qa.double()], 1).to(torch.uint8)


def _decode(q):
    s = q.double() / 255.0
    lin = torch.where(s[:, :3] < 0.04045, s[:, :3] / 12.92, ((s[:, :3] + 0.055) / 1.055) ** 2.4)
    return torch.cat([lin * s[:, 3:], s[:, 3:]], 1)


def _over(top, base):
    return top + (1.0 - top[:, 3:]) * base


def _fold(dst, t, rank, col, front, live=None):
    """Blends col over (or, front to back, under) dst[t] in the order of `rank`."""
    if not t.numel():
        return dst
    for k in range(int(rank.max()) + 1):
        sel = rank == k if live is None else (rank == k) & live
        i = sel.nonzero().squeeze(1)
        if i.numel():
            d, x = dst[t[i]], col[i]
            dst[t[i]] = _over(d, x) if front else _over(x, d)
    return dst


def _rank(t_sorted, T):
    cnt = torch.bincount(t_sorted, minlength=T)
    start = torch.cumsum(cnt, 0) - cnt
    return torch.arange(t_sorted.numel(), device=t_sorted.device) - start[t_sorted], cnt, start


def _k_buffer(case, t, ids, rank, cnt, start, prem, full, K, dst, newest_first, tail):
    """The pixels of more than K fragments through a K-buffer, one fragment at a time; `rank` is the depth order.
    Newest first (the Linked List's composite) the evicted colours are blended front to back into a tail; oldest
    first (the ordered critical sections) each is blended onto dst at once."""
    deep = (cnt > K).nonzero().squeeze(1)
    T = cnt.numel()
    if not tail or not deep.numel():
        return None
    row = torch.full((T,), -1, dtype=torch.int64, device=t.device)
    row[deep] = torch.arange(deep.numel(), device=t.device)
    e = (row[t] >= 0).nonzero().squeeze(1)  # the deep pixels' fragments, in depth order
    by_id = e[torch.sort(ids[e], descending=newest_first).indices]
    by_id = by_id[torch.sort(row[t[by_id]], stable=True).indices]
    step, _, _ = _rank(row[t[by_id]], deep.numel())
    have = torch.full((deep.numel(), K), -1, dtype=torch.int64, device=t.device)
    acc = torch.zeros((deep.numel(), 4), dtype=torch.float64, device=t.device)
    order = torch.sort(step, stable=True).indices
    sizes = torch.bincount(step).tolist()
    at = 0
    for j, n in enumerate(sizes):
        i = by_id[order[at:at + n]]
        at += n
        m, r = row[t[i]], rank[i]
        if j < K:
            have[m, j] = r
            continue
        worst, slot = have[m].max(1)
        out = torch.maximum(worst, r)
        keep = worst > r
        have[m[keep], slot[keep]] = r[keep]
        pos = start[deep[m]] + out
        if newest_first:
            acc[m] = _over(acc[m], prem[pos])
        else:
            dst[deep[m]] = _over(torch.where(keep[:, None], prem[pos], full[pos]), dst[deep[m]])
    if newest_first:
        whole = torch.zeros((T, 4), dtype=torch.float64, device=t.device)
        whole[deep] = acc
        return whole
    return None


def _exact_weighted(f, T, dst):
    d, c = f["depth"].double(), f["rgba"].double()
    t = f["target"].to(torch.int64)
    x = (2.0 + d * 8.0) * 10.0 / 200.0
    dw = (0.03 / (1e-5 + x ** 4)).clamp(1e-2, 3e3)
    aw = (c.max(1).values * 40.0 + 0.01).clamp(max=1.0) ** 2
    acc = torch.zeros((T, 4), dtype=torch.float64, device="cuda").index_add_(0, t, c * (aw * dw)[:, None])
    lr = torch.zeros(T, dtype=torch.float64, device="cuda").index_add_(0, t, torch.log((1.0 - c[:, 3]).clamp(min=0)))
    r = torch.exp(lr)[:, None]
    s = torch.cat([acc[:, :3] / acc[:, 3:].clamp(min=1e-5), r], 1)
    return s * (1.0 - r) + dst * r


def _opaque_planes(f, S, T):
    """Per sample target: the nearest opaque key and colour."""
    clear = int(_key(torch.ones(1, device="cuda")))
    z = torch.full((S * T,), clear, dtype=torch.int64, device="cuda")
    col = torch.full((S * T, 4), BACKGROUND, dtype=torch.float64, device="cuda")
    col[:, 3] = 1.0
    if "opaque" not in f:
        return z, col
    o = f["opaque"]
    key, t = _key(o["depth"]), o["target"].to(torch.int64)
    for s in range(S):
        on = key < clear
        if "mask" in o:
            on &= ((o["mask"] >> s) & 1) == 1
        i = on.nonzero().squeeze(1)
        i = i[torch.sort(key[i], stable=True).indices]
        i = i[torch.sort(t[i], stable=True).indices]
        first = torch.ones(i.numel(), dtype=torch.bool, device="cuda")
        first[1:] = t[i][1:] != t[i][:-1]
        i = i[first]
        z[s * T + t[i]] = key[i]
        col[s * T + t[i]] = o["rgba"][i].double()
    return z, col


def _exact_frame(case, f):
    alg, K, tail = case["alg"], case["layers"], case["tail"]
    T = case["width"] * case["height"] * case["samples"]
    S = max(case["coverage"], 1)
    z, dst = _opaque_planes(f, S, T)
    key, t = _key(f["depth"]), f["target"].to(torch.int64)
    mask = f.get("mask")
    if "opaque" in f:
        if mask is None:
            seen = key < z[t]
        else:
            m = torch.zeros_like(mask)
            for s in range(S):
                m |= ((key < z[s * T + t]).to(torch.int32) << s) & mask
            mask, seen = m, m != 0
        i = seen.nonzero().squeeze(1)
        f = {"depth": f["depth"][i], "rgba": f["rgba"][i], "target": f["target"][i]}
        key, t = key[i], t[i]
        mask = None if mask is None else mask[i]
    if alg == "weighted":
        return _exact_weighted(f, T, dst)
    n = t.numel()
    code = _encode(f["rgba"])
    i = torch.arange(n, device="cuda")
    if alg == "loop64":  # equal depths in the order of the packed colours
        w = code.to(torch.int64)
        i = torch.sort(w[:, 0] | (w[:, 1] << 8) | (w[:, 2] << 16) | (w[:, 3] << 24), stable=True).indices
    i = i[torch.sort(key[i], stable=True).indices]
    i = i[torch.sort(t[i], stable=True).indices]
    del code
    t, key, rgba = t[i], key[i], f["rgba"][i]
    mask = None if mask is None else mask[i]
    prem = _decode(_encode(rgba))
    rank, cnt, start = _rank(t, T)
    if alg == "simple" and int(cnt.max()) > K:
        return None  # the stored set is the first K to arrive: no one answer
    if alg == "loop32":  # one layer per depth, the newest fragment's colour
        new = torch.ones(n, dtype=torch.bool, device="cuda")
        new[1:] = (t[1:] != t[:-1]) | (key[1:] != key[:-1])
        layer = torch.cumsum(new, 0) - 1
        rank = layer - layer[start.clamp(max=max(n - 1, 0))][t]
        last = torch.ones(n, dtype=torch.bool, device="cuda")
        last[:-1] = new[1:]
        live, behind, tail_col = (rank < K) & last, rank >= K, rgba
    else:
        live, behind, tail_col = rank < K, rank >= K, rgba if alg == "simple" else prem
    # the colour pass's tail, oldest first over the destination
    under = None
    if alg == "linkedlist":
        under = _k_buffer(case, t, i, rank, cnt, start, prem, None, K, None, True, tail)
    elif alg == "interlock":
        if mask is not None:
            return None
        _k_buffer(case, t, i, rank, cnt, start, prem, rgba.double(), K, dst, False, tail)
    elif tail:
        b = behind.nonzero().squeeze(1)
        b = b[torch.sort(i[b]).indices]
        b = b[torch.sort(t[b], stable=True).indices]
        order = _rank(t[b], T)[0]
        for s in range(S):
            part = dst[s * T:(s + 1) * T]
            on = None if mask is None else ((mask[b] >> s) & 1) == 1
            _fold(part, t[b], order, tail_col[b].double(), False, on)
    fr = live.nonzero().squeeze(1)
    col = torch.zeros((T, 4), dtype=torch.float64, device="cuda")
    for s in range(S):
        part = torch.zeros((T, 4), dtype=torch.float64, device="cuda")
        on = None if mask is None else ((mask[fr] >> s) & 1) == 1
        col += _fold(part, t[fr], rank[fr], prem[fr], True, on)
    col /= S
    if under is not None:
        col = _over(col, under)
    return _over(col, dst.view(S, T, 4).mean(0))


def exact(case, seed):
    if case["kind"] == "frame":
        p = _scene_of(case, 0, 0, case["spheres"], (0.0, 1.0))
        if case["alg"] != "weighted" and _fragments(p) > 1.2e8:
            return None  # sorting this many fragments and folding them layer by layer takes too long
        image = _exact_frame(case, _frame_inputs(case, seed))
        if image is None:
            return None
        return {"rgba": image, "image": None} if case["coverage"] else image
    if case["kind"] == "batch":
        todo = [(p, _abi.OIT_LINKEDLIST, k) for p, k in _batch_scenes(case, seed)]
    else:
        todo = [(q.scene, q.algorithm, q.layers) for q in _serve_requests(case, seed)]
    if sum(_fragments(p) for p, _, _ in todo) > 1.2e8:
        return None
    names = {v: k for k, v in ALG.items()}
    images = []
    for p, alg, layers in todo:
        c = _frame("", names[alg], layers, p.width, p.height, p.spheres, samples=p.samples)
        images.append(_exact_frame(c, _stream(p)))
    return images
