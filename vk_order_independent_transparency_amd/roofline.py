"""Algorithmic (compulsory) HBM bytes of each kernel and of a whole frame.

One place for the formulas that bench.py's `roofline` block uses.
F = fragments of the frame, P = targets (pixels x samples), K = layers,
N = fragments that end in the colour-pass tail.

Linked List (this build's layout: 8-byte (depth key, colour) node word plus
a 4-byte link word per node, 4-byte head per target):
  clear    : 4P                      (head words)
  store    : 20F in (depth 4 + premultiplied RGBA 16) + 12F out (node + kUnset link)
  link     : 4F in (target) + 8F (head read-modify-write, one per fragment
             without run merging) + 4F out (link word)
  resolve  : 4P (heads) + 12F (nodes) + 16P (RGBA out)
Frame total 60F + 24P. The reference's layout (16-byte uvec4 nodes,
oitLinkedList.frag.glsl:77-82) needs 64F + 24P for the same work; frame
fractions are reported against that figure so the two layouts are compared
on the same work.
"""
from __future__ import annotations

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E, published


def ll_stage_bytes(F: int, P: int, fused: bool = True) -> dict:
    """Per-launch algorithmic bytes. Fused append (default): stream in 24F,
    node word 8F, link word 4F, head read-modify-write 8F. The resetting
    resolve: heads 4P read + 4P reset, nodes 12F read + 4F link reset, 16P out.
    Split append: store 32F (stream 20F in, node 8F + kUnset link 4F out) and
    link 16F (target 4F, head read-modify-write 8F, link 4F)."""
    if fused:
        return {"clear": 0, "store": 44 * F, "resolve": 8 * P + 16 * F + 16 * P}
    return {"clear": 0, "store": 32 * F, "link": 16 * F, "resolve": 8 * P + 16 * F + 16 * P}


def ll_frame_bytes_reference(F: int, P: int) -> int:
    """64F + 24P: the reference node layout's compulsory traffic for one frame."""
    return 64 * F + 24 * P


def tile_stage_bytes(F: int, P: int, runs: int = 0) -> dict:
    """Loop64 and Loop32, which composite tiles of 64 targets: no clear (the
    composite leaves the run structures empty); the listing pass reads the
    targets 4F and writes 8 bytes a run; the composite reads the runs and the
    stream 24F and writes RGBA 16P. Whatever K, with a tail or without (a
    tail's full colours, Loop32's, are read a second time and not counted).
    `runs`: of consecutive fragments of one tile, about F / 30 in raster
    order; without it the bytes that every order needs."""
    return {"clear": 0, "store": 4 * F + 8 * runs, "resolve": 24 * F + 8 * runs + 16 * P}


def loop64_stage_bytes(F: int, P: int, K: int, occupied: int | None = None, tail: bool = True) -> dict:
    """tile_stage_bytes (K, occupied slots and tail make no difference to it)."""
    return tile_stage_bytes(F, P)


def kbuffer_stage_bytes(F: int, P: int, K: int, spin: bool) -> dict:
    aux = 12 if spin else 4
    return {
        "clear": aux * P,
        "store": 24 * F + 12 * min(F, K * P) + 8 * F,
        "resolve": 4 * P + 12 * min(F, K * P) + 16 * P,
    }


def wboit_stage_bytes(F: int, P: int) -> dict:
    """WBOIT: no clear (the composite sets the accumulators it read back to
    the clear values where they are not already; counted here for every
    target, an upper bound); store: stream in 24F + accumulation
    read-modify-write 40F; composite: accumulators read 20P and reset 20P,
    RGBA out 16P."""
    return {
        "clear": 0,
        "store": 24 * F + 40 * F,  # stream in + accumulation read-modify-write
        "resolve": 20 * P + 20 * P + 16 * P,
    }


def loop32_stage_bytes(F: int, P: int, K: int, occupied: int | None = None) -> dict:
    """tile_stage_bytes, likewise."""
    return tile_stage_bytes(F, P)


def interlock_stage_bytes(F: int, P: int) -> dict:
    """Ordered interlock: the Linked List append plus the shaded colour per
    node (16F); the resolve walks the nodes like the Linked List composite."""
    return {"clear": 0, "store": 44 * F + 16 * F, "resolve": 8 * P + 16 * F + 16 * P}


def frac(bytes_: float, seconds: float) -> tuple[float, float]:
    """Returns (GB/s, fraction of the HBM peak)."""
    gbs = bytes_ / seconds / 1e9
    return gbs, gbs / HBM_PEAK_GBS
